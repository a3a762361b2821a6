"""Heap neighbourhoods (RVGP/lib/ptu_dijkstra.pyx:361-394) whose searches end
in the small LDS pool, outgrow it, outgrow the large one, and where the
workspace leaves no room for the list between the two: the pop order equals
the oracle's in every case."""
import numpy as np
import pytest

from oracle import cpu

pytestmark = pytest.mark.gpu


def _graph(kind):
    import scipy.sparse as sp
    rng = np.random.default_rng(3)
    n, D, k = {"surface": (900, 3, 10), "wide": (700, 8, 12), "hub": (1500, 3, 6), "tiny": (5, 2, 2)}[kind]
    X = rng.normal(size=(n, D))
    if kind == "surface":
        X /= np.linalg.norm(X, axis=1, keepdims=True)
    rp, c = cpu.sym_csr(cpu.knn(X, k))
    if kind == "hub":  # two nodes joined to 200 and 600 others
        A = sp.csr_matrix((np.ones(len(c)), c, rp), shape=(n, n)).tolil()
        A[0, 1:201] = A[1:201, 0] = 1
        A[700, 701:1301] = A[701:1301, 700] = 1
        A = A.tocsr()
        A.sort_indices()
        rp, c = A.indptr.astype(np.int32), A.indices.astype(np.int32)
    return X, rp, c


@pytest.mark.parametrize("lanes", [None, 1])
@pytest.mark.parametrize("kind,K", [("surface", 0), ("surface", 15), ("surface", 120), ("wide", 12),
                                    ("wide", 60), ("hub", 25), ("tiny", 4)])
def test_pop_order_in_every_pool(kind, K, lanes):
    import torch
    from rvgp_amd import _lib, ptu_dijkstra
    from rvgp_amd.graph import SymGraph
    X, rp, c = _graph(kind)
    n = len(X)
    g = SymGraph(torch.as_tensor(rp, device="cuda"), torch.as_tensor(c, device="cuda"), n)
    ref, _ = cpu.geo_nbh(X, rp, c, K, centred=False)
    if lanes is None:
        nbh = ptu_dijkstra.geo_nbh_device(g, K)
    else:
        pool = 1 + K * g.max_row()
        size = _lib.lib().rvgp_geo_nbh_ws_bytes(n, lanes, pool)
        ws = torch.empty(size, dtype=torch.uint8, device="cuda")
        nbh = torch.empty((n, K + 1), dtype=torch.int32, device="cuda")
        st = torch.zeros(1, dtype=torch.int32, device="cuda")
        _lib.call("rvgp_geo_nbh", _lib.ptr(g.rowptr), _lib.ptr(g.cols), _lib.ptr(g.weights), n, K, lanes,
                  pool, _lib.ptr(nbh), _lib.ptr(ws), size, _lib.ptr(st), _lib.stream())
        assert int(st.item()) == 0
    np.testing.assert_array_equal(nbh.cpu().numpy(), ref)
