"""rvgp_graph_symmetrize (RVGP/lib/ptu_dijkstra.pyx:84-103) against the oracle's
CSR: row counts about the scan's chunk of 4096, and hubs whose rows are sorted
in registers, in LDS and by insertion."""
import numpy as np
import pytest

from oracle import cpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,k,hubs", [(2, 1, 0), (4095, 3, 0), (4096, 3, 1), (4097, 5, 40), (9000, 20, 700),
                                      (12289, 2, 1023), (12289, 2, 1100), (3000, 70, 0)])
def test_symmetrised_rows(n, k, hubs):
    import torch
    from rvgp_amd import geometry
    rng = np.random.default_rng(n + hubs)
    # k distinct neighbours, never the node itself
    nbr = (np.arange(n)[:, None] + 1 + np.argsort(rng.random((n, min(n - 1, 4 * k))), axis=1)[:, :k]) % n
    if hubs:  # that many nodes have node 0 as their first neighbour
        pick = rng.choice(np.arange(1, n), size=hubs, replace=False)
        pick = pick[~(nbr[pick] == 0).any(axis=1)]
        nbr[pick, 0] = 0
    nbr = np.ascontiguousarray(nbr.astype(np.int32))
    rp, c = geometry.symmetrize_device(torch.as_tensor(nbr, device="cuda"))
    rows = np.repeat(np.arange(n), k)
    pairs = np.unique(np.concatenate([rows.astype(np.int64) * n + nbr.ravel(), nbr.ravel().astype(np.int64) * n + rows,
                                      np.arange(n, dtype=np.int64) * (n + 1)]))
    np.testing.assert_array_equal(rp.cpu().numpy(), np.searchsorted(pairs, np.arange(n + 1, dtype=np.int64) * n))
    np.testing.assert_array_equal(c.cpu().numpy(), pairs % n)
    rp0, c0 = cpu.sym_csr(nbr)
    np.testing.assert_array_equal(rp.cpu().numpy(), rp0)
    np.testing.assert_array_equal(c.cpu().numpy(), c0)
