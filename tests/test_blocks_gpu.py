"""Spatial blocks: the farthest-point loop in registers and over blocks, and the
kNN scan over blocks, against the oracle (bit for bit) at the sizes where their
tiles, block counts and dispatch lines change."""
import numpy as np
import pytest

from oracle import cpu
from tests.util import flat_torus3, torus

pytestmark = pytest.mark.gpu


def _points(n, D, seed):
    if D == 32:
        return flat_torus3(n, seed)
    x = torus(n, seed)
    return np.concatenate([x, x * x], 1)[:, :D] if D > 3 else x[:, :D].copy()


# registers: 256 R points, R = 2 ... 16; blocks: 128, 256, 512 testing threads
@pytest.mark.parametrize("n,D,N", [(1, 3, 1), (63, 3, 63), (512, 3, 100), (513, 2, 100), (1025, 1, 70),
                                   (1536, 3, 90), (2049, 3, 90), (2560, 3, 90), (3329, 3, 90),
                                   (4096, 3, 150), (4097, 3, 150), (16384, 3, 100), (16385, 2, 64),
                                   (512, 32, 120), (1300, 4, 200), (3000, 7, 80), (33000, 3, 70),
                                   (66000, 3, 64)])
def test_fps_forms_match_the_oracle(n, D, N):
    from rvgp_amd import geometry
    x = _points(n, D, n)
    p, lam = geometry.furthest_point_sampling(x, N=N, start_idx=n // 2)
    p_ref, lam_ref = cpu.fps(x, N=N, start_idx=n // 2)
    np.testing.assert_array_equal(p, p_ref)
    np.testing.assert_array_equal(lam, lam_ref)


@pytest.mark.parametrize("n", [300, 4000, 5000])
@pytest.mark.parametrize("scale", [1.0, 1e-160, 1e160])
def test_fps_forms_break_ties_by_index(n, scale):
    """Points of a small lattice, most of them several times over: equal and
    nearly equal squares, distances of 0, squares that under- and overflow."""
    from rvgp_amd import geometry
    x = np.random.default_rng(n).integers(0, 8, (n, 3)) * (0.1 * scale)
    p, lam = geometry.furthest_point_sampling(x, N=n // 4)
    p_ref, lam_ref = cpu.fps(x, N=n // 4)
    np.testing.assert_array_equal(p, p_ref)
    np.testing.assert_array_equal(lam, lam_ref)


@pytest.mark.parametrize("n", [3000, 6000])
def test_fps_forms_stop_at_the_spacing(n):
    from rvgp_amd import geometry
    x = torus(n, 5)
    p, lam = geometry.furthest_point_sampling(x, spacing=0.04)
    p_ref, lam_ref = cpu.fps(x, spacing=0.04)
    np.testing.assert_array_equal(p, p_ref)
    np.testing.assert_array_equal(lam, lam_ref)


@pytest.mark.parametrize("P", [1, 3, 6, 7])
def test_morton_keys_are_the_interleaved_quantised_coordinates(P):
    import torch
    from rvgp_amd import _lib
    Y = torch.as_tensor(np.random.default_rng(P).normal(size=(1000, P)), device="cuda")
    lo, hi = torch.aminmax(Y, dim=0)
    keys = torch.empty(1000, dtype=torch.int64, device="cuda")
    _lib.call("rvgp_morton_keys", _lib.ptr(Y), P, 1000, P, _lib.ptr(lo), _lib.ptr(hi), _lib.ptr(keys),
              _lib.stream())
    bits = min(20, 62 // P)
    q = ((Y - lo) / (hi - lo) * ((1 << bits) - 1)).round().to(torch.int64)
    ref = torch.zeros(1000, dtype=torch.int64, device="cuda")
    for b in range(bits - 1, -1, -1):
        for d in range(P):
            ref = (ref << 1) | ((q[:, d] >> b) & 1)
    assert torch.equal(keys, ref)


# KMAX 16, 24, 32, 64 and the padded dimensions 4, 8, 16, 32, 64; a last block of
# one point, fewer blocks than a workgroup's waves
@pytest.mark.parametrize("n,D,k", [(70, 3, 16), (65, 3, 5), (640, 2, 17), (1000, 8, 24), (1281, 12, 25),
                                   (1500, 32, 32), (900, 40, 33), (700, 6, 64), (2000, 5, 20)])
@pytest.mark.parametrize("kind", ["manifold", "noise", "lattice", "tiny", "far"])
def test_knn_blocks_match_the_scan(n, D, k, kind):
    """rvgp_knn_blocks on every kind of point set, also where nothing can be
    skipped, equals rvgp_knn (which the oracle pins)."""
    import torch
    from rvgp_amd import _lib, geometry
    from rvgp_amd.reorder import SpatialOrder
    rng = np.random.default_rng(n + D)
    x = {"manifold": lambda: np.pad(torus(n, 1), ((0, 0), (0, max(0, D - 3))))[:, :D],
         "noise": lambda: rng.normal(size=(n, D)),
         "lattice": lambda: rng.integers(0, 4, (n, D)) * 1.0,
         "tiny": lambda: rng.normal(size=(n, D)) * 1e-170,   # squares underflow: all distances 0
         "far": lambda: rng.normal(size=(n, D)) + 1e9}[kind]()
    xd = torch.as_tensor(np.ascontiguousarray(x), device="cuda")
    blocks = SpatialOrder(xd, own_axes=D <= 6).blocks(transposed=False)
    nbr = torch.empty((n, k), dtype=torch.int32, device="cuda")
    _lib.call("rvgp_knn_blocks", _lib.ptr(blocks), blocks.numel(), n, D, k, _lib.ptr(nbr), _lib.stream())
    assert torch.equal(nbr, geometry.knn_device(xd, k))


@pytest.mark.parametrize("n,D,k", [(10001, 3, 12), (12000, 32, 20)])
def test_manifold_graph_over_blocks_matches_the_oracle(n, D, k):
    from rvgp_amd import geometry
    x = _points(n, D, 3)
    g = geometry.manifold_graph(x, n_neighbors=k)
    rp, c = cpu.sym_csr(cpu.knn(x, k))
    np.testing.assert_array_equal(g.rowptr.cpu().numpy(), rp)
    np.testing.assert_array_equal(g.cols.cpu().numpy(), c)


# more dimensions than box coordinates: points of a 3-torus in R^32, and clouds
# that fill their space, where no block can be skipped
@pytest.mark.parametrize("n,D,N,kind", [(1500, 32, 400, "torus"), (1500, 32, 400, "cloud"), (2000, 7, 400, "cloud"),
                                        (700, 12, 400, "cloud"), (2100, 64, 400, "cloud")])
def test_fps_over_blocks_by_principal_axes(n, D, N, kind):
    from rvgp_amd import geometry
    assert geometry._fps_blocked(n, D, N)
    x = flat_torus3(n, 1) if kind == "torus" else np.random.default_rng(D).normal(size=(n, D))
    p, lam = geometry.furthest_point_sampling(x, N=N)
    p_ref, lam_ref = cpu.fps(x, N=N)
    np.testing.assert_array_equal(p, p_ref)
    np.testing.assert_array_equal(lam, lam_ref)


def test_fps_of_the_most_points_that_blocks_take():
    """Past 131,072 points a block's coordinates are not kept in LDS."""
    from rvgp_amd import geometry
    x = torus(140001, 3)
    p, lam = geometry.furthest_point_sampling(x, N=70)
    p_ref, lam_ref = cpu.fps(x, N=70)
    np.testing.assert_array_equal(p, p_ref)
    np.testing.assert_array_equal(lam, lam_ref)


@pytest.mark.parametrize("n,D,k", [(12500, 10, 12), (12001, 32, 20)])
def test_graph_of_points_whose_blocks_cannot_be_skipped(n, D, k):
    """A cloud that fills its space: the order says so, and the plain scan runs."""
    import torch
    from rvgp_amd import geometry
    from rvgp_amd.reorder import SpatialOrder
    x = np.random.default_rng(n).normal(size=(n, D))
    xd = torch.as_tensor(x, device="cuda")
    order = SpatialOrder(xd)
    top, prunes = order.prunes(order.blocks(transposed=False), xd.abs().max())
    assert top == np.abs(x).max() and not prunes
    g = geometry.manifold_graph(x, n_neighbors=k)
    rp, c = cpu.sym_csr(cpu.knn(x, k))
    np.testing.assert_array_equal(g.rowptr.cpu().numpy(), rp)
    np.testing.assert_array_equal(g.cols.cpu().numpy(), c)
