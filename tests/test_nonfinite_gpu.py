"""Farthest-point sampling and kNN graphs of points that are not finite, or whose
squares overflow, on every route: registers, spatial blocks and the plain loops."""
import numpy as np
import pytest

from oracle import cpu

pytestmark = pytest.mark.gpu

# registers; blocks by own coordinates; the plain loop (few selections, few points
# of D > 3, and D > 6 where principal axes need finite points)
ROUTES = [(300, 3, 100), (5000, 3, 100), (700, 5, 100), (5000, 3, 20), (300, 7, 30), (700, 7, 100)]


def _points(n, D):
    return np.random.default_rng(n + D).normal(size=(n, D))


@pytest.mark.parametrize("n,D,N", ROUTES)
def test_fps_ends_where_every_distance_is_nan(n, D, N):
    from rvgp_amd import geometry
    x = _points(n, D)
    x[7, D - 1] = np.nan
    perm, lam = geometry.furthest_point_sampling(x, N=N, start_idx=7)
    np.testing.assert_array_equal(perm, [7])
    np.testing.assert_array_equal(lam, [0.0])


@pytest.mark.parametrize("n,D,N", ROUTES)
@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
def test_fps_passes_over_points_that_are_not_finite(n, D, N, bad):
    """A NaN point is never selected; an infinite one always is (its distance to
    itself is NaN, so it stays the farthest), as in the oracle."""
    from rvgp_amd import geometry
    x = _points(n, D)
    x[[3, n // 2, n - 1], [0, D - 1, D // 2]] = bad
    perm, lam = geometry.furthest_point_sampling(x, N=N)
    p_ref, lam_ref = cpu.fps(x, N=N)
    np.testing.assert_array_equal(perm, p_ref)
    np.testing.assert_array_equal(lam, lam_ref)


@pytest.mark.parametrize("n,D,N", [(700, 7, 100), (1500, 12, 300), (5000, 32, 100), (5000, 3, 100)])
@pytest.mark.parametrize("points", [1, 2, 40])
def test_fps_of_points_whose_squares_overflow(n, D, N, points):
    """A few points 1e160 away in one coordinate: the covariance overflows, the
    distances between the others do not."""
    from rvgp_amd import geometry
    x = _points(n, D)
    x[1:1 + points, 2] = 1e160
    perm, lam = geometry.furthest_point_sampling(x, N=N)
    p_ref, lam_ref = cpu.fps(x, N=N)
    np.testing.assert_array_equal(perm, p_ref)
    np.testing.assert_array_equal(lam, lam_ref)


@pytest.mark.parametrize("n,D", [(300, 3), (5000, 3), (10001, 3), (12001, 9)])
@pytest.mark.parametrize("bad", [np.nan, np.inf, 1e160])
def test_knn_refuses_points_without_distances(n, D, bad):
    from rvgp_amd import geometry
    x = _points(n, D)
    x[n // 3, D - 1] = bad
    with pytest.raises(ValueError, match="NaN or infinity|too large"):
        geometry.manifold_graph(x, n_neighbors=5)
