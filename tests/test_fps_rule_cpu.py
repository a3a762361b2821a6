"""Where the farthest-point loop over spatial blocks is taken: sizes well on either
side of its line, timed with points of a surface and of a full-dimensional cloud."""
import pytest

from rvgp_amd.geometry import _fps_blocked


# n, D, selections, the form that was the faster for at least one kind of points
# and not the slower by more than a tenth for the other
@pytest.mark.parametrize("n,D,N,blocked", [
    (512, 64, 64, False), (512, 50, 64, False), (1000, 32, 64, False), (512, 64, 400, False), (512, 16, 64, False),
    (5000, 6, 64, False), (512, 4, 64, False), (4096, 3, 4096, False), (300, 5, 300, False), (60000, 65, 400, False),
    (512, 16, 400, True), (512, 32, 400, True), (2000, 64, 400, True), (5000, 32, 400, True), (20000, 8, 64, True),
    (20000, 4, 64, True), (512, 4, 400, True), (60000, 32, 64, True), (5000, 3, 100, True), (4097, 2, 64, True)])
def test_blocks_are_taken_where_they_pay(n, D, N, blocked):
    assert _fps_blocked(n, D, N) == blocked
