"""Frames applied to many fields at few nodes (2000 fields at 64 sensors), at many
nodes, and with remainders of both."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _apply(mode, T, x, out):
    from rvgp_amd import _lib
    F, n = x.shape[:2]
    _lib.call("rvgp_frame_apply", mode, F, n, T.shape[1], T.shape[2], _lib.ptr(T), T.shape[2], _lib.ptr(x),
              _lib.ptr(out), _lib.stream())


@pytest.mark.parametrize("F,n,D,d", [(2000, 64, 3, 2), (5000, 1, 3, 2), (1, 70000, 3, 2), (301, 77, 9, 3),
                                     (37, 500, 32, 3), (4097, 5, 70, 8), (3, 5, 1, 1)])
def test_frames_of_many_fields(F, n, D, d):
    import torch
    g = torch.Generator("cuda").manual_seed(F)
    T, v, c = (torch.randn(*s, dtype=torch.float64, device="cuda", generator=g)
               for s in ((n, D, d), (F, n, D), (F, n, d)))
    # sums of at most 70 products of numbers of size 1
    for mode, x, ref in ((0, v, (T[None] * v[..., None]).sum(2)), (1, c, (T[None] * c[:, :, None]).sum(3))):
        out = torch.empty_like(ref)
        _apply(mode, T, x, out)
        torch.testing.assert_close(out, ref, rtol=1e-12, atol=1e-11)
    ref = (T[None] * (T[None] * v[..., None]).sum(2)[:, :, None]).sum(3)
    _apply(2, T, v, v)
    torch.testing.assert_close(v, ref, rtol=1e-11, atol=1e-10)


def test_many_fields_at_few_nodes_take_no_longer_than_many_nodes():
    """The same number of rows; one workgroup for all of the fields took 200 times as long."""
    import torch

    def once(F, n):
        T, v = torch.randn(n, 3, 2, dtype=torch.float64, device="cuda"), torch.randn(F, n, 3, dtype=torch.float64, device="cuda")
        out = torch.empty(F, n, 2, dtype=torch.float64, device="cuda")
        _apply(0, T, v, out)
        t = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
        t[0].record()
        for _ in range(20):
            _apply(0, T, v, out)
        t[1].record()
        t[1].synchronize()
        return t[0].elapsed_time(t[1])

    assert np.median([once(2000, 64) for _ in range(3)]) < 20 * np.median([once(1, 128000) for _ in range(3)])
