"""What the heat-kernel series refuses before it hands pointers to the library:
blocks in host memory, and blocks whose rows are not the operator's."""
import pytest
import torch

from rvgp_amd.smoothing import expm_multiply, vector_diffusion_device
from rvgp_amd.sparse import BSR


def _operator(nb, b):
    """The identity, in host memory."""
    i32 = dict(dtype=torch.int32)
    return BSR(torch.arange(nb + 1, **i32), torch.arange(nb, **i32),
               torch.eye(b, dtype=torch.float64).repeat(nb, 1, 1).reshape(-1), None, b)


@pytest.mark.parametrize("b", [1, 3])
def test_blocks_in_host_memory(b):
    with pytest.raises(ValueError, match="device tensor"):
        expm_multiply(_operator(8, b), torch.ones(8 * b, 2, dtype=torch.float64), 0.5, ub=1.0)


@pytest.mark.parametrize("rows", [6, 10, 16])
def test_blocks_of_other_rows(rows):
    with pytest.raises(AssertionError):
        expm_multiply(_operator(8, 1), torch.ones(rows, 2, dtype=torch.float64), 0.5, ub=1.0)


@pytest.mark.parametrize("n,d,perm", [(7, 2, True), (9, 2, True), (7, 2, False), (8, 1, True), (8, 3, False)])
def test_fields_of_other_nodes(n, d, perm):
    p = torch.arange(8) if perm else None
    for c in (torch.ones(n, d, dtype=torch.float64), torch.ones(3, n, d, dtype=torch.float64)):
        with pytest.raises(AssertionError):
            vector_diffusion_device(c, 0.5, _operator(8, 2), _operator(8, 1), perm=p)


def test_no_columns():
    with pytest.raises(ValueError):
        expm_multiply(_operator(8, 1), torch.ones(8, 0, dtype=torch.float64), 0.5, ub=1.0)


def test_the_library_takes_any_even_row_stride():
    """Refused for its buffers alone (16-byte alignment), not for more than 64
    columns: all columns of a series share a launch a term."""
    import ctypes
    from rvgp_amd import _lib
    L = _lib.load_symbols_only()
    active = (ctypes.c_int * 2)(130, 130)
    for ld, word in ((130, b"aligned"), (131, b"even")):
        op = _lib.Series(1, 1, 16, 16, 16, 8, 32, 48, 64, ld, 2, ctypes.addressof(active), 1.0, 0.0)
        assert L.rvgp_cheb_series(1, ctypes.byref(op), None) == _lib.RVGP_EINVAL
        assert word in L.rvgp_last_error()
