"""rvgp_gemm and rvgp_gemm_sym where K is long enough to be split and a caller
may still bring the unsplit product's workspace: against the product in FP64,
with K eps (of the accumulator) sum |a b| as the bound, with and without room
for the split."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("room", [True, False])
@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("M,N,K", [(3, 5, 1025), (64, 64, 1100), (100, 130, 1999), (64, 64, 2047)])
def test_split_products(M, N, K, mode, room):
    import torch
    from rvgp_amd import _lib, dense
    rng = np.random.default_rng(K)
    f32 = mode != dense.GEMM_F64
    out64 = mode != dense.GEMM_F32
    ti = torch.float32 if f32 else torch.float64
    A = torch.as_tensor(rng.normal(size=(K, M)), dtype=ti, device="cuda")
    B = torch.as_tensor(rng.normal(size=(K, N)), dtype=ti, device="cuda")
    C = torch.empty((M, N), dtype=torch.float64 if out64 else torch.float32, device="cuda")
    size = _lib.lib().rvgp_gemm_ws_bytes(mode, M, N, K, 0)
    assert size > 0
    ws = torch.empty(size, dtype=torch.uint8, device="cuda") if room else None
    _lib.call("rvgp_gemm", mode, 1, 0, M, N, K, 1.0, _lib.ptr(A), M, _lib.ptr(B), N, None, 0.0, _lib.ptr(C), N,
              0, _lib.ptr(ws) if room else None, size if room else 0, _lib.stream())
    a, b = A.cpu().numpy().astype(np.float64), B.cpu().numpy().astype(np.float64)
    eps = np.finfo(np.float64 if out64 else np.float32).eps
    assert (np.abs(C.cpu().numpy() - a.T @ b) <= K * eps * (np.abs(a).T @ np.abs(b))).all()


@pytest.mark.parametrize("room", [True, False])
@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("M,K", [(1, 1025), (64, 1300), (130, 2000)])
def test_split_grams(M, K, dtype, room):
    import torch
    from rvgp_amd import _lib, dense
    A = torch.as_tensor(np.random.default_rng(M).normal(size=(K, M)), dtype=getattr(torch, dtype), device="cuda")
    mode = dense.GEMM_F64 if dtype == "float64" else dense.GEMM_F32
    C = torch.empty((M, M), dtype=torch.float64, device="cuda")
    size = _lib.lib().rvgp_gemm_ws_bytes(mode, M, M, K, 0) if room else (0 if dtype == "float64" else 4 * M * M)
    ws = torch.empty(max(size, 1), dtype=torch.uint8, device="cuda")
    _lib.call("rvgp_gemm_sym", mode, M, K, _lib.ptr(A), M, _lib.ptr(A), M, _lib.ptr(C), M, 0, _lib.ptr(ws), size,
              _lib.stream())
    a = A.cpu().numpy().astype(np.float64)
    assert (np.abs(C.cpu().numpy() - a.T @ a) <= K * np.finfo(dtype).eps * (np.abs(a).T @ np.abs(a))).all()
