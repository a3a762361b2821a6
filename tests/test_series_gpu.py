"""The heat kernel's series (rvgp_cheb_series) at every lane mapping -- block
size, number of columns, columns whose series end early, the shared launches of
two series -- and the frame maps at every group size, against plain FP64."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu


def _laplacian(nb, b, seed):
    """A random symmetric PSD block operator with rows of uneven length."""
    rng = np.random.default_rng(seed)
    A = sp.random(nb, nb, density=min(1.0, 6.0 / nb), random_state=seed, format="csr")
    A = sp.kron(abs(A) + abs(A).T + sp.eye(nb), np.ones((b, b))).tocsr()
    A.data = rng.normal(size=A.nnz)
    A = (A + A.T) * 0.5
    return (A + sp.diags(np.asarray(abs(A).sum(1)).ravel() + 0.01)).tocsr()


def _heat(A, x, ts):
    w, V = np.linalg.eigh(A.toarray())
    return np.stack([V @ (np.exp(-t * w) * (V.T @ x[:, c])) for c, t in enumerate(ts)], 1)


@pytest.mark.parametrize("b", [1, 2, 3])
@pytest.mark.parametrize("r", [1, 2, 3, 4, 7, 8, 9, 16, 17, 32, 33, 63, 64, 65, 130])
def test_series_against_the_eigenbasis(b, r):
    import torch
    from rvgp_amd.smoothing import expm_multiply
    from rvgp_amd.sparse import BSR
    nb = 67
    A = _laplacian(nb, b, r)
    rng = np.random.default_rng(r)
    x = rng.normal(size=(nb * b, r))
    B = BSR.from_scipy(A, b)
    # error of the series ~1e-17 |x| per term and FP64 rounding of a few hundred terms
    for ts in ([0.7] * r, list(rng.uniform(0.05, 1.5, r))):
        out = expm_multiply(B, torch.as_tensor(x, device="cuda"), ts if r > 1 else ts[0]).cpu().numpy()
        ref = _heat(A, x, ts)
        assert np.linalg.norm(out - ref) < 1e-12 * np.linalg.norm(x)


@pytest.mark.parametrize("b", [1, 2, 3])
@pytest.mark.parametrize("t", [0.02, 3.0])
def test_two_series_in_one_launch(b, t):
    """One field: the two Laplacians' series share launches, of different lengths."""
    import torch
    from rvgp_amd.smoothing import vector_diffusion_device
    from rvgp_amd.sparse import BSR
    nb = 130
    Lc, L = _laplacian(nb, b, 5) * 0.2, _laplacian(nb, 1, 6)
    c = np.random.default_rng(1).normal(size=(nb, b))
    out = vector_diffusion_device(torch.as_tensor(c, device="cuda"), t, BSR.from_scipy(Lc, b),
                                  BSR.from_scipy(L, 1)).cpu().numpy()
    ref = _heat(Lc, c.reshape(-1, 1), [t]).reshape(nb, b)
    mag = _heat(L, np.stack([np.linalg.norm(c, axis=1), np.ones(nb)], 1), [t, t])
    ref *= (mag[:, 0] / (mag[:, 1] * np.linalg.norm(ref, axis=1)))[:, None]
    np.testing.assert_allclose(out, ref, rtol=1e-8, atol=1e-9 * np.abs(ref).max())


@pytest.mark.parametrize("D,d", [(1, 1), (3, 2), (4, 4), (5, 3), (9, 1), (17, 8), (32, 3), (33, 5), (64, 8), (70, 2)])
@pytest.mark.parametrize("n,F", [(1, 1), (63, 3), (257, 2)])
def test_frame_maps(D, d, n, F):
    import torch
    from rvgp_amd import _lib
    rng = np.random.default_rng(D)
    T, v, c = rng.normal(size=(n, D, d + 1)), rng.normal(size=(F, n, D)), rng.normal(size=(F, n, d))
    Td = torch.as_tensor(T, device="cuda")  # one column more than the frame has
    Q = T[:, :, :d]
    for mode, x, ref in ((0, v, np.einsum("npi,fnp->fni", Q, v)), (1, c, np.einsum("npi,fni->fnp", Q, c)),
                         (2, v, np.einsum("nqi,npi,fnp->fnq", Q, Q, v))):
        xd = torch.as_tensor(x, device="cuda")
        out = torch.empty(ref.shape, dtype=torch.float64, device="cuda")
        _lib.call("rvgp_frame_apply", mode, F, n, D, d, _lib.ptr(Td), d + 1, _lib.ptr(xd), _lib.ptr(out),
                  _lib.stream())
        np.testing.assert_allclose(out.cpu().numpy(), ref, rtol=1e-12, atol=1e-12 * D * d)


@pytest.mark.parametrize("columns", [1, 3, 16])
def test_series_of_one_time_can_be_captured(columns):
    import torch
    from rvgp_amd import smoothing
    from rvgp_amd.sparse import BSR
    A, L = BSR.from_scipy(_laplacian(400, 2, 5), 2), BSR.from_scipy(_laplacian(400, 1, 6), 1)
    X = torch.randn(800, columns, dtype=torch.float64, device="cuda")
    c = torch.randn(400, 2, dtype=torch.float64, device="cuda")
    ub = A.spectral_upper_bound()

    def step():
        return smoothing.expm_multiply(A, X, 0.7, ub=ub), smoothing.vector_diffusion_device(c, 0.7, A, L)

    step()  # the operators' bounds, which a capture cannot compute
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = step()
    for k in range(4):
        X.normal_()
        c.normal_()
        g.replay()
        for got, ref in zip(out, step()):
            assert torch.equal(got, ref), k


def test_series_in_single_precision_can_be_captured():
    """Blocks of other types than FP64 take the block SpMMs, one launch a term for
    one diffusion time."""
    import torch
    from rvgp_amd.smoothing import expm_multiply
    from rvgp_amd.sparse import BSR
    A = _laplacian(300, 3, 9)
    B = BSR.from_scipy(A, 3)
    x = np.random.default_rng(0).normal(size=(900, 4))
    X = torch.as_tensor(x, dtype=torch.float32, device="cuda")
    ub = B.spectral_upper_bound()
    # a few hundred terms of FP32 rounding on values of size 1
    np.testing.assert_allclose(expm_multiply(B, X, 0.7, ub=ub).cpu().numpy(), _heat(A, x, [0.7] * 4), atol=1e-4)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = expm_multiply(B, X, 0.7, ub=ub)
    for _ in range(3):
        X.normal_()
        g.replay()
        assert torch.equal(out, expm_multiply(B, X, 0.7, ub=ub))
