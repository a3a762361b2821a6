"""rvgp_syev (RVGP/geometry.py:73) about the size up to which one workgroup
tridiagonalises, and where the tridiagonal walks end inside a stride: against
numpy.linalg.eigh on random, repeated, decoupled and scaled spectra.  The
bounds are a backward-stable solver's, 1e-12 sqrt(n) |A|, and 1e-10 for the
eigenvectors' orthogonality."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _matrix(kind, n):
    rng = np.random.default_rng(n)
    B = rng.normal(size=(n, n))
    if kind == "random":
        return 0.5 * (B + B.T)
    if kind == "repeated":
        Q, _ = np.linalg.qr(B)
        return (Q * np.sort(rng.integers(0, 4, n).astype(float))) @ Q.T
    if kind == "decoupled":  # a tridiagonal matrix that splits, an isolated zero row
        A = np.diag(rng.normal(size=n)) + np.diag(np.ones(n - 1), 1) + np.diag(np.ones(n - 1), -1)
        A[n // 2, :] = A[:, n // 2] = 0.0
        return A
    return (B + B.T) * float(kind)


@pytest.mark.parametrize("kind", ["random", "repeated", "decoupled", "1e-150", "1e140"])
@pytest.mark.parametrize("n", [2, 7, 8, 9, 33, 63, 66, 128, 129, 191, 192, 193, 200])
def test_syev_sizes_against_numpy(kind, n):
    import torch
    from rvgp_amd import dense
    A = _matrix(kind, n)
    scale = max(np.abs(np.linalg.eigvalsh(A)).max(), 1e-300)
    # a padded leading dimension: the solver reads A by its own
    W = torch.zeros(n, n + 3, dtype=torch.float64, device="cuda")
    W[:, :n] = torch.as_tensor(A)
    w, V = dense.syev(W[:, :n])
    w, V = w.cpu().numpy(), V.cpu().numpy()
    tol = 1e-12 * np.sqrt(n) * scale
    np.testing.assert_allclose(w, np.linalg.eigvalsh(A), rtol=0, atol=tol)
    assert np.abs((A / scale) @ V - V * (w / scale)).max() * scale <= tol
    assert np.abs(V.T @ V - np.eye(n)).max() <= 1e-10
