"""Function-space fits on the k x k system (rvgp_coef_step and its multi-kernel
form) against the oracle's M x M covariance: on both sides of the line where
they start, with singular Phi^T Phi, several right-hand sides, filters that
underflow, and the step's tile edges."""
import numpy as np
import pytest

from oracle import cpu

pytestmark = pytest.mark.gpu

TH = (1.6, 4.0, 0.8, 0.3)


def _problem(M, k, R, rank, seed):
    """Rows with `rank` independent columns (the others repeat them)."""
    rng = np.random.default_rng(seed)
    Phi = rng.normal(size=(M, rank))
    Phi = np.concatenate([Phi, Phi[:, np.arange(k - rank) % rank]], 1)
    lam = np.sort(rng.uniform(0.0, 6.0, k))
    y = Phi @ rng.normal(size=(k, R)) / np.sqrt(k) + 0.3 * rng.normal(size=(M, R))
    return Phi, y, lam


def _engine(Phi, y, lam, **kw):
    import torch
    from rvgp_amd.gp import GPREngine
    e = GPREngine(*(torch.as_tensor(x, device="cuda") for x in (Phi, y, lam)), 500.0, form="function", **kw)
    e.set_theta(TH)
    return e


# the k x k system from M = 2 k on; tiles of 32; a singular Phi^T Phi (rank < k)
@pytest.mark.parametrize("M,k,rank", [(2, 1, 1), (62, 31, 31), (64, 32, 32), (66, 33, 33), (65, 33, 33),
                                      (200, 100, 100), (400, 65, 64), (300, 90, 40), (600, 129, 129)])
@pytest.mark.parametrize("R", [1, 3])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_function_space_on_the_small_system(M, k, rank, R, precision):
    Phi, y, lam = _problem(M, k, R, rank, M + k)
    e = _engine(Phi, y, lam, precision=precision)
    assert e.coef == (M >= 2 * k) and e.fused() == (e.coef and R == 1)
    nlml, gu, out = e.nlml_grad_u(e.u.cpu().numpy())
    S, dS = cpu.spectral_filter(lam, *TH[:3], 500.0)
    ref = cpu.gpr_nlml(Phi, y, S, TH[3])
    gS, gn = cpu.gpr_grad(Phi, y, S, TH[3])
    g = np.append(dS @ gS, gn)
    # both sides work in FP64 on systems of condition <= 1e6
    assert abs(nlml - ref) < 1e-9 * abs(ref)
    np.testing.assert_allclose(out[1:5], g, rtol=1e-8, atol=1e-9 * np.abs(g).max())
    rng = np.random.default_rng(0)
    Ps = np.concatenate([rng.normal(size=(37, rank))] * (1 + k // rank), 1)[:, :k]
    mean, var = e.predict(__import__("torch").as_tensor(Ps, device="cuda"))
    mref, vref = cpu.gpr_predict(Phi, y, S, TH[3], Ps)
    np.testing.assert_allclose(mean.cpu().numpy().reshape(37, R), mref, rtol=1e-8, atol=1e-9 * np.abs(mref).max())
    np.testing.assert_allclose(var.cpu().numpy(), vref.ravel(), rtol=1e-7, atol=1e-9 * np.abs(vref).max())


def test_trial_steps_far_out_stay_finite():
    """A host optimiser's line search visits filters that all but vanish: the
    value is then that of pure noise, on the small system as on the large."""
    Phi, y, lam = _problem(120, 40, 1, 40, 3)
    for u in ([60.0, 20.0, -60.0, 0.5], [129.0, 53.0, -96.0, 0.6], [200.0, 30.0, -700.0, 0.0]):
        v, g, _ = _engine(Phi, y, lam).nlml_grad_u(np.array(u))
        s2 = np.log1p(np.exp(u[3])) + 1e-6
        noise = 0.5 * float((y * y).sum()) / s2 + 60.0 * np.log(2 * np.pi * s2)
        assert np.isfinite(v) and np.all(np.isfinite(g)) and v == pytest.approx(noise, rel=1e-6)


def _extended(Phi, y, lam, th, n_rows):
    """NLML and its gradient in 80 bits: in an orthonormal basis of the rows,
    Phi = Q T, y = Q a + e, the covariance acts as T S T^T + s2 I on a and as s2 on e."""
    X = np.longdouble
    Phi, y, lam = Phi.astype(X), y.astype(X), lam.astype(X)
    nu, kappa, sf, s2 = (X(v) for v in th)
    M, k = Phi.shape
    Q, T = np.zeros((M, k), X), np.zeros((k, k), X)
    for j in range(k):
        v = Phi[:, j].copy()
        for _ in range(3):
            h = Q[:, :j].T @ v
            v, T[:j, j] = v - Q[:, :j] @ h, T[:j, j] + h
        T[j, j] = np.sqrt(v @ v)
        Q[:, j] = v / T[j, j]
    a = Q.T @ y
    e = y - Q @ a
    base = lam + 2 * nu / kappa ** 2
    r = base ** -nu
    dn, dk = -np.log(base) - nu * (2 / kappa ** 2) / base, 4 * nu ** 2 / (kappa ** 3 * base)
    S = sf * X(n_rows) * r / r.sum()
    dS = np.stack([S * (dn - r @ dn / r.sum()), S * (dk - r @ dk / r.sum()), S / sf])
    L = (T * S) @ T.T + s2 * np.eye(k, dtype=X)
    for j in range(k):
        L[j:, j] /= np.sqrt(L[j, j])
        L[j + 1:, j + 1:] -= np.outer(L[j + 1:, j], L[j + 1:, j])
    L = np.tril(L)

    def solve(B):
        B = B.copy()
        for i in range(k):
            B[i] = (B[i] - L[i, :i] @ B[:i]) / L[i, i]
        return B

    Li = solve(np.eye(k, dtype=X))
    z, q = Li @ a, ((Li @ T) ** 2).sum(0)
    p, rhs = T.T @ (Li.T @ z), y.shape[1]
    logdet = 2 * np.log(np.diag(L)).sum() + (M - k) * np.log(s2)
    nlml = ((z * z).sum() + (e * e).sum() / s2 + rhs * (logdet + M * np.log(2 * X(np.pi)))) / 2
    alpha2 = ((Li.T @ z) ** 2).sum() + (e * e).sum() / s2 ** 2
    grad = np.append(dS @ (rhs * q - (p * p).sum(1)), rhs * (M - S @ q) / s2 - alpha2) / 2
    return float(nlml), grad.astype(float), S.astype(float)


# nodes on a part of a circle: the columns are close to dependent, with singular
# values of every size down to rounding
@pytest.mark.parametrize("M,k,part", [(300, 40, 0.5), (240, 60, 0.33)])
@pytest.mark.parametrize("R", [1, 3])
@pytest.mark.parametrize("noise", [0.05, 1e-3])
@pytest.mark.parametrize("s2", [1e-1, 2.5e-3, 1e-4, 2e-6])
def test_nodes_on_a_part_of_the_manifold(M, k, part, R, noise, s2):
    rng = np.random.default_rng(k)
    t, f = 2 * np.pi * part * rng.uniform(size=(M, 1)), np.arange(1, k) // 2 + np.arange(1, k) % 2
    Phi = np.concatenate([np.ones((M, 1)), np.sqrt(2) * np.where(np.arange(1, k) % 2, np.cos(f * t), np.sin(f * t))], 1)
    lam = 0.05 * np.append(0, f) ** 2.0
    y = Phi @ (rng.normal(size=(k, R)) / (1 + 5 * lam[:, None]))
    y = y / np.abs(y).max() + noise * rng.normal(size=(M, R))
    e = _engine(Phi, y, lam)
    th = (1.6, 4.0, 0.8, s2)
    e.set_theta(th)
    assert e.coef
    nlml, _, out = e.nlml_grad_u(e.u.cpu().numpy())
    ref, grad, S = _extended(Phi, y, lam, th, 500.0)
    # rounding of Phi c, where |c| <= |y| / sqrt(ridge G), and of G, against s2, in
    # each of four products
    off = 4 * np.finfo(float).eps * ((y * y).sum() / np.sqrt(1e-9) + R * (Phi * Phi).sum(0) @ S) / s2
    assert abs(nlml - ref) <= off + 1e-9 * abs(ref)
    np.testing.assert_allclose(out[1:4], grad[:3], rtol=1e-7, atol=10 * off)
    np.testing.assert_allclose(out[4], grad[3], rtol=1e-9, atol=off / s2)


# one and several slices of 2048 entries, remainders, the most slices
@pytest.mark.parametrize("k,R", [(1, 1), (3, 7), (33, 64), (64, 32), (150, 2000), (2048, 1100)])
def test_terms_of_the_split_form(k, R):
    import torch
    from rvgp_amd import _lib
    rng = np.random.default_rng(k + R)
    c, g, w, b = (rng.normal(size=(k, R)) for _ in range(4))
    S, ee, s2 = np.exp(rng.normal(size=k)), np.array([3.7]), np.array([0.02])
    S[k // 2], w[k // 2] = 1e-280, 1e-281 * w[k // 2]  # a filter value at its floor
    dev = {n: torch.as_tensor(v, device="cuda") for n, v in dict(c=c, g=g, w=w, b=b, S=S, ee=ee, s2=s2).items()}
    size = _lib.lib().rvgp_coef_terms_ws_bytes(k, R)
    p, ws = torch.empty(k, R, dtype=torch.float64, device="cuda"), torch.empty(size // 8, dtype=torch.float64, device="cuda")
    ya, aa = torch.empty(1, dtype=torch.float64, device="cuda"), torch.empty(1, dtype=torch.float64, device="cuda")
    r = torch.empty_like(p)
    _lib.call("rvgp_coef_terms", k, R, *[_lib.ptr(dev[n]) for n in ("c", "g", "ee", "w", "S", "s2")], _lib.ptr(p),
              _lib.ptr(ya), _lib.ptr(aa), _lib.ptr(ws), size, _lib.stream())
    _lib.call("rvgp_coef_residual", k, R, *[_lib.ptr(dev[n]) for n in ("b", "w", "S", "s2")], _lib.ptr(r), _lib.stream())
    X = np.longdouble
    pr = w / S[:, None]
    np.testing.assert_array_equal(p.cpu().numpy(), pr)
    np.testing.assert_allclose(r.cpu().numpy(), b - s2 * pr, rtol=0, atol=4e-16 * np.abs(b).max())
    d = c.astype(X) - w
    t = (X(3.7) + (g * d).sum()) / X(0.02)
    cp, pd = (c * pr.astype(X)).sum(), (pr * d).sum()
    # sums of k R products of numbers of size 1
    off = 1e-15 * np.sqrt(k * R) * (1 + np.abs(pr).max()) * 10
    assert abs(ya.item() - float(cp + t)) <= off * 60 and abs(aa.item() - float((pd + t) / X(0.02))) <= off * 60 * 60
