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
