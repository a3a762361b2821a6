"""Hyperparameters at which the normalised filter S is not a number, or all but
vanishes: the first fail as a matrix that is not positive definite, the second
give the values of pure noise -- in every form, in one launch or many, with one
right-hand side or several, and in predictions."""
import numpy as np
import pytest

from rvgp_amd.gp import inv_softplus

pytestmark = pytest.mark.gpu


def _engine(form, R, lam=None):
    import torch
    from rvgp_amd.gp import GPREngine
    rng = np.random.default_rng(R)
    lam = np.append(0.0, np.sort(rng.uniform(0.0, 6.0, 39))) if lam is None else lam
    Phi, y = rng.normal(size=(120, 40)), rng.normal(size=(120, R))
    e = GPREngine(*(torch.as_tensor(x, device="cuda") for x in (Phi, y, lam)), 500.0, form=form,
                  lower=(0.0, 0.0, 0.0, 1e-6))
    return e, Phi, y


FORMS = [("function", 1), ("function", 3), ("weight", 1), ("weight", 3)]


# every power of the filter underflows (0 / 0), one overflows (inf / inf), a
# parameter or an eigenvalue is not a number
@pytest.mark.parametrize("form,R", FORMS)
@pytest.mark.parametrize("theta", [(100.0, 0.05, 1.0, 0.3), (200.0, 200.0, 1.0, 0.3), (np.nan, 4.0, 1.0, 0.3), None])
def test_a_filter_that_is_not_a_number_raises(form, R, theta):
    from rvgp_amd.dense import CholeskyError
    lam = None if theta is not None else np.append(np.nan, np.linspace(0.1, 6.0, 39))
    e, _, _ = _engine(form, R, lam)
    u = inv_softplus(np.array(theta or (1.6, 4.0, 0.8, 0.3)) - np.array([0.0, 0.0, 0.0, 1e-6]))
    with pytest.raises(CholeskyError):
        e.nlml_grad_u(u)


@pytest.mark.parametrize("form,R", FORMS)
@pytest.mark.parametrize("u", [[60.0, 20.0, -60.0, 0.5], [129.0, 53.0, -96.0, 0.6], [200.0, 30.0, -700.0, 0.0]])
def test_a_vanishing_filter_gives_pure_noise(form, R, u):
    import torch
    e, Phi, y = _engine(form, R)
    v, g, _ = e.nlml_grad_u(np.array(u))
    s2 = np.log1p(np.exp(u[3])) + 1e-6
    noise = 0.5 * float((y * y).sum()) / s2 + 0.5 * y.size * np.log(2 * np.pi * s2)
    assert v == pytest.approx(noise, rel=1e-6) and np.all(np.isfinite(g))
    mean, var = (x.cpu().numpy() for x in e.predict(torch.as_tensor(Phi[:7], device="cuda")))
    # S is below 1e-20 of the noise
    assert np.abs(mean).max() < 1e-15 and np.abs(var).max() < 1e-15
