"""rvgp_batch_step (RVGP/kernels.py:41-53 with the weight-space NLML) with its
factor in LDS, at the edges of its 16-column blocks, the largest size it takes
and the first beyond it: values and gradients against numpy in FP64, fits that
share a workgroup, and a matrix that is not positive definite.  The systems
have condition numbers below 1e4, so 160 eps cond < 1e-9 bounds the error."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

THETA = np.array([1.7, 2.3, 0.9, 0.4])


def _reference(G, b, yy, M, lam, n_rows, typ):
    nu, kappa, sf, s2 = THETA
    k = len(lam)
    if typ == 0:
        base = lam + 2 * nu / kappa ** 2
        r = base ** -nu
        dn = -np.log(base) - nu * (2 / kappa ** 2) / base
        dk = 4 * nu ** 2 / (kappa ** 3 * base)
    else:
        r, dn, dk = np.exp(-0.5 * lam * kappa ** 2), np.zeros(k), -lam * kappa
    S = sf * n_rows * r / r.sum()
    dS = [S * (dn - (r * dn).sum() / r.sum()), S * (dk - (r * dk).sum() / r.sum()), S / sf]
    A = G + np.diag(s2 / S)
    Ai = np.linalg.inv(A)
    w = Ai @ b
    ld = np.linalg.slogdet(A)[1]
    nlml = 0.5 * (yy - b @ w) / s2 + 0.5 * ((M - k) * np.log(s2) + np.log(S).sum() + ld) + 0.5 * M * np.log(2 * np.pi)
    gS = 0.5 * (1 / S - s2 * np.diag(Ai) / S ** 2 - w ** 2 / S ** 2)
    res2 = yy - 2 * b @ w + w @ G @ w
    gs2 = 0.5 * ((M - k) / s2 + (np.diag(Ai) / S).sum() - res2 / s2 ** 2)
    L = np.linalg.cholesky(A)
    vec = np.stack([S, *dS, gS, np.diag(Ai), np.linalg.solve(L, b), w, G @ w])
    return np.array([nlml, gS @ dS[0], gS @ dS[1], gS @ dS[2], gs2]), L, vec


def _step(Gs, bs, yy, M, lam, n_rows, typ, panel, threads, grid):
    import torch
    from rvgp_amd import _lib
    F, k = bs.shape
    f64 = dict(dtype=torch.float64, device="cuda")
    t = lambda a: torch.as_tensor(np.ascontiguousarray(a), **f64)
    u = t(np.tile(np.log(np.expm1(THETA)), (F, 1)))
    lower, trainable = torch.zeros(4, **f64), torch.ones(4, dtype=torch.int32, device="cuda")
    m1, m2, st = torch.zeros((F, 4), **f64), torch.zeros((F, 4), **f64), torch.zeros(F, **f64)
    out, status = torch.zeros((F, 9), **f64), torch.full((F,), -7, dtype=torch.int32, device="cuda")
    size = _lib.lib().rvgp_batch_step_ws_bytes(F, k)
    ws = torch.empty(size // 8 + 1, **f64)
    lam_, G_, b_, yy_, M_ = t(lam), t(Gs), t(bs), t(yy), t(M)
    p = _lib.ptr
    _lib.call("rvgp_batch_step", F, k, typ, p(lam_), float(n_rows), p(G_), p(b_), p(yy_), p(M_), p(lower), p(u),
              p(trainable), p(m1), p(m2), p(st), 0, 0.1, 0.9, 0.999, 1e-8, panel, threads, grid, p(ws), size,
              p(out), p(status), _lib.stream())
    ws = ws[:size // 8].cpu().numpy().reshape(F, 2 * k * k + 9 * k)
    return out.cpu().numpy(), status.cpu().numpy(), ws[:, :2 * k * k].reshape(F, k, 2 * k), ws[:, 2 * k * k:].reshape(F, 9, k)


@pytest.mark.parametrize("threads", [512, 1024])
@pytest.mark.parametrize("typ", [0, 1])
@pytest.mark.parametrize("k", [1, 5, 16, 17, 48, 120, 129, 144, 159, 160, 161])
def test_step_against_numpy(k, typ, threads):
    rng = np.random.default_rng(k)
    F, rows = 3, 400
    Phi = rng.normal(size=(F, rows, k)) / np.sqrt(rows)
    y = rng.normal(size=(F, rows))
    Gs, bs = np.einsum("fri,frj->fij", Phi, Phi), np.einsum("fri,fr->fi", Phi, y)
    yy, M, lam = (y * y).sum(1), np.full(F, float(rows)), np.sort(rng.uniform(0, 1.0, k))
    out, status, W, vec = _step(Gs, bs, yy, M, lam, rows, typ, 16, threads, 2)
    assert (status == 0).all()
    for f in range(F):
        ref, L, v = _reference(Gs[f], bs[f], yy[f], M[f], lam, rows, typ)
        np.testing.assert_allclose(out[f, :5], ref, rtol=1e-9, atol=1e-9 * np.abs(ref).max())
        # what the step leaves for the predictions: [L | L^-1] and the vectors
        np.testing.assert_allclose(np.tril(W[f, :, :k]), L, rtol=0, atol=1e-9 * np.abs(L).max())
        X = np.linalg.inv(L)
        np.testing.assert_allclose(W[f, :, k:], np.tril(X), rtol=0, atol=1e-9 * np.abs(X).max())
        for q in (0, 5, 6, 7, 8):  # S, diag(A^-1), L^-1 b, w, G w
            np.testing.assert_allclose(vec[f, q], v[q], rtol=0, atol=1e-9 * np.abs(v[q]).max())


@pytest.mark.parametrize("k", [3, 40, 160])
def test_step_reports_a_matrix_that_is_not_positive_definite(k):
    rng = np.random.default_rng(1)
    Gs = np.stack([np.eye(k), np.eye(k)])
    Gs[1, k - 1, k - 1] = -1e6
    bs = rng.normal(size=(2, k))
    status = _step(Gs, bs, np.full(2, 50.0), np.full(2, 200.0), np.linspace(0, 1, k), 200, 0, 16, 512, 2)[1]
    from rvgp_amd import _lib
    assert status[0] == 0 and status[1] != 0


@pytest.mark.parametrize("k", [7, 160, 161])
def test_many_steps_in_one_call_equal_single_calls(k):
    import torch
    from rvgp_amd.batch import BatchedGPR
    rng = np.random.default_rng(k)
    F, rows = 3, 300
    Phi = rng.normal(size=(F, rows, k)) / np.sqrt(rows)
    G, b = np.einsum("fri,frj->fij", Phi, Phi), rng.normal(size=(F, k))
    f64 = dict(dtype=torch.float64, device="cuda")
    e = object.__new__(BatchedGPR)
    e.F, e.k, e.typ, e.n_rows, e.grid, e.panel, e.threads = F, k, 0, float(rows), 2, 16, 512
    e.evals = torch.linspace(0, 1, k, **f64)
    e.G, e.b = torch.as_tensor(G, **f64), torch.as_tensor(b, **f64)
    e.yy, e.M = torch.full((F,), 40.0 + (b * b).sum(), **f64), torch.full((F,), float(rows), **f64)
    e.lower, e.trainable = torch.zeros(4, **f64), torch.ones(4, dtype=torch.int32, device="cuda")
    from rvgp_amd import _lib
    e.ws_bytes = _lib.lib().rvgp_batch_step_ws_bytes(F, k)
    e.out, e.status = torch.zeros((F, 9), **f64), torch.zeros(F, dtype=torch.int32, device="cuda")
    got = []
    for chunks in ([1] * 7, [7], [3, 4]):
        e.ws = torch.zeros(e.ws_bytes // 8, **f64)
        e.u = torch.as_tensor(np.tile(np.log(np.expm1(THETA)), (F, 1)), **f64)
        e.m1, e.m2, e.t = torch.zeros((F, 4), **f64), torch.zeros((F, 4), **f64), torch.zeros(F, **f64)
        for n in chunks:
            e._step(1, 0.05, steps=n)
        got.append([x.cpu().numpy() for x in (e.u, e.t, e.out, e.m1, e.m2, e.ws)])
    assert (got[0][1] == 7).all()
    for other in got[1:]:
        for x, y in zip(got[0], other):
            np.testing.assert_array_equal(x, y)


def test_launch_shapes_are_timed_only_where_they_differ():
    """Up to LDS_MAX_K one kernel serves: nothing to time on a new problem shape."""
    import torch
    import rvgp_amd as RVGP
    from rvgp_amd import autotune
    from tests.util import torus
    d = RVGP.create_data_object(torus(400, 2), n_neighbors=12, n_eigenpairs=20, verbose=False)
    V = torch.randn(3, 400, 3, dtype=torch.float64, device="cuda")
    sets = [np.arange(f, 200 + 7 * f) for f in range(3)]
    gp = RVGP.fit_batched(d, sets, vectors=V, epochs=2)
    assert (gp.panel, gp.threads) == (16, 512)
    assert not [key for key in autotune.table() if key.startswith("batch_step|") and ",k20," in key]
