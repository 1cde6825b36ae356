"""Log-likelihood derivatives in every hyperparameter of every kernel that the library takes
(one or two Matern components, in both orders), at short and long chunks, and of models and
batches at the chunk length that they choose themselves.

Reference: sixth-order central differences of the oracle's FP64 C filter on the same FP32
inputs, steps of 1 % of the hyperparameter.  Truncation (0.01^6 times derivatives of the order
of the value, and binomial factors) and the log-likelihood's rounding over the step (about
1e-14 / 0.01) both stay below 1e-9 of the gradient's norm; the library's own FP64 recursions
are good to 1e-13.  Tolerance: 1e-7 of the gradient's norm."""
import ctypes

import numpy as np
import pytest

from oracle import cfast

TOL = 1e-7
NAMES = ("matern12", "matern32", "matern52")
KERNELS = [(a,) for a in NAMES] + [(a, b) for a in NAMES for b in NAMES]
LS, VAR = (5.0, 2.0), (0.5, 0.7)


def _data(n, seed):
    rng = np.random.default_rng(seed)
    dt = rng.exponential(0.05, n).astype(np.float32)
    dt[0] = 0.0
    x = np.cumsum(dt.astype(np.float64))
    y = (np.sin(0.8 * x) + 0.4 * np.sin(2.9 * x) + 0.1 * rng.standard_normal(n)).astype(np.float32)
    return dt, y, np.full(n, 0.01, np.float32)


def _reference(names, dt, y, r):
    """d log-likelihood / d (lengthscale, variance) of every component."""
    n, k = len(dt), len(names)
    a = [np.asarray(v, np.float64) for v in (dt, y, r)]

    def ll(ls, var):
        return float(cfast.filter_smoother(list(names), ls, var, [0, n], *a)[2][0])

    out = []
    for c in range(k):
        for which in (0, 1):
            h = 0.01 * (LS, VAR)[which][c]
            g = 0.0
            for m, w in ((1, 45.0), (2, -9.0), (3, 1.0)):
                for s in (1, -1):
                    p = [list(LS[:k]), list(VAR[:k])]
                    p[which][c] += s * m * h
                    g += s * w * ll(*p)
            out.append(g / (60.0 * h))
    return np.array(out)


def _kernel(names):
    from bayesnewton_amd import kernels as K
    cls = dict(zip(NAMES, (K.Matern12, K.Matern32, K.Matern52)))
    ks = [cls[m](variance=v, lengthscale=s) for m, v, s in zip(names, VAR, LS)]
    return ks[0] if len(ks) == 1 else K.Sum(ks)


def _library(names, chunk, dt, y, r):
    import torch
    from bayesnewton_amd import _native as nat
    from bayesnewton_amd.plan import SeriesPlan
    kern, L = _kernel(names), nat.lib()
    desc = kern.desc()
    p = SeriesPlan(np.array([0, len(dt)]), chunk_len=chunk)
    t = [p.gather(torch.as_tensor(v).cuda(), pad=q) for v, q in ((dt, 0.0), (y, 0.0), (r, 1.0))]
    ls, var = kern.hypers("cuda")
    ll = torch.zeros(1, dtype=torch.float64, device="cuda")
    g = torch.zeros(2 * desc.n_comp, dtype=torch.float64, device="cuda")
    ws = torch.empty(int(L.bn_grad_workspace_bytes(p.handle, ctypes.byref(desc))), dtype=torch.uint8, device="cuda")
    out = []
    for fill in (0, 255, 85):  # nothing may depend on what the memory held
        ws.fill_(fill)
        nat.check(L.bn_filter_loglik_grad(p.handle, ctypes.byref(desc), nat.ptr(ls), nat.ptr(var), 0, nat.ptr(t[0]),
                                          nat.ptr(t[1]), nat.ptr(t[2]), None, nat.ptr(ll), nat.ptr(g),
                                          nat.ptr(p.workspace(desc)), nat.ptr(ws), nat.stream_ptr()))
        out.append(g.cpu().numpy().copy())
    assert np.array_equal(out[0], out[1]) and np.array_equal(out[0], out[2])
    return out[0]


@pytest.mark.gpu
@pytest.mark.parametrize("names", KERNELS, ids="+".join)
def test_derivatives_of_every_kernel(names):
    dt, y, r = _data(1500, 5)
    want = _reference(names, dt, y, r)
    for chunk in (8, 32, 100, 1500):  # chunks that do and do not fill wavefronts; none scanned
        got = _library(names, chunk, dt, y, r)
        assert np.abs(got - want).max() <= TOL * np.linalg.norm(want), chunk


@pytest.mark.gpu
@pytest.mark.parametrize("names", [("matern32", "matern52"), ("matern52", "matern32"), ("matern52",)], ids="+".join)
@pytest.mark.parametrize("lengths", [(30_000,), (9000, 4500, 130)])
def test_models_at_their_own_chunk_length(names, lengths):
    """The energy's derivatives from models without chunk_len: -d log Z at the model's own sites."""
    from bayesnewton_amd import likelihoods as L, models as M
    xs, ys = [], []
    for i, n in enumerate(lengths):
        dt, y, _ = _data(n, 20 + i)
        xs.append(np.cumsum(dt.astype(np.float64)))
        ys.append(y.astype(np.float64))
    if len(lengths) == 1:
        m = M.MarkovVariationalGP(_kernel(names), L.Gaussian(variance=0.01), xs[0], ys[0])
    else:
        m = M.MarkovVariationalGP.from_series(_kernel(names), L.Gaussian(variance=0.01), xs, ys)
    m.inference(lr=1.0)
    got = m.energy_and_grad_per_series()[1].cpu().numpy()
    assert np.array_equal(got, m.energy_and_grad_per_series()[1].cpu().numpy())
    dt, y, r = (m.plan.scatter(a[None]).cpu().numpy().reshape(-1) for a in (m._dt, m._py, m._pr))
    at = np.concatenate([[0], np.cumsum(lengths)])
    for i in range(len(lengths)):
        s = slice(at[i], at[i + 1])
        want = -_reference(names, dt[s], y[s], r[s])
        assert np.abs(got[i] - want).max() <= TOL * np.linalg.norm(want), i
