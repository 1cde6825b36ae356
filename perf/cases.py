"""Workloads of the Markov-GP framework, each through its public entry points.

A case is a dict of plain values; `kind` says which entry points a pass goes through:

  series   one time series: a site update, the posterior and the energy (models.Markov*GP)
  train    one hyperparameter training step: inference and the energy's gradient
  batch    one model over many uneven series: a site update, the posteriors, the energies
  pass     the fused filter + smoother over a batch of series (ops.filter_smoother)
  filter   the stand-alone Kalman filter and RTS smoother of ops, full states returned
  predict  an update with new data terms, then predictions of y at new times
  field    a space-time model (dense, mean-field or infinite-horizon filter), K runs
"""
import math

import numpy as np
import torch

from bayesnewton_amd import autotune, kernels, likelihoods, models, ops, plan, spacetime


def listed():
    return [
        # a few hundred observations with outliers, the size of a single sensor's day: launch latency
        dict(name="series_300_studentt", kind="series", n=300, kernel="m52", lik="studentt", method="vi", lr=0.5),
        # a regression of ten thousand points, one exact step of conjugate inference
        dict(name="series_10k_gaussian", kind="series", n=10_000, kernel="m52", lik="gaussian", method="vi", lr=1.0),
        # binary labels over a long record, slow and quick components
        dict(name="series_200k_probit", kind="series", n=200_000, kernel="m32+m52", lik="probit", method="newton",
             lr=0.5),
        # hyperparameter learning on half a million points
        dict(name="train_500k", kind="train", n=500_000, kernel="m52"),
        # the fused pass over thousands of series of very uneven length
        dict(name="pass_4096", kind="pass", series=4096, shortest=256, longest=16384, kernel="m52+m32"),
        # a few hundred series with heavy-tailed noise, inference on all of them at once
        dict(name="batch_256_studentt", kind="batch", series=256, shortest=64, longest=4096, kernel="m52+m32",
             lik="studentt", method="vi", lr=0.5),
        # counts: refresh the posterior, then predict on a finer grid
        dict(name="predict_20k_poisson", kind="predict", n=20_000, tests=50_000, kernel="m52+m32", lik="poisson",
             method="newton"),
        # the drop-in operations on one long record
        dict(name="filter_100k", kind="filter", n=100_000, kernel="m32+m52"),
        # a space-time Cox process, one run: an iteration of variational inference
        dict(name="field_1000_steps", kind="field", form="dense", runs=1, steps=1000, grid=8, locations=256,
             lik="poisson", method="vi"),
        # a batch of independent runs, as a training set for the learned start is made
        dict(name="field_32_runs", kind="field", form="dense", runs=32, steps=100, grid=8, locations=256,
             lik="poisson", method="vi"),
        # the same model with the mean-field filter
        dict(name="field_meanfield", kind="field", form="meanfield", runs=4, steps=500, grid=8, locations=256,
             lik="poisson", method="vi"),
        # the steady-state filter on a smaller grid and an odd number of locations
        dict(name="field_steady", kind="field", form="infinite", runs=1, steps=500, grid=6, locations=151,
             lik="poisson", method="vi"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["series", "series", "train", "batch", "pass", "predict", "filter", "field", "field", "field"])
    sum_kernel = rng.choice(["m52", "m32", "m32+m52", "m52+m32"])
    lik = rng.choice(["gaussian", "studentt", "probit", "poisson"])
    if kind == "series":
        return dict(kind=kind, n=_log_int(rng, 200, 250_000), kernel=rng.choice(["m12", sum_kernel]), lik=lik,
                    method=rng.choice(["vi", "newton", "ep"]), lr=rng.choice([0.3, 0.5]))
    if kind == "train":
        return dict(kind=kind, n=_log_int(rng, 1_000, 500_000), kernel=rng.choice(["m52", "m32", "m32+m52"]))
    if kind == "pass":
        return dict(kind=kind, series=_log_int(rng, 16, 4096), shortest=rng.randint(30, 256),
                    longest=_log_int(rng, 500, 8192), kernel=sum_kernel)
    if kind == "batch":
        return dict(kind=kind, series=_log_int(rng, 8, 256), shortest=rng.randint(20, 64),
                    longest=_log_int(rng, 300, 4096), kernel=sum_kernel, lik=lik, method=rng.choice(["vi", "ep"]),
                    lr=0.5)
    if kind == "predict":
        return dict(kind=kind, n=_log_int(rng, 500, 30_000), tests=_log_int(rng, 500, 60_000), kernel=sum_kernel,
                    lik=lik, method=rng.choice(["vi", "newton"]))
    if kind == "filter":
        return dict(kind=kind, n=_log_int(rng, 1_000, 150_000), kernel=sum_kernel)
    form = rng.choice(["dense", "dense", "meanfield", "infinite"])
    grid = rng.choice([3, 4, 5, 6, 7, 8])
    runs = _log_int(rng, 1, 32)
    return dict(kind=kind, form=form, runs=runs, steps=_log_int(rng, 40, max(60, 600 // runs)), grid=grid,
                locations=rng.randint(4 * grid * grid, 256 if grid > 6 else 5 * grid * grid + 20),
                lik=rng.choice(["poisson", "gaussian"]), method=rng.choice(["vi", "newton"]))


# ---- inputs ---------------------------------------------------------------------------
KINDS = {"m12": kernels.Matern12, "m32": kernels.Matern32, "m52": kernels.Matern52}
ORDER = {"m12": 1, "m32": 2, "m52": 3}
NOISE = 0.01          # Gaussian noise variance
SCALE, DF = 0.2, 3.0  # Student's t noise
BINSIZE = 2.0         # expected counts at f = 0


def _parts(case):
    """Component kinds, lengthscales and variances of the case's kernel."""
    names = case["kernel"].split("+")
    ls = [1.0] if len(names) == 1 else [5.0, 2.0]
    return names, ls, [1.0 / len(names)] * len(names)


def _kernel(case):
    ks = [KINDS[k](variance=v, lengthscale=s) for k, s, v in zip(*_parts(case))]
    return ks[0] if len(ks) == 1 else kernels.Sum(ks)


def _likelihood(name):
    return {"gaussian": lambda: likelihoods.Gaussian(variance=NOISE), "probit": likelihoods.Probit,
            "studentt": lambda: likelihoods.StudentsT(scale=SCALE, df=DF),
            "poisson": lambda: likelihoods.Poisson(binsize=BINSIZE)}[name]()


def _steps(n, rate, rng):
    """Uneven steps at `rate` observations a unit of time, as 32-bit numbers; the first is 0."""
    dt = rng.exponential(1.0 / rate, n).astype(np.float32)
    dt[0] = 0.0
    return dt.astype(np.float64)


def _signal(x, rng):
    """A smooth function of time with several periods."""
    f = np.zeros_like(x)
    for w in (0.31, 0.83, 1.7, 2.9):
        f += rng.uniform(0.3, 0.6) * np.sin(w * x + rng.uniform(0, 2 * np.pi))
    return f


def _observe(f, lik, rng):
    if lik == "gaussian":
        y = f + math.sqrt(NOISE) * rng.standard_normal(f.shape)
    elif lik == "studentt":
        y = f + SCALE * rng.standard_t(DF, f.shape)
    elif lik == "probit":
        y = (rng.uniform(size=f.shape) < 0.5 * (1 + np.tanh(0.8 * f))).astype(np.float64)
    else:
        y = rng.poisson(BINSIZE * np.exp(f)).astype(np.float64)
    return y.astype(np.float32).astype(np.float64)


def _series(case, n, rng):
    dt = _steps(n, 20.0, rng)
    x = np.cumsum(dt)
    return x, _observe(_signal(x, rng), case.get("lik", "gaussian"), rng)


def _lengths(case, rng):
    """Lengths spread evenly over their logarithm, in random order: every seed has the same ones."""
    lo, hi = math.log(case["shortest"]), math.log(case["longest"])
    at = (np.arange(case["series"]) + 0.5) / case["series"]
    return rng.permutation(np.floor(np.exp(lo + (hi - lo) * at)).astype(np.int64))


def _batch_hypers(case, rng):
    """One lengthscale a series, unit variances."""
    ls = np.exp(rng.uniform(math.log(0.5), math.log(20.0), case["series"]))
    n = len(case["kernel"].split("+"))
    return np.repeat(ls[:, None], n, 1), np.ones((case["series"], n))


def _batch(case, rng):
    lens = _lengths(case, rng)
    ls, var = _batch_hypers(case, rng)
    xs = [np.cumsum(_steps(n, 10.0, rng)) for n in lens]
    ys = [_observe(_signal(x, rng), case["lik"], rng) for x in xs]
    return xs, ys, ls, var


def _field(case, rng):
    """Grid, times, locations [K, T, R, 2] and counts (or noisy values) of a moving smooth field."""
    g = np.linspace(0.0, 1.0, case["grid"])
    a, b = np.meshgrid(g, g)
    z = np.stack([a.reshape(-1), b.reshape(-1)], 1)
    K, T, R = case["runs"], case["steps"], case["locations"]
    t = np.arange(T, dtype=np.float64)
    r = rng.uniform(0.0, 1.0, (K, T, R, 2)).astype(np.float32).astype(np.float64)
    p = rng.uniform(0, 2 * np.pi, (3, K, 1, 1))
    tt = t[None, :, None]
    f = (0.5 * np.sin(6 * r[..., 0] + 0.10 * tt + p[0]) + 0.5 * np.cos(5 * r[..., 1] - 0.07 * tt + p[1])
         + 0.4 * np.sin(0.05 * tt + p[2]))
    return z, t, r, _observe(f, case["lik"], rng)


def _test_times(case, x, rng):
    return rng.uniform(x[0] - 1.0, x[-1] + 1.0, case["tests"])


def _gpu(x, dtype):
    return torch.as_tensor(np.ascontiguousarray(x), dtype=dtype, device="cuda")


MODELS = {"vi": models.MarkovVariationalGP, "newton": models.MarkovLaplaceGP, "ep": models.MarkovExpectationPropagationGP}
FIELDS = {("dense", "vi"): spacetime.SpaceTimeVariationalGP, ("dense", "newton"): spacetime.SpaceTimeLaplaceGP,
          ("meanfield", "vi"): spacetime.SpaceTimeVariationalMeanFieldGP,
          ("meanfield", "newton"): spacetime.SpaceTimeLaplaceMeanFieldGP,
          ("infinite", "vi"): spacetime.SpaceTimeVariationalInfiniteHorizonGP,
          ("infinite", "newton"): spacetime.SpaceTimeLaplaceInfiniteHorizonGP}
FIELD_LS = (10.0, 0.3)  # in time and in space


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    state = {"case": case}
    if kind in ("series", "train", "predict"):
        x, y = _series(case, case["n"], rng)
        state["model"] = MODELS[case.get("method", "vi")](_kernel(case), _likelihood(case.get("lik", "gaussian")), x, y)
        if kind == "predict":
            state["tests"] = _test_times(case, x, rng)
    elif kind == "batch":
        xs, ys, ls, var = _batch(case, rng)
        state["model"] = MODELS[case["method"]].from_series(_kernel(case), _likelihood(case["lik"]), xs, ys,
                                                            lengthscale=ls, variance=var)
    elif kind == "pass":
        dt, y, off, ls, var = _pass_inputs(case, rng)
        # the chunk length whose chunks fill the GPU in one round, as a program sizes a batch of its own
        lens = np.diff(off)
        units = torch.cuda.get_device_properties(0).multi_processor_count
        p = plan.SeriesPlan(off, chunk_len=autotune.fill_chunk_len(lens, units))
        f32, f64 = torch.float32, torch.float64
        state.update(plan=p, desc=_kernel(case).desc(), ls=_gpu(ls, f64), var=_gpu(var, f64),
                     dt=p.gather(_gpu(dt, f32)), y=p.gather(_gpu(y, f32)),
                     r=p.gather(torch.full((off[-1],), NOISE, dtype=f32, device="cuda"), pad=1.0),
                     mean=torch.zeros(p.n_slots, dtype=f32, device="cuda"),
                     v=torch.zeros(p.n_slots, dtype=f32, device="cuda"))
    elif kind == "filter":
        dt, y, r = _filter_inputs(case, rng)
        state.update(kernel=_kernel(case), dt=_gpu(dt, torch.float64), after=_gpu(np.append(dt[1:], 0.0), torch.float64),
                     y=_gpu(y, torch.float64)[:, None, None], r=_gpu(r, torch.float64)[:, None, None])
    else:
        z, t, r, y = _field(case, rng)
        kern = kernels.SpatioTemporalKernel(kernels.Matern32(variance=1.0, lengthscale=FIELD_LS[0]),
                                            kernels.Matern32(variance=1.0, lengthscale=FIELD_LS[1]), z=z)
        state["model"] = FIELDS[case["form"], case["method"]].from_runs(
            kern, _likelihood(case["lik"]), [t] * case["runs"], list(r), list(y))
    return state


def _pass_inputs(case, rng):
    lens = _lengths(case, rng)
    off = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    ls, var = _batch_hypers(case, rng)
    n = int(off[-1])
    dt = rng.standard_exponential(n, dtype=np.float32) * np.float32(0.1)
    dt[off[:-1]] = 0.0
    w = np.repeat(1.0 / ls[:, 0], lens).astype(np.float32)
    y = np.sin(w * np.cumsum(dt)) + np.float32(math.sqrt(NOISE)) * rng.standard_normal(n, dtype=np.float32)
    return dt, y.astype(np.float32), off, ls, var


def _filter_inputs(case, rng):
    dt = _steps(case["n"], 20.0, rng)
    y = _observe(_signal(np.cumsum(dt), rng), "gaussian", rng)
    r = rng.uniform(0.5 * NOISE, 2 * NOISE, case["n"]).astype(np.float32).astype(np.float64)
    return dt, y, r


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "pass":
        return ops.filter_smoother(state["plan"], state["desc"], state["ls"], state["var"], state["dt"], state["y"],
                                   state["r"], hyper_stride=state["ls"].shape[1], post_mean=state["mean"],
                                   post_var=state["v"])
    if kind == "filter":
        ell, (fm, fP) = ops.kalman_filter(state["dt"], state["kernel"], state["y"], state["r"], parallel=True)
        sm, sP, gain = ops.rauch_tung_striebel_smoother(state["after"], state["kernel"], fm, fP, return_full=True,
                                                        parallel=True)
        return ell, fm, fP, sm, sP, gain
    m = state["model"]
    if kind == "train":
        m.inference(lr=1.0)
        e, g = m.energy_and_grad()
        return e, g, m.posterior_mean, m.posterior_variance
    if kind == "predict":
        m.inference(lr=0.5)
        return m.predict_y(state["tests"])
    if kind == "field":
        m.inference(lr=0.2 if case["lik"] == "poisson" else 1.0)
        return m.energy_per_run(), m.posterior_mean, m.posterior_variance, m.site_nat
    m.inference(lr=case["lr"])
    e = m.energy() if kind == "series" else m.energy_per_series()
    return e, m.posterior_mean, m.posterior_variance


# ---- work of one pass -------------------------------------------------------------------
def work(case):
    if case["kind"] == "field":
        K, T, R, M = case["runs"], case["steps"], case["locations"], case["grid"] ** 2
        D = 2 * M
        # projection of the locations on the grid and back (two directions, symmetric results), twice:
        # the update and the energy
        sites = 2 * R * M * M * 3
        if case["form"] == "dense":
            # update of rank M of a symmetric D x D covariance; gain and two symmetric products back
            walk = 2 * D * M * M + M ** 3 + D * D * M + 2 * D ** 3 // 3 + 4 * D ** 3
            stored = D * (D + 1)
        elif case["form"] == "meanfield":
            walk, stored = 2 * M ** 3 + 100 * M, 12 * M
        else:
            walk, stored = 2 * M ** 3 + 4 * D * M + 2 * D * D, 2 * D
        steps = K * T
        return dict(flops=float(steps * (sites + walk)),
                    bytes=float(8 * steps * (2 * R * M + 6 * R + 3 * M * M + stored)))
    d = sum(ORDER[k] for k in case["kernel"].split("+"))
    walk = 18 * d ** 3  # filter and smoother of one step, symmetric d x d covariances
    if case["kind"] in ("pass", "batch"):
        lo, hi = case["shortest"], case["longest"]
        n = case["series"] * (hi - lo) / math.log(hi / lo) if hi > lo else case["series"] * hi
    else:
        n = case["n"]
    if case["kind"] == "pass":
        return dict(flops=n * walk, bytes=n * 20.0)
    if case["kind"] == "filter":
        return dict(flops=float(n * walk), bytes=8.0 * n * (3 + 2 * d + 3 * d * d))
    sites = 20 * 20 if case.get("lik") in ("probit", "studentt") else 40
    flops, moved = n * (walk + 2.0 * sites), n * (4 + 8 * 4 + 8 * 2 + 16 + 24)
    if case["kind"] == "train":
        flops += 3 * n * 10.0 * d ** 3
    if case["kind"] == "predict":
        flops += case["tests"] * 20.0 * d ** 3
        moved += case["tests"] * 24.0 + 8.0 * n * (d + 2 * d * d)
    return dict(flops=float(flops), bytes=float(moved))


# ---- the same results in 64 bits, plain torch ----------------------------------------------
LOG2PI = math.log(2 * math.pi)
GH_X, GH_W = np.polynomial.hermite.hermgauss(20)
GH_X, GH_W = GH_X * math.sqrt(2.0), GH_W / math.sqrt(math.pi)
GL_X, GL_W = np.polynomial.legendre.leggauss(12)
DEVICE = "cuda" if torch.cuda.is_available() else "cpu"


def _d(a):
    """A double tensor (complex numbers stay complex) on the device that the exact results are made on."""
    if not isinstance(a, torch.Tensor):
        a = torch.as_tensor(np.asarray(a))
    return a.to(DEVICE, a.dtype if a.is_complex() or a.dtype == torch.bool else torch.float64)


def _t(a):
    return a.transpose(-1, -2)


def _mv(a, x):
    return (a @ x[..., None])[..., 0]


def _outer(a, b):
    return a[..., :, None] * b[..., None, :]


def _spd_solve(a, b):
    """a^-1 b for many small positive definite a, all at once (Gauss-Jordan, pivots on the diagonal)."""
    d = a.shape[-1]
    x = torch.cat([a, b], -1)
    for k in range(d):
        row = x[..., k, :] / x[..., k, k, None]
        x = x - _outer(x[..., :, k], row)
        x[..., k, :] = row
    return x[..., d:]


def _component(name, ls, var, dt):
    """A(dt), Q(dt) and the stationary covariance of one Matern component; ls, var: arrays over dt's shape."""
    d = ORDER[name]
    lam = {1: 1.0, 2: math.sqrt(3.0), 3: math.sqrt(5.0)}[d] / ls

    def matrix(rows):
        return torch.stack([torch.stack(torch.broadcast_tensors(*r), -1) for r in rows], -2)

    def trans(s):
        e, x = torch.exp(-lam * s), lam * s
        if d == 1:
            return matrix([[e]])
        if d == 2:
            return matrix([[e * (1 + x), e * s], [-e * x * lam, e * (1 - x)]])
        return matrix([[e * (1 + x + 0.5 * x * x), e * s * (1 + x), 0.5 * e * s * s],
                       [-0.5 * e * x * x * lam, e * (1 + x - x * x), e * s * (1 - 0.5 * x)],
                       [e * lam * lam * x * (0.5 * x - 1), e * lam * x * (x - 3), e * (1 - 2 * x + 0.5 * x * x)]])

    one = torch.ones_like(lam * dt)
    zero = 0 * one
    if d == 1:
        pinf = [[var * one]]
    elif d == 2:
        pinf = [[var * one, zero], [zero, var * lam ** 2 * one]]
    else:
        k = var * lam ** 2 / 3 * one
        pinf = [[var * one, zero, -k], [zero, k, zero], [-k, zero, var * lam ** 4 * one]]
    pinf, A = matrix(pinf), trans(dt)
    # Q = integral of (last column of A(s)) outer itself times the spectral density: no cancellation at short
    # steps; the difference Pinf - A Pinf A' at long ones
    density = (2 * lam * var, 4 * lam ** 3 * var, 16.0 / 3.0 * lam ** 5 * var)[d - 1]
    Q = 0
    for gx, gw in zip(GL_X, GL_W):
        a = trans(0.5 * (1 + gx) * dt)[..., -1]
        Q = Q + (0.5 * gw * density * dt)[..., None, None] * _outer(a, a)
    x = lam * dt
    far = ((x.real if x.is_complex() else x) > 1.0)[..., None, None]
    return A, torch.where(far, pinf - A @ pinf @ _t(A), Q), pinf


class _Prior:
    """State-space form of a sum of components; hyperparameters [S, n_comp]."""

    def __init__(self, names, ls, var):
        self.names, self.ls, self.var = names, _d(ls), _d(var)
        self.d = sum(ORDER[n] for n in names)
        at = [sum(ORDER[m] for m in names[:i]) for i in range(len(names))]
        self.parts = list(zip(names, at))
        self.H = torch.zeros(self.d, dtype=self.ls.dtype, device=DEVICE)
        self.H[at] = 1.0

    def steps(self, dt, series):
        """A, Q and Pinf for steps dt [rows, ...]; series: the series of each row."""
        out = [torch.zeros(dt.shape + (self.d, self.d), dtype=self.ls.dtype, device=DEVICE) for _ in range(3)]
        for i, (n, o) in enumerate(self.parts):
            shape = (-1,) + (1,) * (dt.dim() - 1)
            got = _component(n, self.ls[series, i].reshape(shape), self.var[series, i].reshape(shape), dt)
            for a, b in zip(out, got):
                a[..., o:o + ORDER[n], o:o + ORDER[n]] = b
        return out


def _smooth(prior, dt, y, r, masked, keep=False, loglik_only=False):
    """Filter and smoother of S series [S, N], cut into pieces whose maps are chained, so that the steps of all pieces
    run side by side.  Rows shorter than N end in masked steps with dt = 0 and r = inf.  masked: no log-likelihood
    term.  Returns log-likelihoods [S] and the smoothed f (mean, variance) or, with keep, the filtered and smoothed
    states (means, covariances) and the smoother's gains."""
    S, N = dt.shape
    L = N if N <= 400 or S >= 64 else int(math.ceil(math.sqrt(N * 1.5)))
    C = -(-N // L)
    B, d, H = S * C, prior.d, prior.H
    kind = H.dtype

    def cut(a, v):  # [L, B]
        return torch.cat([a, torch.full((S, C * L - N), v, dtype=a.dtype, device=DEVICE)], 1).reshape(B, L).t()

    cy, cm, w = cut(y, 0.0), cut(masked, True), 1.0 / cut(r, math.inf)  # precision: 0 where padded
    series = torch.arange(S, device=DEVICE).repeat_interleave(C)

    def tables(steps):
        return [a.transpose(0, 1).contiguous() for a in prior.steps(cut(steps, 0.0).t(), series)[:2]]

    As, Qs = tables(dt)
    m0 = torch.zeros((S, d), dtype=kind, device=DEVICE)
    P0 = prior.steps(dt[:, :1], torch.arange(S, device=DEVICE))[2][:, 0]

    def update(P, m, k):
        """P H', 1 / (H P H' + r) and the innovation of step k."""
        ph = P @ H
        return ph, w[k] / (1 + w[k] * (ph @ H)), cy[k] - m @ H

    starts = [(m0, P0)]
    if C > 1:
        F = torch.eye(d, dtype=kind, device=DEVICE).expand(B, d, d)
        b, V = torch.zeros((B, d), dtype=kind, device=DEVICE), torch.zeros((B, d, d), dtype=kind, device=DEVICE)
        J, eta = V, b
        for k in range(L):
            F, b, V = As[k] @ F, _mv(As[k], b), As[k] @ V @ _t(As[k]) + Qs[k]
            ph, g, e = update(V, b, k)
            hf, g1, g2 = H @ F, g[:, None], g[:, None, None]
            J, eta = J + g2 * _outer(hf, hf), eta + g1 * e[:, None] * hf
            b, F, V = b + g1 * e[:, None] * ph, F - g2 * _outer(ph, hf), V - g2 * _outer(ph, ph)
        F, b, V, J, eta = (a.reshape((S, C) + a.shape[1:]) for a in (F, b, V, J, eta))
        eye = torch.eye(d, dtype=kind, device=DEVICE)
        for c in range(C - 1):
            m1 = torch.cat([P0, (m0 + _mv(P0, eta[:, c]))[..., None]], -1)
            m1 = torch.linalg.solve((eye + P0 @ J[:, c]).cpu(), m1.cpu()).to(DEVICE)
            m0, P0 = _mv(F[:, c], m1[..., d]) + b[:, c], F[:, c] @ m1[..., :d] @ _t(F[:, c]) + V[:, c]
            P0 = 0.5 * (P0 + _t(P0))
            starts.append((m0, P0))
    m, P = (torch.stack(a, 1).flatten(0, 1) for a in zip(*starts))
    ll = torch.zeros(B, dtype=kind, device=DEVICE)
    fm, fP = [], []
    for k in range(L):
        m, P = _mv(As[k], m), As[k] @ P @ _t(As[k]) + Qs[k]
        ph, g, e = update(P, m, k)
        one = torch.where(cm[k], 1.0, g)
        ll = ll + torch.where(cm[k], 0.0, -0.5 * (LOG2PI - torch.log(one) + g * e * e))
        m, P = m + (g * e)[:, None] * ph, P - g[:, None, None] * _outer(ph, ph)
        P = 0.5 * (P + _t(P))
        if not loglik_only:
            fm.append(m)
            fP.append(P)
    ll = ll.reshape(S, C).sum(1)
    if loglik_only:
        return ll
    fm, fP = torch.stack(fm), torch.stack(fP)
    As, Qs = tables(torch.cat([dt[:, 1:], torch.zeros_like(dt[:, :1])], 1))
    AP = As @ fP
    ahead = AP @ _t(As) + Qs
    gains = _t(_spd_solve(ahead, AP))
    drift, rest = fm - _mv(gains, _mv(As, fm)), fP - gains @ ahead @ _t(gains)
    del AP, ahead, As, Qs
    sm, sP = fm[-1].reshape(S, C, d)[:, -1], fP[-1].reshape(S, C, d, d)[:, -1]
    ends = [(sm, sP)]
    if C > 1:
        E = torch.eye(d, dtype=kind, device=DEVICE).expand(B, d, d)
        g0, V = torch.zeros((B, d), dtype=kind, device=DEVICE), torch.zeros((B, d, d), dtype=kind, device=DEVICE)
        for k in range(L - 1, -1, -1):
            G = gains[k]
            E, g0, V = G @ E, drift[k] + _mv(G, g0), rest[k] + G @ V @ _t(G)
        E, g0, V = (a.reshape((S, C) + a.shape[1:]) for a in (E, g0, V))
        for c in range(C - 1, 0, -1):
            sm, sP = g0[:, c] + _mv(E[:, c], sm), V[:, c] + E[:, c] @ sP @ _t(E[:, c])
            ends.append((sm, sP))
    sm, sP = (torch.stack(a[::-1], 1).flatten(0, 1) for a in zip(*ends))
    om, oP = [], []
    for k in range(L - 1, -1, -1):
        sm, sP = drift[k] + _mv(gains[k], sm), rest[k] + gains[k] @ sP @ _t(gains[k])
        sP = 0.5 * (sP + _t(sP))
        om.append(sm if keep else sm @ H)
        oP.append(sP if keep else (sP @ H) @ H)

    def rows(a):
        return a.transpose(0, 1).reshape((S, C * L) + a.shape[2:])[:, :N]

    om, oP = rows(torch.stack(om[::-1])), rows(torch.stack(oP[::-1]))
    return (ll, rows(fm), rows(fP), om, oP, rows(gains)) if keep else (ll, om, oP)


def _log_p(lik, y, f):
    """log p(y | f) and its first two derivatives in f."""
    if lik == "gaussian":
        return -0.5 * (LOG2PI + math.log(NOISE)) - 0.5 * (y - f) ** 2 / NOISE, (y - f) / NOISE, -1.0 / NOISE + 0 * f
    if lik == "poisson":
        mu = BINSIZE * torch.exp(f)
        return y * torch.log(mu) - mu - torch.lgamma(y + 1.0), y - mu, -mu
    e = y - f
    if lik == "studentt":
        q = DF * SCALE ** 2
        c = math.lgamma(0.5 * (DF + 1)) - math.lgamma(0.5 * DF) - 0.5 * math.log(q * math.pi)
        return (c - 0.5 * (DF + 1) * torch.log1p(e * e / q), (DF + 1) * e / (q + e * e),
                (DF + 1) * (e * e - q) / (q + e * e) ** 2)
    s, eps = torch.where(y == 1, 1.0, -1.0).double(), 1e-3
    p = eps + (1 - 2 * eps) * torch.special.ndtr(s * f)
    j = s * (1 - 2 * eps) * torch.exp(-0.5 * f * f) / math.sqrt(2 * math.pi) / p
    return torch.log(p), j, -f * j - j * j


def _expect(lik, y, m, v):
    """E log p under N(m, v) and its derivative and second derivative in m."""
    if lik == "gaussian":
        ll, j, h = _log_p(lik, y, m)
        return ll - 0.5 * v / NOISE, j, h
    if lik == "poisson":
        mu = BINSIZE * torch.exp(m + 0.5 * v)
        return y * math.log(BINSIZE) + y * m - mu - torch.lgamma(y + 1.0), y - mu, -mu
    E, J, H = 0.0, 0.0, 0.0
    for x, w in zip(GH_X, GH_W):
        p = w * _log_p(lik, y, torch.sqrt(v) * x + m)[0]
        E, J, H = E + p, J + x * p / torch.sqrt(v), H + (x * x - 1) * p / v
    return E, J, H


def _match(lik, y, m, v):
    """log of E p under N(m, v) and its derivatives in m."""
    if lik == "gaussian":
        s = NOISE + v
        return -0.5 * (LOG2PI + torch.log(s) + (y - m) ** 2 / s), (y - m) / s, -1 / s
    Z, J, H = 0.0, 0.0, 0.0
    for x, w in zip(GH_X, GH_W):
        p = w * torch.exp(_log_p(lik, y, torch.sqrt(v) * x + m)[0])
        Z, J, H = Z + p, J + x * p / torch.sqrt(v), H + (x * x - 1) * p / v
    Z = Z.clamp(min=1e-8)
    return torch.log(Z), J / Z, H / Z - (J / Z) ** 2


def _cavity(m, v, n1, n2):
    q = 1.0 / (v + 1e-8)
    cv = 1.0 / (q - n2)
    return cv * (q * m - n1), cv


def _site(method, lik, y, m, v, n1, n2, lr):
    if method == "ep":
        m, v = _cavity(m, v, n1, n2)
        _, j, h = _match(lik, y, m, v)
        scale = (1 / v) / (h + 1 / v)
        j, h = scale * j, scale * h
    else:
        _, j, h = _expect(lik, y, m, v) if method == "vi" else _log_p(lik, y, m)
    h = torch.where(-h < 0, -1e-2, h)
    return (1 - lr) * n1 + lr * (j - h * m), (1 - lr) * n2 + lr * -h


def _energy(method, lik, y, m, v, n1, n2, ll, real):
    """Energies of the rows; real: which entries are observations."""
    if method == "ep":
        cm, cv = _cavity(m, v, n1, n2)
        s = 1 / n2 + cv
        pseudo = -0.5 * (LOG2PI + torch.log(s) + (n1 / n2 - cm) ** 2 / s)
        return -(ll + torch.where(real, _match(lik, y, cm, cv)[0] - pseudo, 0.0).sum(1))
    data = _expect(lik, y, m, v)[0] if method == "vi" else _log_p(lik, y, m)[0]
    ed = -0.5 * (LOG2PI - torch.log(n2) + n2 * ((n1 / n2 - m) ** 2 + v))
    return -(torch.where(real, data - ed, 0.0).sum(1) + ll)


def _iterate(case, prior, dt, y, real, lr):
    """The pass on a new model: sites N(0, 1e2), posterior, site update.  Returns the sites both ways."""
    def sites(n1, n2):
        return torch.where(real, n1 / n2, 0.0), torch.where(real, 1 / n2, math.inf)

    n1, n2 = torch.zeros_like(y), torch.full_like(y, 1e-2)
    _, m, v = _smooth(prior, dt, *sites(n1, n2), ~real)
    n1, n2 = _site(case.get("method", "vi"), case.get("lik", "gaussian"), y, m, v, n1, n2, lr)
    return n1, n2, sites(n1, n2)


def _f32(a):
    return np.asarray(a, np.float32).astype(np.float64)


def _exact_series(case, rng):
    names, ls, var = _parts(case)
    x, y = _series(case, case["n"], rng)
    dt, y = _d(_f32(np.diff(x, prepend=x[0])))[None], _d(y)[None]
    real = torch.ones_like(y, dtype=torch.bool)
    prior = _Prior(names, [ls], [var])
    kind = case["kind"]
    lr = {"train": 1.0, "predict": 0.5}.get(kind, case.get("lr"))
    n1, n2, (py, pr) = _iterate(case, prior, dt, y, real, lr)
    if kind == "predict":
        return _exact_predict(case, prior, _d(x), dt, py, pr, _d(_test_times(case, x, rng)))
    ll, m, v = _smooth(prior, dt, py, pr, ~real)
    e = _energy(case.get("method", "vi"), case.get("lik", "gaussian"), y, m, v, n1, n2, ll, real)[0]
    m, v = m.reshape(-1, 1, 1), v.reshape(-1, 1, 1)
    if kind == "series":
        return e, m, v
    # derivatives of the log-likelihood in every hyperparameter by a complex step, chained through softplus
    grad = []
    for i in range(len(names)):
        for which, value in ((0, ls[i]), (1, var[i])):
            h = [np.array([ls], complex), np.array([var], complex)]
            h[which][0, i] += 1e-30j
            g = float(_smooth(_Prior(names, *h), dt, py, pr, ~real, loglik_only=True)[0].imag) / 1e-30
            grad.append(g * math.expm1(-value))
    g = float((0.5 / NOISE - 0.5 * ((y[0] - m[:, 0, 0]) ** 2 + v[:, 0, 0]) / NOISE ** 2).sum())
    grad.append(g * -math.expm1(-NOISE))
    return float(e), np.array(grad), m, v


def _exact_predict(case, prior, x, dt, py, pr, tests):
    _, _, _, sm, sP, gain = _smooth(prior, dt, py, pr, torch.zeros_like(py, dtype=torch.bool), keep=True)
    d, H = prior.d, prior.H
    one = torch.zeros(1, dtype=torch.long, device=DEVICE)
    Pinf = prior.steps(torch.zeros_like(dt[:, :1]), one)[2][0]
    zero = torch.zeros_like(sm[0, :1])
    m = torch.cat([zero, sm[0], zero])
    P = torch.cat([Pinf, sP[0], Pinf])
    G = torch.cat([torch.zeros_like(Pinf), gain[0]])
    xs = torch.cat([_d([-1e10]), x, _d([1e10])])
    k = torch.searchsorted(xs, tests) - 1
    Af, Qf, _ = (a[0] for a in prior.steps((tests - xs[k])[None], one))
    Ab, Qb, _ = (a[0] for a in prior.steps((xs[k + 1] - tests)[None], one))
    AQ = Ab @ Qf
    V = _spd_solve(Qb + Ab @ _t(AQ) + 1e-8 * torch.eye(d, dtype=torch.float64, device=DEVICE), Ab)
    W = Qf @ _t(V)
    T = Qf - _t(AQ) @ V @ Qf
    u = H @ torch.cat([Af - W @ Ab @ Af, W], -1)
    cross = G[k] @ P[k + 1]
    cov = torch.cat([torch.cat([P[k], cross], -1), torch.cat([_t(cross), P[k + 1]], -1)], -2)
    mean = (u * torch.cat([m[k], m[k + 1]], -1)).sum(-1)
    var = (_mv(cov, u) * u).sum(-1) + (T @ H) @ H
    if case["lik"] == "gaussian":
        return mean, var + NOISE
    ey = ey2 = 0.0
    for gx, gw in zip(GH_X, GH_W):
        f = torch.sqrt(var) * gx + mean
        if case["lik"] == "poisson":
            mu = s2 = BINSIZE * torch.exp(f)
        elif case["lik"] == "studentt":
            mu, s2 = f, SCALE ** 2 * DF / (DF - 2)
        else:
            mu = 1e-3 + (1 - 2e-3) * torch.special.ndtr(f)
            s2 = mu - mu * mu
        ey, ey2 = ey + gw * mu, ey2 + gw * (s2 + mu * mu)
    return ey, ey2 - ey * ey


def _rows(parts, fill):
    """Series of uneven length as the rows of one array."""
    out = np.full((len(parts), max(len(p) for p in parts)), fill)
    for row, p in zip(out, parts):
        row[:len(p)] = p
    return _d(out)


def _exact_batch(case, rng):
    xs, ys, ls, var = _batch(case, rng)
    dt, y = _rows([_f32(np.diff(x, prepend=x[0])) for x in xs], 0.0), _rows(ys, 0.0)
    real = _rows([np.ones(len(x)) for x in xs], 0.0) > 0
    prior = _Prior(case["kernel"].split("+"), ls, var)
    n1, n2, (py, pr) = _iterate(case, prior, dt, y, real, case["lr"])
    ll, m, v = _smooth(prior, dt, py, pr, ~real)
    e = _energy(case["method"], case["lik"], y, m, v, n1, n2, ll, real)
    return e, m[real].reshape(-1, 1, 1), v[real].reshape(-1, 1, 1)


def _exact_pass(case, rng):
    """The log-likelihoods (the moments come in the plan's own layout)."""
    dt, y, off, ls, var = _pass_inputs(case, rng)
    cut = lambda a: np.split(a, off[1:-1])  # noqa: E731
    real = _rows(cut(np.ones_like(y)), 0.0) > 0
    r = torch.where(real, float(np.float32(NOISE)), math.inf).double()
    return _smooth(_Prior(case["kernel"].split("+"), ls, var), _rows(cut(dt), 0.0), _rows(cut(y), 0.0), r, ~real,
                   loglik_only=True)


def _exact_filter(case, rng):
    dt, y, r = (_d(a)[None] for a in _filter_inputs(case, rng))
    names, ls, var = _parts(case)
    ll, fm, fP, sm, sP, gain = _smooth(_Prior(names, [ls], [var]), dt, y, r, torch.zeros_like(y, dtype=torch.bool),
                                       keep=True)
    return ll[0], fm[0, :, :, None], fP[0], sm[0, :, :, None], sP[0], gain[0]


def _exact_field(case, rng):
    """One pass of the dense model, runs side by side, state (f, f') of every grid point."""
    z, t, r, y = _field(case, rng)
    K, T, R, M = case["runs"], case["steps"], case["locations"], len(z)
    lik, lr = case["lik"], 0.2 if case["lik"] == "poisson" else 1.0
    z, r, y = _d(z), _d(r), _d(y)

    def cov(a, b):
        d2 = ((a[..., :, None, :] - b[..., None, :, :]) ** 2).sum(-1)
        s = math.sqrt(3.0) / FIELD_LS[1] * torch.sqrt(d2.clamp(min=1e-36))
        return (1 + s) * torch.exp(-s)

    def lower_solve(L, b):
        return torch.linalg.solve_triangular(L, b, upper=False)

    def chol_solve(L, b):
        return torch.linalg.solve_triangular(_t(L), lower_solve(L, b), upper=True)

    eye = torch.eye(M, dtype=torch.float64, device=DEVICE)
    B = cov(r, z) @ _t(lower_solve(torch.linalg.cholesky(cov(z, z)), eye)).contiguous()  # [K, T, R, M]
    Bt = _t(B).contiguous()
    c = 1.0 - (Bt ** 2).sum(-2)
    one = _d([1.0])
    A, Q, Pinf = (torch.kron(a[0], eye) for a in _component("m32", FIELD_LS[0] * one, one, one))

    def project(n1, n2):
        N2, N1 = Bt @ (n2[..., None] * B) + 1e-12 * eye, Bt @ n1[..., None]
        W = torch.stack([torch.linalg.cholesky(N2[:, k]) for k in range(T)], 1)
        return W, torch.stack([lower_solve(W[:, k], N1[:, k])[..., 0] for k in range(T)], 1)

    def posterior(W, q):
        m, P = torch.zeros_like(Pinf[:1]).expand(K, -1), Pinf.expand(K, -1, -1)
        ll, kept = 0.0, []
        for k in range(T):
            if k:
                m, P = m @ A.t(), A @ P @ A.t() + Q
            U = P[:, :, :M] @ W[:, k]
            G = torch.linalg.cholesky(eye + _t(W[:, k]) @ U[:, :M])
            e = q[:, k] - _mv(_t(W[:, k]), m[:, :M])
            V = lower_solve(G, torch.cat([_t(U), e[..., None]], -1))
            V, e = V[..., :-1], V[..., -1]
            ll = ll - 0.5 * ((e * e).sum(-1) + M * LOG2PI) - torch.log(G.diagonal(dim1=1, dim2=2)).sum(-1)
            ll = ll + torch.log(W[:, k].diagonal(dim1=1, dim2=2)).sum(-1)
            m, P = m + _mv(_t(V), e), P - _t(V) @ V
            kept.append((m, P))
        out = [(m[:, :M], P[:, :M, :M])]
        for fm, fP in reversed(kept[:-1]):
            AP = A @ fP
            ahead = AP @ A.t() + Q
            G = _t(chol_solve(torch.linalg.cholesky(ahead), AP))
            m, P = fm + _mv(G, m - fm @ A.t()), fP + G @ (P - ahead) @ _t(G)
            P = 0.5 * (P + _t(P))
            out.append((m[:, :M], P[:, :M, :M]))
        return (ll,) + tuple(torch.stack(a[::-1], 1) for a in zip(*out))

    def marginals(pm, pP):
        return _mv(B, pm), ((B @ pP) * B).sum(-1) + c

    n1, n2 = torch.zeros_like(y), torch.full_like(y, 1e-2)
    _, pm, pP = posterior(*project(n1, n2))
    n1, n2 = _site(case["method"], lik, y, *marginals(pm, pP), n1, n2, lr)
    W, q = project(n1, n2)
    ll, pm, pP = posterior(W, q)
    m, v = marginals(pm, pP)
    data = (_expect(lik, y, m, v) if case["method"] == "vi" else _log_p(lik, y, m))[0].sum((1, 2))
    q = q - _mv(_t(W), pm)
    ed = -0.5 * ((q ** 2).sum((1, 2)) + T * M * LOG2PI + (W * (pP @ W)).sum((1, 2, 3)))
    ed = ed + torch.log(W.diagonal(dim1=2, dim2=3)).sum((1, 2))
    return -(data - (ed - ll)), pm[..., None], pP, (n1, n2)


def exact(case, seed):
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    if kind in ("series", "train", "predict"):
        return _exact_series(case, rng)
    if kind == "filter":
        return _exact_filter(case, rng)
    if kind == "batch":
        return _exact_batch(case, rng)
    if kind == "pass":
        return (None, None, _exact_pass(case, rng)) if case["series"] * case["longest"] <= 4_000_000 else None
    # the mean-field and steady-state filters are approximations, given by their own recursions alone
    return _exact_field(case, rng) if case["form"] == "dense" else None
