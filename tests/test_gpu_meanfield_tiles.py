"""The mean-field recursions at the edges of their tiles (8 steps, 32 or 64 lanes) against the
FP64 oracle, and lanes of several runs in one workgroup against the runs by themselves.  FP64
on both sides: 1e-8 relative on the blocks, as for the other mean-field operations; the same
operations in the same order for runs taken together or alone: 1e-12."""
import numpy as np
import pytest

from oracle import kernels as OK, ops as OP

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return np.max(np.abs(a - b)) / np.max(np.abs(b))


@pytest.mark.parametrize("kt", [1, 2])
@pytest.mark.parametrize("M,N", [(1, 1), (1, 17), (2, 8), (3, 9), (33, 7), (64, 16), (64, 25)])
def test_recursions_match_oracle(kt, M, N):
    from bayesnewton_amd import kernels as K, ops
    rng = np.random.default_rng(100 * M + N)
    z = rng.uniform(size=(M, 2))
    gt, ot = ((K.Matern12, OK.Matern12), (K.Matern32, OK.Matern32))[kt - 1]
    gk = K.SpatioTemporalKernel(gt(variance=1.3, lengthscale=2.0), K.Matern32(variance=1.0, lengthscale=0.4), z=z)
    ok = OK.SpatioTemporalKernel(ot(1.3, 2.0), OK.Matern32(1.0, 0.4), z)
    dt = np.concatenate([[0.0], rng.uniform(0.1, 1.5, N - 1)])
    y = rng.standard_normal((N, M, 1))
    G = rng.standard_normal((N, M, M)) * (0.8 / np.sqrt(M))
    R = G @ np.swapaxes(G, -1, -2) + np.eye(M) * rng.uniform(0.05, 0.5, (N, 1, 1))
    _, (fm, fP) = ops.kalman_filter_meanfield(dt, gk, y, R, parallel=True)
    _, (ofm, ofP) = OP.kalman_filter_meanfield(dt, ok, y, R, parallel=True)
    assert _rel(fm.cpu().numpy(), ofm) < 1e-8 and _rel(fP.cpu().numpy(), ofP) < 1e-8
    after = np.concatenate([dt[1:], [0.0]])
    got = ops.rauch_tung_striebel_smoother_meanfield(after, gk, ofm, ofP, return_full=True, parallel=True)
    want = OP.rauch_tung_striebel_smoother_meanfield(after, ok, ofm, ofP, return_full=True, parallel=True)
    for a, b in zip(got, want):
        assert a.shape == b.shape and _rel(a.cpu().numpy(), b) < 1e-8


@pytest.mark.parametrize("M,runs,T", [(1, 40, 9), (2, 33, 7), (9, 15, 17), (64, 3, 8)])
def test_runs_together_equal_runs_alone(M, runs, T):
    from bayesnewton_amd import kernels as K, likelihoods as L, spacetime as S
    rng = np.random.default_rng(M)
    g = np.linspace(0.0, 1.0, 8)
    z = np.stack([a.ravel() for a in np.meshgrid(g, g)], 1)[:M]
    nr = 4 * M + 3
    ts = [np.cumsum(rng.integers(1, 4, T)).astype(np.float64) for _ in range(runs)]
    rs = [rng.uniform(size=(T, nr, 2)).astype(np.float32).astype(np.float64) for _ in range(runs)]
    ys = [rng.poisson(2.0, (T, nr)).astype(np.float64) for _ in range(runs)]

    def model(sel):
        k = K.SpatioTemporalKernel(K.Matern32(variance=1.0, lengthscale=5.0), K.Matern32(variance=1.0, lengthscale=0.3),
                                   z=z)
        m = S.SpaceTimeVariationalMeanFieldGP.from_runs(k, L.Poisson(binsize=2.0), [ts[i] for i in sel],
                                                        [rs[i] for i in sel], [ys[i] for i in sel])
        m.inference(lr=0.3)
        return m.posterior_mean.cpu().numpy(), m.energy_per_run().cpu().numpy()

    mean, e = model(range(runs))
    for i in (0, runs // 2, runs - 1):
        m1, e1 = model([i])
        assert _rel(mean[i], m1.reshape(mean[i].shape)) < 1e-12
        assert abs(e[i] - e1[0]) <= 1e-12 * abs(e1[0])
