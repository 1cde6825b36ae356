"""The space-time kernels at the edges of their 16-wide tiles: numbers of inducing points
around multiples of 16, both temporal state sizes, the shortest runs, against the FP64 oracle.

Tolerance 1e-6 of the field's scale: FP64 throughout on both sides, and the oracle's explicit
inverse of B' diag(nat2) B (condition up to about 1e7 on these grids) limits the agreement to
about 1e7 * 2e-16 with two orders of headroom.
"""
import numpy as np
import pytest

from oracle import kernels as OK, likelihoods as OL, models as OM

pytestmark = pytest.mark.gpu

TOL = 1e-6


def _case(M, kt, T, seed=11):
    from bayesnewton_amd import kernels as K, likelihoods as L, models as GM
    g = np.linspace(0.0, 1.0, 8)
    a, b = np.meshgrid(g, g)
    z = np.stack([a.ravel(), b.ravel()], 1)[:M]
    rng = np.random.default_rng(seed)
    nr = 4 * M + 3
    t = np.cumsum(rng.integers(1, 4, T)).astype(np.float64)
    r = rng.uniform(size=(T, nr, 2)).astype(np.float32).astype(np.float64)
    f = np.sin(0.3 * t)[:, None] + np.cos(3.0 * r[..., 0]) * np.sin(2.0 * r[..., 1])
    y = rng.poisson(2.0 * np.exp(f)).astype(np.float64)
    gt, ot = ((K.Matern12, OK.Matern12), (K.Matern32, OK.Matern32))[kt - 1]
    gk = K.SpatioTemporalKernel(gt(variance=1.2, lengthscale=6.0), K.Matern32(variance=0.9, lengthscale=0.25), z=z)
    ok = OK.SpatioTemporalKernel(ot(1.2, 6.0), OK.Matern32(0.9, 0.25), z, sparse=True, conditional="Full")
    gm = GM.MarkovVariationalGP(gk, L.Poisson(binsize=2.0), t, y, R=r)
    om = OM.MarkovGP(ok, OL.Poisson(2.0), t[:, None], y, R=r, inference="VI")
    return gm, om


def _close(got, want):
    got, want = got.cpu().numpy(), np.asarray(want)
    assert got.shape == want.shape
    assert np.max(np.abs(got - want)) <= TOL * np.max(np.abs(want))


@pytest.mark.parametrize("kt", [1, 2])
@pytest.mark.parametrize("M", [1, 2, 15, 16, 17, 31, 32, 33, 48, 49, 63, 64])
def test_inducing_points_around_tiles(M, kt):
    gm, om = _case(M, kt, 6)
    for _ in range(2):
        gm.inference(lr=0.2)
        om.inference(lr=0.2)
    _close(gm.posterior_mean, om.posterior_mean)
    _close(gm.posterior_variance, om.posterior_variance)
    assert abs(float(gm.energy()) - om.energy()) <= TOL * abs(om.energy())


@pytest.mark.parametrize("T", [1, 2, 3, 9, 10, 11, 40])
def test_run_lengths_around_one_chunk(T):
    """Up to 9 steps back one chunk is walked; longer runs are cut into chunks."""
    gm, om = _case(20, 2, T)
    gm.inference(lr=0.2)
    om.inference(lr=0.2)
    _close(gm.posterior_mean, om.posterior_mean)
    _close(gm.posterior_variance, om.posterior_variance)
    assert abs(float(gm.compute_log_lik()) - om.compute_log_lik()) <= TOL * abs(om.compute_log_lik())


def test_many_runs_in_blocks_of_steps():
    """130 runs of 24 steps at M = 64 go back in two blocks of steps, one chunk each; two runs in
    one block of several chunks.  Same arithmetic up to the order of the covariance sums: 1e-10."""
    from bayesnewton_amd import kernels as K, likelihoods as L, spacetime as S
    g = np.linspace(0.0, 1.0, 8)
    a, b = np.meshgrid(g, g)
    z = np.stack([a.ravel(), b.ravel()], 1)
    rng = np.random.default_rng(5)
    T, nr = 24, 200
    t = np.arange(T, dtype=np.float64)
    r = rng.uniform(size=(2, T, nr, 2)).astype(np.float32).astype(np.float64)
    y = rng.poisson(2.0 * np.exp(np.sin(4 * r[..., 0]))).astype(np.float64)
    out = []
    for n in (130, 2):
        kern = K.SpatioTemporalKernel(K.Matern32(variance=1.0, lengthscale=8.0),
                                      K.Matern32(variance=1.0, lengthscale=0.25), z=z)
        idx = [i % 2 for i in range(n)]
        m = S.SpaceTimeVariationalGP.from_runs(kern, L.Poisson(binsize=2.0), [t] * n, [r[i] for i in idx],
                                               [y[i] for i in idx])
        m.inference(lr=0.2, return_terms=False)
        m.inference(lr=0.2, return_terms=False)
        out.append((m.posterior_mean[-2:].cpu().numpy(), m.posterior_variance[-2:].cpu().numpy()))
    for x, w in zip(*out):
        assert np.max(np.abs(x - w)) <= 1e-10 * np.max(np.abs(w))


def test_blocks_of_several_chunks():
    """One run of 2,700 steps at M = 64 goes back in two blocks of steps, two such runs in three,
    every block in several chunks: the ends of blocks and chunks lie elsewhere, and only the
    order of the covariance sums differs, 1e-10.  The first steps see all of them."""
    from bayesnewton_amd import kernels as K, likelihoods as L, spacetime as S
    g = np.linspace(0.0, 1.0, 8)
    z = np.stack([a.ravel() for a in np.meshgrid(g, g)], 1)
    rng = np.random.default_rng(6)
    T, nr = 2700, 70
    t = np.cumsum(rng.integers(1, 3, T)).astype(np.float64)
    r = rng.uniform(size=(T, nr, 2)).astype(np.float32).astype(np.float64)
    y = np.sin(4 * r[..., 0] + 0.05 * t[:, None]) + 0.3 * rng.standard_normal((T, nr))
    out = []
    for n in (1, 2):
        kern = K.SpatioTemporalKernel(K.Matern32(variance=1.0, lengthscale=300.0),
                                      K.Matern32(variance=1.0, lengthscale=0.25), z=z)
        m = S.SpaceTimeVariationalGP.from_runs(kern, L.Gaussian(variance=0.09), [t] * n, [r] * n, [y] * n)
        m.inference(lr=1.0, return_terms=False)
        out.append([a.reshape(n, T, -1)[-1].cpu().numpy() for a in (m.posterior_mean, m.posterior_variance)])
    for a, b in zip(*out):
        for s in (slice(0, 60), slice(60, 120), slice(1200, 1500), slice(2500, 2700)):
            assert np.max(np.abs(a[s] - b[s])) <= 1e-10 * np.max(np.abs(b[s]))


@pytest.mark.parametrize("M", [9, 33])
@pytest.mark.parametrize("noise", [1e-2, 1e-4, 1e-6])
def test_equal_times_and_precise_observations(M, noise):
    """Steps of length zero: the predicted covariance is the filtered one, as small as the noise
    where the sites determine the field, and the gain is the identity.  The oracle agrees with
    the dense posterior to 1e-15 / noise; the library has the same terms: 1e-8."""
    from bayesnewton_amd import kernels as K, likelihoods as L, models as GM
    g = np.linspace(0.0, 1.0, 8)
    z = np.stack([a.ravel() for a in np.meshgrid(g, g)], 1)[:M]
    rng = np.random.default_rng(3)
    t = np.array([0.0, 0.0, 1.0, 1.0, 1.0, 2.0, 5.0, 5.0, 6.0])
    T, nr = len(t), 4 * M + 3
    r = rng.uniform(size=(T, nr, 2)).astype(np.float32).astype(np.float64)
    f = np.sin(0.3 * t)[:, None] + np.cos(3.0 * r[..., 0]) * np.sin(2.0 * r[..., 1])
    y = (f + np.sqrt(noise) * rng.standard_normal((T, nr))).astype(np.float32).astype(np.float64)
    gk = K.SpatioTemporalKernel(K.Matern32(variance=1.2, lengthscale=6.0), K.Matern32(variance=0.9, lengthscale=0.25), z=z)
    ok = OK.SpatioTemporalKernel(OK.Matern32(1.2, 6.0), OK.Matern32(0.9, 0.25), z, sparse=True, conditional="Full")
    gm = GM.MarkovVariationalGP(gk, L.Gaussian(variance=noise), t, y, R=r)
    om = OM.MarkovGP(ok, OL.Gaussian(noise), t[:, None], y, R=r, inference="VI")
    for m in (gm, om):
        m.inference(lr=1.0)
    for got, want in ((gm.posterior_mean, om.posterior_mean), (gm.posterior_variance, om.posterior_variance)):
        got, want = got.cpu().numpy(), np.asarray(want)
        assert np.max(np.abs(got - want)) <= 1e-8 * np.max(np.abs(want))
    assert abs(float(gm.energy()) - om.energy()) <= 1e-8 * abs(om.energy())
