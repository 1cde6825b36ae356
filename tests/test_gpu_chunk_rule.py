"""The chunk length that models and single operations choose, at the edges of its rule."""
import numpy as np
import pytest
import torch

from bayesnewton_amd.plan import default_chunk_len, model_chunk_len


@pytest.mark.parametrize("lengths", [[], [0], [1], [31, 32], [33], [4095], [4000, 96], [131072], [131073], [458753],
                                     [3840] * 4096, [40_000_000], [5_000_000] * 10])
def test_rule_bounds_each_series_to_its_scan(lengths):
    c = model_chunk_len(lengths)
    nmax = max([1] + lengths)
    assert 1 <= c <= max(32, 128, -(-nmax // 16384))
    assert -(-nmax // c) <= 128 * 128
    if nmax <= 32:
        assert c == nmax
    elif sum(lengths) < 4096:
        assert c == default_chunk_len(lengths)
    assert model_chunk_len(lengths, parallel=False) == default_chunk_len(lengths, parallel=False)


@pytest.mark.parametrize("lengths,longer", [([2000] * 1000, False), ([2000] * 2000, False), ([2000] * 3670, False),
                                            ([2000] * 3671, True), ([3840] * 4096, True)])
def test_chunks_longer_than_the_default(lengths, longer):
    """Only under a sum, from 128 * 57344 = 7,340,032 steps on: elsewhere they slow the site update."""
    for d in (1, 2, 3):
        assert model_chunk_len(lengths, state_dim=d) == 32
    for d in (4, 5, 6):
        assert model_chunk_len(lengths, state_dim=d) == (128 if longer else 32)
    assert model_chunk_len([40_000_000], state_dim=5) == -(-40_000_000 // 16384)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 32, 33, 4095, 4096, 4097, 131073])
def test_parallel_filter_at_the_rule_edges_equals_the_sequential_one(n):
    """FP64 on both sides: the two orders of the same sums agree to 1e-9."""
    from bayesnewton_amd import kernels as K, ops
    rng = np.random.default_rng(n)
    dt = torch.as_tensor(rng.uniform(0.05, 0.5, n), dtype=torch.float64, device="cuda")
    y = torch.as_tensor(rng.standard_normal(n), dtype=torch.float64, device="cuda")
    r = torch.full((n,), 0.1, dtype=torch.float64, device="cuda")
    k = K.Matern52(variance=1.0, lengthscale=2.0)
    a, (am, aP) = ops.kalman_filter(dt, k, y, r, parallel=True)
    b, (bm, bP) = ops.kalman_filter(dt, k, y, r, parallel=False)
    assert abs(float(a) - float(b)) <= 1e-9 * abs(float(b))
    assert float((am - bm).abs().max()) <= 1e-9 * float(bm.abs().max())
    assert float((aP - bP).abs().max()) <= 1e-9 * float(bP.abs().max())


@pytest.mark.gpu
@pytest.mark.parametrize("n,runs", [(4095, 1), (4096, 1), (5000, 2)])
@pytest.mark.parametrize("two", [False, True])
def test_lengths_that_models_take(n, runs, two):
    """One rule for one series and for batches, under one component and under a sum."""
    from bayesnewton_amd import kernels as K, likelihoods as L, models as M
    k = K.Matern32(variance=1.0, lengthscale=1.0)
    if two:
        k = K.Sum([k, K.Matern52(variance=0.5, lengthscale=4.0)])
    x = np.arange(n) * 0.1
    lik = L.Gaussian(variance=0.01)
    m = (M.MarkovVariationalGP(k, lik, x, np.sin(x)) if runs == 1
         else M.MarkovVariationalGP.from_series(k, lik, [x] * runs, [np.sin(x)] * runs))
    assert m.plan.chunk_len == model_chunk_len([n] * runs)
