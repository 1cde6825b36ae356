"""The plan that a model's gradient runs on: the model's own chunks, or chunks of the default
length where the model has so many short ones that they fill the chip several times over."""
import numpy as np
import pytest


def _model(lengths, two, seed=3, **kw):
    from bayesnewton_amd import kernels as K, likelihoods as L, models as M
    k = K.Matern32(variance=1.0, lengthscale=1.0)
    if two:
        k = K.Sum([K.Matern52(variance=0.5, lengthscale=5.0), K.Matern32(variance=0.5, lengthscale=2.0)])
    rng = np.random.default_rng(seed)
    xs = [np.cumsum(rng.exponential(0.05, n)) for n in lengths]
    ys = [np.sin(x) + 0.1 * rng.standard_normal(len(x)) for x in xs]
    for y in ys:
        y[::7] = np.nan
    return M.MarkovVariationalGP.from_series(k, L.Gaussian(variance=0.01), xs, ys, **kw)


@pytest.mark.gpu
@pytest.mark.parametrize("lengths,two,moves", [([130] * 1030, True, True), ([130] * 1029, True, False),
                                               ([130] * 3000, False, False), ([30] * 6000, True, False),
                                               ([3000, 1, 140] * 60, True, True)])
def test_gradient_on_the_default_length_equals_the_one_on_own_chunks(lengths, two, moves):
    """20 lanes a chunk at D = 5: 17 chunks of 8 steps in 130, 350,200 lanes in 1030 such series.
    FP64 on both plans and the same FP32 pseudo observations: 1e-10 of the gradient's norm."""
    m = _model(lengths, two)
    m.inference(lr=1.0)
    E, g, gl = m.energy_and_grad_per_series()
    assert (m._grad_plan is not m.plan) == moves
    assert m._grad_plan.chunk_len == (32 if moves else m.plan.chunk_len)
    fixed = _model(lengths, two, chunk_len=m.plan.chunk_len)  # an explicit length is kept
    fixed.inference(lr=1.0)
    E1, g1, gl1 = fixed.energy_and_grad_per_series()
    assert fixed._grad_plan is fixed.plan
    assert float((g - g1).norm()) <= 1e-10 * float(g1.norm())
    assert float((E - E1).norm()) <= 1e-10 * float(E1.norm())
    assert float((gl - gl1).norm()) <= 1e-10 * float(gl1.norm())
    m.inference(lr=0.5)  # new pseudo observations reach the other plan
    fixed.inference(lr=0.5)
    g, g1 = m.energy_and_grad_per_series()[1], fixed.energy_and_grad_per_series()[1]
    assert float((g - g1).norm()) <= 1e-10 * float(g1.norm())
