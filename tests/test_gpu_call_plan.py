"""Plans that live for one call: their tables are written by a kernel, in the stream's order.
They must be the tables that a kept plan holds, so both give the same bits."""
import ctypes

import numpy as np
import pytest
import torch

from bayesnewton_amd import _native as nat
from bayesnewton_amd.plan import SeriesPlan


@pytest.mark.parametrize("n,chunk", [(0, 8), (-1, 8), (10, 0), (10, (1 << 24) + 1), (128 * 128 * 4 + 1, 4)])
def test_refusals(n, chunk):
    assert nat.lib().bn_plan_single_bytes(n, chunk) == -1
    h = ctypes.c_void_p()
    assert nat.lib().bn_plan_create_single(n, chunk, 256, 1 << 40, None, ctypes.byref(h)) != 0
    assert h.value is None


@pytest.mark.gpu
@pytest.mark.parametrize("n,chunk", [(1, 1), (1, 8), (2, 1), (63, 1), (64, 1), (65, 1), (129, 1), (500, 4), (512, 4),
                                     (513, 4), (770, 3), (4097, 8), (128 * 128 * 4, 4), (300, 300), (300, 1000)])
def test_tables_equal_the_kept_plan(n, chunk):
    from bayesnewton_amd import kernels as K, ops
    dev = torch.device("cuda", torch.cuda.current_device())
    kept = SeriesPlan(np.array([0, n], dtype=np.int64), chunk_len=chunk)
    made = SeriesPlan.for_call(n, chunk, dev)
    for name in ("n_slots", "n_chunks", "n_tiles", "n_steps", "n_series", "chunk_len"):
        assert getattr(kept, name) == getattr(made, name), name
    rng = np.random.default_rng(n + chunk)
    dt, y, r = (torch.as_tensor(a, device=dev) for a in (rng.uniform(0.05, 0.5, n), rng.standard_normal(n),
                                                         rng.uniform(0.05, 0.2, n)))
    k = K.Matern32(variance=1.0, lengthscale=2.0)
    out = []
    for plan in (kept, made):
        e, (m, P) = ops.kalman_filter(dt, k, y, r, plan=plan)
        out.append((e, m, P) + tuple(ops.rauch_tung_striebel_smoother(dt, k, m, P, return_full=True, plan=plan)))
    for a, b in zip(*out):
        assert torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("n,chunk", [(1, 1), (16, 1), (17, 1), (1000, 3), (4097, 2)])
def test_gradient_composes_in_the_kept_plans_order(n, chunk):
    """16 elements a level, whoever made the plan: the same bits."""
    from bayesnewton_amd import kernels as K
    dev = torch.device("cuda", torch.cuda.current_device())
    rng = np.random.default_rng(n)
    rows = [torch.as_tensor(a.astype(np.float32), device=dev)
            for a in (rng.uniform(0.05, 0.5, n), rng.standard_normal(n), rng.uniform(0.05, 0.2, n))]
    k, out = K.Matern32(variance=1.0, lengthscale=2.0), []
    desc, (ls, var), L = k.desc(), k.hypers(dev), nat.lib()
    for plan in (SeriesPlan(np.array([0, n], dtype=np.int64), chunk_len=chunk), SeriesPlan.for_call(n, chunk, dev)):
        dt, y, r = (plan.gather(a, pad=1.0) for a in rows)
        res = torch.zeros(3, dtype=torch.float64, device=dev)
        gws = torch.empty(int(L.bn_grad_workspace_bytes(plan.handle, ctypes.byref(desc))), dtype=torch.uint8, device=dev)
        nat.check(L.bn_filter_loglik_grad(plan.handle, ctypes.byref(desc), nat.ptr(ls), nat.ptr(var), 0, nat.ptr(dt),
                                          nat.ptr(y), nat.ptr(r), None, nat.ptr(res), nat.ptr(res[1:]),
                                          nat.ptr(plan.workspace(desc)), nat.ptr(gws), nat.stream_ptr()))
        out.append(res.cpu())
    assert torch.equal(*out) and bool(torch.isfinite(out[0]).all())


@pytest.mark.gpu
def test_calls_on_other_streams():
    from bayesnewton_amd import kernels as K, ops
    rng = np.random.default_rng(3)
    k = K.Sum([K.Matern32(variance=1.0, lengthscale=2.0), K.Matern52(variance=0.5, lengthscale=0.4)])
    sets = [[torch.as_tensor(a, device="cuda") for a in (rng.uniform(0.05, 0.5, n), rng.standard_normal(n),
                                                         rng.uniform(0.05, 0.2, n))] for n in (700, 20_000, 5000)]
    want = [ops.kalman_filter(*(s[0], k) + tuple(s[1:]), parallel=True) for s in sets]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in sets]
    got = []
    for _ in range(5):
        for s, st in zip(sets, streams):
            with torch.cuda.stream(st):
                got.append(ops.kalman_filter(s[0], k, s[1], s[2], parallel=True))
    torch.cuda.synchronize()
    for i, (e, (m, P)) in enumerate(got):
        we, (wm, wP) = want[i % 3]
        assert torch.equal(e, we) and torch.equal(m, wm) and torch.equal(P, wP)
