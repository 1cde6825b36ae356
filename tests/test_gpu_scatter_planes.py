"""The conversion of float32 planes to float64 rows of the series."""
import numpy as np
import pytest
import torch

from bayesnewton_amd.plan import SeriesPlan


@pytest.mark.gpu
@pytest.mark.parametrize("lengths,chunk", [([1], 1), ([70, 1, 33], 8), ([0, 5, 0], 4), ([300, 129], 128)])
@pytest.mark.parametrize("w", [1, 3])
def test_planes_to_double_rows(lengths, chunk, w):
    off = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int64)
    plan = SeriesPlan(off, chunk_len=chunk)
    x = torch.randn(int(off[-1]), w, device="cuda")
    t = plan.gather(x, pad=7.0)
    out = plan.scatter_planes(t)
    assert out.dtype == torch.float64 and out.shape == (w, int(off[-1]))
    assert torch.equal(out, plan.scatter(t).double().t())
    assert torch.equal(out, x.double().t())


def test_planes_of_other_types_are_refused():
    plan = object.__new__(SeriesPlan)  # the check comes before any use of the plan
    for dtype in (torch.float64, torch.float16, torch.int32):
        with pytest.raises(TypeError):
            plan.scatter_planes(torch.zeros(1, 8, dtype=dtype))


@pytest.mark.gpu
@pytest.mark.parametrize("lengths,chunk", [([1], 1), ([7], 100), ([70, 1, 33], 8), ([0, 5, 0], 4), ([300, 129, 2, 64], 3),
                                           ([513], 4), ([4000], 4000)])
@pytest.mark.parametrize("w", [2, 5, 25, 36, 100, 101])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_rows_of_words_to_planes_and_back(lengths, chunk, w, dtype):
    off = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int64)
    plan = SeriesPlan(off, chunk_len=chunk)
    x = torch.randn(int(off[-1]), w, device="cuda", dtype=dtype)
    t = plan.gather(x, pad=7.0)
    assert torch.equal(t, torch.cat([plan.gather(x[:, f].contiguous(), pad=7.0) for f in range(w)]))
    back = plan.scatter(t)
    assert back.shape == x.shape and torch.equal(back, x)
