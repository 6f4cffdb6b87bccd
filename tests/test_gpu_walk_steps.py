"""The transmittance walk of alpha2weight (eight steps at a time, a rest of up to three by
itself) against the sequential
recurrence T = float(double(T) (1 - double(alpha))), to the bit: segments around eight and 64
samples, walks that end at every step of an eight, a NaN."""
import pytest
import torch

from voxurf_amd import render_utils_cuda as ru

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("back", [3, 1, 2])
def test_walk_ends_at_every_step(dev, dtype, back):
    """Ray r of length r: alphas that bring T below 1e-3 at step r - back or never, and a NaN."""
    g = torch.Generator().manual_seed(3)
    alpha, ids = [], []
    for r in range(150):
        a = torch.rand(r, generator=g, dtype=torch.float64) * 0.02
        if r > 3 and r % 2:
            a[r - back] = 0.9999
        if r == 77:
            a[20] = float("nan")
        alpha.append(a)
        ids += [r] * r
    alpha = torch.cat(alpha).to(dtype)
    ids = torch.tensor(ids)
    w, T, last, i0, i1 = ru.alpha2weight(alpha.to(dev), ids.to(dev), 151)
    f32 = lambda v: float(torch.tensor(v, dtype=torch.float64).float())
    pos = 0
    for r in range(150):
        t, end = 1.0, pos + r
        for i in range(pos, pos + r):
            assert torch.equal(T[i].cpu(), torch.tensor(t, dtype=dtype)) or t != t
            if t == t:
                assert torch.equal(w[i].cpu(), torch.tensor(t, dtype=dtype) * alpha[i]) or r == 77
            t = f32(t * (1.0 - float(alpha[i])))
            if t < 1e-3:
                end = i + 1
                break
        if r:
            assert int(i1[r]) == end and (float(last[r]) == t or t != t)
        assert bool((w[end:pos + r] == 0).all())
        pos += r
    assert float(last[150]) == 1.0
