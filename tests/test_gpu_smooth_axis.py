"""Separable smoothing (vx_smooth3d) by vectors of a plane, against a float64 restatement: every
number of taps, rows of whole vectors and not, sides shorter than the taps, several channels,
unaligned buffers.  Three sums of up to nine products each: 3 x 10 roundings of 2^-24 of the
largest magnitude (taps sum to one)."""
import numpy as np
import pytest
import torch

from voxurf_amd._lib import call, dtype_code, ptr, stream_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [1, 3, 5, 7, 9])
@pytest.mark.parametrize("shape", [(1, 40, 36, 64), (3, 17, 5, 33), (1, 1, 2, 4), (2, 64, 64, 128),
                                   (1, 3, 3, 8)])
@pytest.mark.parametrize("off", [0, 1])
def test_smooth3d(dev, k, shape, off):
    n = int(np.prod(shape))
    g = torch.Generator(device=dev).manual_seed(k)
    x = torch.randn(n + 1, generator=g, device=dev)[off:off + n]
    o, t = torch.empty(n + 1, device=dev)[off:off + n], torch.empty(n, device=dev)
    taps = np.random.RandomState(k).rand(k)
    taps /= taps.sum()
    call("vx_smooth3d", dtype_code(x), ptr(x), ptr(o), ptr(t), *shape, taps.ctypes.data, k, 0, stream_of(x))
    q, w, r = x.double().reshape(shape).cpu(), torch.tensor(taps), k // 2
    for axis in (3, 2, 1):
        idx = torch.arange(shape[axis])
        q = sum(w[i] * q.index_select(axis, (idx + i - r).clamp(0, shape[axis] - 1)) for i in range(k))
    assert float((o.double().cpu().reshape(shape) - q).abs().max()) <= 30 * 2.0 ** -24 * float(x.abs().max())
