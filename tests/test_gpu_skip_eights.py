"""Empty space told by eights of steps (the brick of the fifth of them, while four steps are at
most 4.5 voxels long) and, for longer steps, sample by sample: every output of the fused walk
equals the full walk's (counts, statistics, slots, page flags), over step sizes on both sides
of that line, grids with unequal and odd sides, rays through corners of the box and past it."""
import dataclasses

import pytest
import torch

from voxurf_amd import scene
from voxurf_amd.fused import FusedFineTrainer

from .test_gpu_skip import _walk

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("stepsize,shape,n", [
    (0.5, (96, 96, 96), 700), (0.25, (64, 90, 130), 300), (1.1, (100, 70, 64), 300),
    (1.2, (96, 96, 96), 300), (3.0, (96, 80, 96), 300), (0.5, (97, 65, 33), 257)])
def test_eights_equal_full_walk(dev, stepsize, shape, n):
    R = max(shape)
    cfg = dataclasses.replace(scene.FINE, R=R, world_size=shape, n_rays=n, stepsize=stepsize)
    x, y, z = torch.meshgrid(*[torch.linspace(-1, 1, s, dtype=torch.float64) for s in shape],
                             indexing="ij")
    sdf = torch.sqrt(x * x + y * y + z * z) - 0.5 + 0.02 * torch.sin(9 * x) * torch.sin(7 * y + z)
    k0 = torch.randn((1, cfg.feat_dim, *shape), generator=torch.Generator().manual_seed(1)) * 0.1
    t = FusedFineTrainer(cfg, sdf.float()[None, None].contiguous(), k0,
                         scene.mlp_params(cfg.mlp_in, cfg.mlp_width, cfg.mlp_depth, seed=1), device=dev)
    o, d, v = scene.rays(n, seed=R)
    # a third towards the box's corners and edges, some of them past it
    g = torch.Generator().manual_seed(n)
    aim = torch.sign(torch.randn((n // 3, 3), generator=g)) * (0.9 + 0.2 * torch.rand((n // 3, 3), generator=g))
    d[:n // 3] = torch.nn.functional.normalize(aim - o[:n // 3], dim=-1)
    v[:n // 3] = d[:n // 3]
    o, d, v = (a.to(dev).contiguous() for a in (o, d, v))
    t.prime_touched([(o, d, v)])
    a, b = _walk(t, o, d, v, False), _walk(t, o, d, v, True)
    assert int(a["cnt"].sum()) > 0
    for k in a:
        assert torch.equal(a[k], b[k]), k
