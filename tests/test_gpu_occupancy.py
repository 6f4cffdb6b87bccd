"""The ray pre-filter with the MaskCache's occupancy bits against the same walk without them
(every sample looked up): identical hits, for caches of every shape the walk accepts -- odd and
tiny grids, boxes off the scene's, nearest lookups, thresholds where no density or every
density passes, non-finite densities."""
import pytest
import torch

from voxurf_amd import rays as vr, scene
from voxurf_amd._lib import call, lib, ptr, stream_of
from voxurf_amd.maskcache import MaskCache

pytestmark = pytest.mark.gpu


def _every_sample(mc, o, d, near, stepdist):
    box, params, args = vr._prefilter_args(mc, [-1.0] * 3, [1.0] * 3, near, stepdist)
    hit = torch.empty(o.shape[0], dtype=torch.bool, device=o.device)
    call("vx_hit_coarse_geo", ptr(o), ptr(d), o.shape[0], box.data_ptr(), params.data_ptr(), *args,
         ptr(hit), None, stream_of(o))
    return hit


def _density(kind, shape, g):
    x = [torch.linspace(-1, 1, n) if n > 1 else torch.zeros(1) for n in shape]
    r = (x[0][:, None, None] ** 2 + x[1][None, :, None] ** 2 + x[2] ** 2).sqrt()
    noise = torch.randn(shape, generator=g)
    if kind == "shell":
        return torch.where((r - 0.5).abs() < 0.1, 5.0, -20.0) + 0.1 * noise
    if kind == "sparse":
        return torch.where(torch.rand(shape, generator=g) < 2e-3, 3.0, -8.0) + noise
    if kind == "edge":      # densities around the value whose alpha is the threshold
        return -2.3 + 1e-3 * noise - 3.0 * (r > 0.3)
    d = torch.where(torch.rand(shape, generator=g) < 0.01, 2.0, -9.0) + noise
    d[torch.rand(shape, generator=g) < 0.01] = float("nan")
    d[torch.rand(shape, generator=g) < 0.01] = float("-inf")
    d[torch.rand(shape, generator=g) < 1e-3] = float("inf")
    return d


@pytest.mark.parametrize("kind", ["shell", "sparse", "edge", "nonfinite"])
@pytest.mark.parametrize("shape,ks", [((100, 100, 100), 3), ((33, 17, 64), 1), ((1, 2, 5), 1),
                                      ((130, 260, 20), 1)])
@pytest.mark.parametrize("opts", [dict(), dict(nearest=True), dict(act_shift=0.0),
                                  dict(thres=0.5, ratio=0.3), dict(thres=0.0), dict(thres=1.0),
                                  dict(box=((-0.4, -0.3, -0.2), (0.5, 0.9, 0.6))),
                                  dict(box=((-3.0, -2.0, -1.5), (1.2, 4.0, 2.0)))])
def test_occupancy_gives_the_same_hits(dev, kind, shape, ks, opts, monkeypatch):
    monkeypatch.setattr(vr, "OCC_RAYS", 0)   # the walk with occupancy bits for any number of rays
    g = torch.Generator().manual_seed(sum(shape) + len(kind))
    box = opts.get("box", ((-1.0, -1.0, -1.0), (1.0, 1.0, 1.0)))
    mc = MaskCache(density=_density(kind, shape, g)[None, None], ks=ks, xyz_min=box[0],
                   xyz_max=box[1], act_shift=opts.get("act_shift", -4.6),
                   voxel_size_ratio=opts.get("ratio", 1.0),
                   mask_cache_thres=opts.get("thres", 1e-3), nearest=opts.get("nearest", False)).to(dev)
    o, d, _ = scene.rays(2000, seed=3, jitter=0.4)
    d[:40] = torch.eye(3).repeat(14, 1)[:40]           # axis-parallel directions
    d[40:60, 1] = 0.0
    o[60:200] = torch.rand((140, 3), generator=g) * 1.6 - 0.8   # origins inside the box
    o, d = o.to(dev).contiguous(), d.to(dev).contiguous()
    for near, stepdist in ((0.0, 1.0 / 64), (0.3, 1.0 / 301), (0.0, 0.31)):
        hit = vr.hit_coarse_geo(mc, [-1.0] * 3, [1.0] * 3, o, d, near, stepdist)
        assert torch.equal(hit, _every_sample(mc, o, d, near, stepdist))


@pytest.mark.parametrize("H,W,focal", [(1, 1, 30.0), (37, 61, 50.0), (64, 8, 900.0), (41, 130, 6.0)])
@pytest.mark.parametrize("kind", ["shell", "sparse", "nonfinite"])
@pytest.mark.parametrize("eye", [(0.0, -3.0, 0.5), (0.2, 0.1, 0.05), (30.0, 4.0, -2.0)])
def test_view_gives_the_same_hits(dev, H, W, focal, kind, eye):
    """Every pixel's flag of a view (narrow, wide, from inside the box, from afar) is that of
    its ray looked up at every sample; with the NDC warp too."""
    import numpy as np
    g = torch.Generator().manual_seed(H + W)
    mc = MaskCache(density=_density(kind, (100, 90, 101), g)[None, None], ks=1,
                   xyz_min=[-1.0, -1.1, -1.0], xyz_max=[1.0, 1.0, 1.2], act_shift=-4.6,
                   voxel_size_ratio=1.0).to(dev)
    e = torch.tensor(eye)
    fwd = -e / e.norm()
    right = torch.linalg.cross(fwd, torch.tensor([0.0, 0.0, 1.0]))
    right = right / right.norm()
    c2w = torch.stack([right, torch.linalg.cross(right, fwd), -fwd, e], 1)
    K = np.array([[focal, 0, W / 2], [0, focal, H / 2], [0, 0, 1]])
    box, params, args = vr._prefilter_args(mc, [-1.0] * 3, [1.0] * 3, 0.0, 1.0 / 200)
    occ = vr._occupancy(mc, args)
    for ndc in (False, True):
        cam = vr.camera_params(H, W, K, c2w, False, False, False, "center", ndc)
        flag = torch.empty(H * W, dtype=torch.int64, device=dev)
        call("vx_view_hit_coarse_geo_occ", cam.data_ptr(), box.data_ptr(), params.data_ptr(), *args,
             ptr(occ), ptr(flag), stream_of(flag))
        o, d, _ = vr.get_rays_of_a_view(H, W, K, c2w.to(dev), ndc, False, False, False)
        want = _every_sample(mc, o.reshape(-1, 3), d.reshape(-1, 3), 0.0, 1.0 / 200)
        assert torch.equal(flag != 0, want)


@pytest.mark.parametrize("dist", [30.0, 1e3, 4.9e3, 4e4, 3e5])
@pytest.mark.parametrize("stepdist", [1.0 / 200, 0.05, 0.31])
@pytest.mark.parametrize("kind", ["shell", "sparse", "grains"])
def test_view_from_very_far(dev, dist, stepdist, kind):
    """Every pixel's flag from cameras so far off that their rays' coordinates are rounded to a
    good part of a cell, or to several; tiles of a fifth of a brick and of five."""
    import numpy as np
    g = torch.Generator().manual_seed(17)
    shape = (200, 190, 201)
    if kind == "grains":     # lone lattice points: bricks that few rays meet
        dens = torch.where(torch.rand(shape, generator=g) < 2e-4, 5.0, -20.0)
    else:
        dens = _density(kind, shape, g)
    mc = MaskCache(density=dens[None, None], ks=1, xyz_min=[-1.0, -1.1, -1.0],
                   xyz_max=[1.0, 1.0, 1.2], act_shift=-4.6, voxel_size_ratio=1.0).to(dev)
    box, params, args = vr._prefilter_args(mc, [-1.0] * 3, [1.0] * 3, 0.0, stepdist)
    occ = vr._occupancy(mc, args)
    H = W = 240
    for way, zoom in (((0.0, -1.0, 0.1), 1000.0), ((0.5, 0.6, -0.7), 1000.0), ((-1.0, 0.0, 0.003), 300.0),
                      ((0.31, -0.9, 0.2), 40.0)):
        focal = zoom * dist
        K = np.array([[focal, 0, W / 2], [0, focal, H / 2], [0, 0, 1]])
        e = torch.tensor(way) / torch.tensor(way).norm() * dist
        fwd = -e / e.norm()
        right = torch.linalg.cross(fwd, torch.tensor([0.0, 0.0, 1.0]))
        right = right / right.norm()
        c2w = torch.stack([right, torch.linalg.cross(right, fwd), -fwd, e], 1)
        cam = vr.camera_params(H, W, K, c2w, False, False, False, "center", False)
        flag, want = (torch.empty(H * W, dtype=torch.int64, device=dev) for _ in range(2))
        call("vx_view_hit_coarse_geo_occ", cam.data_ptr(), box.data_ptr(), params.data_ptr(), *args,
             ptr(occ), ptr(flag), stream_of(flag))
        call("vx_view_hit_coarse_geo", cam.data_ptr(), box.data_ptr(), params.data_ptr(), *args,
             ptr(want), stream_of(flag))
        assert torch.equal(flag, want), int((flag != want).sum())


def test_occupancy_bytes(dev):
    # bricks grow until their bits fit the LDS copy: at most 2^17 of them
    geom = torch.tensor([1, 700, 700, 700, 1, 490000, 700, 1], dtype=torch.int64)
    assert 0 < lib().vx_maskcache_occupancy_bytes(geom.data_ptr()) <= 9 << 17
    assert lib().vx_maskcache_occupancy_bytes(None) == -1


def test_few_rays_take_no_occupancy(dev, monkeypatch):
    """Small calls look every sample up, a wavefront a ray, without a pass over the cache's grid;
    the flags on both sides of the line are the same."""
    made = []
    make = vr._occupancy
    monkeypatch.setattr(vr, "_occupancy", lambda *a: made.append(1) or make(*a))
    g = torch.Generator().manual_seed(5)
    mc = MaskCache(density=_density("shell", (64, 64, 64), g)[None, None], ks=3, xyz_min=[-1.0] * 3,
                   xyz_max=[1.0] * 3, act_shift=-4.6, voxel_size_ratio=1.0).to(dev)
    o, d, _ = scene.rays(40000, seed=3, jitter=0.4)
    o, d = o.to(dev).contiguous(), d.to(dev).contiguous()
    hit = vr.hit_coarse_geo(mc, [-1.0] * 3, [1.0] * 3, o, d, 0.0, 1.0 / 64)
    assert made == [1]
    for n in (0, 1, 1000, 8192):
        few = vr.hit_coarse_geo(mc, [-1.0] * 3, [1.0] * 3, o[:n], d[:n], 0.0, 1.0 / 64)
        assert torch.equal(few, hit[:n])
    assert made == [1]

    class Model:
        mask_cache, xyz_min, xyz_max, voxel_size = mc, [-1.0] * 3, [1.0] * 3, 1.0 / 32

    c2w = torch.tensor([[1.0, 0, 0, 0], [0, 0, -1, -3.0], [0, 1, 0, 0.1]])
    K = [[60.0, 0, 32], [0, 60.0, 24], [0, 0, 1]]
    img = torch.rand((48, 64, 3), generator=g).to(dev)

    def views(pixels):
        monkeypatch.setattr(vr, "OCC_PIXELS", pixels)
        return vr.get_training_rays_in_maskcache_sampling(
            [img, img[:, :9]], [c2w] * 2, [(48, 64), (48, 9)], [K] * 2, False, False, False, False,
            Model, dict(near=0.0, stepsize=0.5))

    few = views(vr.OCC_PIXELS)
    assert made == [1]
    # one of the two views past the line, then both: the bits are made once a call
    for pixels, calls in ((1000, 2), (100, 3)):
        some = views(pixels)
        assert len(made) == calls and some[4] == few[4]
        assert all(torch.equal(a, b) for a, b in zip(some[:4], few[:4]))
    assert 0 < few[4][0] < 48 * 64
