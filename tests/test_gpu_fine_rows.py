"""The survivor rows of the fine steps (vx_fused_fine_gather, vx_voxurf_gather) from made-up
walk-range slots, against a float64 restatement: which slots become rows and in which order,
and every column, over channel layouts, row counts around the tiles of 64 and 32 rows, rays
without and with more survivors than sixteen, and an output capacity below the row count.

Tolerances: a lattice index is good to a few ulp of 24 (1e-5), which the grids' slopes (up to
about 4 per cell for k0, 0.1 for the SDF) carry into the values; an argument below 2^5 to 4e-6."""
import pytest
import torch
import torch.nn.functional as F

from voxurf_amd._lib import call, ptr, stream_of
from voxurf_amd.total_variation_cuda import grid_geom

pytestmark = pytest.mark.gpu
R, CAP, THRES = 24, 90, 1e-4
MN, MX = [-1.0, -1.1, -0.9], [1.0, 1.2, 1.1]


def _slots(dev, n_rays, seed):
    """Slots of n_rays rays: survivors have T = 1 and an alpha past the
    threshold; T = 1e-9 in half of the others."""
    g = torch.Generator().manual_seed(seed)
    m1 = torch.randint(0, 30, (n_rays,), generator=g)
    m1[n_rays // 2] = CAP
    m1[0] = 0
    keep = torch.rand(n_rays, CAP, generator=g) < 0.6
    keep[n_rays // 2] = True
    keep &= torch.arange(CAP) < m1[:, None]
    mn, mx = torch.tensor(MN), torch.tensor(MX)
    p = mn + (mx - mn) * (torch.rand(n_rays, CAP, 3, generator=g) * 1.04 - 0.02)
    grad = torch.randn(n_rays, CAP, 3, generator=g)
    s4 = torch.cat([p, torch.where(keep, 1.0, 1e-9)[..., None]], -1)
    g4 = torch.cat([grad, torch.rand(n_rays, CAP, 1, generator=g) * 1e-3], -1)
    vd = F.normalize(torch.randn(n_rays, 3, generator=g), dim=-1)
    # NeuS alpha of the slots with T = 1: samples that look along the gradient do not survive
    ic = -F.relu(-(grad.double() * vd.double()[:, None]).sum(-1)) * 0.02 * 0.5
    sdf = g4[..., 3].double()
    c, nx = ((sdf - ic) * 64).sigmoid(), ((sdf + ic) * 64).sigmoid()
    keep &= (c - nx + 1e-5) / (c + 1e-5) > THRES
    cnt = keep.sum(1)
    stats = torch.stack([m1, m1, m1], 1).int()
    rid, slot = keep.nonzero(as_tuple=True)
    d = dict(s4=s4, g4=g4, vd=vd, cnt=cnt, off=cnt.cumsum(0), stats=stats.contiguous())
    return {k: v.to(dev) for k, v in d.items()}, p[keep].double(), g4[keep].double(), \
        vd[rid].double(), rid


def _trilinear(grid, idx):
    """grid [C, X, Y, Z] at continuous indices [m, 3] (zero outside), float64."""
    size = torch.tensor(grid.shape[1:], dtype=torch.float64)
    n = (idx / (size - 1) * 2 - 1).flip(-1)
    out = F.grid_sample(grid[None].double(), n[None, None, None], align_corners=True)
    return out[0, :, 0, 0].T


def _pe(x, nf):
    a = (x[:, :, None] * 2.0 ** torch.arange(nf)).flatten(1)
    return torch.cat([x, a.sin(), a.cos()], 1)


def _grid(dev, C, inner, seed):
    g = torch.Generator().manual_seed(seed)
    k0 = torch.randn(C, R, R + 1, R + 2, generator=g)
    d = k0.to(dev)
    if inner:
        d = d.permute(1, 2, 3, 0).contiguous().permute(3, 0, 1, 2)
    return k0, d[None]


def _fixed():
    box = torch.tensor(MN + MX)
    params = torch.tensor([0.02, 0.05, 64.0, THRES, 0.1, 4.0])
    return box, params


@pytest.mark.parametrize("C,inner,nf,n_rays,room", [
    (12, True, 4, 40, 0), (12, False, 4, 7, 0), (6, True, 4, 300, 0), (5, True, 2, 33, 0),
    (1, False, 0, 12, 0), (16, True, 4, 200, 1000), (12, True, 4, 64, 64), (12, True, 3, 50, 65)])
def test_rgbnet_rows(dev, C, inner, nf, n_rays, room):
    d, p, g4, vd, rid = _slots(dev, n_rays, seed=C + n_rays)
    k0, k0d = _grid(dev, C, inner, seed=3)
    sdf = torch.zeros((1, 1, R, R + 1, R + 2), device=dev)
    total = len(rid)
    rows = min(room or total, total)
    xs = 64
    X = torch.full((total + 3, xs), 7.0, device=dev)
    P4, G4 = (torch.full((total + 3, 4), 7.0, device=dev) for _ in range(2))
    ids = torch.full((total + 3,), 7, dtype=torch.int32, device=dev)
    box, params = _fixed()
    kg, sg = grid_geom(k0d), grid_geom(sdf)
    call("vx_fused_fine_gather", ptr(k0d), kg.data_ptr(), sg.data_ptr(), box.data_ptr(),
         params.data_ptr(), ptr(d["vd"]), n_rays, CAP, nf, ptr(d["s4"]), ptr(d["g4"]),
         ptr(d["stats"]), ptr(d["cnt"]), ptr(d["off"]), xs, rows, ptr(X), ptr(P4), ptr(G4),
         ptr(ids), None, stream_of(X))
    assert bool((X[rows:] == 7).all()) and bool((P4[rows:] == 7).all()) and bool((ids[rows:] == 7).all())
    X, P4, G4, ids = X[:rows].cpu(), P4[:rows].cpu(), G4[:rows].cpu(), ids[:rows].cpu()
    assert torch.equal(ids, rid[:rows].int())
    assert torch.equal(P4[:, :3], p[:rows].float()) and torch.equal(G4, g4[:rows].float())
    mn, mx = torch.tensor(MN).double(), torch.tensor(MX).double()
    size = torch.tensor(k0.shape[1:]).double()
    idx = (p - mn) / (mx - mn) * (size - 1)
    n = g4[:, :3] / (g4[:, :3].norm(dim=1, keepdim=True) + 1e-5)
    want = torch.cat([_trilinear(k0, idx), n, _pe(vd, nf)], 1)[:rows]
    w = want.shape[1]
    assert float((X[:, :C] - want[:, :C]).abs().max()) < 2e-4
    assert float((X[:, C:w] - want[:, C:]).abs().max()) < 2e-5
    assert bool((X[:, w:] == 0).all())


@pytest.mark.parametrize("C,inner,cfg,disp,n_rays,room", [
    (12, True, (5, 4, 1), (0.5, 1.0, 1.5, 2.0), 40, 0), (6, False, (5, 1, 2), (0.5, 1.0), 9, 0),
    (5, True, (0, 0, 2), (1.0,), 33, 32), (6, True, (2, 3, 1), (0.5, 1.0, 2.5), 150, 900)])
def test_voxurf_rows(dev, C, inner, cfg, disp, n_rays, room):
    d, p, g4, vd, rid = _slots(dev, n_rays, seed=C + n_rays)
    p = torch.minimum(torch.maximum(p, torch.tensor(MN).double()), torch.tensor(MX).double())
    d["s4"][..., :3] = torch.minimum(torch.maximum(d["s4"][..., :3], torch.tensor(MN, device=dev)),
                                     torch.tensor(MX, device=dev))
    k0, k0d = _grid(dev, C, inner, seed=4)
    ax = [torch.arange(s, dtype=torch.float32) for s in (R, R + 1, R + 2)]
    x, y, z = torch.meshgrid(*ax, indexing="ij")
    sdf = 0.08 * ((x - 3.3) ** 2 + (y + 2.1) ** 2 + (z - 30.7) ** 2).sqrt()
    sd = sdf.to(dev)[None, None].contiguous()
    nd, (pp, vp, kp) = len(disp), cfg
    total = len(rid)
    rows = min(room or total, total)
    xs, ks = 104, 64
    X, XK = (torch.full((total + 3, s), 7.0, device=dev) for s in (xs, ks))
    P4, G4 = (torch.full((total + 3, 4), 7.0, device=dev) for _ in range(2))
    ids = torch.full((total + 3,), 7, dtype=torch.int32, device=dev)
    box, params = _fixed()
    row_cfg = torch.tensor([pp, vp, kp, nd, xs, ks], dtype=torch.int32)
    dd = torch.tensor(disp)
    kg, sg = grid_geom(k0d), grid_geom(sd)
    call("vx_voxurf_gather", ptr(sd), sg.data_ptr(), ptr(k0d), kg.data_ptr(), box.data_ptr(),
         params.data_ptr(), row_cfg.data_ptr(), dd.data_ptr(), ptr(d["vd"]), n_rays, CAP,
         ptr(d["s4"]), ptr(d["g4"]), ptr(d["stats"]), ptr(d["cnt"]), ptr(d["off"]), rows, ptr(X),
         ptr(XK), ptr(P4), ptr(G4), ptr(ids), stream_of(X))
    assert bool((X[rows:] == 7).all()) and bool((XK[rows:] == 7).all())
    X, XK, ids = X[:rows].cpu(), XK[:rows].cpu(), ids[:rows].cpu()
    assert torch.equal(ids, rid[:rows].int())
    mn, mx = torch.tensor(MN).double(), torch.tensor(MX).double()
    size = torch.tensor(sdf.shape).double()
    u = (p - mn) / (mx - mn)
    idx = u * (size - 1)
    feat, grads = [], []
    for a in (2, 1, 0):  # zyx
        for e in disp:
            lo, hi = idx.clone(), idx.clone()
            lo[:, a] = (lo[:, a] - e).clamp(0, float(size[a] - 1))
            hi[:, a] = (hi[:, a] + e).clamp(0, float(size[a] - 1))
            fm, fp = (_trilinear(sdf[None], i)[:, 0] for i in (lo, hi))
            feat.append((fm, fp))
            grads.append((fp - fm) / (hi - lo)[:, a] / 0.05)
    cols = [feat[a * nd + j][s] for a in range(3) for s in range(2) for j in range(nd)]
    g = torch.stack(grads, 1).reshape(-1, 3, nd)
    g = g / (g.norm(dim=1, keepdim=True) + 1e-5)
    want = torch.cat([_pe(u, pp), _pe(vd, vp), g4[:, 3:], torch.stack(cols, 1), g.flatten(1)], 1)[:rows]
    w = want.shape[1]
    assert float((X[:, :w] - want).abs().max()) < 1e-4
    assert bool((X[:, w:] == 0).all())
    want = torch.cat([_trilinear(k0, idx), _pe(u, pp), _pe(vd, kp), g4[:, :3]], 1)[:rows]
    w = want.shape[1]
    assert float((XK[:, :C] - want[:, :C]).abs().max()) < 2e-4
    assert float((XK[:, C:w] - want[:, C:]).abs().max()) < 2e-5
    assert bool((XK[:, w:] == 0).all())
