"""Marching cubes on bit rows (vx_mc_classify / vx_mc_write) against the per-point passes
(vx_mc_count, a scan, vx_mc_emit): the same vertices and triangles in the same order, exactly,
at row lengths around the 64-point words; and the row-wise lattice field against the drop-in
grid_sample at torch.linspace's points, bit for bit."""
import numpy as np
import pytest
import torch

from voxurf_amd import functional, mesh
from voxurf_amd._lib import VoxhipError, call, lib, ptr, stream_of

pytestmark = pytest.mark.gpu


def _per_point(u, iso, bounds):
    nx, ny, nz = u.shape
    n, dev, st = u.numel(), u.device, stream_of(u)
    count, edges = (torch.from_numpy(t).to(dev) for t in mesh.mc_tables_host())
    cnt = torch.empty((2, n), dtype=torch.int64, device=dev)
    call("vx_mc_count", ptr(u), nx, ny, nz, iso, ptr(count), ptr(edges), ptr(cnt[0]), ptr(cnt[1]), st)
    incl = cnt.cumsum(1)
    nv, nf = incl[:, -1].tolist()
    verts = torch.empty((max(nv, 1), 3), dtype=torch.float64, device=dev)
    faces = torch.empty((max(nf, 1), 3), dtype=torch.int64, device=dev)
    b = np.asarray(bounds, dtype=np.float64)
    call("vx_mc_emit", ptr(u), nx, ny, nz, iso, ptr(count), ptr(edges), ptr(incl[0]), ptr(incl[1]),
         b.ctypes.data, ptr(verts), ptr(faces), st)
    return verts[:nv], faces[:nf]


@pytest.mark.parametrize("shape", [(1, 1, 1), (2, 2, 2), (3, 1, 65), (1, 4, 64), (5, 3, 63),
                                   (4, 6, 64), (3, 5, 65), (7, 9, 127), (6, 5, 128), (4, 7, 130),
                                   (40, 33, 70)])
@pytest.mark.parametrize("kind", ["noise", "smooth", "nan"])
def test_groups_match_per_point(dev, shape, kind):
    g = torch.Generator().manual_seed(sum(shape))
    u = torch.rand(shape, generator=g) * 2 - 1
    if kind == "smooth":
        ax = [torch.linspace(-1, 1, n) for n in shape]
        u = (ax[0][:, None, None] ** 2 + ax[1][None, :, None] ** 2 + ax[2] ** 2) - 0.6 + 1e-3 * u
    if kind == "nan":
        u[torch.rand(shape, generator=g) < 0.05] = float("nan")
        u[torch.rand(shape, generator=g) < 0.05] = float("inf")
    u = u.to(dev).contiguous()
    bounds = [-1.0, -2.0, 0.5, 1.0, 2.5, 1.7]
    v, f = mesh.marching_cubes(u, 0.1, bounds[:3], bounds[3:])
    rv, rf = _per_point(u, 0.1, bounds)
    assert v.shape == rv.shape and f.shape == rf.shape
    assert torch.equal(f, rf)
    assert torch.equal(torch.nan_to_num(v, nan=77.0), torch.nan_to_num(rv, nan=77.0))


def test_a_dense_field_is_no_slower(dev):
    """Noise, every point of which is listed, on a lattice of few workgroups: writing its mesh takes
    at most twice the per-point passes' time (one workgroup a list took ten times it)."""
    u = (torch.rand((64, 64, 64), generator=torch.Generator().manual_seed(0)) * 2 - 1).to(dev)
    n, st = u.numel(), stream_of(u)
    count, edges = (torch.from_numpy(t).to(dev) for t in mesh.mc_tables_host())
    cnt = torch.empty((2, n), dtype=torch.int64, device=dev)
    call("vx_mc_count", ptr(u), 64, 64, 64, 0.0, ptr(count), ptr(edges), ptr(cnt[0]), ptr(cnt[1]), st)
    incl = cnt.cumsum(1)
    nv, nf = incl[:, -1].tolist()
    ws = torch.empty(lib().vx_mc_workspace_bytes(64, 64, 64) // 8, dtype=torch.int64, device=dev)
    tot = torch.empty(2, dtype=torch.int64, device=dev)
    call("vx_mc_classify", ptr(u), 64, 64, 64, 0.0, ptr(count), ptr(ws), ptr(tot), st)
    assert tot.tolist() == [nv, nf]
    verts = torch.empty((nv, 3), dtype=torch.float64, device=dev)
    faces = torch.empty((nf, 3), dtype=torch.int64, device=dev)
    forms = [lambda: call("vx_mc_write", ptr(u), 64, 64, 64, 0.0, ptr(count), ptr(edges), ptr(ws), nv,
                          nf, None, ptr(verts), ptr(faces), st),
             lambda: call("vx_mc_emit", ptr(u), 64, 64, 64, 0.0, ptr(count), ptr(edges), ptr(incl[0]),
                          ptr(incl[1]), None, ptr(verts), ptr(faces), st)]
    best = [1e9, 1e9]
    for _ in range(10):
        for k, form in enumerate(forms):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            for _ in range(5):
                form()
            b.record()
            torch.cuda.synchronize()
            best[k] = min(best[k], a.elapsed_time(b))
    assert best[0] <= 2 * best[1], best


def test_bad_sizes_are_refused(dev):
    for shape in [(0, 2, 2), (65536, 1, 1)]:
        with pytest.raises(VoxhipError):
            mesh.marching_cubes(torch.zeros(shape, device=dev))
    assert lib().vx_mc_workspace_bytes(2, 2, 0) == -1


@pytest.mark.parametrize("grid,res", [((9, 7, 5), (20, 17, 65)), ((33, 40, 29), (12, 9, 300)),
                                      ((1, 2, 3), (5, 8, 7)), ((16, 16, 16), (16, 1, 16))])
@pytest.mark.parametrize("order", [(0, 1, 2), (2, 0, 1)])
def test_field_matches_grid_sample(dev, grid, res, order):
    g = torch.Generator().manual_seed(3)
    sdf = torch.randn([grid[a] for a in order], generator=g)
    sdf = sdf.permute([order.index(a) for a in range(3)])[None, None].to(dev)
    assert sdf.shape[-3:] == grid
    mn, mx = [-1.0, -1.2, -0.7], [1.0, 0.9, 1.1]
    bmin, bmax = [-1.1, -1.2, -0.6], [0.95, 1.0, 1.1]   # partly outside the grid's box
    u = mesh.extract_fields(sdf, mn, mx, bmin, bmax, res)
    axes = [torch.linspace(a, b, n) for a, b, n in zip(bmin, bmax, res)]
    pts = torch.stack(torch.meshgrid(*axes, indexing="ij"), -1).reshape(-1, 3).to(dev)
    want = functional.grid_sample(sdf, pts, torch.tensor(mn, device=dev), torch.tensor(mx, device=dev))
    assert torch.equal(u.reshape(-1), (-1.0 * want).reshape(-1))
