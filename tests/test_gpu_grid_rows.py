"""The row forms of the grid operators (channels innermost, rows of z) against the general
strided ones: the same bits where no sum is reordered (lookup, total variation, the lattice
query), float64 to rounding where it is (the scatters); at the channel counts, strides, bases
and sizes around the rules that choose them."""
import pytest
import torch
import torch.nn.functional as F

from voxurf_amd import functional as vf, scene, serve
from voxurf_amd._lib import call, dtype_code, ptr, stream_of
from voxurf_amd.total_variation_cuda import grid_geom

pytestmark = pytest.mark.gpu


def _points(n, g, dtype):
    """Runs of neighbouring points, some outside the box, some on lattice planes."""
    o = torch.rand((n // 5 + 1, 1, 3), generator=g, dtype=torch.float64) * 2.4 - 1.2
    p = (o + torch.arange(5).reshape(1, 5, 1) * 0.011).reshape(-1, 3)[:n]
    p[::17] = p[::17].round()
    return p.to(dtype)


def _rows_grid(C, shape, pad, g, dtype):
    """[1, C, *shape] with channel stride 1 inside a wider channels-innermost array."""
    X, Y, Z = shape
    big = torch.randn((X, Y, Z, C + pad), generator=g, dtype=torch.float64).to(dtype)
    return big, pad // 2


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("C,pad", [(2, 0), (2, 1), (3, 0), (4, 0), (4, 2), (4, 4), (6, 0), (8, 8),
                                   (12, 0), (12, 2), (16, 0), (17, 0), (33, 0), (64, 0), (65, 0)])
@pytest.mark.parametrize("n", [1, 63, 257])
def test_lookup_and_scatter(dev, C, pad, n, dtype):
    g = torch.Generator().manual_seed(100 * C + n)
    big, off = _rows_grid(C, (9, 7, 11), pad, g, dtype)
    rows = big.to(dev)[..., off:off + C].permute(3, 0, 1, 2)[None]
    assert rows.stride(1) == 1
    plain = rows.contiguous()                       # the general order
    mn, mx = torch.tensor([-1.0, -1.1, -0.9]).to(dev, dtype), torch.tensor([1.0, 0.9, 1.2]).to(dev, dtype)
    pts = _points(n, g, dtype).to(dev)
    out = vf.grid_sample(rows, pts, mn, mx)
    assert torch.equal(out, vf.grid_sample(plain, pts, mn, mx))
    # the adjoint, with zero rows among the gradients
    go = torch.randn((n, C), generator=g, dtype=torch.float64)
    go[::7] = 0
    go = go.to(dev, dtype)
    gbig = torch.zeros_like(big).to(dev)
    grows = gbig[..., off:off + C].permute(3, 0, 1, 2)[None]
    geom = grid_geom(grows)  # host array: must outlive the call
    call("vx_grid_sample_bwd", dtype_code(rows), ptr(grows), geom.data_ptr(), ptr(pts), ptr(mn),
         ptr(mx), n, ptr(go), stream_of(rows))
    ref = plain.double().cpu().requires_grad_(True)
    q = ((pts.double().cpu() - mn.double().cpu()) / (mx - mn).double().cpu()).flip(-1) * 2 - 1
    F.grid_sample(ref, q.reshape(1, 1, 1, -1, 3), align_corners=True).reshape(C, -1).T.backward(
        go.double().cpu())
    # one rounding per term and addition, at most a few hundred of magnitude max |go|
    # (float32 coordinates: weights off by 2^-20 on this grid)
    tol = (1e-4 if dtype == torch.float32 else 1e-12) * float(go.abs().max() + 1)
    assert float((grows.double().cpu() - ref.grad).abs().max()) <= tol
    if pad:   # nothing outside the grid's own channels
        gbig[..., off:off + C] = 0
        assert not gbig.any()


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("n", [1, 2, 64, 65, 255, 256, 257, 321, 1000])
@pytest.mark.parametrize("which", ["both", "sdf", "grad"])
def test_sdf_scatter_runs(dev, n, which, dtype):
    """With and without (zero) neighbour-value gradients: the plain form and the runs' (from 256
    samples on)."""
    g = torch.Generator().manual_seed(n)
    shape = (1, 1, 13, 9, 11)
    mn, mx = torch.full((3,), -1.0).to(dev, dtype), torch.full((3,), 1.0).to(dev, dtype)
    pts = _points(n, g, dtype).clamp(-1, 1).to(dev).contiguous()
    gs = torch.randn(n, generator=g, dtype=torch.float64)
    gg = torch.randn((n, 3), generator=g, dtype=torch.float64)
    gs[::3] = 0
    gg[::3] = 0
    gs[::4] = 0
    gs, gg = gs.to(dev, dtype), gg.to(dev, dtype)
    feat = torch.zeros((n, 6), dtype=dtype, device=dev)
    res = []
    for f in (feat, None):
        out = torch.zeros(shape, dtype=dtype, device=dev)
        geom = grid_geom(out)  # host array: must outlive the call
        call("vx_sdf_grad_bwd", dtype_code(out), ptr(out), geom.data_ptr(), ptr(pts), ptr(mn),
             ptr(mx), 0.15, n, ptr(gs) if which != "grad" else None,
             ptr(gg) if which != "sdf" else None, ptr(f), stream_of(out))
        res.append(out.double())
    tol = (2e-5 if dtype == torch.float32 else 1e-13) * float(res[0].abs().max() + 1e-30)
    assert float((res[0] - res[1]).abs().max()) <= tol


def test_sdf_gradient_without_neighbour_values(dev):
    """The autograd function passes no gradient for outputs nobody used."""
    g = torch.Generator().manual_seed(0)
    grid = torch.randn((1, 1, 8, 9, 10), generator=g, dtype=torch.float64).to(dev).requires_grad_(True)
    pts = _points(50, g, torch.float64).clamp(-1, 1).to(dev)
    mn, mx = torch.full((3,), -1.0, device=dev), torch.full((3,), 1.0, device=dev)
    outs = []
    for k in range(3):
        grid.grad = None
        s, gr, f = vf.SdfGradSample.apply(grid, pts, mn, mx, 0.2)
        (s.sum() * 0 + [s.sum(), gr.pow(2).sum(), s.sum() + (f * f).sum()][k]).backward()
        outs.append(grid.grad.clone())
    grid.grad = None
    s, gr, f = vf.SdfGradSample.apply(grid, pts, mn, mx, 0.2)
    gr.pow(2).sum().backward()                      # s and f without a gradient
    assert torch.allclose(grid.grad, outs[1], rtol=1e-12, atol=1e-12)


@pytest.mark.parametrize("C", [1, 3, 12])
@pytest.mark.parametrize("inner", [False, True])
@pytest.mark.parametrize("shape", [(1, 1, 1), (2, 3, 5), (5, 1, 255), (3, 4, 256), (4, 5, 257)])
@pytest.mark.parametrize("masked,dense", [(False, 1), (False, 0), (True, 1), (True, 0)])
def test_total_variation_rows(dev, C, inner, shape, masked, dense):
    g = torch.Generator().manual_seed(C + sum(shape))
    X, Y, Z = shape
    full = (X, Y, Z, C) if inner else (C, X, Y, Z)
    val = [torch.randn(full, generator=g) for _ in range(3)]
    val[1][torch.rand(full, generator=g) < 0.5] = 0
    val[2] = (val[2] > 0).float()
    res = [_tv(dev, val, inner, masked, dense, (0.3, 0.5, 0.7), long) for long in (False, True)]
    assert torch.equal(*res)


def _tv(dev, val, inner, masked, dense, w, long):
    """The gradient val[1] (parameters val[0], mask val[2]) with the total variation's added;
    long: in rows one element longer, which only the strided kernel takes."""
    full = val[0].shape

    def view(t):
        if long:
            w = torch.zeros((*full[:-1], full[-1] + 1), dtype=t.dtype)
            w[..., :full[-1]] = t
            t = w.to(dev)[..., :full[-1]]
        else:
            t = t.to(dev)
        return (t.permute(3, 0, 1, 2) if inner else t)[None]

    p, gr, m = (view(v) for v in val)
    geom = grid_geom(p)
    args = (dtype_code(p), ptr(p), ptr(gr), *([ptr(m)] if masked else []), geom.data_ptr(), *w, dense,
            stream_of(p))
    call("vx_total_variation_add_grad_new" if masked else "vx_total_variation_add_grad", *args)
    return gr.contiguous()


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("C,inner", [(1, False), (3, False), (3, True), (4, True)])
@pytest.mark.parametrize("shape", [(6, 5, 8), (5, 4, 7)])
@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("dense", [0, 1])
def test_total_variation_that_cancels(dev, dtype, C, inner, shape, masked, dense):
    """Whole numbers (differences clamped to -1, 0 or 1, weights of 6 / 6), the gradient of every
    other element minus its term: the sums are exact, and an element that had a gradient holds
    exactly zero afterwards; one without stays as it is where only those are taken."""
    g = torch.Generator().manual_seed(C + sum(shape))
    X, Y, Z = shape
    full = (X, Y, Z, C) if inner else (C, X, Y, Z)
    p = torch.randint(-3, 4, full, generator=g).to(dtype)
    mask = (torch.rand(full, generator=g) < 0.7).to(dtype)
    zero = torch.zeros(full, dtype=dtype)
    w = (6.0, 6.0, 6.0)
    term = _tv(dev, [p, zero, mask], inner, masked, 1, w, True).cpu()
    term = (term[0].permute(1, 2, 3, 0) if inner else term[0]).contiguous()
    own = torch.rand(full, generator=g) < 0.5
    assert int((own & (term != 0)).sum()) > 10
    val = [p, torch.where(own, -term, zero), mask]
    res = [_tv(dev, val, inner, masked, dense, w, long) for long in (False, True)]
    want = torch.where(own, zero, term if dense else zero)
    want = (want.permute(3, 0, 1, 2) if inner else want)[None].to(dev)
    for r in res:
        assert torch.equal(r, want)


@pytest.mark.parametrize("tile,origin,res", [(1, (0, 0, 0), 8), (5, (3, 0, 2), 40), (63, (1, 4, 0), 70),
                                             (64, (10, 20, 30), 100), (65, (-2, 0, 7), 66),
                                             (4, (0.5, 1.25, 2), 9)])
def test_sdf_query(dev, tile, origin, res):
    import dataclasses
    cfg = dataclasses.replace(scene.FINE, R=40, feat_dim=3)
    sc = serve.ResidentScene(cfg, scene.sdf_grid(40), scene.feature_grid(40, 3),
                             scene.mlp_params(cfg.mlp_in, 192, 4), device=dev)
    s, n = sc.sdf_query(res, origin, tile)
    ax = [-1.0 + 2.0 * (torch.arange(tile, device=dev, dtype=torch.float32) + o) / (res - 1)
          for o in origin]
    pts = torch.stack(torch.meshgrid(*ax, indexing="ij"), -1).reshape(-1, 3).contiguous()
    rs, rg, _ = vf.SdfGradSample.apply(sc.sdf, pts, sc.xyz_min, sc.xyz_max, cfg.voxel_size)
    assert torch.equal(s, rs)
    # (outside the box the clamped neighbours coincide: no direction, in either form)
    want = rg / (rg.norm(dim=-1, keepdim=True) + 1e-5)
    assert torch.allclose(n, want, rtol=1e-6, atol=1e-7, equal_nan=True)


def test_sdf_query_forms(dev):
    """A tile given as a float (as arange takes it), origins in tensors, an empty tile, and a
    default device other than the host's."""
    import dataclasses
    cfg = dataclasses.replace(scene.FINE, R=24, feat_dim=3)
    sc = serve.ResidentScene(cfg, scene.sdf_grid(24), scene.feature_grid(24, 3),
                             scene.mlp_params(cfg.mlp_in, 192, 4), device=dev)
    want = sc.sdf_query(30, (1, 2, 3), 5)
    forms = [((1, 2, 3), 5.0), (torch.tensor([1, 2, 3]), 5), (torch.tensor([1.0, 2.0, 3.0]).to(dev), 4.5)]
    for origin, tile in forms:
        assert all(torch.equal(a, b) for a, b in zip(sc.sdf_query(30, origin, tile), want))
    with torch.device(dev):
        assert all(torch.equal(a, b) for a, b in zip(sc.sdf_query(30, (1, 2, 3), 5), want))
    s, n = sc.sdf_query(30, (1, 2, 3), 0)
    assert s.shape == (0,) and n.shape == (0, 3)
