"""The work this framework is used for, as cases that can be timed and checked.

Each case is one call (or one step) through the package's public entry points on a
synthetic scene: a perturbed sphere of radius 0.5 in the box [-1, 1]^3 whose ripple
phases come from the seed, feature grids N(0, 0.1^2), rays as a training batch (random
rays from the radius-3 sphere) or as the pixels of a pinhole view.  `exact` restates a
case in float64 with plain torch operations.

Kinds
  fine_step     one fused fine training step (forward, backward, Adam), mid-training
  coarse_grads  the coarse stage through the drop-in modules: forward, loss, backward, TV
  render        a resident scene rendered for a batch of rays (serving, evaluation)
  rgbnet        the colour MLP alone, forward and backward (or forward only)
  lookup        DenseGrid: trilinear feature lookup at surface samples and its adjoint
  ray_ops       the drop-in ray operators: sampling, alpha -> weight, compositing
  prefilter     the training rays of one view that hit the coarse geometry
  mesh          surface extraction: smoothing, lattice query, marching cubes
  regularise    the fine stage's grid regularisers added to the SDF gradient
  sdf_query     an SDF / normal query of one lattice tile (serving)
"""
import dataclasses
import math

import numpy as np
import torch
import torch.nn.functional as F

from voxurf_amd import (functional, grid, mesh, mlp, model, rays, render_utils_cuda, scene, serve,
                        smooth)
from voxurf_amd.fused import FusedFineTrainer
from voxurf_amd.fused_voxurf import FusedVoxurfTrainer
from voxurf_amd.maskcache import MaskCache

DEV = "cuda:0"
BOX = (-1.0, 1.0)


# ---- the cases ----------------------------------------------------------------------------

def listed():
    return [
        # the headline training step: 256^3 grids, 8192 rays
        dict(name="fine step 8192 rays", kind="fine_step", model="plain", R=256, rays=8192),
        # the coarse stage's step up to its gradients, at its own grid and batch size
        dict(name="coarse step 8192 rays", kind="coarse_grads", R=96, rays=8192),
        # an interactive preview tile: latency, launches
        dict(name="render 1000 rays", kind="render", model="plain", R=256, rays=1000,
             extras=False),
        # one evaluation chunk of the reference fine model with normals and depth
        dict(name="render fine model 8192 rays", kind="render", model="voxurf", R=256, rays=8192,
             extras=True),
        # a full batch of the render server
        dict(name="render 131072 rays", kind="render", model="plain", R=256, rays=131072,
             extras=False),
        # the colour MLP on one training step's survivors
        dict(name="rgbnet train 100003 rows", kind="rgbnet", rows=100003, inputs=42,
             dtype="float32", train=True),
        # the feature grid's lookup and scatter on a step's survivors
        dict(name="lookup 12 channels", kind="lookup", R=256, channels=12, points=100001),
        # the drop-in ray operators on a small batch
        dict(name="ray operators 1024 rays", kind="ray_ops", R=96, rays=1024),
        # the ray pre-filter of one full-size training view
        dict(name="prefilter 1200 x 1600", kind="prefilter", R=256, H=1200, W=1600),
        # the mesh of a fitted scene at the usual evaluation lattice
        dict(name="mesh 512", kind="mesh", R=256, resolution=512),
        # the dense regularisers of a fine step
        dict(name="regularise 256", kind="regularise", R=256),
        # a lattice tile query of the server
        dict(name="sdf query 64", kind="sdf_query", R=256, tile=64),
    ]


def _between(rng, lo, hi):
    """A whole number in [lo, hi], spread over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["fine_step", "coarse_grads", "render", "rgbnet", "lookup", "ray_ops",
                       "prefilter", "mesh", "regularise", "sdf_query"])
    R = rng.choice([96, 127, 128, 160, 192, 200, 255, 256])
    if kind == "fine_step":
        m = rng.choice(["plain", "plain", "voxurf"])
        return dict(kind=kind, model=m, R=max(R, 128), rays=_between(rng, 1024, 8192))
    if kind == "coarse_grads":
        return dict(kind=kind, R=rng.randint(64, 100), rays=_between(rng, 512, 8192))
    if kind == "render":
        m = rng.choice(["plain", "voxurf"])
        return dict(kind=kind, model=m, R=R, extras=rng.random() < 0.5,
                    rays=_between(rng, 256, 131072 if m == "plain" else 40000))
    if kind == "rgbnet":
        return dict(kind=kind, rows=_between(rng, 1000, 400000), inputs=rng.choice([42, 54, 79]),
                    dtype=rng.choice(["float32", "float32", "float32", "bfloat16"]),
                    train=rng.random() < 0.7)
    if kind == "lookup":
        return dict(kind=kind, R=R, channels=rng.choice([1, 3, 6, 12]),
                    points=_between(rng, 1000, 400000))
    if kind == "ray_ops":
        return dict(kind=kind, R=rng.randint(64, 256), rays=_between(rng, 128, 16384))
    if kind == "prefilter":
        H = _between(rng, 200, 1200)
        return dict(kind=kind, R=R, H=H, W=H * 4 // 3)
    if kind == "mesh":
        return dict(kind=kind, R=R, resolution=_between(rng, 64, 500))
    if kind == "regularise":
        return dict(kind=kind, R=rng.randint(64, 256))
    return dict(kind=kind, R=R, tile=rng.choice([32, 48, 63, 64]))


def work(case):
    return _WORK[case["kind"]](case)


def prepare(case, seed):
    with torch.no_grad():
        return dict(case=case, **_PREPARE[case["kind"]](case, seed))


def run(state):
    return _RUN[state["case"]["kind"]](state)


def exact(case, seed):
    f = _EXACT.get(case["kind"])
    return f(case, prepare(case, seed)) if f else None


# ---- scenes, rays -------------------------------------------------------------------------

def _gen(seed, tag):
    g = torch.Generator(device=DEV)
    g.manual_seed((seed * 1000003 + tag) & 0x7FFFFFFF)
    return g


def _sdf(R, seed):
    """[1, 1, R, R, R]: a sphere of radius 0.5 with ripples of the seed's phases."""
    ph = torch.rand(3, generator=_gen(seed, 1), device=DEV, dtype=torch.float64) * 2 * math.pi
    x = torch.linspace(*BOX, R, device=DEV, dtype=torch.float64)
    r = torch.sqrt(x[:, None, None] ** 2 + x[None, :, None] ** 2 + x[None, None, :] ** 2)
    s = [torch.sin(8 * x + p) for p in ph]
    s = r - 0.5 + 0.02 * s[0][:, None, None] * s[1][None, :, None] * s[2][None, None, :]
    return s.float()[None, None].contiguous()


def _features(R, C, seed):
    """[1, C, R, R, R] in the package's layout (channels innermost for C > 1)."""
    f = torch.randn((1, R, R, R, C), generator=_gen(seed, 2), device=DEV) * 0.1
    return f.permute(0, 4, 1, 2, 3)


def _mlp_params(width_in, depth, seed, tag):
    """[(W, b)] with nn.Linear's default scale."""
    g, dims, out = _gen(seed, tag), [width_in] + [192] * (depth - 1) + [3], []
    for a, b in zip(dims[:-1], dims[1:]):
        k = 1.0 / math.sqrt(a)
        out.append(((torch.rand((b, a), generator=g, device=DEV) * 2 - 1) * k,
                    (torch.rand(b, generator=g, device=DEV) * 2 - 1) * k))
    return out


def _training_rays(n, seed, tag=0):
    """n rays from the radius-3 sphere toward the origin with jitter."""
    g = _gen(seed, 100 + tag)
    u = torch.randn((n, 3), generator=g, device=DEV, dtype=torch.float64)
    u = u / u.norm(dim=-1, keepdim=True)
    d = -u + 0.05 * torch.randn((n, 3), generator=g, device=DEV, dtype=torch.float64)
    d = (d / d.norm(dim=-1, keepdim=True)).float().contiguous()
    return (3.0 * u).float().contiguous(), d, d


def _camera(H, W, seed):
    """(K, c2w) of a view from the radius-3 sphere in which the object fills most of the
    shorter side."""
    g = torch.Generator()
    g.manual_seed(seed * 7919 + 5)
    eye = torch.randn(3, generator=g, dtype=torch.float64)
    eye = 3.0 * eye / eye.norm()
    fwd = -eye / eye.norm()
    up = torch.tensor([0.0, 0.0, 1.0] if abs(float(fwd[2])) < 0.99 else [0.0, 1.0, 0.0],
                      dtype=torch.float64)
    right = torch.linalg.cross(fwd, up)
    right = right / right.norm()
    c2w = torch.stack([right, torch.linalg.cross(right, fwd), -fwd, eye], 1).float()
    f = 1.17 * 2 * min(H, W)
    return np.array([[f, 0, W / 2], [0, f, H / 2], [0, 0, 1]]), c2w


def _view_rays(n, seed):
    """n rays of a view, in pixel order."""
    W = max(1, int(round(math.sqrt(n * 4 / 3))))
    H = (n + W - 1) // W
    K, c2w = _camera(H, W, seed)
    o, d, v = rays.get_rays_of_a_view(H, W, K, c2w.to(DEV), False, False, False, False)
    return tuple(t.reshape(-1, 3)[:n].contiguous() for t in (o, d, v))


def _targets(o, d, seed, tag):
    """Colours a trained scene is near to: grey where the ray meets the object, with noise."""
    hit = (torch.linalg.cross(o, d).norm(dim=-1, keepdim=True) < 0.5).float()
    noise = torch.randn(o.shape, generator=_gen(seed, 200 + tag), device=DEV)
    return (hit * (0.5 + 0.05 * noise)).contiguous()


def _fine_cfg(case, **kw):
    base = scene.VOXURF if case["model"] == "voxurf" else scene.FINE
    return dataclasses.replace(base, R=case["R"], n_rays=case["rays"], inv_s=float(case["R"]), **kw)


# ---- fine_step ----------------------------------------------------------------------------

def _fine_prepare(case, seed):
    # learning rates as the schedule leaves them late in training (a tenth of the first),
    # and a few steps behind it, so that the moments and the touched pages are in use
    base = scene.VOXURF if case["model"] == "voxurf" else scene.FINE
    cfg = _fine_cfg(case, lr_sdf=base.lr_sdf * 0.1, lr_k0=base.lr_k0 * 0.1,
                    lr_mlp=base.lr_mlp * 0.1, lr_k_mlp=base.lr_k_mlp * 0.1)
    sdf, k0 = _sdf(case["R"], seed), _features(case["R"], cfg.feat_dim, seed)
    params = _mlp_params(cfg.mlp_in, cfg.mlp_depth, seed, 41)
    if case["model"] == "voxurf":
        t = FusedVoxurfTrainer(cfg, sdf, k0, params,
                               _mlp_params(cfg.k_mlp_in, cfg.k_mlp_depth, seed, 43), device=DEV)
        t.global_step = 10000
    else:
        t = FusedFineTrainer(cfg, sdf, k0, params, device=DEV)
    batches = []
    for i in range(4):
        o, d, v = _training_rays(case["rays"], seed, i)
        batches.append((o, d, v, _targets(o, d, seed, i)))
    for b in batches:
        t.step(*b)
    return dict(trainer=t, batches=batches, next=[0], weights=dict(t.state_dict()))


def _fine_run(s):
    i = s["next"][0]
    s["next"][0] = (i + 1) % len(s["batches"])
    out = s["trainer"].step(*s["batches"][i])
    return dict(loss=out["loss"], rgb=out["rgb_marched"], weights=s["weights"])


def _survivors(case):
    """About twelve samples a ray carry weight at 256^3."""
    return max(1, int(12 * case["rays"] * case["R"] / 256))


def _mlp_flops(rows, inputs):
    return 2.0 * rows * (inputs * 192 + 2 * 192 * 192 + 192 * 3)


def _shell(R):
    """Voxels within a few voxels of the surface."""
    return 4 * math.pi * (R / 4) ** 2 * 12


def _fine_work(case):
    m, R = _survivors(case), case["R"]
    C, f = (6, _mlp_flops(m, 79) + _mlp_flops(m, 54)) if case["model"] == "voxurf" else \
        (12, _mlp_flops(m, 42))
    return dict(bytes=case["rays"] * 60 + 24.0 * _shell(R) * (C + 1), flops=3 * f)


# ---- coarse_grads -------------------------------------------------------------------------

def _coarse_prepare(case, seed):
    cfg = dataclasses.replace(scene.COARSE, R=case["R"], n_rays=case["rays"])
    m = model.VoxurfCoarse(cfg, _sdf(case["R"], seed), _features(case["R"], 3, seed)).to(DEV)
    o, d, v = _training_rays(case["rays"], seed)
    return dict(model=m, cfg=cfg, rays=(o, d, v), target=_targets(o, d, seed, 0))


def _coarse_run(s):
    m = s["model"]
    m.sdf.grid.grad = m.k0.grid.grad = None
    out = m(*s["rays"])
    loss = F.mse_loss(out["rgb_marched"], s["target"])
    loss.backward()
    m.total_variation_add_grad(s["cfg"].tv_weight, True)
    return dict(loss=loss.detach(), rgb=out["rgb_marched"].detach(), sdf=m.sdf.grid.grad,
                k0=m.k0.grid.grad)


def _coarse_work(case):
    n, R = case["rays"] * 1.2 * case["R"], case["R"]
    return dict(bytes=case["rays"] * 60 + 8.0 * 4 * R ** 3, flops=n * 400)


def _coarse_exact(case, s):
    m, cfg = s["model"], s["cfg"]
    sdf = m.sdf.grid.detach().double().requires_grad_(True)
    k0 = m.k0.grid.detach().double().contiguous().requires_grad_(True)
    o, d, v = (t.double() for t in s["rays"])
    n = o.shape[0]
    pts, rid, _ = _sample64(o, d, cfg.stepdist)
    val, grad = _sdf_grad64(sdf, pts, cfg.voxel_size)
    alpha = _neus64(v[rid], val, grad, cfg.stepdist, cfg.inv_s)
    w, _ = _weights64(alpha, rid, n)
    keep = w.detach() > cfg.fast_color_thres
    pts, rid, alpha = pts[keep], rid[keep], alpha[keep]
    w, last = _weights64(alpha, rid, n)
    rgb = torch.sigmoid(_tri64(k0, pts))
    out = torch.zeros((n, 3), device=DEV, dtype=torch.float64).index_add(0, rid, w[:, None] * rgb)
    out = out.clamp(0, 1)
    loss = F.mse_loss(out, s["target"].double())
    loss.backward()
    for p in (sdf, k0):
        _tv_add64(p.detach(), p.grad, cfg.tv_weight)
    return dict(loss=loss.detach(), rgb=out.detach(), sdf=sdf.grad, k0=k0.grad)


# ---- render -------------------------------------------------------------------------------

def _render_prepare(case, seed):
    cfg = _fine_cfg(case)
    sdf, k0 = _sdf(case["R"], seed), _features(case["R"], cfg.feat_dim, seed)
    params = _mlp_params(cfg.mlp_in, cfg.mlp_depth, seed, 41)
    if case["model"] == "voxurf":
        kp = _mlp_params(cfg.k_mlp_in, cfg.k_mlp_depth, seed, 43)
        sc = serve.ResidentVoxurfScene(cfg, sdf, k0, params, kp, 1.0 / case["R"], device=DEV)
        nets = (params, kp)
    else:
        sc = serve.ResidentScene(cfg, sdf, k0, params, device=DEV)
        nets = (params,)
    ws = serve.Workspace(torch.device(DEV), sc.cap)
    ws.ensure(case["rays"])
    return dict(scene=sc, ws=ws, cfg=cfg, nets=nets, rays=_view_rays(case["rays"], seed))


def _render_run(s):
    x = s["case"]["extras"]
    return s["scene"].render_full(*s["rays"], s["ws"], render_grad=x, render_depth=x)


def _render_work(case):
    m = 0.6 * _survivors(case)
    C, f = (6, _mlp_flops(m, 79) + _mlp_flops(m, 54)) if case["model"] == "voxurf" else \
        (12, _mlp_flops(m, 42))
    grids = min(_shell(case["R"]), 8.0 * m) * (C + 1)
    return dict(bytes=case["rays"] * 52 + 4.0 * grids, flops=f)


@torch.no_grad()
def _render_exact(case, s):
    cfg, sc = s["cfg"], s["scene"]
    sdf, k0 = sc.sdf.double(), sc.k0.double().contiguous()
    nets = [[(W.double(), b.double()) for W, b in p] for p in s["nets"]]
    inv_s = float(sc.params[2])
    parts = []
    for a in range(0, case["rays"], 4096):
        o, d, v = (t[a:a + 4096].double() for t in s["rays"])
        n = o.shape[0]
        pts, rid, step = _sample64(o, d, cfg.stepdist)
        # far from the surface alpha is below the threshold whatever the gradient
        near = _tri64(sdf, pts)[:, 0] < 0.12 + 20.0 / inv_s
        pts, rid, step = pts[near], rid[near], step[near]
        val, grad = _sdf_grad64(sdf, pts, cfg.voxel_size)
        alpha = _neus64(v[rid], val, grad, cfg.stepdist, inv_s)
        k = alpha > cfg.fast_color_thres
        pts, rid, step, val, grad, alpha = (t[k] for t in (pts, rid, step, val, grad, alpha))
        w, last = _weights64(alpha, rid, n)
        k = w > cfg.fast_color_thres
        pts, rid, step, val, grad, w = (t[k] for t in (pts, rid, step, val, grad, w))

        def march(c):
            return torch.zeros((n, c.shape[1]), device=DEV, dtype=torch.float64).index_add(
                0, rid, w[:, None] * c)
        feat = _tri64(k0, pts)
        r = dict(alphainv_cum=last, normal_marched=None, depth=None)
        if case["model"] == "voxurf":
            xyz = (pts + 1) / 2
            fs, gs = zip(*[_displaced64(sdf, pts, cfg.voxel_size, q) for q in cfg.grad_feat])
            X = torch.cat([_pe64(xyz, cfg.pos_pe), _pe64(v, cfg.view_pe)[rid], val[:, None],
                           torch.stack(fs, -1).flatten(1), torch.stack(gs, -1).flatten(1)], -1)
            logit = _mlp64(X, nets[0])
            XK = torch.cat([feat, _pe64(xyz, cfg.pos_pe), _pe64(v, cfg.k_view_pe)[rid], grad,
                            logit], -1)
            r["rgb_marched"] = march(torch.sigmoid(logit + _mlp64(XK, nets[1]))).clamp(0, 1)
            r["rgb_marched0"] = march(torch.sigmoid(logit))
        else:
            nrm = grad / (grad.norm(dim=-1, keepdim=True) + 1e-5)
            X = torch.cat([feat, nrm, _pe64(v, cfg.view_pe)[rid]], -1)
            r["rgb_marched"] = march(torch.sigmoid(_mlp64(X, nets[0])))
        if case["extras"]:
            r["normal_marched"] = march(grad / (grad.norm(dim=-1, keepdim=True) + 1e-6))
            r["depth"] = march((step * cfg.stepdist)[:, None])[:, 0]
        parts.append(r)
    return {k: None if parts[0][k] is None else torch.cat([p[k] for p in parts])
            for k in parts[0]}


# ---- rgbnet -------------------------------------------------------------------------------

def _rgbnet_prepare(case, seed):
    params = _mlp_params(case["inputs"], 4, seed, 41)
    net = mlp.RgbNet(case["inputs"], 192, 4, params=params,
                     compute_dtype=getattr(torch, case["dtype"])).to(DEV)
    g = _gen(seed, 3)
    # features of the grid's scale beside unit-scale encodings, as the fine rows are
    x = torch.randn((case["rows"], case["inputs"]), generator=g, device=DEV)
    x[:, :12] *= 0.1
    # the output gradient of a mean squared error: small residuals of one sign
    go = (torch.rand((case["rows"], 3), generator=g, device=DEV) + 0.05) / (10 * case["rows"])
    return dict(net=net, params=params, x=x, go=go)


def _rgbnet_run(s):
    net = s["net"]
    if not s["case"]["train"]:
        with torch.no_grad():
            return dict(logits=net(s["x"]))
    x = s["x"].requires_grad_(True)
    x.grad = None
    for p in net.parameters():
        p.grad = None
    logits = net(x)
    logits.backward(s["go"])
    return dict(logits=logits.detach(), x=x.grad, params=[p.grad for p in net.parameters()])


def _rgbnet_work(case):
    r, k = case["rows"], case["inputs"]
    f, b = _mlp_flops(r, k), r * (k + 3) * 4.0
    return dict(bytes=2 * b, flops=3 * f) if case["train"] else dict(bytes=b, flops=f)


def _rgbnet_exact(case, s):
    ps = [t.double().requires_grad_(case["train"]) for wb in s["params"] for t in wb]
    x = s["x"].detach().double().requires_grad_(case["train"])
    logits = _mlp64(x, list(zip(ps[0::2], ps[1::2])))
    if not case["train"]:
        return dict(logits=logits)
    if case["dtype"] == "bfloat16":   # gradients of the rounded network are another function's
        return dict(logits=logits.detach(), x=None, params=[None] * len(ps))
    logits.backward(s["go"].double())
    return dict(logits=logits.detach(), x=x.grad, params=[p.grad for p in ps])


# ---- lookup -------------------------------------------------------------------------------

def _lookup_prepare(case, seed):
    R, C, P = case["R"], case["channels"], case["points"]
    g = grid.DenseGrid(C, [R] * 3, [-1.0] * 3, [1.0] * 3).to(DEV)
    g.grid.data.copy_(_features(R, C, seed))
    # survivors of training rays: twelve half-voxel steps each, around the surface
    n = (P + 11) // 12
    o, d, _ = _training_rays(n, seed)
    t = 2.5 + (torch.arange(12, device=DEV) - 6) / R
    pts = (o[:, None] + d[:, None] * t[None, :, None]).reshape(-1, 3)[:P].contiguous()
    shape = (P, C) if C > 1 else (P,)
    return dict(grid=g, pts=pts, go=torch.randn(shape, generator=_gen(seed, 4), device=DEV) * 1e-4)


def _lookup_run(s):
    s["grid"].grid.grad = None
    out = s["grid"](s["pts"])
    out.backward(s["go"])
    return dict(out=out.detach(), grid=s["grid"].grid.grad)


def _lookup_work(case):
    C, P, R = case["channels"], case["points"], case["R"]
    return dict(bytes=P * (24.0 + 8 * C) + 4.0 * C * R ** 3 + min(8.0 * P, _shell(R)) * 4 * C,
                flops=32.0 * P * C)


def _lookup_exact(case, s):
    g = s["grid"].grid.detach().double().contiguous().requires_grad_(True)
    out = _tri64(g, s["pts"].double()).reshape(s["go"].shape)
    out.backward(s["go"].double())
    return dict(out=out.detach(), grid=g.grad)


# ---- ray_ops ------------------------------------------------------------------------------

def _ray_ops_prepare(case, seed):
    # one set of rays in the seed's order and mirroring, which leave the number of samples
    # (the size of most outputs) as it is
    o, d, _ = _training_rays(case["rays"], 0)
    g = _gen(seed, 5)
    order = torch.randperm(case["rays"], generator=g, device=DEV)
    mirror = torch.randint(0, 2, (3,), generator=g, device=DEV) * 2.0 - 1.0
    o, d = (o[order] * mirror).contiguous(), (d[order] * mirror).contiguous()
    stepdist = 1.0 / case["R"]
    mn = torch.full((3,), BOX[0], device=DEV)
    mx = torch.full((3,), BOX[1], device=DEV)
    # in-box samples with an opacity that rises across the surface, in ray order
    pts, out, rid, _, _, _, _ = render_utils_cuda.sample_pts_on_rays(o, d, mn, mx, 0.0, 1e9,
                                                                     stepdist)
    pts, rid = pts[~out], rid[~out].contiguous()
    alpha = torch.sigmoid((0.5 - pts.norm(dim=-1)) * case["R"] / 2 - 2) * \
        (0.1 + 0.5 * torch.rand(rid.shape, generator=g, device=DEV))
    return dict(rays=(o, d, mn, mx), stepdist=stepdist, alpha=alpha.contiguous(), rid=rid,
                rgb=torch.rand((rid.shape[0], 3), generator=g, device=DEV),
                go=torch.randn((case["rays"], 3), generator=g, device=DEV) * 1e-3,
                gl=torch.randn(case["rays"], generator=g, device=DEV) * 1e-3)


def _ray_ops_run(s):
    n = s["case"]["rays"]
    pts, out, rid, step, n_steps, t_min, t_max = render_utils_cuda.sample_pts_on_rays(
        *s["rays"], 0.0, 1e9, s["stepdist"])
    alpha = s["alpha"].requires_grad_(True)
    rgb = s["rgb"].requires_grad_(True)
    alpha.grad = rgb.grad = None
    w, last = functional.Alphas2Weights.apply(alpha, s["rid"], n)
    marched = functional.segment_coo(w[:, None] * rgb, s["rid"], dim_size=n)
    torch.autograd.backward([marched, last], [s["go"], s["gl"]])
    return dict(pts=pts, out=out, rid=rid, step=step, n_steps=n_steps, t_min=t_min, t_max=t_max,
                weights=w.detach(), last=last.detach(), marched=marched.detach(), alpha=alpha.grad,
                rgb=rgb.grad)


def _ray_ops_work(case):
    n = case["rays"] * 1.5 * case["R"]
    return dict(bytes=case["rays"] * 100 + n * (29.0 + 12 + 40), flops=n * 60)


def _ray_ops_exact(case, s):
    n = case["rays"]
    alpha = s["alpha"].detach().double().requires_grad_(True)
    rgb = s["rgb"].detach().double().requires_grad_(True)
    w, last = _weights64(alpha, s["rid"], n)
    marched = torch.zeros((n, 3), device=DEV, dtype=torch.float64).index_add(
        0, s["rid"], w[:, None] * rgb)
    torch.autograd.backward([marched, last], [s["go"].double(), s["gl"].double()])
    o, d = (t.double() for t in s["rays"][:2])
    t0, t1 = _slab64(o, d)
    steps = _steps64(d, t0, t1, s["stepdist"])
    rid = torch.repeat_interleave(torch.arange(n, device=DEV), steps)
    step = torch.arange(rid.numel(), device=DEV) - (torch.cumsum(steps, 0) - steps)[rid]
    pts = _points64(o, d, t0, rid, step, s["stepdist"])
    return dict(pts=pts, out=None, rid=None, step=None, n_steps=None, t_min=t0, t_max=t1,
                weights=w.detach(), last=last.detach(), marched=marched.detach(), alpha=alpha.grad,
                rgb=rgb.grad)


# ---- prefilter ----------------------------------------------------------------------------

class _Occupied:
    """What the pre-filter asks of a model."""

    def __init__(self, cache, voxel_size):
        self.mask_cache, self.voxel_size = cache, voxel_size
        self.xyz_min, self.xyz_max = cache.xyz_min, cache.xyz_max


def _prefilter_prepare(case, seed):
    # coarse occupancy: a shell around the surface on a 100^3 density grid.  The view is the
    # same for every seed (it sets how many rays are kept), its picture is not.
    dens = torch.where(_sdf(100, 0).abs() < 0.1, 5.0, -20.0)
    mc = MaskCache(density=dens, xyz_min=[-1.0] * 3, xyz_max=[1.0] * 3, act_shift=-4.6,
                   voxel_size_ratio=1.0).to(DEV)
    K, c2w = _camera(case["H"], case["W"], 0)
    img = torch.rand((case["H"], case["W"], 3), generator=_gen(seed, 6), device=DEV)
    return dict(model=_Occupied(mc, 2.0 / case["R"]), K=K, c2w=c2w, img=img)


def _prefilter_run(s):
    c = s["case"]
    rgb, o, d, v, kept = rays.get_training_rays_in_maskcache_sampling(
        [s["img"]], [s["c2w"]], [(c["H"], c["W"])], [s["K"]], False, False, False, False,
        s["model"], dict(near=0.0, stepsize=0.5))
    return dict(rgb=rgb, rays_o=o, rays_d=d, viewdirs=v, kept=kept)


def _prefilter_work(case):
    n = case["H"] * case["W"]
    return dict(bytes=n * (12.0 + 0.4 * 48) + 4e6, flops=n * 0.5 * case["R"] * 20)


@torch.no_grad()
def _prefilter_exact(case, s):
    H, W, K = case["H"], case["W"], torch.tensor(s["K"], device=DEV).float().double()
    c2w, mc = s["c2w"].to(DEV).double(), s["model"].mask_cache
    dens, stepdist = mc.density.double(), 0.5 * s["model"].voxel_size
    p = torch.arange(H * W, device=DEV)
    i, j = (p % W).double() + 0.5, (p // W).double() + 0.5
    cam = torch.stack([(i - K[0, 2]) / K[0, 0], -(j - K[1, 2]) / K[1, 1], -torch.ones_like(i)], -1)
    d = cam @ c2w[:3, :3].T
    o = c2w[:3, 3].expand_as(d)
    keep = []
    for a in range(0, H * W, 32768):
        pts, rid, _ = _sample64(o[a:a + 32768], d[a:a + 32768], stepdist)
        x = _tri64(dens, pts)[:, 0] + mc.act_shift
        alpha = 1 - torch.exp(-F.softplus(x) * mc.voxel_size_ratio)
        hit = torch.zeros(min(32768, H * W - a), device=DEV, dtype=torch.bool)
        hit[rid[alpha >= mc.mask_cache_thres]] = True
        keep.append(hit)
    keep = torch.cat(keep)
    v = d / d.norm(dim=-1, keepdim=True)
    return dict(rgb=s["img"].reshape(-1, 3)[keep].double(), rays_o=o[keep], rays_d=d[keep],
                viewdirs=v[keep], kept=[None])


# ---- mesh ---------------------------------------------------------------------------------

def _mesh_prepare(case, seed):
    # one object (its shape sets how many vertices there are) at the seed's place and size
    # in the world
    c = torch.rand(3, generator=_gen(seed, 8), device=DEV).cpu()
    k = 1.0 + float(c[0])
    return dict(sdf=_sdf(case["R"], 0), world=(c - 0.9 * k, c + 0.9 * k),
                smooth=smooth.GaussianConv3d(3, 0.5))


def _mesh_run(s):
    u = mesh.extract_fields(s["smooth"](s["sdf"]), [-1.0] * 3, [1.0] * 3, [-0.9] * 3, [0.9] * 3,
                            s["case"]["resolution"])
    return mesh.marching_cubes(u, 0.0, *s["world"])


def _mesh_work(case):
    n = case["resolution"]
    return dict(bytes=4.0 * case["R"] ** 3 + 0.95 * n * n * (24 + 48), flops=n ** 3 * 20.0)


@torch.no_grad()
def _mesh_exact(case, s):
    n = case["resolution"]
    x = np.arange(-1, 2, dtype=np.float64)
    t = torch.tensor(np.exp(-(x ** 2) / (2 * 0.5 ** 2)), device=DEV)
    t = t / t.sum()
    g = F.pad(s["sdf"].double(), (1,) * 6, mode="replicate")
    for a in (2, 3, 4):
        k = g.shape[a] - 2
        g = sum(t[i] * g.narrow(a, i, k) for i in range(3))
    ax = torch.linspace(-0.9, 0.9, n, device=DEV, dtype=torch.float64)
    u = []
    for i in range(n):
        pts = torch.stack(torch.meshgrid(ax[i:i + 1], ax, ax, indexing="ij"), -1).reshape(-1, 3)
        u.append(-_tri64(g, pts)[:, 0].reshape(n, n))
    u = torch.stack(u)
    ids, verts = [], []
    for a in range(3):
        lo, hi = u.narrow(a, 0, n - 1), u.narrow(a, 1, n - 1)
        c = ((lo < 0) != (hi < 0)).nonzero()
        f1, f2 = lo[tuple(c.T)], hi[tuple(c.T)]
        v = c.double()
        v[:, a] += (0 - f1) / (f2 - f1)
        ids.append(((c[:, 0] * n + c[:, 1]) * n + c[:, 2]) * 3 + a)
        verts.append(v)
    order = torch.cat(ids).argsort()
    lo, hi = (b.to(DEV).double() for b in s["world"])
    return [torch.cat(verts)[order] / (n - 1) * (hi - lo) + lo, None]


# ---- regularise ---------------------------------------------------------------------------

def _regularise_prepare(case, seed):
    R = case["R"]
    g = grid.DenseGrid(1, [R] * 3, [-1.0] * 3, [1.0] * 3).to(DEV)
    sdf = _sdf(R, seed)
    # a grid in training: rough at the scale of an Adam step
    noise = torch.randn(sdf.shape, generator=_gen(seed, 7), device=DEV)
    g.grid.data.copy_(sdf + noise * 1e-3)
    # the data term's gradient: near the surface only
    g.grid.grad = torch.where(sdf.abs() < 4.0 / R, noise * 1e-5, torch.zeros_like(noise))
    x = torch.linspace(*BOX, R, device=DEV)
    mask = (x[:, None, None] ** 2 + x[None, :, None] ** 2 + x[None, None, :] ** 2).sqrt() < 0.9
    return dict(grid=g, mask=mask, count=int(mask.sum()), loss=torch.empty(1, device=DEV),
                ws=smooth.smooth_grad_tv_workspace(g.grid.data))


def _regularise_run(s):
    g, tv, R = s["grid"], scene.FINE_TV, s["case"]["R"]
    smooth.smooth_grad_tv_add_grad(g.grid, g.grid.grad, 2.0 / R, s["mask"],
                                   tv["weight_tv_density"] * tv["smooth_grad_tv"],
                                   mask_count=s["count"], loss=s["loss"], workspace=s["ws"])
    w = tv["weight_tv_density"] * tv["sdf_tv"] / 8192 * R / 128
    g.total_variation_add_grad(w, w, w, True)
    return dict(loss=s["loss"], grad=g.grid.grad)


def _regularise_work(case):
    n = float(case["R"]) ** 3
    return dict(bytes=n * (4 + 1 + 8), flops=n * 80)


def _regularise_exact(case, s):
    R, tv = case["R"], scene.FINE_TV
    x = s["grid"].grid.detach().double()
    p = x.clone().requires_grad_(True)
    vs, q = 2.0 / R, p[0, 0]
    G = [F.pad((q[2:] - q[:-2]) / 2 / vs, (0, 0, 0, 0, 1, 1)),
         F.pad((q[:, 2:] - q[:, :-2]) / 2 / vs, (0, 0, 1, 1)),
         F.pad((q[:, :, 2:] - q[:, :, :-2]) / 2 / vs, (1, 1))]
    loss = 0
    for c in G:
        with torch.no_grad():
            m = F.pad(c[None, None], (1,) * 6, mode="replicate")
            for a in (2, 3, 4):
                k = m.shape[a] - 2
                m = 0.25 * m.narrow(a, 0, k) + 0.5 * m.narrow(a, 1, k) + 0.25 * m.narrow(a, 2, k)
        loss = loss + ((m[0, 0] - c)[s["mask"]] ** 2).sum()
    loss = loss / (3 * s["count"]) * tv["weight_tv_density"] * tv["smooth_grad_tv"]
    loss.backward()
    grad = s["grid"].grid.grad.double() + p.grad
    _tv_add64(x, grad, tv["weight_tv_density"] * tv["sdf_tv"] / 8192 * R / 128)
    return dict(loss=loss.detach().reshape(1), grad=grad)


# ---- sdf_query ----------------------------------------------------------------------------

def _query_prepare(case, seed):
    cfg = dataclasses.replace(scene.FINE, R=case["R"], inv_s=float(case["R"]), feat_dim=3)
    sc = serve.ResidentScene(cfg, _sdf(case["R"], seed), _features(case["R"], 3, seed),
                             _mlp_params(cfg.mlp_in, cfg.mlp_depth, seed, 41), device=DEV)
    return dict(scene=sc, res=512, origin=(100 + seed % 50, 200, 250))


def _query_run(s):
    return s["scene"].sdf_query(s["res"], s["origin"], s["case"]["tile"])


def _query_work(case):
    n = float(case["tile"]) ** 3
    return dict(bytes=n * (16 + 4.0 * (case["R"] / 512) ** 3), flops=n * 150)


@torch.no_grad()
def _query_exact(case, s):
    ax = [-1 + 2 * (torch.arange(case["tile"], device=DEV, dtype=torch.float64) + o) /
          (s["res"] - 1) for o in s["origin"]]
    pts = torch.stack(torch.meshgrid(*ax, indexing="ij"), -1).reshape(-1, 3)
    val, grad = _sdf_grad64(s["scene"].sdf.double(), pts, s["scene"].cfg.voxel_size)
    return [val, grad / (grad.norm(dim=-1, keepdim=True) + 1e-5)]


# ---- the path in float64, in plain torch --------------------------------------------------

def _tri64(g, pts):
    """Trilinear lookup of g [1, C, X, Y, Z] at pts in the box, zero outside -> [P, C]."""
    out = F.grid_sample(g, pts.flip(-1).reshape(1, 1, 1, -1, 3), mode="bilinear",
                        align_corners=True)
    return out.reshape(g.shape[1], -1).T


def _displaced64(sdf, pts, voxel_size, q):
    """SDF at +-q voxels along z, y, x (clamped to the grid) and the normalised gradient."""
    f, gr = _stencil64(sdf, pts, voxel_size, q)
    return f, gr / (gr.norm(dim=-1, keepdim=True) + 1e-5)


def _stencil64(sdf, pts, voxel_size, q):
    size = torch.tensor([s - 1 for s in sdf.shape[-3:]], device=DEV, dtype=torch.float64)
    ind = (pts + 1) / 2 * size
    f, gr = [], []
    for a in (2, 1, 0):
        side, at = [], []
        for sg in (-1, 1):
            e = ind.clone()
            e[:, a] += sg * q
            e = torch.minimum(e.clamp(min=0), size)
            at.append(e[:, a])
            side.append(_tri64(sdf, e / size * 2 - 1)[:, 0])
        f += side
        gr.append((side[1] - side[0]) / (at[1] - at[0]) / voxel_size)
    return torch.stack(f, 1), torch.stack(gr, 1)


def _sdf_grad64(sdf, pts, voxel_size):
    """Centre value and the central-difference gradient (x, y, z) at one voxel."""
    _, gr = _stencil64(sdf, pts, voxel_size, 1.0)
    return _tri64(sdf, pts)[:, 0], gr.flip(-1)


def _slab64(o, d):
    v = torch.where(d == 0, torch.full_like(d, 1e-6), d)
    a, b = (BOX[1] - o) / v, (BOX[0] - o) / v
    t0 = torch.minimum(a, b).amax(-1).clamp(0.0, 1e9)
    t1 = torch.maximum(a, b).amin(-1).clamp(0.0, 1e9)
    return t0, t1


def _steps64(d, t0, t1, stepdist):
    return ((t1 - t0) * d.norm(dim=-1) / stepdist).ceil().clamp(min=1).long()


def _points64(o, d, t0, rid, step, stepdist):
    start, unit = o + d * t0[:, None], d / d.norm(dim=-1, keepdim=True)
    return start[rid] + unit[rid] * (step * stepdist)[:, None]


def _sample64(o, d, stepdist):
    """In-box samples of the rays: points, ray and step numbers."""
    t0, t1 = _slab64(o, d)
    steps = _steps64(d, t0, t1, stepdist)
    rid = torch.repeat_interleave(torch.arange(o.shape[0], device=DEV), steps)
    step = torch.arange(rid.numel(), device=DEV) - (torch.cumsum(steps, 0) - steps)[rid]
    pts = _points64(o, d, t0, rid, step, stepdist)
    k = ((pts >= BOX[0]) & (pts <= BOX[1])).all(-1)
    return pts[k], rid[k], step[k]


def _neus64(dirs, val, grad, dist, inv_s):
    h = -torch.relu(-(dirs * grad).sum(-1)) * dist * 0.5
    c, nx = torch.sigmoid((val - h) * inv_s), torch.sigmoid((val + h) * inv_s)
    return ((c - nx + 1e-5) / (c + 1e-5)).clip(0.0, 1.0)


def _weights64(alpha, rid, n):
    """weight = T alpha with T the product of (1 - alpha) before the sample; a ray ends
    once T < 1e-3."""
    steps = torch.bincount(rid, minlength=n)
    first = torch.cumsum(steps, 0) - steps
    at = torch.arange(rid.numel(), device=DEV) - first[rid]
    width = int(steps.max()) if steps.numel() else 0
    q = torch.ones((n, width + 1), device=DEV, dtype=torch.float64)
    q = q.index_put((rid, at + 1), 1 - alpha)
    T = torch.cumprod(q, 1)
    ends = (T.detach() < 1e-3).to(torch.int8)
    stop = torch.where(ends.any(1), ends.argmax(1), steps)
    last = T.gather(1, stop[:, None])[:, 0]
    w = T[rid, at] * alpha
    return torch.where(at < stop[rid], w, torch.zeros_like(w)), last


def _pe64(x, freqs):
    e = (x.unsqueeze(-1) * torch.tensor([2.0 ** i for i in range(freqs)], device=DEV,
                                        dtype=torch.float64)).flatten(-2)
    return torch.cat([x, e.sin(), e.cos()], -1)


def _mlp64(x, params):
    for i, (W, b) in enumerate(params):
        x = x @ W.T + b
        if i + 1 < len(params):
            x = torch.relu(x)
    return x


def _tv_add64(p, grad, w):
    """Total variation's gradient with differences clamped to one, w / 6 on each axis."""
    for a in (2, 3, 4):
        k = p.shape[a] - 1
        t = (p.narrow(a, 1, k) - p.narrow(a, 0, k)).clamp(-1, 1) * (w / 6)
        grad.narrow(a, 1, k).add_(t)
        grad.narrow(a, 0, k).sub_(t)


_PREPARE = dict(fine_step=_fine_prepare, coarse_grads=_coarse_prepare, render=_render_prepare,
                rgbnet=_rgbnet_prepare, lookup=_lookup_prepare, ray_ops=_ray_ops_prepare,
                prefilter=_prefilter_prepare, mesh=_mesh_prepare, regularise=_regularise_prepare,
                sdf_query=_query_prepare)
_RUN = dict(fine_step=_fine_run, coarse_grads=_coarse_run, render=_render_run,
            rgbnet=_rgbnet_run, lookup=_lookup_run, ray_ops=_ray_ops_run,
            prefilter=_prefilter_run, mesh=_mesh_run, regularise=_regularise_run,
            sdf_query=_query_run)
_WORK = dict(fine_step=_fine_work, coarse_grads=_coarse_work, render=_render_work,
             rgbnet=_rgbnet_work, lookup=_lookup_work, ray_ops=_ray_ops_work,
             prefilter=_prefilter_work, mesh=_mesh_work, regularise=_regularise_work,
             sdf_query=_query_work)
_EXACT = dict(coarse_grads=_coarse_exact, render=_render_exact, rgbnet=_rgbnet_exact,
              lookup=_lookup_exact, ray_ops=_ray_ops_exact, prefilter=_prefilter_exact,
              mesh=_mesh_exact, regularise=_regularise_exact, sdf_query=_query_exact)
