"""Voxurf coarse/fine forward passes and training steps on the HIP ops.

VoxurfFine / VoxurfCoarse keep the reference models' parameter names (sdf.grid, k0.grid,
rgbnet.*), buffers (xyz_min, xyz_max, viewfreq) and call structure
(lib/voxurf_fine.py:620-802, lib/voxurf_coarse.py:513-619): ray sampling ->
in-bbox compaction -> SDF value and 6-neighbour gradient -> NeuS alpha ->
alpha/weight compactions -> Alphas2Weights -> feature lookup -> rgbnet ->
segment-sum compositing.  Every step of it runs on the HIP kernels of libvoxhip.so
through the autograd Functions of voxurf_amd.functional; this is the "store-all" path
(every sample's intermediates are kept for backward, as the reference does).  The fused
per-ray path lives in voxurf_amd.fused.
"""
import torch
import torch.nn as nn
import torch.nn.functional as F

from . import render_utils_cuda as ru
from .functional import (Alphas2Weights, NeusAlpha, SampleSdfs, SdfGradSample, segment_coo,
                         select_rows)
from .grid import DenseGrid
from .mlp import RgbNet
from .scene import SceneConfig


class _VoxurfBase(nn.Module):
    def __init__(self, cfg: SceneConfig, sdf_grid=None, k0_grid=None):
        super().__init__()
        self.cfg = cfg
        ws = list(cfg.grid_shape)
        mn, mx = list(cfg.box[:3]), list(cfg.box[3:])
        self.register_buffer("xyz_min", torch.tensor(mn))
        self.register_buffer("xyz_max", torch.tensor(mx))
        self.world_size = torch.tensor(ws)
        self.voxel_size = cfg.voxel_size
        self.sdf = DenseGrid(1, ws, mn, mx)
        self.k0 = DenseGrid(cfg.feat_dim, ws, mn, mx)
        if sdf_grid is not None:
            self.sdf.grid.data.copy_(sdf_grid)
        if k0_grid is not None:
            self.k0.grid.data.copy_(k0_grid)
        self.s_val = nn.Parameter(torch.ones(1) / cfg.inv_s, requires_grad=False)

    @property
    def inv_s(self):
        return self.cfg.inv_s

    def sample_ray(self, rays_o, rays_d, stepsize):
        """lib/voxurf_fine.py:593-617 (far forced to 1e9)."""
        stepdist = self.cfg.stepdist
        ray_pts, mask_outbbox, ray_id, step_id, N_steps, t_min, t_max = ru.sample_pts_on_rays(
            rays_o.contiguous(), rays_d.contiguous(), self.xyz_min, self.xyz_max, 0.0, 1e9,
            stepdist)
        mask_inbbox = ~mask_outbbox
        ray_pts, ray_id, step_id = select_rows(mask_inbbox, ray_pts, ray_id, step_id)
        if getattr(self, "mask_cache", None) is not None:
            # known free space from the coarse geometry (lib/voxurf_fine.py:631-636)
            mask = self.mask_cache(ray_pts)
            ray_pts, ray_id, step_id = select_rows(mask, ray_pts, ray_id, step_id)
            mask_outbbox[~mask_outbbox] |= ~mask
        return ray_pts, ray_id, step_id, mask_outbbox, N_steps

    def hit_coarse_geo(self, rays_o, rays_d, near, far, stepsize, **render_kwargs):
        """lib/voxurf_fine.py:579-591: whether each ray has an in-box sample (far forced to
        1e9) that passes the MaskCache."""
        from .rays import hit_coarse_geo
        return hit_coarse_geo(self.mask_cache, self.xyz_min, self.xyz_max, rays_o, rays_d, near,
                              stepsize * self.voxel_size)

    def sdf_and_gradient(self, ray_pts):
        sdf, gradient, _ = SdfGradSample.apply(self.sdf.grid, ray_pts, self.xyz_min, self.xyz_max,
                                                self.voxel_size)
        return sdf, gradient

    def total_variation_add_grad(self, weight, dense_mode=True):
        self.sdf.total_variation_add_grad(weight, weight, weight, dense_mode)
        self.k0.total_variation_add_grad(weight, weight, weight, dense_mode)


class VoxurfFine(_VoxurfBase):
    """Fine stage: 12-channel k0, rgbnet(k0 | normal | view PE) (lib/voxurf_fine.py)."""

    def __init__(self, cfg: SceneConfig, sdf_grid=None, k0_grid=None, mlp_params=None,
                 mlp_dtype=torch.float32):
        super().__init__(cfg, sdf_grid, k0_grid)
        self.register_buffer("viewfreq", torch.tensor([2.0 ** i for i in range(cfg.view_pe)]))
        self.rgbnet = RgbNet(cfg.mlp_in, cfg.mlp_width, cfg.mlp_depth, params=mlp_params,
                             compute_dtype=mlp_dtype)

    def forward(self, rays_o, rays_d, viewdirs, bg=0.0):
        cfg = self.cfg
        N = len(rays_o)
        ray_pts, ray_id, step_id, mask_outbbox, N_steps = self.sample_ray(rays_o, rays_d,
                                                                          cfg.stepsize)
        sdf, gradient = self.sdf_and_gradient(ray_pts)
        alpha = NeusAlpha.apply(viewdirs, ray_id, sdf, gradient, cfg.stepdist, self.inv_s)
        m = alpha > cfg.fast_color_thres
        alpha, ray_id, ray_pts, gradient, step_id = select_rows(m, alpha, ray_id, ray_pts, gradient,
                                                                step_id)
        weights, alphainv_last = Alphas2Weights.apply(alpha, ray_id, N)
        m = weights > cfg.fast_color_thres
        weights, ray_id, ray_pts, gradient, step_id = select_rows(m, weights, ray_id, ray_pts,
                                                                  gradient, step_id)
        k0 = self.k0(ray_pts)
        normal = gradient / (gradient.norm(dim=-1, keepdim=True) + 1e-5)
        vemb = (viewdirs.unsqueeze(-1) * self.viewfreq).flatten(-2)
        vemb = torch.cat([viewdirs, vemb.sin(), vemb.cos()], -1)
        rgb_feat = torch.cat([k0, normal, vemb[ray_id]], -1)
        rgb = torch.sigmoid(self.rgbnet(rgb_feat))
        rgb_marched = segment_coo(weights.unsqueeze(-1) * rgb, ray_id,
                                  out=torch.zeros([N, 3], device=rgb.device), reduce="sum")
        rgb_marched = rgb_marched + alphainv_last[..., None] * bg
        return dict(rgb_marched=rgb_marched, alphainv_cum=alphainv_last, weights=weights,
                    ray_id=ray_id, n_samples=int(ray_id.numel()))


def positional_embedding(x, freq):
    """[x, sin(x (x) F), cos(x (x) F)] with x (x) F laid out component-major
    ((x[..., None] * F).flatten(-2)), lib/voxurf_fine.py:694-698."""
    emb = (x.unsqueeze(-1) * freq).flatten(-2)
    return torch.cat([x, emb.sin(), emb.cos()], -1)


class Voxurf(_VoxurfBase):
    """The reference fine model (lib/voxurf_fine.py `Voxurf`, forward :620-793) as
    configs/dtu_e2e/fine.py trains it (SceneConfig.model == "voxurf"): rgbnet on
    xyz PE | view PE | centre sdf | sample_sdfs features and normalised gradients at the
    grad_feat displacements, and the residual k_rgbnet on k0 | xyz PE | view PE |
    gradient | rgb_logit.detach(), whose sigmoid(rgb_logit.detach() + k_rgbnet(.)) is the
    rendered colour.  State-dict keys follow the reference (sdf.grid, k0.grid, rgbnet.*,
    k_rgbnet.*, posfreq, viewfreq, k_posfreq, k_viewfreq, s_val)."""

    def __init__(self, cfg: SceneConfig, sdf_grid=None, k0_grid=None, mlp_params=None,
                 k_mlp_params=None, mlp_dtype=torch.float32):
        if cfg.model != "voxurf":
            raise ValueError("Voxurf needs a SceneConfig with model='voxurf'")
        super().__init__(cfg, sdf_grid, k0_grid)
        self.register_buffer("posfreq", torch.tensor([2.0 ** i for i in range(cfg.pos_pe)]))
        self.register_buffer("viewfreq", torch.tensor([2.0 ** i for i in range(cfg.view_pe)]))
        self.register_buffer("k_posfreq", torch.tensor([2.0 ** i for i in range(cfg.pos_pe)]))
        self.register_buffer("k_viewfreq", torch.tensor([2.0 ** i for i in range(cfg.k_view_pe)]))
        self.rgbnet = RgbNet(cfg.mlp_in, cfg.mlp_width, cfg.mlp_depth, params=mlp_params,
                             compute_dtype=mlp_dtype)
        self.k_rgbnet = RgbNet(cfg.k_mlp_in, cfg.mlp_width, cfg.k_mlp_depth,
                               params=k_mlp_params, compute_dtype=mlp_dtype)
        if k_mlp_params is None:
            # the reference never zeroes k_rgbnet's last bias (it re-zeroes rgbnet's)
            nn.init.uniform_(self.k_rgbnet[-1].bias, -cfg.mlp_width ** -0.5,
                             cfg.mlp_width ** -0.5)
        # s_val is a plain tensor, not a registered parameter: the reference's
        # nn.Parameter(...).cuda() returns an unregistered copy, so its state dict has no
        # s_val (lib/voxurf_fine.py:61-62)
        s0 = cfg.s_start if cfg.s_ratio > 0 else 1.0 / cfg.inv_s
        del self.s_val
        self.s_val = torch.ones(1) * s0

    def set_step(self, global_step):
        """The s_val schedule of a training forward at `global_step`
        (lib/voxurf_fine.py:466-469); returns inv_s."""
        s_val, inv_s = self.cfg.s_val_at(global_step)
        self.s_val = torch.ones(1) * s_val
        return inv_s

    @property
    def inv_s(self):
        # evaluation uses the stored s_val (lib/voxurf_fine.py:476), in float32
        return float(torch.ones(1) / self.s_val.float().cpu())

    def forward(self, rays_o, rays_d, viewdirs, global_step=None, bg=0.0, render_grad=False,
                render_depth=False):
        cfg = self.cfg
        N = len(rays_o)
        inv_s = self.set_step(global_step) if global_step is not None else self.inv_s
        ray_pts, ray_id, step_id, mask_outbbox, N_steps = self.sample_ray(rays_o, rays_d,
                                                                          cfg.stepsize)
        sdf, gradient = self.sdf_and_gradient(ray_pts)
        dist = cfg.stepdist
        alpha = NeusAlpha.apply(viewdirs, ray_id, sdf, gradient, dist, inv_s)
        m = alpha > cfg.fast_color_thres
        alpha, ray_id, ray_pts, step_id, gradient, sdf = select_rows(m, alpha, ray_id, ray_pts,
                                                                     step_id, gradient, sdf)
        weights, alphainv_last = Alphas2Weights.apply(alpha, ray_id, N)
        m = weights > cfg.fast_color_thres
        weights, ray_id, ray_pts, step_id, gradient, sdf = select_rows(m, weights, ray_id, ray_pts,
                                                                       step_id, gradient, sdf)
        k0 = self.k0(ray_pts)
        if k0.dim() == 1:
            k0 = k0[:, None]
        all_feat, all_grad = SampleSdfs.apply(self.sdf.grid, ray_pts, self.xyz_min, self.xyz_max,
                                              sorted(cfg.grad_feat), self.voxel_size, True)
        rays_xyz = (ray_pts - self.xyz_min) / (self.xyz_max - self.xyz_min)
        xyz_emb = positional_embedding(rays_xyz, self.posfreq)
        vemb = positional_embedding(viewdirs, self.viewfreq)
        rgb_feat = torch.cat([xyz_emb, vemb[ray_id], sdf[:, None], all_feat, all_grad], -1)
        rgb_logit = self.rgbnet(rgb_feat)
        rgb = torch.sigmoid(rgb_logit)
        k_xyz_emb = positional_embedding(rays_xyz, self.k_posfreq)
        k_vemb = positional_embedding(viewdirs, self.k_viewfreq)
        k_feat = torch.cat([k0, k_xyz_emb, k_vemb[ray_id], gradient, rgb_logit.detach()], -1)
        k_rgb = torch.sigmoid(rgb_logit.detach() + self.k_rgbnet(k_feat))
        zeros = torch.zeros([N, 3], device=rgb.device)
        k_rgb_marched = (segment_coo(weights.unsqueeze(-1) * k_rgb, ray_id, out=zeros,
                                     reduce="sum") + alphainv_last[..., None] * bg).clamp(0, 1)
        rgb_marched = segment_coo(weights.unsqueeze(-1) * rgb, ray_id, out=zeros,
                                  reduce="sum") + alphainv_last[..., None] * bg
        out = dict(rgb_marched=k_rgb_marched, rgb_marched0=rgb_marched,
                   alphainv_cum=alphainv_last, weights=weights, ray_id=ray_id,
                   n_samples=int(ray_id.numel()), normal_marched=None, depth=None)
        if render_grad:
            normal = gradient / (gradient.norm(2, -1, keepdim=True) + 1e-6)
            out["normal_marched"] = segment_coo(weights.unsqueeze(-1) * normal, ray_id,
                                                out=zeros, reduce="sum")
        if render_depth:
            with torch.no_grad():
                out["depth"] = segment_coo(weights * step_id * dist, ray_id,
                                           out=torch.zeros([N], device=rgb.device), reduce="sum")
        return out


def _mesh_color_forward(self, ray_pts):
    """lib/voxurf_fine.py:804-892: the colour of surface points (mesh vertices) seen along
    their inward normal: the rows of both colour networks at each point with the view
    direction -normal (normal = gradient / (|gradient| + 1e-5) of the 6-neighbour SDF
    gradient), rgb = sigmoid(rgb_logit + k_rgbnet(.)) (the same networks as forward())."""
    cfg = self.cfg
    ray_pts = ray_pts.reshape(-1, 3).contiguous()
    sdf, gradient = self.sdf_and_gradient(ray_pts)
    viewdirs = -(gradient / (gradient.norm(dim=-1, keepdim=True) + 1e-5))
    k0 = self.k0(ray_pts)
    if k0.dim() == 1:
        k0 = k0[:, None]
    all_feat, all_grad = SampleSdfs.apply(self.sdf.grid, ray_pts, self.xyz_min, self.xyz_max,
                                          sorted(cfg.grad_feat), self.voxel_size, True)
    rays_xyz = (ray_pts - self.xyz_min) / (self.xyz_max - self.xyz_min)
    xyz_emb = positional_embedding(rays_xyz, self.posfreq)
    vemb = positional_embedding(viewdirs, self.viewfreq)
    rgb_feat = torch.cat([xyz_emb, vemb, sdf[:, None], all_feat, all_grad], -1)
    rgb_logit = self.rgbnet(rgb_feat)
    k_xyz_emb = positional_embedding(rays_xyz, self.k_posfreq)
    k_vemb = positional_embedding(viewdirs, self.k_viewfreq)
    k_feat = torch.cat([k0, k_xyz_emb, k_vemb, gradient, rgb_logit.detach()], -1)
    return torch.sigmoid(rgb_logit.detach() + self.k_rgbnet(k_feat))


Voxurf.mesh_color_forward = _mesh_color_forward


def voxurf_loss(out, target, cfg):
    """run.py:604-633 without the regularisers: weight_main * MSE(rgb_marched) +
    weight_entropy_last * the binary entropy of alphainv_cum[..., -1] (the last ray's
    alphainv_last: the fine model's alphainv_cum is [N]) + weight_rgb0 * MSE(rgb_marched0)."""
    loss = cfg.weight_main * F.mse_loss(out["rgb_marched"], target)
    if cfg.weight_entropy_last > 0:
        pout = out["alphainv_cum"][..., -1].clamp(1e-6, 1 - 1e-6)
        ent = -(pout * torch.log(pout) + (1 - pout) * torch.log(1 - pout)).mean()
        loss = loss + cfg.weight_entropy_last * ent
    if cfg.weight_rgb0 > 0 and out.get("rgb_marched0") is not None:
        loss = loss + F.mse_loss(out["rgb_marched0"], target) * cfg.weight_rgb0
    return loss


class VoxurfCoarse(_VoxurfBase):
    """Coarse stage: colour = sigmoid(k0) with a 3-channel k0 (lib/voxurf_coarse.py)."""

    def forward(self, rays_o, rays_d, viewdirs, bg=0.0):
        cfg = self.cfg
        N = len(rays_o)
        ray_pts, ray_id, step_id, mask_outbbox, N_steps = self.sample_ray(rays_o, rays_d,
                                                                          cfg.stepsize)
        sdf, gradient = self.sdf_and_gradient(ray_pts)
        alpha = NeusAlpha.apply(viewdirs, ray_id, sdf, gradient, cfg.stepdist, self.inv_s)
        weights, alphainv_last = Alphas2Weights.apply(alpha, ray_id, N)
        m = weights > cfg.fast_color_thres
        ray_pts, ray_id, alpha = select_rows(m, ray_pts, ray_id, alpha)
        weights, alphainv_last = Alphas2Weights.apply(alpha, ray_id, N)
        rgb = torch.sigmoid(self.k0(ray_pts))
        rgb_marched = segment_coo(weights.unsqueeze(-1) * rgb, ray_id,
                                  out=torch.zeros([N, 3], device=rgb.device), reduce="sum")
        cum_w = segment_coo(weights.unsqueeze(-1), ray_id,
                            out=torch.zeros([N, 1], device=rgb.device), reduce="sum")
        rgb_marched = (rgb_marched + (1 - cum_w) * bg).clamp(0, 1)
        return dict(rgb_marched=rgb_marched, alphainv_cum=alphainv_last, weights=weights,
                    ray_id=ray_id, n_samples=int(ray_id.numel()))


class Trainer:
    """The training step of run.py:600-659 around a VoxurfFine/VoxurfCoarse model:
    forward, MSE loss, backward, TV gradient (if cfg.tv_weight > 0), Adam
    (utils.Adam, betas (0.9, 0.99)) with per-module learning rates."""

    def __init__(self, model, cfg: SceneConfig):
        from .optim import Adam
        self.model = model
        self.cfg = cfg
        groups = [dict(params=[model.sdf.grid], lr=cfg.lr_sdf, name="sdf"),
                  dict(params=[model.k0.grid], lr=cfg.lr_k0, name="k0")]
        if hasattr(model, "rgbnet") and cfg.lr_mlp > 0:
            groups.append(dict(params=list(model.rgbnet.parameters()), lr=cfg.lr_mlp,
                               name="rgbnet"))
        if hasattr(model, "k_rgbnet") and cfg.lr_k_mlp > 0:
            groups.append(dict(params=list(model.k_rgbnet.parameters()), lr=cfg.lr_k_mlp,
                               name="k_rgbnet"))
        self.opt = Adam(groups, betas=(0.9, 0.99))
        self.global_step = 0

        self.last_profile = {}
        self.last_counts = {}

    def step(self, rays_o, rays_d, viewdirs, target, profile=False, global_step=None):
        self.global_step = self.global_step + 1 if global_step is None else global_step
        self.opt.zero_grad(set_to_none=True)
        if isinstance(self.model, Voxurf):
            out = self.model(rays_o, rays_d, viewdirs, global_step=self.global_step,
                             bg=self.cfg.bg)
            loss = voxurf_loss(out, target, self.cfg)
        else:
            out = self.model(rays_o, rays_d, viewdirs, bg=self.cfg.bg)
            loss = F.mse_loss(out["rgb_marched"], target)
        loss.backward()
        if self.cfg.tv_weight > 0:
            self.model.total_variation_add_grad(self.cfg.tv_weight, True)
        if profile:
            self.grads_snapshot = dict(
                sdf=self.model.sdf.grid.grad.clone(), k0=self.model.k0.grid.grad.clone(),
                mlp=[p.grad.clone() for p in self.model.rgbnet.parameters()]
                if hasattr(self.model, "rgbnet") else [],
                k_mlp=[p.grad.clone() for p in self.model.k_rgbnet.parameters()]
                if hasattr(self.model, "k_rgbnet") else [])
            self.opt.profile_events = {}
        self.opt.step()
        if profile:
            torch.cuda.synchronize()
            e0, e1 = self.opt.profile_events[id(self.model.k0.grid)]
            self.last_profile = {"adam_k0_ms": e0.elapsed_time(e1)}
            self.opt.profile_events = None
            self.last_counts = {"m2": out["n_samples"]}
        out["loss"] = loss.detach()
        return out
