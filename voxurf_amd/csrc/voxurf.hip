// Fused colour side of the reference fine model (gfx950): lib/voxurf_fine.py:678-763 as
// configs/dtu_e2e/fine.py trains it.  Two MLPs share the survivor rows:
//   rgbnet   on X  = [xyz PE | view PE | sdf | sample_sdfs feat (6 nd) | normalised grad (3 nd)]
//   k_rgbnet on XK = [k0 (C) | xyz PE | k view PE | gradient (3) | rgb_logit.detach() (3)]
// and the rendered colour is sigmoid(rgb_logit.detach() + k_rgbnet(XK)), clamped after
// compositing; rgb_marched0 (sigmoid(rgb_logit) composited) feeds the second MSE term.
//
// The per-ray forward, the survivor scan and the SDF backward are the plain fine step's
// (fused.hip).  Here: the row builder (tiles of 32 survivor rows put together in LDS, a lane
// per displaced SDF sample of sample_sdfs, sine and cosine), the compositing with both colour terms, the loss and the entropy of the last
// ray, and the adjoint of the rows (k0 scatter, the raw-gradient and centre-SDF
// adjoints handed to the SDF backward, and the displaced-sample scatter of sample_sdfs).
// Every per-value formula is the drop-in ops' own (voxel.h), so the rows equal the
// op-by-op path's.
#include "fine.h"

namespace vx {

constexpr int kVxMaxDisp = 4;

struct VoxurfRowDesc {
  int pos_pe, view_pe, k_view_pe, nd;
  float disp[kVxMaxDisp];
  int xstride, kstride;
  // column offsets
  int x_view, x_sdf, x_feat, x_grad, x_end;
  int k_pos, k_view, k_grad, k_logit, k_end;
};

// One lane's share of sample_sdfs for one row: lane l < 3 nd takes axis a = l / nd and
// displacement j = l % nd, i.e. the samples at -d and +d along a (zyx index space) and
// the unnormalised gradient component (f+ - f-) / diff / voxel_size, as k_sdfs_fwd.
struct HierLane {
  float fm, fp, df, r;
  int a, j;
  bool on;
};

__device__ __forceinline__ void hier_lane(const FusedGeom& G, const VoxurfRowDesc& D,
                                          const float q[3], int l, HierLane& h) {
#pragma clang fp contract(off)
  h.on = l < 3 * D.nd;
  h.a = h.on ? l / D.nd : 0;
  h.j = h.on ? l % D.nd : 0;
  h.fm = h.fp = h.r = 0.f;
  h.df = 1.f;
  if (!h.on) return;
  float ind[3];
  zyx_index(q, G.mn, G.mx, G.gs, ind);
  const float d = D.disp[h.j];
  float cm, cp;
  h.fm = sample_displaced(G.sdf, G.gs, ind, h.a, -d, cm);
  h.fp = sample_displaced(G.sdf, G.gs, ind, h.a, d, cp);
  h.df = clamped_diff(ind, h.a, d, G.gs);
  h.r = ((h.fp - h.fm) / h.df) / G.voxel_size;
}

// Rows X and XK of the survivors, 32 a workgroup and pass, put together in LDS (dynamic: the
// two tiles of rows) and written out in one run each.  Every value is a lane's own task: the
// 6 nd displaced samples of a row (minus and plus in neighbouring lanes), the sines and
// cosines (once for both rows), four channels of k0.  A wavefront per ray with sixteen lanes a
// row before, twelve of them taking two samples in turn and each working out its columns'
// embeddings with runtime divisions, was bound by those instructions: 491 us for 96,000 rows
// of an 8192-ray chunk, 51 so.  XK's logit columns are left zero (vx_voxurf_logit_cols
// fills them after rgbnet's forward).
constexpr int kVxRowTile = 32;

__global__ void __launch_bounds__(256) k_voxurf_rows(
    FusedGeom G, VoxurfRowDesc D, const float* __restrict__ viewdirs, int64_t n_rays,
    const int64_t* __restrict__ off_incl, int64_t max_rows, float* __restrict__ X,
    float* __restrict__ XK, const float4* __restrict__ P4, const float4* __restrict__ G4,
    const int* __restrict__ rid) {
  extern __shared__ float4 tiles[];
  __shared__ float raw[kVxRowTile][3 * kVxMaxDisp];  // unnormalised gradients [axis][displacement]
  __shared__ float ind[kVxRowTile][4], unit[kVxRowTile][4], dir[kVxRowTile][4];
  __shared__ float4 pos[kVxRowTile], grad[kVxRowTile];
  float* xr = reinterpret_cast<float*>(tiles);
  float* kr = xr + kVxRowTile * D.xstride;
  const int tid = threadIdx.x, C = G.gk.C, nd = D.nd;
  const bool vec4 = G.gk.sc == 1 && (C & 3) == 0 && ((G.gk.sx | G.gk.sy | G.gk.sz) & 3) == 0 &&
                    (reinterpret_cast<uintptr_t>(G.k0) & 15) == 0;
  const int64_t total = off_incl[n_rays - 1];
  const int64_t rows = total < max_rows ? total : max_rows;
  for (int64_t row0 = blockIdx.x * (int64_t)kVxRowTile; row0 < rows;
       row0 += gridDim.x * (int64_t)kVxRowTile) {
    const int m = (int)(rows - row0 < kVxRowTile ? rows - row0 : kVxRowTile);
    for (int i = tid; i < kVxRowTile * (D.xstride + D.kstride) / 4; i += 256)
      tiles[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (tid < m) {
#pragma clang fp contract(off)
      const float4 a = P4[row0 + tid];
      const int64_t r = min(max(rid[row0 + tid], 0), (int)n_rays - 1);
      const float q[3] = {a.x, a.y, a.z};
      float id[3];
      zyx_index(q, G.mn, G.mx, G.gs, id);
      for (int e = 0; e < 3; ++e) {
        ind[tid][e] = id[e];
        unit[tid][e] = (q[e] - G.mn[e]) / (G.mx[e] - G.mn[e]);  // for the xyz PE
        dir[tid][e] = viewdirs[3 * r + e];
      }
      pos[tid] = a;
      grad[tid] = G4[row0 + tid];
    }
    __syncthreads();
    // sample_sdfs: the value at -d (even tasks) and +d (odd) along each axis, and the
    // gradient component (f+ - f-) / diff / voxel_size, as k_sdfs_fwd
    const int n6 = 6 * nd;
    for (int i = tid; i < m * n6; i += 256) {
#pragma clang fp contract(off)
      const int row = (int)((unsigned)i / (unsigned)n6), t = i - row * n6;
      const int sgn = t & 1, hl = t >> 1, a = (int)((unsigned)hl / (unsigned)nd), j = hl - a * nd;
      const float id[3] = {ind[row][0], ind[row][1], ind[row][2]};
      const float d = D.disp[j];
      float cl;
      const float f = sample_displaced(G.sdf, G.gs, id, a, sgn ? d : -d, cl);
      xr[row * D.xstride + D.x_feat + (2 * a + sgn) * nd + j] = f;
      const float fm = __shfl_xor(f, 1, 64);
      if (sgn) raw[row][hl] = ((f - fm) / clamped_diff(id, a, d, G.gs)) / G.voxel_size;
    }
    const int np3 = 3 * D.pos_pe;
    for (int i = tid; i < m * np3; i += 256) {
#pragma clang fp contract(off)
      const int row = (int)((unsigned)i / (unsigned)np3), t = i - row * np3;
      const int comp = (int)((unsigned)t / (unsigned)D.pos_pe), f = t - comp * D.pos_pe;
      const float arg = unit[row][comp] * (float)(1 << f);
      const float sn = sinf(arg), cs = cosf(arg);
      float* x = xr + row * D.xstride + 3 + t;
      float* k = kr + row * D.kstride + D.k_pos + 3 + t;
      x[0] = sn;
      x[np3] = cs;
      k[0] = sn;
      k[np3] = cs;
    }
    const int nv = max(D.view_pe, D.k_view_pe), nv3 = 3 * nv;
    for (int i = tid; i < m * nv3; i += 256) {
#pragma clang fp contract(off)
      const int row = (int)((unsigned)i / (unsigned)nv3), t = i - row * nv3;
      const int comp = (int)((unsigned)t / (unsigned)nv), f = t - comp * nv;
      const float arg = dir[row][comp] * (float)(1 << f);
      const float sn = sinf(arg), cs = cosf(arg);
      if (f < D.view_pe) {
        float* x = xr + row * D.xstride + D.x_view + 3 + comp * D.view_pe + f;
        x[0] = sn;
        x[3 * D.view_pe] = cs;
      }
      if (f < D.k_view_pe) {
        float* k = kr + row * D.kstride + D.k_view + 3 + comp * D.k_view_pe + f;
        k[0] = sn;
        k[3 * D.k_view_pe] = cs;
      }
    }
    const int nch = vec4 ? C >> 2 : C;
    for (int i = 255 - tid; i < m * nch; i += 256) {
      const int row = (int)((unsigned)i / (unsigned)nch), ch = i - row * nch;
      const float4 q = pos[row];
      Tri<float> t;
      t.init(world_to_index(q.x, G.mn[0], G.mx[0] - G.mn[0], G.gk.X),
             world_to_index(q.y, G.mn[1], G.mx[1] - G.mn[1], G.gk.Y),
             world_to_index(q.z, G.mn[2], G.mx[2] - G.mn[2], G.gk.Z));
      float* k = kr + row * D.kstride;
      if (vec4) *reinterpret_cast<float4*>(k + 4 * ch) = tri_gather4(G.k0, G.gk, t, 4 * ch);
      else k[ch] = tri_gather(G.k0, G.gk, t, ch);
    }
    for (int i = tid; i < m * 4; i += 256) {
      const int row = i >> 2, e = i & 3;
      float* x = xr + row * D.xstride;
      float* k = kr + row * D.kstride;
      const float4 g = grad[row];
      if (e < 3) {
        x[e] = k[D.k_pos + e] = unit[row][e];
        x[D.x_view + e] = k[D.k_view + e] = dir[row][e];
        k[D.k_grad + e] = e == 0 ? g.x : (e == 1 ? g.y : g.z);
      } else {
        x[D.x_sdf] = g.w;
      }
    }
    __syncthreads();
    // normalised over the three axes of each displacement
    for (int i = tid; i < m * nd; i += 256) {
#pragma clang fp contract(off)
      const int row = (int)((unsigned)i / (unsigned)nd), j = i - row * nd;
      const float r0 = raw[row][j], r1 = raw[row][nd + j], r2 = raw[row][2 * nd + j];
      const float nrm = sqrtf(r0 * r0 + r1 * r1 + r2 * r2) + 1e-5f;
      float* x = xr + row * D.xstride + D.x_grad + j;
      x[0] = r0 / nrm;
      x[nd] = r1 / nrm;
      x[2 * nd] = r2 / nrm;
    }
    __syncthreads();
    float4* xo = reinterpret_cast<float4*>(X + row0 * D.xstride);
    float4* ko = reinterpret_cast<float4*>(XK + row0 * D.kstride);
    for (int i = tid; i < m * D.xstride / 4; i += 256) xo[i] = tiles[i];
    for (int i = tid; i < m * D.kstride / 4; i += 256) ko[i] = reinterpret_cast<float4*>(kr)[i];
    __syncthreads();
  }
}

// XK[:, k_logit .. k_logit + 3) = rgb logits (the detached k_rgbnet input).
__global__ void k_voxurf_logit_cols(int64_t m, const int64_t* __restrict__ m_dev,
                                    const float* __restrict__ lg, float* __restrict__ XK,
                                    int kstride, int lcol) {
  if (m_dev) m = *m_dev < m ? *m_dev : m;
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= 3 * m) return;
  const int64_t j = i / 3;
  const int c = (int)(i % 3);
  XK[j * kstride + lcol + c] = lg[j * 3 + c];
}

// Compositing of both colour terms, the loss and the colour-side adjoints (sixteen lanes
// per ray):
//   rgb0_j = sigmoid(lg_j), krgb_j = sigmoid(lg_j + klg_j)        (lib/voxurf_fine.py:718-751)
//   rgb_marched0 = sum w rgb0 + last bg,  rgb_marched = clamp(sum w krgb + last bg, 0, 1)
//   loss = w_main MSE(rgb_marched) + w_rgb0 MSE(rgb_marched0) + w_ent H(clamp(last[N-1]))
//   (run.py:604-633); per ray loss_r = w_main |rgbm - t|^2 + w_rgb0 |rgbm0 - t|^2 (+ the
//   entropy term / inv_count on the last ray), summed and scaled by inv_count later.
//   gk = w_main 2 (rgbm - t) inv_count [0 <= pre-clamp <= 1],  g0 = w_rgb0 2 (rgbm0 - t) inv_count
//   dlg0_j = w g0 rgb0 (1 - rgb0),  dlgk_j = w gk krgb (1 - krgb)  (the logit is detached
//   in the k branch), gw_j = <gk, krgb> + <g0, rgb0>, glast = bg (sum gk + sum g0) (+ the
//   entropy's derivative log((1 - p) / p) on the last ray), S_r = sum gw_j w_j.
__global__ void __launch_bounds__(256) k_voxurf_composite(
    int64_t n_rays, const int64_t* __restrict__ cnt, const int64_t* __restrict__ off_incl,
    const float* __restrict__ lg, const float* __restrict__ klg, const float4* __restrict__ P4,
    const float* __restrict__ last, const float* __restrict__ target, float bg, float inv_count,
    float w_main, float w_rgb0, float w_ent, float* __restrict__ rgb_out,
    float* __restrict__ rgb0_out, float* __restrict__ dlg0, float* __restrict__ dlgk,
    float* __restrict__ gw, float* __restrict__ glast, float* __restrict__ S,
    float* __restrict__ loss_r, int64_t max_rows) {
  constexpr int SEG = 16;
  const int lane = threadIdx.x & 63, grp = lane / SEG, sl = lane % SEG;
  const int64_t groups = (int64_t)gridDim.x * (blockDim.x >> 6) * (64 / SEG);
  auto seg_sum = [&](float v) {
#pragma unroll
    for (int off = SEG / 2; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
  };
  for (int64_t r0 = ((int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) * (64 / SEG);
       r0 < n_rays; r0 += groups) {
    const int64_t r = r0 + grp;
    const bool ok = r < n_rays;
    const int64_t c = ok && off_incl[r] <= max_rows ? cnt[r] : 0;
    const int64_t o = ok ? off_incl[r] - cnt[r] : 0;
    float acc0[3] = {0.f, 0.f, 0.f}, acck[3] = {0.f, 0.f, 0.f};
    for (int64_t j = o + sl; j < o + c; j += SEG) {
      const float w = P4[j].w;
      for (int ch = 0; ch < 3; ++ch) {
        const float l0 = lg[j * 3 + ch];
        acc0[ch] += w * (1.f / (1.f + expf(-l0)));
        acck[ch] += w * (1.f / (1.f + expf(-(l0 + klg[j * 3 + ch]))));
      }
    }
    for (int ch = 0; ch < 3; ++ch) {
      acc0[ch] = seg_sum(acc0[ch]);
      acck[ch] = seg_sum(acck[ch]);
    }
    if (!ok) continue;
    const float lr = last[r];
    float gk[3], g0[3], l = 0.f;
    for (int ch = 0; ch < 3; ++ch) {
      const float v0 = acc0[ch] + lr * bg;
      const float vk = acck[ch] + lr * bg;
      const float rk = vk < 0.f ? 0.f : (vk > 1.f ? 1.f : vk);
      if (sl == 0) {
        rgb_out[3 * r + ch] = rk;
        rgb0_out[3 * r + ch] = v0;
      }
      if (target) {
        const float dk = rk - target[3 * r + ch], d0 = v0 - target[3 * r + ch];
        l += w_main * (dk * dk) + w_rgb0 * (d0 * d0);
        gk[ch] = (vk >= 0.f && vk <= 1.f) ? w_main * (2.f * dk * inv_count) : 0.f;
        g0[ch] = w_rgb0 * (2.f * d0 * inv_count);
      }
    }
    if (!target) continue;
    float gl = (gk[0] + gk[1] + gk[2] + g0[0] + g0[1] + g0[2]) * bg;
    if (r == n_rays - 1 && w_ent > 0.f) {
      // H(p) = -(p log p + (1 - p) log(1 - p)) of p = clamp(last, 1e-6, 1 - 1e-6);
      // dH/dp = log(1 - p) - log(p), passed by the clamp where 1e-6 <= last <= 1 - 1e-6
      const float p = lr < 1e-6f ? 1e-6f : (lr > 1.f - 1e-6f ? 1.f - 1e-6f : lr);
      const float ent = -(p * logf(p) + (1.f - p) * logf(1.f - p));
      l += w_ent * ent / inv_count;
      if (lr >= 1e-6f && lr <= 1.f - 1e-6f) gl += w_ent * (logf(1.f - p) - logf(p));
    }
    if (sl == 0) {
      loss_r[r] = l;
      glast[r] = gl;
    }
    float s = 0.f;
    for (int64_t j = o + sl; j < o + c; j += SEG) {
      const float w = P4[j].w;
      float gwj = 0.f;
      for (int ch = 0; ch < 3; ++ch) {
        const float l0 = lg[j * 3 + ch];
        const float rgb0 = 1.f / (1.f + expf(-l0));
        const float krgb = 1.f / (1.f + expf(-(l0 + klg[j * 3 + ch])));
        gwj += gk[ch] * krgb + g0[ch] * rgb0;
        dlg0[j * 3 + ch] = (w * g0[ch]) * (rgb0 * (1.f - rgb0));
        dlgk[j * 3 + ch] = (w * gk[ch]) * (krgb * (1.f - krgb));
      }
      gw[j] = gwj;
      s += gwj * w;
    }
    s = seg_sum(s);
    if (sl == 0) S[r] = s;
  }
}

// Adjoint of the rows, four rows per pass, sixteen lanes per row:
//   k0_grad += trilinear scatter of dXK[:, 0:C];
//   dgf [M,3] = dXK[:, k_grad .. k_grad+3) (the raw gradient's adjoint), dsf [M] =
//   dX[:, x_sdf] (the centre SDF's): both go to the SDF backward at the row's sample;
//   sdf_grad += the adjoint of sample_sdfs (k_sdfs_bwd's arithmetic): lane l < 3 nd takes
//   axis a and displacement j, recomputes its pair of displaced samples, the normalised
//   gradient's adjoint across the three axes, and scatters f- and f+.
__global__ void __launch_bounds__(256) k_voxurf_feat_bwd(
    FusedGeom G, VoxurfRowDesc D, int64_t m, const int64_t* __restrict__ m_dev,
    const float* __restrict__ dX, const float* __restrict__ dXK, const float4* __restrict__ P4,
    float* __restrict__ k0_grad, float* __restrict__ sdf_grad, float* __restrict__ dgf,
    float* __restrict__ dsf) {
  if (m_dev) m = *m_dev < m ? *m_dev : m;
  const int C = G.gk.C;
  const int lane = threadIdx.x & 63, grp = lane >> 4, cl = lane & 15;
  const int64_t groups = (int64_t)gridDim.x * (blockDim.x >> 6) * 4;
  for (int64_t j = ((int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) * 4 + grp;
       j - grp < m; j += groups) {
    const bool valid = j < m;
    const float4 a = P4[valid ? j : 0];
    const float q[3] = {a.x, a.y, a.z};
    // k0 scatter, lane cl < C takes channel cl
    if (valid && cl < C) {
      const float go = dXK[j * D.kstride + cl];
      if (go != 0.f) {
        Tri<float> t;
        t.init(world_to_index(q[0], G.mn[0], G.mx[0] - G.mn[0], G.gk.X),
               world_to_index(q[1], G.mn[1], G.mx[1] - G.mn[1], G.gk.Y),
               world_to_index(q[2], G.mn[2], G.mx[2] - G.mn[2], G.gk.Z));
        tri_scatter(k0_grad, G.gk, t, cl, go);
      }
    }
    if (valid && cl == 0) {
      for (int e = 0; e < 3; ++e) dgf[3 * j + e] = dXK[j * D.kstride + D.k_grad + e];
      dsf[j] = dX[j * D.xstride + D.x_sdf];
    }
    // sample_sdfs adjoint
    HierLane h;
    hier_lane(G, D, q, valid ? cl : 64, h);
    const int gbase = grp * 16;
    float gg = 0.f;
    if (h.on && valid) gg = dX[j * D.xstride + D.x_grad + h.a * D.nd + h.j];
    const float r0 = __shfl(h.r, gbase + h.j, 64), r1 = __shfl(h.r, gbase + D.nd + h.j, 64),
                r2 = __shfl(h.r, gbase + 2 * D.nd + h.j, 64);
    const float g0 = __shfl(gg, gbase + h.j, 64), g1 = __shfl(gg, gbase + D.nd + h.j, 64),
                g2 = __shfl(gg, gbase + 2 * D.nd + h.j, 64);
    if (h.on && valid) {
#pragma clang fp contract(off)
      // y = r / (|r| + eps):  dr = (gy - r (r . gy) / (|r| (|r| + eps))) / (|r| + eps)
      const float nr = sqrtf(r0 * r0 + r1 * r1 + r2 * r2);
      const float den = nr + 1e-5f;
      const float dot = r0 * g0 + r1 * g1 + r2 * g2;
      const float kk = nr > 0.f ? dot / (nr * den) : 0.f;
      const float ga = (gg - h.r * kk) / den;
      const float gd = ga / h.df / G.voxel_size;
      const float gm = dX[j * D.xstride + D.x_feat + (2 * h.a) * D.nd + h.j] - gd;
      const float gp = dX[j * D.xstride + D.x_feat + (2 * h.a + 1) * D.nd + h.j] + gd;
      float ind[3];
      zyx_index(q, G.mn, G.mx, G.gs, ind);
      const float d = D.disp[h.j];
      scatter_displaced(sdf_grad, G.gs, ind, h.a, -d, gm);
      scatter_displaced(sdf_grad, G.gs, ind, h.a, d, gp);
    }
  }
}


// Render outputs besides the colour (lib/voxurf_fine.py:765-777, asked for with
// render_grad / render_depth at run.py:1052-1054), sixteen lanes per ray:
//   normal_marched[r] = sum_j w_j g_j / (|g_j| + 1e-6)      (g: the raw SDF gradient)
//   depth[r]          = sum_j w_j step_id_j dist             (dist = stepdist)
// The step id of a row is recovered from its point: p = start + dir (stepdist s) with
// |dir| = 1, so s = rint(<p - start, dir> / stepdist) (the rounding error of p is far
// below half a step).
__global__ void __launch_bounds__(256) k_render_extras(
    FusedGeom G, int64_t n_rays, const int64_t* __restrict__ cnt,
    const int64_t* __restrict__ off_incl, const float4* __restrict__ P4,
    const float4* __restrict__ G4, const float* __restrict__ rays_o,
    const float* __restrict__ rays_d, float* __restrict__ normal, float* __restrict__ depth,
    int64_t max_rows) {
  constexpr int SEG = 16;
  const int lane = threadIdx.x & 63, grp = lane / SEG, sl = lane % SEG;
  const int64_t groups = (int64_t)gridDim.x * (blockDim.x >> 6) * (64 / SEG);
  for (int64_t r0 = ((int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) * (64 / SEG);
       r0 < n_rays; r0 += groups) {
    const int64_t r = r0 + grp;
    const bool ok = r < n_rays;
    const int64_t c = ok && off_incl[r] <= max_rows ? cnt[r] : 0;
    const int64_t o = ok ? off_incl[r] - cnt[r] : 0;
    float start[3] = {0.f, 0.f, 0.f}, dir[3] = {0.f, 0.f, 1.f};
    if (ok) {
      int64_t ns;
      ray_setup(G, rays_o + 3 * r, rays_d + 3 * r, start, dir, ns);
    }
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    for (int64_t j = o + sl; j < o + c; j += SEG) {
#pragma clang fp contract(off)
      const float4 a = P4[j], b = G4[j];
      const float nr = sqrtf(b.x * b.x + b.y * b.y + b.z * b.z) + 1e-6f;
      acc[0] += a.w * (b.x / nr);
      acc[1] += a.w * (b.y / nr);
      acc[2] += a.w * (b.z / nr);
      const float t = (a.x - start[0]) * dir[0] + (a.y - start[1]) * dir[1] + (a.z - start[2]) * dir[2];
      const float sid = rintf(t / G.stepdist);
      acc[3] += (a.w * sid) * G.stepdist;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int off = SEG / 2; off >= 1; off >>= 1) acc[e] += __shfl_xor(acc[e], off, 64);
    if (ok && sl == 0) {
      if (normal)
        for (int e = 0; e < 3; ++e) normal[3 * r + e] = acc[e];
      if (depth) depth[r] = acc[3];
    }
  }
}

static int voxurf_desc(VoxurfRowDesc& D, const FusedGeom& G, const int* cfg, const float* disp) {
  // cfg = {pos_pe, view_pe, k_view_pe, nd, xstride, kstride}
  D.pos_pe = cfg[0];
  D.view_pe = cfg[1];
  D.k_view_pe = cfg[2];
  D.nd = cfg[3];
  D.xstride = cfg[4];
  D.kstride = cfg[5];
  VX_CHECK_ARG(D.nd >= 1 && D.nd <= kVxMaxDisp, "voxurf rows: 1 to %d displacements", kVxMaxDisp);
  VX_CHECK_ARG(D.pos_pe >= 0 && D.pos_pe <= 16 && D.view_pe >= 0 && D.view_pe <= 16 &&
                   D.k_view_pe >= 0 && D.k_view_pe <= 16,
               "voxurf rows: PE frequencies out of range");
  for (int i = 0; i < D.nd; ++i) {
    VX_CHECK_ARG(disp[i] > 0.f, "voxurf rows: displacements must be positive");
    D.disp[i] = disp[i];
  }
  for (int i = D.nd; i < kVxMaxDisp; ++i) D.disp[i] = 0.f;
  D.x_view = 3 + 6 * D.pos_pe;
  D.x_sdf = D.x_view + 3 + 6 * D.view_pe;
  D.x_feat = D.x_sdf + 1;
  D.x_grad = D.x_feat + 6 * D.nd;
  D.x_end = D.x_grad + 3 * D.nd;
  D.k_pos = G.gk.C;
  D.k_view = D.k_pos + 3 + 6 * D.pos_pe;
  D.k_grad = D.k_view + 3 + 6 * D.k_view_pe;
  D.k_logit = D.k_grad + 3;
  D.k_end = D.k_logit + 3;
  VX_CHECK_ARG(D.x_end <= D.xstride && D.xstride % 4 == 0 && D.xstride <= 128,
               "voxurf rows: rgbnet row (%d columns) does not fit xstride %d", D.x_end, D.xstride);
  VX_CHECK_ARG(D.k_end <= D.kstride && D.kstride % 4 == 0 && D.kstride <= 64,
               "voxurf rows: k_rgbnet row (%d columns) does not fit kstride %d", D.k_end, D.kstride);
  VX_CHECK_ARG(G.gs.C == 1, "voxurf rows: the SDF grid must have one channel");
  VX_CHECK_ARG(G.gk.C >= 1 && G.gk.C <= 16, "voxurf rows: 1 to 16 k0 channels");
  return VX_OK;
}

}  // namespace vx

using namespace vx;

extern "C" {

int vx_voxurf_gather(const float* sdf, const int64_t* sdf_geom, const float* k0,
                     const int64_t* k0_geom, const float* box, const float* params,
                     const int* row_cfg, const float* disp, const float* viewdirs,
                     int64_t n_rays, int cap, const void* s4, const void* g4, const int* stats,
                     const int64_t* cnt, const int64_t* off_incl, int64_t max_rows, float* X,
                     float* XK, void* P4, void* G4, int* rid, void* stream) {
  FusedGeom G;
  if (int st = fused_geom(G, sdf, sdf_geom, k0, k0_geom, box, params)) return st;
  VoxurfRowDesc D;
  if (int st = voxurf_desc(D, G, row_cfg, disp)) return st;
  VX_CHECK_ARG(cap >= 1 && n_rays >= 0, "voxurf_gather: bad sizes");
  if (n_rays == 0) return VX_OK;
  hipStream_t st = (hipStream_t)stream;
  launch_survivors(G, viewdirs, n_rays, cap, s4, g4, stats, cnt, off_incl, max_rows, P4, G4, rid,
                   nullptr, st);
  if (max_rows > 0)
    k_voxurf_rows<<<grid_for(max_rows, kVxRowTile, 1 << 12), 256,
                    kVxRowTile * (D.xstride + D.kstride) * 4, st>>>(
        G, D, viewdirs, n_rays, off_incl, max_rows, X, XK, (const float4*)P4, (const float4*)G4, rid);
  return launch_status("voxurf_gather");
}

int vx_voxurf_logit_cols(int64_t m, const int64_t* m_dev, const float* logits, float* XK,
                         int kstride, int col, void* stream) {
  VX_CHECK_ARG(m >= 0 && col >= 0 && col + 3 <= kstride, "voxurf_logit_cols: bad sizes");
  if (m == 0) return VX_OK;
  k_voxurf_logit_cols<<<grid_for(3 * m, 256), 256, 0, (hipStream_t)stream>>>(m, m_dev, logits, XK,
                                                                            kstride, col);
  return launch_status("voxurf_logit_cols");
}

int vx_voxurf_composite(int64_t n_rays, const int64_t* cnt, const int64_t* off_incl,
                        const float* logits, const float* k_logits, const void* P4,
                        const float* last, const float* target, float bg, float w_main,
                        float w_rgb0, float w_ent, float* rgb, float* rgb0, float* dlogit0,
                        float* dlogitk, float* gw, float* glast, float* S, float* loss_r,
                        int64_t max_rows, void* stream) {
  VX_CHECK_ARG(n_rays >= 0, "voxurf_composite: n_rays < 0");
  if (n_rays == 0) return VX_OK;
  const float inv_count = 1.f / (3.f * (float)n_rays);
  k_voxurf_composite<<<grid_for(n_rays, 16, 1 << 16), 256, 0, (hipStream_t)stream>>>(
      n_rays, cnt, off_incl, logits, k_logits, (const float4*)P4, last, target, bg, inv_count,
      w_main, w_rgb0, w_ent, rgb, rgb0, dlogit0, dlogitk, gw, glast, S, loss_r, max_rows);
  return launch_status("voxurf_composite");
}

int vx_voxurf_feat_bwd(const float* sdf, const int64_t* sdf_geom, const int64_t* k0_geom,
                       const float* box, const float* params, const int* row_cfg,
                       const float* disp, int64_t m, const int64_t* m_dev, const float* dX,
                       const float* dXK, const void* P4, float* k0_grad, float* sdf_grad,
                       float* dgf, float* dsf, void* stream) {
  FusedGeom G;
  if (int st = fused_geom(G, sdf, sdf_geom, nullptr, k0_geom, box, params)) return st;
  VoxurfRowDesc D;
  if (int st = voxurf_desc(D, G, row_cfg, disp)) return st;
  VX_CHECK_ARG(m >= 0, "voxurf_feat_bwd: m < 0");
  if (m == 0) return VX_OK;
  k_voxurf_feat_bwd<<<grid_for(m, 16, 1 << 16), 256, 0, (hipStream_t)stream>>>(
      G, D, m, m_dev, dX, dXK, (const float4*)P4, k0_grad, sdf_grad, dgf, dsf);
  return launch_status("voxurf_feat_bwd");
}

int vx_fused_render_extras(const float* box, const float* params, int64_t n_rays,
                           const int64_t* cnt, const int64_t* off_incl, const void* P4,
                           const void* G4, const float* rays_o, const float* rays_d,
                           float* normal, float* depth, int64_t max_rows, void* stream) {
  FusedGeom G;
  const int64_t geom[8] = {1, 1, 1, 1, 1, 1, 1, 1};
  if (int st = fused_geom(G, nullptr, geom, nullptr, nullptr, box, params)) return st;
  VX_CHECK_ARG(n_rays >= 0, "fused_render_extras: n_rays < 0");
  if (n_rays == 0) return VX_OK;
  k_render_extras<<<grid_for(n_rays, 16, 1 << 16), 256, 0, (hipStream_t)stream>>>(
      G, n_rays, cnt, off_incl, (const float4*)P4, (const float4*)G4, rays_o, rays_d, normal,
      depth, max_rows);
  return launch_status("fused_render_extras");
}

}  // extern "C"
