// Per-ray geometry shared by the fine-stage kernels: the SDF / feature grid
// descriptors, the bounding box and sampling constants, and the optional MaskCache
// (coarse occupancy) test, with the host helpers that fill them from the C-ABI arguments.
#pragma once
#include "voxel.h"

namespace vx {

struct FusedGeom {
  const float* sdf;       // [X, Y, Z] contiguous
  GridDesc gs;
  const float* k0;        // [C, X, Y, Z] with strides
  GridDesc gk;
  float mn[3], mx[3];
  float stepdist, voxel_size, inv_s, thres, near_, far_;
  // optional MaskCache (coarse occupancy); mc == nullptr disables it
  const float* mc;
  GridDesc gm;
  float mc_shift, mc_ratio, mc_thres, mc_mn[3], mc_mx[3];
  int mc_nearest;
  // optional empty-space bounds (vx_sdf_skip_bounds): per brick of 8^3 cells, a lower
  // bound on the SDF and an upper bound on the length of its central-difference gradient
  // over every voxel a sample in the brick can read; skip == nullptr disables skipping
  const float4* skip;
  int skx, sky, skz;
  float skip_xmin;
  float skip_scale[3];  // voxels per world unit
};

constexpr int kSkipShift = 3;  // empty-space bricks of 8^3 cells

// Empty space along a ray, eight steps at a time.  A sample provably has NeuS alpha <= thres,
// so that it takes no part in the walk (lib/voxurf_fine.py keeps alpha > thres only), when with
// c = sigmoid(prev inv_s), n = sigmoid(next inv_s), alpha = (c - n + 1e-5) / (c + 1e-5) and
// next = sdf - |h| <= prev, |h| = |cos| dist / 2 <= |viewdir| |grad| dist / 2, next inv_s >=
// x_min = ln(1 / (thres - 2e-5)) + 1: c - n <= e^-x_min (plus float rounding) and alpha stays
// below thres.
//
// A brick's bounds on the SDF and its gradient hold over the voxels from 8 below its first
// cell to 8 above its last, and a sample reads from 2 below its cell to 3 above it: they hold
// for every sample within five cells of the brick.  So the brick of the fifth of eight steps
// speaks for all eight while four steps are no longer than 4.5 voxels along any axis (the
// index of that step need not be exact either).
constexpr int kSkipGroup = 8;
struct SkipRay {
  float b[3], a[3];  // index of step s along axis k: b + a s
  float hfac;        // |viewdir| dist / 2 (with a margin)
  bool on, eights;   // empty space is known; eight steps at a time
};

__device__ __forceinline__ void skip_ray(const FusedGeom& G, const float start[3],
                                         const float dir[3], const float* vd, SkipRay& k) {
  k.on = k.eights = false;
  if (!G.skip) return;
  k.on = true;
  k.hfac = sqrtf(vd[0] * vd[0] + vd[1] * vd[1] + vd[2] * vd[2]) * G.stepdist * 0.5f * (1.f + 1e-4f);
  float longest = 0.f;
  for (int e = 0; e < 3; ++e) {
    k.b[e] = (start[e] - G.mn[e]) * G.skip_scale[e];
    k.a[e] = dir[e] * G.stepdist * G.skip_scale[e];
    longest = fmaxf(longest, fabsf(k.a[e]));
  }
  k.eights = longest * (kSkipGroup / 2) <= 4.5f;
}

__device__ __forceinline__ bool skip_at(const FusedGeom& G, const SkipRay& k, int64_t step) {
  const float s = (float)(int)step;
  const int bx = min(max(sat_f2i(floorf(fmaf(k.a[0], s, k.b[0]))) >> kSkipShift, 0), G.skx - 1);
  const int by = min(max(sat_f2i(floorf(fmaf(k.a[1], s, k.b[1]))) >> kSkipShift, 0), G.sky - 1);
  const int bz = min(max(sat_f2i(floorf(fmaf(k.a[2], s, k.b[2]))) >> kSkipShift, 0), G.skz - 1);
  const float4 b = G.skip[((int64_t)bx * G.sky + by) * G.skz + bz];
  return (b.x * (1.f - 1e-6f) - k.hfac * b.y) * G.inv_s >= G.skip_xmin;
}

// MaskCache.forward for one point (lib/voxurf_fine.py:930-942), as vx_maskcache_alpha: the
// density at a continuous index of the cache's grid, and whether its alpha passes.
__device__ __forceinline__ void maskcache_index(const FusedGeom& G, const float q[3], float f[3]) {
  f[0] = world_to_index(q[0], G.mc_mn[0], G.mc_mx[0] - G.mc_mn[0], G.gm.X);
  f[1] = world_to_index(q[1], G.mc_mn[1], G.mc_mx[1] - G.mc_mn[1], G.gm.Y);
  f[2] = world_to_index(q[2], G.mc_mn[2], G.mc_mx[2] - G.mc_mn[2], G.gm.Z);
}

__device__ __forceinline__ float maskcache_density(const FusedGeom& G, const float f[3]) {
  if (G.mc_nearest) {
    const int x = sat_f2i(rintf(f[0])), y = sat_f2i(rintf(f[1])), z = sat_f2i(rintf(f[2]));
    return in_grid<float>(x, y, z, G.gm) ? G.mc[x * G.gm.sx + y * G.gm.sy + z * G.gm.sz] : 0.f;
  }
  Tri<float> t;
  t.init(f[0], f[1], f[2]);
  return tri_gather(G.mc, G.gm, t, 0);
}

__device__ __forceinline__ bool maskcache_alpha_pass(const FusedGeom& G, float d) {
#pragma clang fp contract(off)
  const float x = d + G.mc_shift;
  const float sp = x > 20.f ? x : log1pf(expf(x));
  return 1.f - expf(-sp * G.mc_ratio) >= G.mc_thres;
}

__device__ __forceinline__ bool maskcache_pass(const FusedGeom& G, const float q[3]) {
  float f[3];
  maskcache_index(G, q, f);
  return maskcache_alpha_pass(G, maskcache_density(G, f));
}

__device__ __forceinline__ void ray_setup(const FusedGeom& G, const float* o, const float* d,
                                          float* start, float* dir, int64_t& n) {
  float tmin, tmax;
  ray_t_minmax<float>(o, d, G.mn, G.mx, G.near_, G.far_, tmin, tmax);
  n = ray_n_samples<float>(d, tmin, tmax, G.stepdist);
  ray_start_dir<float>(o, d, tmin, start, dir);
}

__device__ __forceinline__ uint64_t lanemask_lt(int lane) {
  return lane ? ((~0ull) >> (64 - lane)) : 0ull;
}

// Alpha and weight of a stored walk-range sample, recomputed with the forward's own
// arithmetic (bit-identical to the walk's values).
struct SlotSample {
  float q[3], grad[3], sdf, myT, alpha, w;
  NeusFwd<float> nf;
};

__device__ __forceinline__ void load_slot(const FusedGeom& G, const float* vd, float4 a, float4 b,
                                          SlotSample& ss) {
#pragma clang fp contract(off)
  ss.q[0] = a.x;
  ss.q[1] = a.y;
  ss.q[2] = a.z;
  ss.myT = a.w;
  ss.grad[0] = b.x;
  ss.grad[1] = b.y;
  ss.grad[2] = b.z;
  ss.sdf = b.w;
  ss.nf = neus_fwd<float>(vd, ss.grad, ss.sdf, G.stepdist, G.inv_s);
  ss.alpha = clip01(ss.nf.a);
  ss.w = ss.myT * ss.alpha;
}

// Host side: fill a FusedGeom from the C-ABI arguments.
static inline int fused_geom(FusedGeom& G, const float* sdf, const int64_t* sdf_geom,
                             const float* k0, const int64_t* k0_geom, const float* box,
                             const float* params) {
  // box = {mn x,y,z, mx x,y,z}; params = {stepdist, voxel_size, inv_s, thres, near, far}
  G.sdf = sdf;
  G.k0 = k0;
  auto desc = [](const int64_t* s, GridDesc& g) {
    g.C = (int)s[0];
    g.X = (int)s[1];
    g.Y = (int)s[2];
    g.Z = (int)s[3];
    g.sc = s[4];
    g.sx = s[5];
    g.sy = s[6];
    g.sz = s[7];
  };
  desc(sdf_geom, G.gs);
  if (k0_geom) desc(k0_geom, G.gk);
  else G.gk = G.gs;
  VX_CHECK_ARG(G.gs.C == 1, "fused: the SDF grid must have one channel");
  for (int i = 0; i < 3; ++i) {
    G.mn[i] = box[i];
    G.mx[i] = box[3 + i];
  }
  G.stepdist = params[0];
  G.voxel_size = params[1];
  G.inv_s = params[2];
  G.thres = params[3];
  G.near_ = params[4];
  G.far_ = params[5];
  G.mc = nullptr;
  G.skip = nullptr;
  G.skx = G.sky = G.skz = 0;
  G.skip_xmin = 0.f;
  return VX_OK;
}

// Empty-space bounds of vx_sdf_skip_bounds for this SDF grid (may be NULL: no skipping).
// Skipping needs thres > 2.5e-5 (the bound leaves alpha below thres only then) and
// inv_s > 0; otherwise the bounds are ignored.
static inline void fused_skip(FusedGeom& G, const void* bounds) {
  G.skip = nullptr;
  if (!bounds || !(G.thres > 2.5e-5f) || !(G.inv_s > 0.f)) return;
  G.skip = static_cast<const float4*>(bounds);
  G.skx = (G.gs.X + (1 << kSkipShift) - 1) >> kSkipShift;
  G.sky = (G.gs.Y + (1 << kSkipShift) - 1) >> kSkipShift;
  G.skz = (G.gs.Z + (1 << kSkipShift) - 1) >> kSkipShift;
  G.skip_xmin = logf(1.f / (G.thres - 2e-5f)) + 1.f;
  const int size[3] = {G.gs.X, G.gs.Y, G.gs.Z};
  for (int e = 0; e < 3; ++e) G.skip_scale[e] = (float)(size[e] - 1) / (G.mx[e] - G.mn[e]);
}

// mc_params = {act_shift, voxel_size_ratio, thres, nearest, xyz_min[3], xyz_max[3]}
static inline int fused_maskcache(FusedGeom& G, const float* mc, const int64_t* mc_geom,
                                  const float* mc_params) {
  if (!mc) return VX_OK;
  VX_CHECK_ARG(mc_geom && mc_params, "fused: mask cache geometry/parameters missing");
  G.mc = mc;
  G.gm.C = (int)mc_geom[0];
  G.gm.X = (int)mc_geom[1];
  G.gm.Y = (int)mc_geom[2];
  G.gm.Z = (int)mc_geom[3];
  G.gm.sc = mc_geom[4];
  G.gm.sx = mc_geom[5];
  G.gm.sy = mc_geom[6];
  G.gm.sz = mc_geom[7];
  VX_CHECK_ARG(G.gm.C == 1, "fused: the mask-cache density must have one channel");
  G.mc_shift = mc_params[0];
  G.mc_ratio = mc_params[1];
  G.mc_thres = mc_params[2];
  G.mc_nearest = mc_params[3] != 0.f;
  for (int i = 0; i < 3; ++i) {
    G.mc_mn[i] = mc_params[4 + i];
    G.mc_mx[i] = mc_params[7 + i];
  }
  return VX_OK;
}

// Survivor rows P4 = (x, y, z, weight), G4 = (gradient, sdf), rid of the walk-range slots
// (k_survivors in fused.hip); n_rays > 0.
void launch_survivors(const FusedGeom& G, const float* viewdirs, int64_t n_rays, int cap,
                      const void* s4, const void* g4, const int* stats, const int64_t* cnt,
                      const int64_t* off_incl, int64_t max_rows, void* P4, void* G4, int* rid,
                      uint32_t* pages, hipStream_t st);

}  // namespace vx
