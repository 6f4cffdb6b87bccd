// Camera rays and the MaskCache ray pre-filter of the fine stage (gfx950).
//
// get_rays_of_a_view (lib/voxurf_fine.py:1001-1068) builds the rays of one pinhole view
// with ~15 full-image torch passes; here one thread makes one pixel's ray in registers.
// hit_coarse_geo (lib/voxurf_fine.py:579-591) samples every step of every ray, then looks
// up the MaskCache at every in-box point and scatters the hits; here one thread walks one
// ray, jumps over the bricks of the coarse grid in which no sample can pass, and stops at the
// first step that passes the mask; few rays take a wavefront each, 64 steps at a time, until
// one passes.
// get_training_rays_in_maskcache_sampling (lib/voxurf_fine.py:1127-1164) becomes, per
// view: hit flags straight from the camera (no ray arrays), an inclusive scan, and a
// compaction that rebuilds the kept rays with the same arithmetic and writes them in
// pixel order, as the reference's boolean indexing does.
#include <math.h>

#include "fine.h"

namespace vx {

struct Camera {
  int H, W;
  float fx, fy, cx, cy;  // K[0][0], K[1][1], K[0][2], K[1][2]
  float R[9];            // c2w[:3, :3], row-major
  float t[3];            // c2w[:3, 3]
  float off;             // 0.5 (pixel centres) or 0 (left-top corners)
  int inverse_y, flip_x, flip_y;
  int ndc;
  float ndc_c0, ndc_c1, ndc_near;  // -1/(W/(2 focal)), -1/(H/(2 focal)), near plane
};

// NDC warp of one ray (lib/voxurf_fine.py:1042-1059), in the reference's operation
// order: shift the origin to z = -near, then project.
__device__ __forceinline__ void ndc_ray(float c0, float c1, float near_, float o[3], float d[3]) {
#pragma clang fp contract(off)
  const float t = -(near_ + o[2]) / d[2];
  const float ox = o[0] + t * d[0], oy = o[1] + t * d[1], oz = o[2] + t * d[2];
  const float o0 = c0 * ox / oz;
  const float o1 = c1 * oy / oz;
  const float o2 = 1.f + 2.f * near_ / oz;
  const float d0 = c0 * (d[0] / d[2] - ox / oz);
  const float d1 = c1 * (d[1] / d[2] - oy / oz);
  const float d2 = -2.f * near_ / oz;
  o[0] = o0;
  o[1] = o1;
  o[2] = o2;
  d[0] = d0;
  d[1] = d1;
  d[2] = d2;
}

// Ray of pixel (row, col) (lib/voxurf_fine.py:1001-1029, 1062-1068): camera-frame
// direction from the pixel coordinate, rotated by c2w (sum of the three products in
// index order), viewdir = d / |d| before the optional NDC warp.
__device__ __forceinline__ void camera_ray(const Camera& c, int row, int col, float o[3],
                                           float d[3], float v[3]) {
#pragma clang fp contract(off)
  const float i = (float)(c.flip_x ? c.W - 1 - col : col) + c.off;
  const float j = (float)(c.flip_y ? c.H - 1 - row : row) + c.off;
  float dir[3];
  dir[0] = (i - c.cx) / c.fx;
  if (c.inverse_y) {
    dir[1] = (j - c.cy) / c.fy;
    dir[2] = 1.f;
  } else {
    dir[1] = -((j - c.cy) / c.fy);
    dir[2] = -1.f;
  }
  for (int r = 0; r < 3; ++r) {
    d[r] = (dir[0] * c.R[3 * r] + dir[1] * c.R[3 * r + 1]) + dir[2] * c.R[3 * r + 2];
    o[r] = c.t[r];
  }
  const float nrm = sqrtf((d[0] * d[0] + d[1] * d[1]) + d[2] * d[2]);
  v[0] = d[0] / nrm;
  v[1] = d[1] / nrm;
  v[2] = d[2] / nrm;
  if (c.ndc) ndc_ray(c.ndc_c0, c.ndc_c1, c.ndc_near, o, d);
}

__global__ void __launch_bounds__(256) k_camera_rays(Camera c, float* __restrict__ rays_o,
                                                     float* __restrict__ rays_d,
                                                     float* __restrict__ viewdirs) {
  const int64_t n = (int64_t)c.H * c.W;
  for (int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; p < n;
       p += (int64_t)gridDim.x * blockDim.x) {
    float o[3], d[3], v[3];
    camera_ray(c, (int)(p / c.W), (int)(p % c.W), o, d, v);
    for (int k = 0; k < 3; ++k) {
      rays_o[3 * p + k] = o[k];
      rays_d[3 * p + k] = d[k];
      viewdirs[3 * p + k] = v[k];
    }
  }
}

__global__ void __launch_bounds__(256) k_ndc_rays(int64_t n, float c0, float c1, float near_,
                                                  const float* __restrict__ o_in,
                                                  const float* __restrict__ d_in,
                                                  float* __restrict__ o_out,
                                                  float* __restrict__ d_out) {
  for (int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; p < n;
       p += (int64_t)gridDim.x * blockDim.x) {
    float o[3] = {o_in[3 * p], o_in[3 * p + 1], o_in[3 * p + 2]};
    float d[3] = {d_in[3 * p], d_in[3 * p + 1], d_in[3 * p + 2]};
    ndc_ray(c0, c1, near_, o, d);
    for (int k = 0; k < 3; ++k) {
      o_out[3 * p + k] = o[k];
      d_out[3 * p + k] = d[k];
    }
  }
}

// ---- occupancy of the MaskCache -----------------------------------------------------------
// Bricks of 2^shift cells of the cache's grid (cells 0 .. X - 2 of an axis), of 4 x 4 x 4
// blocks each.  A block's bit is clear when the density of every lattice point of its cells
// is below d_clear, under which no interpolated density passes: alpha rises with the density,
// and an interpolation stays below the largest of its corners.  A sample that rounding puts
// past the grid by up to `margin` cells mixes in a little of the 0 read there, which
// d_clear <= d_lo allows for; samples further out are always looked up.  d_lo and d_hi come
// from inverting alpha(d) = thres in double with a margin far above the float formula's
// error, so that the float test itself decides between them and only there.
struct Occupancy {
  const uint32_t* bits;      // brick has a block that may pass; nullptr: not known
  const uint32_t* near;      // it or one of the 26 around it has
  const uint64_t* blocks;    // its blocks: bit 16 x + 4 y + z
  int shift, bx, by, bz;     // bricks per axis
  float d_lo, d_hi;          // densities below / above which the test is known
  float d_clear;             // densities of clear blocks lie below
  int inner;                 // the scene's box lies in the cache's
  float margin[3];           // cells by which a sample's index may be off the straight line
};

constexpr int kOccShift = 2;             // bricks of 4^3 cells (at least)
constexpr int kOccMaxBits = 1 << 17;     // twice 16 KB of LDS

// One workgroup per word of 32 bricks, a wave per two of them, a lane per block of a brick.
__global__ void __launch_bounds__(1024) k_occupancy(const float* __restrict__ mc, GridDesc g,
                                                    Occupancy oc, uint32_t* __restrict__ bits,
                                                    uint64_t* __restrict__ blocks) {
  __shared__ uint32_t word;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (threadIdx.x == 0) word = 0u;
  __syncthreads();
  const int sub = 1 << (oc.shift - 2);   // cells per block and axis
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const int b = blockIdx.x * 32 + wave * 2 + e;
    if (b >= oc.bx * oc.by * oc.bz) break;
    const int z0 = ((b % oc.bz) << oc.shift) + (lane & 3) * sub,
              y0 = ((b / oc.bz % oc.by) << oc.shift) + (lane >> 2 & 3) * sub,
              x0 = ((b / (oc.bz * oc.by)) << oc.shift) + (lane >> 4) * sub;
    bool any = false;
    for (int dx = 0; dx <= sub; ++dx)
      for (int dy = 0; dy <= sub; ++dy)
        for (int dz = 0; dz <= sub; ++dz) {
          const int x = x0 + dx, y = y0 + dy, z = z0 + dz;
          if (in_grid<float>(x, y, z, g)) any |= !(mc[x * g.sx + y * g.sy + z * g.sz] < oc.d_clear);
        }
    const uint64_t m = __ballot(any);
    if (lane == 0) {
      blocks[b] = m;
      if (m) atomicOr(&word, 1u << (wave * 2 + e));
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) bits[blockIdx.x] = word;
}

// near[brick]: a set bit among the brick and the 26 around it.  One thread per brick.
__global__ void __launch_bounds__(256) k_occupancy_near(Occupancy oc, const uint32_t* __restrict__ bits,
                                                        uint32_t* __restrict__ near) {
  const int nb = oc.bx * oc.by * oc.bz, b = blockIdx.x * 256 + threadIdx.x;
  bool any = false;
  if (b < nb) {
    const int z = b % oc.bz, y = b / oc.bz % oc.by, x = b / (oc.bz * oc.by);
#pragma unroll
    for (int k = 0; k < 27; ++k) {
      const int i = min(max(x + k / 9 - 1, 0), oc.bx - 1), j = min(max(y + k / 3 % 3 - 1, 0), oc.by - 1),
                l = min(max(z + k % 3 - 1, 0), oc.bz - 1);
      const int id = (i * oc.by + j) * oc.bz + l;
      any |= bits[id >> 5] >> (id & 31) & 1u;
    }
  }
  const uint64_t m = __ballot(any);
  if ((threadIdx.x & 63) == 0) {
    const int w = b >> 5, words = (nb + 31) >> 5;
    if (w < words) near[w] = (uint32_t)m;
    if (w + 1 < words) near[w + 1] = (uint32_t)(m >> 32);
  }
}

// Does any in-box sample of the ray pass the MaskCache?  Samples exactly as
// sample_pts_on_rays.  The wave looks 64 at a time up and leaves at the first chunk that
// holds a passing one.
__device__ __forceinline__ bool wave_hits(const FusedGeom& G, const float* o, const float* d,
                                          int lane) {
  float start[3], dir[3];
  int64_t n;
  ray_setup(G, o, d, start, dir, n);
  for (int64_t base = 0; base < n; base += 64) {
    const int64_t s = base + lane;
    bool pass = false;
    if (s < n) {
      float q[3];
      if (!sample_point<float>(start, dir, G.mn, G.mx, G.stepdist, s, q[0], q[1], q[2]))
        pass = maskcache_pass(G, q);
    }
    if (__ballot(pass)) return true;
  }
  return false;
}

// One wavefront per ray: hit (bool bytes) and/or flag (int64 0/1) per ray.
__global__ void __launch_bounds__(256) k_hit_rays_wave(FusedGeom G, const float* __restrict__ rays_o,
                                                       const float* __restrict__ rays_d,
                                                       int64_t n_rays, uint8_t* __restrict__ hit,
                                                       int64_t* __restrict__ flag) {
  const int lane = threadIdx.x & 63;
  const int64_t waves = (int64_t)gridDim.x * (blockDim.x >> 6);
  for (int64_t r = blockIdx.x * (int64_t)(blockDim.x >> 6) + (threadIdx.x >> 6); r < n_rays;
       r += waves) {
    const bool h = wave_hits(G, rays_o + 3 * r, rays_d + 3 * r, lane);
    if (lane == 0) {
      if (hit) hit[r] = h;
      if (flag) flag[r] = h;
    }
  }
}

// The same for a view, each pixel's ray made by every lane of its wave (a few dozen flops,
// cheaper than a broadcast).
__global__ void __launch_bounds__(256) k_hit_camera_wave(FusedGeom G, Camera c,
                                                         int64_t* __restrict__ flag) {
  const int lane = threadIdx.x & 63;
  const int64_t n = (int64_t)c.H * c.W;
  const int64_t waves = (int64_t)gridDim.x * (blockDim.x >> 6);
  for (int64_t p = blockIdx.x * (int64_t)(blockDim.x >> 6) + (threadIdx.x >> 6); p < n; p += waves) {
    float o[3], d[3], v[3];
    camera_ray(c, (int)(p / c.W), (int)(p % c.W), o, d, v);
    const bool h = wave_hits(G, o, d, lane);
    if (lane == 0) flag[p] = h;
  }
}

// The same question with occupancy bits, a thread a ray: a sample is looked up only where its
// block's bit is set or the block is in doubt: the walk follows the straight line through the cache's
// grid, which a sample's own index is off by less than `margin` cells, and from a sample
// inside a clear brick or block by more than that it goes on with the first one that is not.
// A lookup on that line decides too, unless the margin could change the answer: then the
// sample's own index and the cache's own formula do.  Steps s0 .. n - 1.  Bound by instruction issue (the bits
// are in LDS, the densities in L2), so the walk is free of branches: with them, and with the
// exact lookup for every candidate, the same walk took 1,470 us for the view below.
__device__ __forceinline__ bool ray_hits(const FusedGeom& G, const Occupancy& oc,
                                         const uint32_t* bits, const float* start,
                                         const float* dir, int64_t s0, int64_t n) {
  const int size[3] = {G.gm.X, G.gm.Y, G.gm.Z};
  // index of the line at the first step, cells per step, steps per cell; the margin at the
  // side where it leaves a box
  float p0[3], rate[3], inv[3], far[3];
  bool line = n < (1 << 24);  // (float) s is exact
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const float cells = (float)(size[a] - 1) / (G.mc_mx[a] - G.mc_mn[a]);
    p0[a] = (start[a] - G.mc_mn[a]) * cells;
    rate[a] = dir[a] * G.stepdist * cells;
    // an axis the line hardly moves along is never left; the sign of inf / inf is the rate's
    inv[a] = fabsf(rate[a]) > 1e-20f ? 1.f / rate[a] : (rate[a] < 0.f ? -1e20f : 1e20f);
    far[a] = rate[a] < 0.f ? oc.margin[a] : -oc.margin[a];
    line = line && fabsf(p0[a]) < 1e6f && fabsf(rate[a]) < 1e6f;
  }
  const float brick = (float)(1 << oc.shift), rbrick = 1.f / brick;
  const float block = (float)(1 << (oc.shift - 2)), rblock = 1.f / block;
  const float sum_margin = oc.margin[0] + oc.margin[1] + oc.margin[2];
  for (int64_t s = s0; s < n; ++s) {
    float p[3];
    bool known = false;   // the line's cell is the sample's own
    if (line) {
      // the lanes of a wave jump until each has a sample to look up, then look up together
      for (;;) {
        const float sf = (float)(int)s;
        float b[3];
        bool in = true;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          p[a] = fmaf(rate[a], sf, p0[a]);
          in = in && p[a] >= 0.f && p[a] < (float)(size[a] - 1);
          b[a] = floorf(p[a] * rbrick);
        }
        in = in && s < n;
        const int id = in ? ((int)b[0] * oc.by + (int)b[1]) * oc.bz + (int)b[2] : 0;
        const bool set = bits[id >> 5] >> (id & 31) & 1u;
        const float width = set ? block : brick, rwidth = set ? rblock : rbrick;
        float k = 1e6f, c[3];
        bool inside = in;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          c[a] = floorf(p[a] * rwidth);
          const float r = fmaf(-width, c[a], p[a]);   // cells into the box, exact
          // its end, or the grid's
          const float e = fminf(width, fmaf(-width, c[a], (float)(size[a] - 1)));
          inside = inside && r >= oc.margin[a] && r <= e - oc.margin[a];
          k = fminf(k, ((rate[a] < 0.f ? 0.f : e) + far[a] - r) * inv[a]);
        }
        bool clear = !set;
        if (in && set) {
          const int q = ((int)c[0] & 3) << 4 | ((int)c[1] & 3) << 2 | ((int)c[2] & 3);
          clear = !(oc.blocks[id] >> q & 1);
        }
        if (!(inside && clear)) {
          known = inside;
          break;
        }
        s += 1 + (int)fmaxf(k, 0.f);
      }
      if (s >= n) break;
    }
    if (known && !G.mc_nearest && oc.shift == kOccShift) {
      // inside one cell: the line's interpolation, off by at most the margins times the
      // corners' spread
      const int x0 = (int)floorf(p[0]), y0 = (int)floorf(p[1]), z0 = (int)floorf(p[2]);
      const float u = p[0] - floorf(p[0]), v = p[1] - floorf(p[1]), w = p[2] - floorf(p[2]);
      {  // (a known cell lies in the grid)
        const float* g = G.mc + (x0 * G.gm.sx + y0 * G.gm.sy + z0 * G.gm.sz);
        float e[8], lo = INFINITY, hi = -INFINITY;
        bool nan = false;
#pragma unroll
        for (int c = 0; c < 8; ++c) {
          e[c] = g[(c >> 2) * G.gm.sx + (c >> 1 & 1) * G.gm.sy + (c & 1) * G.gm.sz];
          lo = fminf(lo, e[c]);
          hi = fmaxf(hi, e[c]);
          nan = nan || e[c] != e[c];
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) e[c] = e[2 * c] + w * (e[2 * c + 1] - e[2 * c]);
#pragma unroll
        for (int c = 0; c < 2; ++c) e[c] = e[2 * c] + v * (e[2 * c + 1] - e[2 * c]);
        const float dens = e[0] + u * (e[1] - e[0]);
        const float err = (hi - lo) * sum_margin + 4e-6f * fmaxf(fabsf(hi), fabsf(lo));
        if (!nan && err < 1e30f) {
          if (dens - err > oc.d_hi) {
            // the sample passes if it lies in the scene's box
            float q[3];
            if (!sample_point<float>(start, dir, G.mn, G.mx, G.stepdist, s, q[0], q[1], q[2])) return true;
            continue;
          }
          if (dens + err < oc.d_lo) continue;
        }
      }
    }
    float q[3], f[3];
    if (sample_point<float>(start, dir, G.mn, G.mx, G.stepdist, s, q[0], q[1], q[2])) continue;
    maskcache_index(G, q, f);
    const float dens = maskcache_density(G, f);
    if (dens > oc.d_hi) return true;
    if (!(dens < oc.d_lo) && maskcache_alpha_pass(G, dens)) return true;
  }
  return false;
}

// The workgroup's copy of `words` (dynamic LDS from word `at`).
__device__ __forceinline__ const uint32_t* occ_to_lds(const uint32_t* words, int n, int at) {
  extern __shared__ uint32_t occ_lds[];
  for (int i = threadIdx.x; i < n; i += blockDim.x) occ_lds[at + i] = words[i];
  return occ_lds + at;
}

// One thread per ray: hit (bool bytes) and/or flag (int64 0/1) per ray.
__global__ void __launch_bounds__(256) k_hit_rays(FusedGeom G, Occupancy oc,
                                                  const float* __restrict__ rays_o,
                                                  const float* __restrict__ rays_d, int64_t n_rays,
                                                  uint8_t* __restrict__ hit,
                                                  int64_t* __restrict__ flag) {
  const int words = (oc.bx * oc.by * oc.bz + 31) >> 5;
  const uint32_t* bits = occ_to_lds(oc.bits, words, 0);
  __syncthreads();
  for (int64_t r = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; r < n_rays;
       r += (int64_t)gridDim.x * blockDim.x) {
    const float o[3] = {rays_o[3 * r], rays_o[3 * r + 1], rays_o[3 * r + 2]};
    const float d[3] = {rays_d[3 * r], rays_d[3 * r + 1], rays_d[3 * r + 2]};
    float start[3], dir[3];
    int64_t n;
    ray_setup(G, o, d, start, dir, n);
    const bool h = ray_hits(G, oc, bits, start, dir, 0, n);
    if (hit) hit[r] = h;
    if (flag) flag[r] = h;
  }
}

// The same, with each pixel's ray made by its thread; a wave takes 8 x 8 pixels.  The rays of
// a pinhole camera's tile stay close together: the 64 lanes first look at 64 stretches of the
// tile's middle ray, each whether the bricks around it are clear (`near`) as far as the
// tile's rays reach, and the walks cover only what lies between the first and the last
// stretch in doubt -- nothing, for most tiles beside the object.
// Measured on 1.92 M rays of a 1200 x 1600 view at half-voxel steps of 256^3: a wavefront per
// ray that looked every sample up (64 at a time, eight loads, exp and log1p each) 5,480 us;
// a thread per ray jumping over clear bricks and blocks 1,200 us (410 M vector instructions,
// 140 jumps a wave); with the tiles' stretches 614 us (205 M).  Five waves a SIMD: with the
// registers for four the view took 30 us longer.
__global__ void __launch_bounds__(256, 5) k_hit_camera(FusedGeom G, Occupancy oc, Camera c,
                                                    int64_t* __restrict__ flag) {
  const int words = (oc.bx * oc.by * oc.bz + 31) >> 5;
  const uint32_t* bits = occ_to_lds(oc.bits, words, 0);
  const uint32_t* near = occ_to_lds(oc.near, words, words);
  __syncthreads();
  const int tw = (c.W + 7) >> 3, th = (c.H + 7) >> 3, lane = threadIdx.x & 63;
  const int64_t waves = (int64_t)gridDim.x * (blockDim.x >> 6);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  for (int64_t t = (int64_t)blockIdx.x * (blockDim.x >> 6) + wave; t < (int64_t)tw * th; t += waves) {
    const int tr = (int)((uint32_t)t / (uint32_t)tw), tc = (int)(t - (int64_t)tr * tw);
    // (pixels past the edge repeat the edge's, so that every lane takes part)
    const int row = tr * 8 + (lane >> 3), col = tc * 8 + (lane & 7);
    float o[3], d[3], v[3], start[3], dir[3];
    camera_ray(c, min(row, c.H - 1), min(col, c.W - 1), o, d, v);
    int64_t n, s0 = 0;
    ray_setup(G, o, d, start, dir, n);
    if (oc.inner && !c.ndc) {
      // distances from the camera at which this ray's samples begin and end
      float t0 = 0.f, dev = 0.f, mid[3];
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        t0 = fmaf(start[a] - o[a], dir[a], t0);
        mid[a] = __shfl(dir[a], 36, 64);
        dev += fabsf(dir[a] - mid[a]);
      }
      const float t1 = t0 + (float)n * G.stepdist;
      float lo = t0, hi = t1, far = dev;
#pragma unroll
      for (int k = 1; k < 64; k <<= 1) {
        lo = fminf(lo, __shfl_xor(lo, k, 64));
        hi = fmaxf(hi, __shfl_xor(hi, k, 64));
        far = fmaxf(far, __shfl_xor(far, k, 64));
      }
      const float len = (hi - lo) * (1.f / 64.f), at = lo + ((float)lane + 0.5f) * len;
      const float reach = 0.51f * len + far * fmaxf(fabsf(lo), fabsf(hi));
      const int size[3] = {G.gm.X, G.gm.Y, G.gm.Z};
      const int nb[3] = {oc.bx, oc.by, oc.bz};
      const float brick = (float)(1 << oc.shift);
      bool doubt = false;
      int b[3];
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        const float cells = (float)(size[a] - 1) / (G.mc_mx[a] - G.mc_mn[a]);
        // (the rays' samples lie in the grid, whatever their surroundings)
        const float p = fminf(fmaxf((o[a] + mid[a] * at - G.mc_mn[a]) * cells, 0.f), (float)(size[a] - 1));
        doubt = doubt || !(reach * fabsf(cells) + oc.margin[a] + 0.01f < brick);
        b[a] = min((int)(p / brick), nb[a] - 1);
      }
      if (!doubt) {
        const int id = (b[0] * oc.by + b[1]) * oc.bz + b[2];
        doubt = near[id >> 5] >> (id & 31) & 1u;
      }
      const uint64_t m = __ballot(doubt);
      if (hi * (1.f / G.stepdist) < 1e6f && lo > -1e6f * G.stepdist) {
        if (m == 0) {
          n = 0;
        } else {
          const int first = __ffsll((unsigned long long)m) - 1, last = 63 - __clzll((long long)m);
          const float per = 1.f / G.stepdist;
          s0 = max((int64_t)0, (int64_t)((lo + (float)first * len - t0) * per) - 2);
          n = min(n, (int64_t)((lo + (float)(last + 1) * len - t0) * per) + 3);
        }
      }
    }
    if (row < c.H && col < c.W)
      flag[(int64_t)row * c.W + col] = ray_hits(G, oc, bits, start, dir, s0, n);
  }
}

// Kept pixels of one view, in pixel order: row incl[p] - 1 of the outputs receives the
// pixel's colour and rebuilt ray when its flag (incl[p] - incl[p - 1]) is set.
__global__ void __launch_bounds__(256) k_compact_view(Camera c, const float* __restrict__ rgb,
                                                      const int64_t* __restrict__ incl,
                                                      float* __restrict__ rgb_out,
                                                      float* __restrict__ o_out,
                                                      float* __restrict__ d_out,
                                                      float* __restrict__ v_out) {
  const int64_t n = (int64_t)c.H * c.W;
  for (int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; p < n;
       p += (int64_t)gridDim.x * blockDim.x) {
    const int64_t prev = p ? incl[p - 1] : 0;
    if (incl[p] == prev) continue;
    float o[3], d[3], v[3];
    camera_ray(c, (int)(p / c.W), (int)(p % c.W), o, d, v);
    const int64_t k = prev;
    for (int j = 0; j < 3; ++j) {
      rgb_out[3 * k + j] = rgb[3 * p + j];
      o_out[3 * k + j] = o[j];
      d_out[3 * k + j] = d[j];
      v_out[3 * k + j] = v[j];
    }
  }
}

}  // namespace vx

using namespace vx;

// cam = {H, W, fx, fy, cx, cy, R[9], t[3], off, inverse_y, flip_x, flip_y, ndc, ndc_c0,
// ndc_c1, ndc_near} as 26 floats (host memory).
static int camera_from(Camera& c, const float* cam) {
  VX_CHECK_ARG(cam, "camera: parameters missing");
  c.H = (int)cam[0];
  c.W = (int)cam[1];
  VX_CHECK_ARG(c.H >= 0 && c.W >= 0 && (float)c.H == cam[0] && (float)c.W == cam[1],
               "camera: H and W must be non-negative integers");
  c.fx = cam[2];
  c.fy = cam[3];
  c.cx = cam[4];
  c.cy = cam[5];
  for (int i = 0; i < 9; ++i) c.R[i] = cam[6 + i];
  for (int i = 0; i < 3; ++i) c.t[i] = cam[15 + i];
  c.off = cam[18];
  c.inverse_y = cam[19] != 0.f;
  c.flip_x = cam[20] != 0.f;
  c.flip_y = cam[21] != 0.f;
  c.ndc = cam[22] != 0.f;
  c.ndc_c0 = cam[23];
  c.ndc_c1 = cam[24];
  c.ndc_near = cam[25];
  return VX_OK;
}

// Sampling geometry of the pre-filter: box {mn, mx}, params {stepdist, near}.
static int prefilter_geom(FusedGeom& G, const float* box, const float* params, const float* mc,
                          const int64_t* mc_geom, const float* mc_params) {
  VX_CHECK_ARG(box && params, "hit_coarse_geo: box/parameters missing");
  VX_CHECK_ARG(mc, "hit_coarse_geo: the mask cache is required");
  G = FusedGeom{};
  for (int i = 0; i < 3; ++i) {
    G.mn[i] = box[i];
    G.mx[i] = box[3 + i];
  }
  G.stepdist = params[0];
  G.near_ = params[1];
  G.far_ = 1e9f;
  return fused_maskcache(G, mc, mc_geom, mc_params);
}

// Occupancy bricks and the known densities of a MaskCache (host side); occ: what
// vx_maskcache_occupancy filled, the blocks of every brick and then the bricks' bits, or NULL
// (then only the densities are used).
static Occupancy occupancy_of(const FusedGeom& G, const void* occ) {
  Occupancy oc{};
  const int size[3] = {G.gm.X, G.gm.Y, G.gm.Z};
  auto bricks = [&](int a) { return ((size[a] > 1 ? size[a] - 2 : 0) >> oc.shift) + 1; };
  for (oc.shift = kOccShift; (int64_t)bricks(0) * bricks(1) * bricks(2) > kOccMaxBits;) ++oc.shift;
  oc.bx = bricks(0);
  oc.by = bricks(1);
  oc.bz = bricks(2);
  const double ratio = G.mc_ratio, shift = G.mc_shift, thres = G.mc_thres;
  // density at which alpha reaches t (0 < t < 1): softplus(x) = -log(1 - t) / ratio, with the
  // softplus that is x above 20
  auto density = [&](double t, double side) {
    const double sp = -log1p(-t) / ratio;
    const double x = sp > 20.0 ? sp : log(expm1(sp));
    const double d = x - shift;
    return d + side * (1e-3 + 1e-5 * (fabs(x) + fabs(shift) + fabs(d)));
  };
  oc.d_lo = -INFINITY;
  oc.d_hi = INFINITY;
  // the float formula's alpha is off by less than 5e-7
  if (ratio > 0 && isfinite(ratio) && isfinite(shift) && thres - 1e-6 > 0 && thres < 1.0) {
    const double lo = density(thres - 1e-6, -1.0);
    if (isfinite(lo)) oc.d_lo = (float)lo;
    if (thres + 1e-6 < 1.0) {
      const double hi = density(thres + 1e-6, 1.0);
      if (isfinite(hi)) oc.d_hi = (float)hi;
    }
  }
  bool plain = isfinite(oc.d_lo);
  oc.inner = 1;
  float margins = 0.f;
  for (int a = 0; a < 3; ++a) {
    // rounding of a sample's index: a few parts in 2^24 of the coordinates' size, in cells
    const float far = fmaxf(fmaxf(fabsf(G.mn[a]), fabsf(G.mx[a])),
                            fmaxf(fabsf(G.mc_mn[a]), fabsf(G.mc_mx[a])));
    oc.margin[a] = 1e-4f + 4e-6f * (float)size[a] * (1.f + far / (G.mc_mx[a] - G.mc_mn[a]));
    plain = plain && size[a] > 1 && oc.margin[a] > 0.f && oc.margin[a] < 0.1f;
    margins += oc.margin[a];
    const float slack = 0.5f * oc.margin[a] * (G.mc_mx[a] - G.mc_mn[a]) / (float)(size[a] - 1);
    if (!(G.mn[a] >= G.mc_mn[a] - slack && G.mx[a] <= G.mc_mx[a] + slack)) oc.inner = 0;
  }
  oc.d_clear = oc.d_lo < 0.f ? oc.d_lo / (1.f - margins) : oc.d_lo;
  if (plain && occ) {
    oc.blocks = (const uint64_t*)occ;
    const int64_t nb = (int64_t)oc.bx * oc.by * oc.bz;
    oc.bits = (const uint32_t*)(oc.blocks + nb);
    oc.near = oc.bits + cdiv(nb, 32);
  }
  return oc;
}

// LDS of `arrays` copies of the bits.
static size_t occ_lds_bytes(const Occupancy& oc, int arrays) {
  return (size_t)cdiv((int64_t)oc.bx * oc.by * oc.bz, 32) * 4 * arrays;
}

extern "C" {

int vx_camera_rays(const float* cam, float* rays_o, float* rays_d, float* viewdirs, void* stream) {
  Camera c;
  if (int st = camera_from(c, cam)) return st;
  const int64_t n = (int64_t)c.H * c.W;
  if (n == 0) return VX_OK;
  k_camera_rays<<<grid_for(n, 256), 256, 0, (hipStream_t)stream>>>(c, rays_o, rays_d, viewdirs);
  return launch_status("camera_rays");
}

int vx_ndc_rays(int64_t n, float c0, float c1, float near_, const float* rays_o,
                const float* rays_d, float* o_out, float* d_out, void* stream) {
  VX_CHECK_ARG(n >= 0, "ndc_rays: n < 0");
  if (n == 0) return VX_OK;
  k_ndc_rays<<<grid_for(n, 256), 256, 0, (hipStream_t)stream>>>(n, c0, c1, near_, rays_o, rays_d,
                                                                o_out, d_out);
  return launch_status("ndc_rays");
}

int64_t vx_maskcache_occupancy_bytes(const int64_t* mc_geom) {
  if (!mc_geom || mc_geom[1] < 1 || mc_geom[2] < 1 || mc_geom[3] < 1) return -1;
  FusedGeom G{};
  G.gm.X = (int)mc_geom[1];
  G.gm.Y = (int)mc_geom[2];
  G.gm.Z = (int)mc_geom[3];
  const Occupancy oc = occupancy_of(G, nullptr);
  const int64_t nb = (int64_t)oc.bx * oc.by * oc.bz;
  return 8 * nb + 8 * cdiv(nb, 32);
}

int vx_maskcache_occupancy(const float* mc, const int64_t* mc_geom, const float* mc_params,
                           void* occ, void* stream) {
  VX_CHECK_ARG(mc && occ, "maskcache_occupancy: missing argument");
  VX_CHECK_ARG(((uintptr_t)occ & 7) == 0, "maskcache_occupancy: occ must be 8-byte aligned");
  FusedGeom G{};
  if (int st = fused_maskcache(G, mc, mc_geom, mc_params)) return st;
  const Occupancy oc = occupancy_of(G, nullptr);
  const int64_t nb = (int64_t)oc.bx * oc.by * oc.bz;
  uint64_t* blocks = (uint64_t*)occ;
  uint32_t* bits = (uint32_t*)(blocks + nb);
  hipStream_t st = (hipStream_t)stream;
  k_occupancy<<<(unsigned)cdiv(nb, 32), 1024, 0, st>>>(G.mc, G.gm, oc, bits, blocks);
  k_occupancy_near<<<(unsigned)cdiv(nb, 256), 256, 0, st>>>(oc, bits, bits + cdiv(nb, 32));
  return launch_status("maskcache_occupancy");
}

int vx_hit_coarse_geo_occ(const float* rays_o, const float* rays_d, int64_t n_rays,
                          const float* box, const float* params, const float* mc,
                          const int64_t* mc_geom, const float* mc_params, const void* occ,
                          uint8_t* hit, int64_t* flag, void* stream) {
  FusedGeom G;
  if (int st = prefilter_geom(G, box, params, mc, mc_geom, mc_params)) return st;
  VX_CHECK_ARG(n_rays >= 0, "hit_coarse_geo: n_rays < 0");
  if (n_rays == 0) return VX_OK;
  VX_CHECK_ARG(hit || flag, "hit_coarse_geo: no output");
  const Occupancy oc = occupancy_of(G, occ);
  if (oc.bits)
    k_hit_rays<<<grid_for(n_rays, 256), 256, occ_lds_bytes(oc, 1), (hipStream_t)stream>>>(
        G, oc, rays_o, rays_d, n_rays, hit, flag);
  else
    k_hit_rays_wave<<<grid_for(n_rays, 4, 1 << 16), 256, 0, (hipStream_t)stream>>>(
        G, rays_o, rays_d, n_rays, hit, flag);
  return launch_status("hit_coarse_geo");
}

int vx_hit_coarse_geo(const float* rays_o, const float* rays_d, int64_t n_rays, const float* box,
                      const float* params, const float* mc, const int64_t* mc_geom,
                      const float* mc_params, uint8_t* hit, int64_t* flag, void* stream) {
  return vx_hit_coarse_geo_occ(rays_o, rays_d, n_rays, box, params, mc, mc_geom, mc_params,
                               nullptr, hit, flag, stream);
}

int vx_view_hit_coarse_geo_occ(const float* cam, const float* box, const float* params,
                               const float* mc, const int64_t* mc_geom, const float* mc_params,
                               const void* occ, int64_t* flag, void* stream) {
  Camera c;
  if (int st = camera_from(c, cam)) return st;
  FusedGeom G;
  if (int st = prefilter_geom(G, box, params, mc, mc_geom, mc_params)) return st;
  const int64_t n = (int64_t)c.H * c.W;
  if (n == 0) return VX_OK;
  const Occupancy oc = occupancy_of(G, occ);
  if (!oc.bits) {
    k_hit_camera_wave<<<grid_for(n, 4, 1 << 16), 256, 0, (hipStream_t)stream>>>(G, c, flag);
    return launch_status("view_hit_coarse_geo");
  }
  const int64_t tiles = cdiv(c.W, 8) * cdiv(c.H, 8);
  VX_CHECK_ARG(tiles < ((int64_t)1 << 32), "hit_coarse_geo: view too large");
  // a tile per wave: the walks along the object's outline are ten times the others', and a
  // grid of resident blocks ended with the waves that had met several of them
  k_hit_camera<<<grid_for(tiles, 4), 256, occ_lds_bytes(oc, 2), (hipStream_t)stream>>>(G, oc, c, flag);
  return launch_status("view_hit_coarse_geo");
}

int vx_view_hit_coarse_geo(const float* cam, const float* box, const float* params,
                           const float* mc, const int64_t* mc_geom, const float* mc_params,
                           int64_t* flag, void* stream) {
  return vx_view_hit_coarse_geo_occ(cam, box, params, mc, mc_geom, mc_params, nullptr, flag,
                                    stream);
}

int vx_view_compact_rays(const float* cam, const float* rgb, const int64_t* incl, float* rgb_out,
                         float* o_out, float* d_out, float* v_out, void* stream) {
  Camera c;
  if (int st = camera_from(c, cam)) return st;
  const int64_t n = (int64_t)c.H * c.W;
  if (n == 0) return VX_OK;
  k_compact_view<<<grid_for(n, 256), 256, 0, (hipStream_t)stream>>>(c, rgb, incl, rgb_out, o_out,
                                                                    d_out, v_out);
  return launch_status("view_compact_rays");
}

}  // extern "C"
