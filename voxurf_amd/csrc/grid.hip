// Dense voxel-grid kernels (gfx950): trilinear gather and its scatter-add adjoint, the
// 6-neighbour SDF stencil (centre value + clamped central differences), the dense
// central-difference gradient grid, and the total-variation gradient.
//
// A grid is [C, X, Y, Z] with arbitrary element strides (sc, sx, sy, sz): the
// reference's contiguous [1, C, X, Y, Z] layout (sc = XYZ, sz = 1) and the
// channels-last layout used for multi-channel feature grids (sc = 1, sz = C) are both
// served by the same kernels.  The interpolation reproduces F.grid_sample(...,
// mode='bilinear', align_corners=True, padding_mode='zeros') on a 5-D input: the same
// normalise/unnormalise chain, corner order and weight products (contraction off), so
// results agree with PyTorch's CPU kernel to rounding of the final sum.
#include "voxel.h"

namespace vx {

// ---- DenseGrid.forward / backward (lib/grid.py:47-58) ----------------------------

template <typename T>
__global__ void k_tri_fwd(const T* __restrict__ grid, GridDesc g, const T* __restrict__ xyz,
                          const T* __restrict__ mn, const T* __restrict__ mx, int64_t n,
                          T* __restrict__ out) {
  const T ex = mx[0] - mn[0], ey = mx[1] - mn[1], ez = mx[2] - mn[2];
  for (int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; p < n;
       p += (int64_t)gridDim.x * blockDim.x) {
    Tri<T> t;
    t.init(world_to_index(xyz[3 * p], mn[0], ex, g.X), world_to_index(xyz[3 * p + 1], mn[1], ey, g.Y),
           world_to_index(xyz[3 * p + 2], mn[2], ez, g.Z));
    for (int c = 0; c < g.C; ++c) out[p * g.C + c] = tri_gather(grid, g, t, c);
  }
}

// The same for channels-innermost grids (channel stride 1): a lane per point and V
// neighbouring channels, 16-byte corner loads where C, the strides and the base allow V = 4
// (or 8-byte ones, V = 2), so that a point's lanes read one run per corner and write one run.
// A lane per point that looped over the channels read 64 scattered lines per load: 38 us for
// 100 k points of a 256^3 x 12 grid, against 13 us here.  Each channel is summed as above.
template <typename T, int V>
struct alignas(V * sizeof(T)) ChanVec {
  T v[V];
};

template <typename T, int V>
__global__ void __launch_bounds__(256) k_tri_fwd_rows(const T* __restrict__ grid, GridDesc g,
                                                      const T* __restrict__ xyz,
                                                      const T* __restrict__ mn,
                                                      const T* __restrict__ mx, int64_t n,
                                                      T* __restrict__ out) {
#pragma clang fp contract(off)
  using Vec = ChanVec<T, V>;
  const T ex = mx[0] - mn[0], ey = mx[1] - mn[1], ez = mx[2] - mn[2];
  const int cv = g.C / V;
  const int64_t total = n * cv;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t p = total <= 0x7fffffff ? (int64_t)((uint32_t)i / (uint32_t)cv) : i / cv;
    const int c = (int)(i - p * cv) * V;
    Tri<T> t;
    t.init(world_to_index(xyz[3 * p], mn[0], ex, g.X), world_to_index(xyz[3 * p + 1], mn[1], ey, g.Y),
           world_to_index(xyz[3 * p + 2], mn[2], ez, g.Z));
    Vec v[8];
    bool in[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int x = t.x0 + (k >> 2), y = t.y0 + (k >> 1 & 1), z = t.z0 + (k & 1);
      in[k] = in_grid<T>(x, y, z, g);
      v[k] = *reinterpret_cast<const Vec*>(grid + c + clamp_index(x, g.X) * g.sx +
                                           clamp_index(y, g.Y) * g.sy + clamp_index(z, g.Z) * g.sz);
    }
    Vec acc;
#pragma unroll
    for (int e = 0; e < V; ++e) acc.v[e] = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      if (!in[k]) continue;
      const T w = t.w(k >> 2, k >> 1 & 1, k & 1);
#pragma unroll
      for (int e = 0; e < V; ++e) acc.v[e] += v[k].v[e] * w;
    }
    *reinterpret_cast<Vec*>(out + p * g.C + c) = acc;
  }
}

// Its adjoint: L lanes per point (the power of two that holds the channels), a lane per
// channel, so that an atomic instruction's lanes hit one run per point.  Consecutive points
// (a ray's samples, half a voxel apart) often share their cell: the 64 / L points of a pass
// that do add their corner terms across the lane groups first, and the first of them issues
// the atomics.  Bound by the rate of scattered atomic requests: a lane per point and its own
// 8 C atomics took 480 us for 100 k points x 12 channels, this 44 us.
template <typename T, int L>
__global__ void __launch_bounds__(256) k_tri_bwd_rows(T* __restrict__ grad, GridDesc g,
                                                      const T* __restrict__ xyz,
                                                      const T* __restrict__ mn,
                                                      const T* __restrict__ mx, int64_t n,
                                                      const T* __restrict__ gout) {
#pragma clang fp contract(off)
  constexpr int P = 64 / L;  // points per pass
  const T ex = mx[0] - mn[0], ey = mx[1] - mn[1], ez = mx[2] - mn[2];
  const int lane = threadIdx.x & 63, grp = lane / L, ch = lane % L;
  const int64_t waves = (int64_t)gridDim.x * (blockDim.x >> 6);
  for (int64_t base = ((int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) * P; base < n;
       base += waves * P) {
    const int64_t p = base + grp;
    const bool valid = p < n;
    const int64_t q = valid ? p : n - 1;
    Tri<T> t;
    t.init(world_to_index(xyz[3 * q], mn[0], ex, g.X), world_to_index(xyz[3 * q + 1], mn[1], ey, g.Y),
           world_to_index(xyz[3 * q + 2], mn[2], ez, g.Z));
    const T go = valid && ch < g.C ? gout[q * g.C + ch] : (T)0;
    T v[8];
#pragma unroll
    for (int b = 0; b < 8; ++b) v[b] = go == (T)0 ? (T)0 : t.w(b >> 2, (b >> 1) & 1, b & 1) * go;
    // runs of points in one cell among the pass's groups
    const int px = __shfl(t.x0, (lane - L) & 63, 64), py = __shfl(t.y0, (lane - L) & 63, 64),
              pz = __shfl(t.z0, (lane - L) & 63, 64);
    const bool same = grp > 0 && valid && px == t.x0 && py == t.y0 && pz == t.z0;
    const uint64_t heads = __ballot(!same);
    if (heads != ~0ull) {
      // the run of this group ends before the next head
      const uint64_t later = lane - ch + L < 64 ? heads >> (lane - ch + L) << (lane - ch + L) : 0;
      const int end = later ? __ffsll((unsigned long long)later) - 1 : 64;  // first lane of it
#pragma unroll
      for (int off = L; off < 64; off <<= 1) {
        const bool take = lane + off < end;
#pragma unroll
        for (int b = 0; b < 8; ++b) {
          const T o = __shfl_down(v[b], off, 64);
          if (take) v[b] += o;
        }
      }
    }
    if (valid && !same && ch < g.C) {
#pragma unroll
      for (int b = 0; b < 8; ++b) {
        const int x = t.x0 + (b >> 2), y = t.y0 + ((b >> 1) & 1), z = t.z0 + (b & 1);
        if (v[b] != (T)0 && in_grid<T>(x, y, z, g))
          atomic_add(&grad[ch + x * g.sx + y * g.sy + z * g.sz], v[b]);
      }
    }
  }
}

template <typename T>
__global__ void k_tri_bwd(T* __restrict__ grad, GridDesc g, const T* __restrict__ xyz,
                          const T* __restrict__ mn, const T* __restrict__ mx, int64_t n,
                          const T* __restrict__ gout) {
  const T ex = mx[0] - mn[0], ey = mx[1] - mn[1], ez = mx[2] - mn[2];
  for (int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; p < n;
       p += (int64_t)gridDim.x * blockDim.x) {
    Tri<T> t;
    t.init(world_to_index(xyz[3 * p], mn[0], ex, g.X), world_to_index(xyz[3 * p + 1], mn[1], ey, g.Y),
           world_to_index(xyz[3 * p + 2], mn[2], ez, g.Z));
    for (int c = 0; c < g.C; ++c) tri_scatter(grad, g, t, c, gout[p * g.C + c]);
  }
}

// ---- sample_sdfs (lib/voxurf_fine.py:537-577) -------------------------------------
// For each point and displacement d in `disp[0..nd)`, the SDF is sampled at the 6
// points ind +- d along each index axis (zyx order), each component clamped to
// [0, size-1] in index space, then mapped back through the normalised coordinate
// (all_ind / (size-1)) * 2 - 1 before grid_sample unnormalises it again.
//   feat[p, k*nd + j]   k = 0..5 : (-z, +z, -y, +y, -x, +x)
//   grad[p, a*nd + j]   a = 0..2 : (z, y, x),  (f[+] - f[-]) / (ind[+] - ind[-]) / voxel_size
// optionally normalised per displacement: grad / (|grad| + 1e-5).

template <typename T>
__global__ void k_sdfs_fwd(const T* __restrict__ grid, GridDesc g, const T* __restrict__ xyz,
                           const T* __restrict__ mn, const T* __restrict__ mx,
                           const T* __restrict__ disp, int nd, T voxel_size, int use_norm,
                           int64_t n, T* __restrict__ feat, T* __restrict__ grad) {
#pragma clang fp contract(off)
  for (int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; p < n;
       p += (int64_t)gridDim.x * blockDim.x) {
    T ind[3];
    zyx_index(xyz + 3 * p, mn, mx, g, ind);
    for (int j = 0; j < nd; ++j) {
      const T d = disp[j];
      T gr[3];
      for (int a = 0; a < 3; ++a) {
        T cm, cp;
        const T fm = sample_displaced(grid, g, ind, a, -d, cm);
        const T fp = sample_displaced(grid, g, ind, a, d, cp);
        feat[p * 6 * nd + (2 * a) * nd + j] = fm;
        feat[p * 6 * nd + (2 * a + 1) * nd + j] = fp;
        const T df = clamped_diff(ind, a, d, g);
        gr[a] = ((fp - fm) / df) / voxel_size;
      }
      if (use_norm) {
        const T nrm = sqrt(gr[0] * gr[0] + gr[1] * gr[1] + gr[2] * gr[2]) + (T)1e-5;
        for (int a = 0; a < 3; ++a) gr[a] = gr[a] / nrm;
      }
      for (int a = 0; a < 3; ++a) grad[p * 3 * nd + a * nd + j] = gr[a];
    }
  }
}

template <typename T>
__global__ void k_sdfs_bwd(T* __restrict__ ggrid, const T* __restrict__ grid, GridDesc g,
                           const T* __restrict__ xyz, const T* __restrict__ mn,
                           const T* __restrict__ mx, const T* __restrict__ disp, int nd,
                           T voxel_size, int use_norm, int64_t n, const T* __restrict__ gfeat,
                           const T* __restrict__ ggrad) {
#pragma clang fp contract(off)
  for (int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; p < n;
       p += (int64_t)gridDim.x * blockDim.x) {
    T ind[3];
    zyx_index(xyz + 3 * p, mn, mx, g, ind);
    for (int j = 0; j < nd; ++j) {
      const T d = disp[j];
      T df[3], gg[3];
      for (int a = 0; a < 3; ++a) {
        df[a] = clamped_diff(ind, a, d, g);
        gg[a] = ggrad ? ggrad[p * 3 * nd + a * nd + j] : (T)0;
      }
      if (use_norm && ggrad) {
        // y = r / (|r| + eps):  dr = (gy - r (r . gy) / (|r| (|r| + eps))) / (|r| + eps)
        T r[3];
        for (int a = 0; a < 3; ++a) {
          T cm, cp;
          const T fm = sample_displaced(grid, g, ind, a, -d, cm);
          const T fp = sample_displaced(grid, g, ind, a, d, cp);
          r[a] = ((fp - fm) / df[a]) / voxel_size;
        }
        const T nr = sqrt(r[0] * r[0] + r[1] * r[1] + r[2] * r[2]);
        const T den = nr + (T)1e-5;
        const T dot = r[0] * gg[0] + r[1] * gg[1] + r[2] * gg[2];
        const T k = nr > (T)0 ? dot / (nr * den) : (T)0;
        for (int a = 0; a < 3; ++a) gg[a] = (gg[a] - r[a] * k) / den;
      }
      for (int a = 0; a < 3; ++a) {
        const T gd = gg[a] / df[a] / voxel_size;  // d grad / d f[+] ; -gd for f[-]
        const T gm = (gfeat ? gfeat[p * 6 * nd + (2 * a) * nd + j] : (T)0) - gd;
        const T gp = (gfeat ? gfeat[p * 6 * nd + (2 * a + 1) * nd + j] : (T)0) + gd;
        scatter_displaced(ggrid, g, ind, a, -d, gm);
        scatter_displaced(ggrid, g, ind, a, d, gp);
      }
    }
  }
}

// ---- Voxurf.grid_sampler(sample_ret, sample_grad) (lib/voxurf_fine.py:502-534) ------
// Centre SDF value plus the displacement-1 stencil in one pass:
//   sdf [n], grad [n,3] (xyz order, unnormalised), feat [n,6] (-x,+x,-y,+y,-z,+z).

template <typename T>
__global__ void k_sdf_grad_fwd(const T* __restrict__ grid, GridDesc g, const T* __restrict__ xyz,
                               const T* __restrict__ mn, const T* __restrict__ mx, T voxel_size,
                               int64_t n, T* __restrict__ sdf, T* __restrict__ grad,
                               T* __restrict__ feat) {
  for (int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; p < n;
       p += (int64_t)gridDim.x * blockDim.x) {
    const T q[3] = {xyz[3 * p], xyz[3 * p + 1], xyz[3 * p + 2]};
    T s, gr[3], f[6];
    sdf7(grid, g, q, mn, mx, voxel_size, s, gr, f);
    sdf[p] = s;
    for (int c = 0; c < 3; ++c) grad[3 * p + c] = gr[c];
    if (feat)
      for (int c = 0; c < 6; ++c) feat[6 * p + c] = f[c];
  }
}

template <typename T>
__global__ void k_sdf_grad_bwd(T* __restrict__ ggrid, GridDesc g, const T* __restrict__ xyz,
                               const T* __restrict__ mn, const T* __restrict__ mx, T voxel_size,
                               int64_t n, const T* __restrict__ gsdf, const T* __restrict__ ggrad,
                               const T* __restrict__ gfeat) {
  for (int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; p < n;
       p += (int64_t)gridDim.x * blockDim.x) {
    const T q[3] = {xyz[3 * p], xyz[3 * p + 1], xyz[3 * p + 2]};
    const T gg[3] = {ggrad ? ggrad[3 * p] : (T)0, ggrad ? ggrad[3 * p + 1] : (T)0,
                     ggrad ? ggrad[3 * p + 2] : (T)0};
    sdf7_scatter(ggrid, g, q, mn, mx, voxel_size, gsdf ? gsdf[p] : (T)0, gg,
                 gfeat ? gfeat + 6 * p : (const T*)nullptr);
  }
}

// The adjoint without the neighbour values' gradients (gfeat), for consecutive samples of
// rays.  A sample adds to 32 voxels (sdf7_terms): as 32 atomics of a lane they are 32
// scattered requests, and the rate of those bounds the scatter (359 us for the 1.5 M samples
// of a coarse step, of which one in six has a gradient).  Here a wave leaves its samples'
// terms in LDS, and half a wave takes a run of samples in one cell, a lane per voxel: the
// run's terms are added first, and the voxels of a z line (12 lines per cell) go out as one
// request.  Measured 136 us.
constexpr int kScatterThreads = 256;
template <typename T>
__global__ void __launch_bounds__(kScatterThreads) k_sdf_grad_bwd_runs(
    T* __restrict__ ggrid, GridDesc g, const T* __restrict__ xyz, const T* __restrict__ mn,
    const T* __restrict__ mx, T voxel_size, int64_t n, const T* __restrict__ gsdf,
    const T* __restrict__ ggrad) {
#pragma clang fp contract(off)
  constexpr int kStride = 33;  // odd: the lanes' rows spread over the banks
  __shared__ T terms[kScatterThreads * kStride];
  __shared__ int cell[kScatterThreads * 3];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, half = lane >> 5, vl = lane & 31;
  T* tw = terms + wave * 64 * kStride;
  int* cw = cell + wave * 64 * 3;
  // this lane's voxel of a cell's 32 (offsets from the cell): the order of Sdf7Terms
  int dx, dy, dz;
  if (vl < 8) {
    dx = vl >> 2;
    dy = vl >> 1 & 1;
    dz = vl & 1;
  } else {
    const int c = (vl - 8) >> 3, side = (vl >> 2) & 1, j = vl & 3;
    const int lo = c == 0 ? 1 : 0, hi = c == 2 ? 1 : 2;
    int v[3] = {0, 0, 0};
    v[c] = side ? 2 : -1;
    v[lo] += j >> 1;
    v[hi] += j & 1;
    dx = v[0];
    dy = v[1];
    dz = v[2];
  }
  const int64_t waves = (int64_t)gridDim.x * (kScatterThreads >> 6);
  for (int64_t base = ((int64_t)blockIdx.x * (kScatterThreads >> 6) + wave) * 64; base < n;
       base += waves * 64) {
    const int64_t p = base + lane;
    const T gs = p < n && gsdf ? gsdf[p] : (T)0;
    const T gg[3] = {p < n && ggrad ? ggrad[3 * p] : (T)0, p < n && ggrad ? ggrad[3 * p + 1] : (T)0,
                     p < n && ggrad ? ggrad[3 * p + 2] : (T)0};
    const bool act = gs != (T)0 || gg[0] != (T)0 || gg[1] != (T)0 || gg[2] != (T)0;
    const uint64_t acts = __ballot(act);
    if (acts == 0) continue;
    int x0 = 0, y0 = 0, z0 = 0;
    if (act) {
      const T q[3] = {xyz[3 * p], xyz[3 * p + 1], xyz[3 * p + 2]};
      Sdf7Terms<T> o;
      sdf7_terms(ggrid, g, q, mn, mx, voxel_size, gs, gg, o);
      x0 = o.x0;
      y0 = o.y0;
      z0 = o.z0;
      T* row = tw + lane * kStride;
#pragma unroll
      for (int b = 0; b < 8; ++b) row[b] = o.acc[b];
#pragma unroll
      for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int sd = 0; sd < 2; ++sd)
#pragma unroll
          for (int j = 0; j < 4; ++j) row[8 + 8 * c + 4 * sd + j] = o.out[c][sd][j];
      cw[3 * lane] = x0;
      cw[3 * lane + 1] = y0;
      cw[3 * lane + 2] = z0;
    }
    const int px = __shfl_up(x0, 1, 64), py = __shfl_up(y0, 1, 64), pz = __shfl_up(z0, 1, 64);
    const bool prev = lane > 0 && (acts >> (lane - 1) & 1);
    const bool head = act && !(prev && px == x0 && py == y0 && pz == z0);
    // runs: from each head up to the next head or gap
    const uint64_t heads = __ballot(head), stops = heads | ~acts;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // the terms, for the other lanes
    uint64_t todo = heads;
    while (todo) {
      // one run for each half of the wave
      const int first = __ffsll((unsigned long long)todo) - 1;
      todo &= todo - 1;
      const int second = todo ? __ffsll((unsigned long long)todo) - 1 : -1;
      todo &= todo - 1;
      const int r = half ? second : first;
      if (r < 0) continue;
      const uint64_t after = r < 63 ? stops >> (r + 1) : 0;
      const int end = after ? r + __ffsll((unsigned long long)after) : 64;
      T sum = tw[r * kStride + vl];
      for (int k = r + 1; k < end; ++k) sum += tw[k * kStride + vl];
      const int x = cw[3 * r] + dx, y = cw[3 * r + 1] + dy, z = cw[3 * r + 2] + dz;
      if (sum != (T)0 && in_grid<T>(x, y, z, g))
        atomic_add(&ggrid[x * g.sx + y * g.sy + z * g.sz], sum);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  }
}

// ---- neus_sdf_gradient 'interpolate' (lib/voxurf_fine.py:440-450) ------------------
// out[a] = (s[+1] - s[-1]) / 2 / voxel_size along axis a, 0 on that axis' boundary faces.
// Launched as a 3-D grid (z chunks of 256 threads, y, x): no index division.

template <typename T>
__global__ void __launch_bounds__(256) k_dense_grad_fwd(const T* __restrict__ s, int X, int Y, int Z,
                                                        T vs, T* __restrict__ out) {
#pragma clang fp contract(off)
  const int z = blockIdx.x * blockDim.x + threadIdx.x, y = blockIdx.y, x = blockIdx.z;
  if (z >= Z) return;
  const int64_t N = (int64_t)X * Y * Z;
  const int64_t sx = (int64_t)Y * Z, sy = Z;
  const int64_t i = x * sx + y * sy + z;
  out[i] = (x > 0 && x < X - 1) ? ((s[i + sx] - s[i - sx]) / (T)2) / vs : (T)0;
  out[N + i] = (y > 0 && y < Y - 1) ? ((s[i + sy] - s[i - sy]) / (T)2) / vs : (T)0;
  out[2 * N + i] = (z > 0 && z < Z - 1) ? ((s[i + 1] - s[i - 1]) / (T)2) / vs : (T)0;
}

// ---- total_variation_add_grad (lib/cuda/total_variation_kernel.cu:13-66) ----------
// Weights arrive already divided by 6.  Axis weights follow the reference exactly: the
// plain kernel uses wz on both the contiguous (k) and outermost (i) axes and wy on j;
// the masked kernel uses wx, wy, wz on k, j, i.

template <typename T, bool kMasked>
__global__ void k_tv(const T* __restrict__ param, T* __restrict__ grad, const T* __restrict__ mask,
                     GridDesc g, float wk, float wj, float wi, int dense) {
#pragma clang fp contract(off)
  const int64_t N = (int64_t)g.C * g.X * g.Y * g.Z;
  for (int64_t idx = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; idx < N;
       idx += (int64_t)gridDim.x * blockDim.x) {
    // logical (c, i, j, k) -> address via strides
    const int k = (int)(idx % g.Z);
    const int j = (int)(idx / g.Z % g.Y);
    const int i = (int)(idx / g.Z / g.Y % g.X);
    const int c = (int)(idx / g.Z / g.Y / g.X);
    const int64_t a = c * g.sc + i * g.sx + j * g.sy + k * g.sz;
    if (!dense && grad[a] == (T)0) continue;
    const T p = param[a];
    float add = 0;
    // grad_to_add (float) += w * clamp(p - p_nb, -1, 1) [* mask[a] * mask[nb]], the
    // product formed in the tensor type.
    auto term = [&](bool has, int64_t nb, float w) {
      if (!has) return;
      T v = p - param[nb];
      v = v < (T)-1 ? (T)-1 : (v > (T)1 ? (T)1 : v);
      T t = (T)w * v;
      if (kMasked) t = (t * mask[a]) * mask[nb];
      add = (float)((T)add + t);
    };
    term(k > 0, a - g.sz, wk);
    term(k < g.Z - 1, a + g.sz, wk);
    term(j > 0, a - g.sy, wj);
    term(j < g.Y - 1, a + g.sy, wj);
    term(i > 0, a - g.sx, wi);
    term(i < g.X - 1, a + g.sx, wi);
    grad[a] += (T)add;
  }
}

// The same for the two layouts the grids have, rows of z (and of the channels, innermost):
// C_in is the channels of a row's point (C when they are innermost, else 1, with the channel
// an outer index), so a row has Z C_in elements, the z neighbours lie C_in apart, and a plane
// of one x is Y rows on end.  A thread takes V elements of a plane on `depth` planes in turn,
// keeping the plane before and the one after in registers.
// Bound by HBM reads: the strided form above, and one element per thread of this one, read
// every x and y neighbour again on another XCD (a block's neighbours run on the next XCDs,
// each with its own L2): 119 and 108 us at 256^3, where reading param once and the gradient
// twice takes 40.  Vectors of a row, 16 planes on end: 51 us.
template <typename T, int V>
struct TvVec {
  T v[V];
};

// V neighbouring elements at p, of which those with index >= lo and < hi may be read.
template <typename T, int V>
__device__ __forceinline__ TvVec<T, V> tv_load(const T* __restrict__ p, int lo, int hi) {
  TvVec<T, V> r;
  if (lo <= 0 && hi >= V) {
    __builtin_memcpy(&r, p, sizeof(r));   // (elements aligned, the vector perhaps not)
  } else {
#pragma unroll
    for (int e = 0; e < V; ++e) r.v[e] = e >= lo && e < hi ? p[e] : (T)0;
  }
  return r;
}

template <typename T, bool kMasked, int V>
__global__ void __launch_bounds__(256) k_tv_rows(const T* __restrict__ param, T* __restrict__ grad,
                                                 const T* __restrict__ mask, int X, int Y, int row,
                                                 int C_in, int depth, float wk, float wj, float wi,
                                                 int dense) {
#pragma clang fp contract(off)
  const int64_t plane = (int64_t)Y * row;
  const int64_t f = ((int64_t)blockIdx.x * 256 + threadIdx.x) * V;
  if (f >= plane) return;
  const int y = (int)(f / row), l = (int)(f - (int64_t)y * row);
  const int x0 = blockIdx.y * depth, x1 = min(x0 + depth, X);
  const T* pm = param + (int64_t)blockIdx.z * X * plane + f;
  const T* mm = kMasked ? mask + (int64_t)blockIdx.z * X * plane + f : nullptr;
  T* gm = grad + (int64_t)blockIdx.z * X * plane + f;
  // elements e of the vector with a z neighbour below (e >= below) and above (e < above)
  const int below = C_in - l, above = row - C_in - l;
  using Vec = TvVec<T, V>;
  auto at = [&](const T* p, int x) { return tv_load<T, V>(p + x * plane, 0, V); };
  Vec prev{}, cur, next{}, mprev{}, mcur{}, mnext{};
  if (x0 > 0) {
    prev = at(pm, x0 - 1);
    if (kMasked) mprev = at(mm, x0 - 1);
  }
  cur = at(pm, x0);
  if (kMasked) mcur = at(mm, x0);
  for (int x = x0; x < x1; ++x) {
    if (x + 1 < X) {
      next = at(pm, x + 1);
      if (kMasked) mnext = at(mm, x + 1);
    }
    Vec g = tv_load<T, V>(gm + x * plane, 0, V);
    // the elements that take the term, told from the gradient before it is added: a sum that
    // cancels to zero is stored like any other
    unsigned take = 0u;
#pragma unroll
    for (int e = 0; e < V; ++e) take |= (dense || g.v[e] != (T)0 ? 1u : 0u) << e;
    if (take) {
      const T* p = pm + x * plane;
      const T* m = kMasked ? mm + x * plane : nullptr;
      const Vec zl = tv_load<T, V>(p - C_in, below, V), zh = tv_load<T, V>(p + C_in, 0, above);
      const Vec yl = y > 0 ? tv_load<T, V>(p - row, 0, V) : Vec{},
                yh = y < Y - 1 ? tv_load<T, V>(p + row, 0, V) : Vec{};
      Vec mzl{}, mzh{}, myl{}, myh{};
      if (kMasked) {
        mzl = tv_load<T, V>(m - C_in, below, V);
        mzh = tv_load<T, V>(m + C_in, 0, above);
        if (y > 0) myl = tv_load<T, V>(m - row, 0, V);
        if (y < Y - 1) myh = tv_load<T, V>(m + row, 0, V);
      }
#pragma unroll
      for (int e = 0; e < V; ++e) {
        if (!(take >> e & 1u)) continue;
        const T c = cur.v[e];
        float add = 0;
        auto term = [&](bool has, T nb, T mnb, float w) {
#pragma clang fp contract(off)
          if (!has) return;
          T v = c - nb;
          v = v < (T)-1 ? (T)-1 : (v > (T)1 ? (T)1 : v);
          T t = (T)w * v;
          if (kMasked) t = (t * mcur.v[e]) * mnb;
          add = (float)((T)add + t);
        };
        term(e >= below, zl.v[e], mzl.v[e], wk);
        term(e < above, zh.v[e], mzh.v[e], wk);
        term(y > 0, yl.v[e], myl.v[e], wj);
        term(y < Y - 1, yh.v[e], myh.v[e], wj);
        term(x > 0, prev.v[e], mprev.v[e], wi);
        term(x < X - 1, next.v[e], mnext.v[e], wi);
        g.v[e] += (T)add;
      }
      T* o = gm + x * plane;
      if (dense) {
        __builtin_memcpy(o, &g, sizeof(g));
      } else {
#pragma unroll
        for (int e = 0; e < V; ++e)
          if (take >> e & 1u) o[e] = g.v[e];
      }
    }
    prev = cur;
    cur = next;
    if (kMasked) {
      mprev = mcur;
      mcur = mnext;
    }
  }
}

// Launches k_tv_rows if the grid's strides have the row form (false: other orders and sizes
// past a launch's limits take the strided kernel).  Vectors of four when a row holds whole
// ones; as many planes per thread as leave eight blocks per CU.
template <typename T, bool kMasked>
static bool tv_rows(const GridDesc& g, const T* param, T* grad, const T* mask, float wk, float wj,
                    float wi, int dense, hipStream_t st) {
  const int64_t X = g.X, Y = g.Y, Z = g.Z, C = g.C;
  const bool inner = C > 1 && g.sc == 1;
  const int64_t c_in = inner ? C : 1, outer = inner ? 1 : C, row = Z * c_in;
  if (g.sz != c_in || g.sy != row || g.sx != Y * row) return false;
  if (!inner && C > 1 && g.sc != X * Y * row) return false;
  if (row > 0x3fffffff || X > 65535 || outer > 65535) return false;
  const int v = row % 4 == 0 ? 4 : 1;
  const int64_t per_plane = cdiv(Y * row, 256 * v);
  int64_t depth = per_plane * X * outer / 2048;
  depth = depth < 1 ? 1 : (depth > 16 ? 16 : depth);
  if (per_plane > 0x7fffffff) return false;
  const dim3 blocks((unsigned)per_plane, (unsigned)cdiv(X, depth), (unsigned)outer);
  if (v == 4)
    k_tv_rows<T, kMasked, 4><<<blocks, 256, 0, st>>>(param, grad, mask, g.X, g.Y, (int)row, (int)c_in,
                                                     (int)depth, wk, wj, wi, dense);
  else
    k_tv_rows<T, kMasked, 1><<<blocks, 256, 0, st>>>(param, grad, mask, g.X, g.Y, (int)row, (int)c_in,
                                                     (int)depth, wk, wj, wi, dense);
  return true;
}

// Adjoint of k_dense_grad_fwd: gs[i] += sum_a (g_a[i - e_a] - g_a[i + e_a]) / 2 / vs over
// interior entries.  Bound by HBM: at 256^3 the three gradient grids read once and gs read and
// written are 335 MB.  A thread per element, its block's neighbours in x and y on other XCDs,
// read them again and took 143 us; vectors of a plane on 16 planes in turn, as k_tv_rows, 64
// (5.2 TB/s; a large copy, half of whose bytes are writes, reaches 5.0).
template <typename T, int V>
__global__ void __launch_bounds__(256) k_dense_grad_bwd(const T* __restrict__ go, int X, int Y, int Z,
                                                        int depth, T vs, T* __restrict__ gs) {
#pragma clang fp contract(off)
  const int64_t plane = (int64_t)Y * Z, N = X * plane;
  const int64_t f = ((int64_t)blockIdx.x * 256 + threadIdx.x) * V;
  if (f >= plane) return;
  const int y = (int)(f / Z), z = (int)(f - (int64_t)y * Z);
  const int x0 = blockIdx.y * depth, x1 = min(x0 + depth, X);
  using Vec = TvVec<T, V>;
  auto at = [&](const T* p) { return tv_load<T, V>(p, 0, V); };
  Vec prev{}, cur{}, next{};
  if (x0 > 0) prev = at(go + (x0 - 1) * plane + f);
  cur = at(go + x0 * plane + f);
  for (int x = x0; x < x1; ++x) {
    const int64_t i = x * plane + f;
    next = Vec{};
    if (x + 1 < X) next = at(go + i + plane);
    const Vec yl = y - 1 > 0 ? at(go + N + i - Z) : Vec{}, yh = y + 1 < Y - 1 ? at(go + N + i + Z) : Vec{};
    const Vec zl = tv_load<T, V>(go + 2 * N + i - 1, 1 - z, V),
              zh = tv_load<T, V>(go + 2 * N + i + 1, 0, Z - 1 - z);
    Vec g = at(gs + i);
#pragma unroll
    for (int e = 0; e < V; ++e) {
      T acc = 0;
      if (x - 1 > 0) acc += (prev.v[e] / (T)2) / vs;
      if (x + 1 < X - 1) acc -= (next.v[e] / (T)2) / vs;
      if (y - 1 > 0) acc += (yl.v[e] / (T)2) / vs;
      if (y + 1 < Y - 1) acc -= (yh.v[e] / (T)2) / vs;
      if (z + e - 1 > 0) acc += (zl.v[e] / (T)2) / vs;
      if (z + e + 1 < Z - 1) acc -= (zh.v[e] / (T)2) / vs;
      g.v[e] += acc;
    }
    __builtin_memcpy(gs + i, &g, sizeof(g));
    prev = cur;
    cur = next;
  }
}

template <typename T>
static void dense_grad_bwd(const T* go, int X, int Y, int Z, T vs, T* gs, hipStream_t st) {
  const int v = Z % 4 == 0 ? 4 : 1;
  const int64_t per_plane = cdiv((int64_t)Y * Z, 256 * v);
  int64_t depth = per_plane * X / 2048;  // enough blocks for the chip first
  depth = depth < 1 ? 1 : (depth > 16 ? 16 : depth);
  const dim3 blocks((unsigned)per_plane, (unsigned)cdiv(X, depth));
  if (v == 4) k_dense_grad_bwd<T, 4><<<blocks, 256, 0, st>>>(go, X, Y, Z, (int)depth, vs, gs);
  else k_dense_grad_bwd<T, 1><<<blocks, 256, 0, st>>>(go, X, Y, Z, (int)depth, vs, gs);
}

// ---- SDF and unit normal on a lattice tile (lib/dvgo_ori.py:679-693 with the normal of
// lib/voxurf_fine.py:502-534) --------------------------------------------------------------
// One thread per point of the tile (3-D launch: z chunks of 64, y, x), its lattice point
// (-1 + 2 i / (res - 1) per axis, as a product with the reciprocal) made in registers; normal = grad / (|grad| + 1e-5).
struct QueryArgs {
  const float* sdf;
  GridDesc g;
  float mn[3], mx[3], voxel_size, step;  // step: 1 / (res - 1)
  float o[3];
  int tile;
  float* out;
  float* normal;
};

__global__ void __launch_bounds__(64) k_sdf_query(QueryArgs a) {
#pragma clang fp contract(off)
  const int k = blockIdx.x * 64 + threadIdx.x, j = blockIdx.y, i = blockIdx.z;
  if (k >= a.tile) return;
  const float q[3] = {-1.f + 2.f * ((float)i + a.o[0]) * a.step, -1.f + 2.f * ((float)j + a.o[1]) * a.step,
                      -1.f + 2.f * ((float)k + a.o[2]) * a.step};
  float s, gr[3];
  sdf7<float>(a.sdf, a.g, q, a.mn, a.mx, a.voxel_size, s, gr, nullptr);
  const int64_t p = ((int64_t)i * a.tile + j) * a.tile + k;
  const float den = sqrtf(gr[0] * gr[0] + gr[1] * gr[1] + gr[2] * gr[2]) + 1e-5f;
  a.out[p] = s;
  for (int c = 0; c < 3; ++c) a.normal[3 * p + c] = gr[c] / den;
}

// ---- MaskCache.forward (lib/voxurf_fine.py:930-942, lib/dvgo_ori.py:440-473) --------
// density at the point (trilinear, or nearest lattice point with round-half-to-even as
// grid_sample's 'nearest'), alpha = 1 - exp(-softplus(density + act_shift) * ratio)
// with torch's softplus (threshold 20), out = alpha >= thres.
template <typename T>
__device__ __forceinline__ T softplus20(T x) {
  return x > (T)20 ? x : log1p(exp(x));
}

template <typename T>
__global__ void k_maskcache_alpha(const T* __restrict__ dens, GridDesc g, const T* __restrict__ xyz,
                                  const T* __restrict__ mn, const T* __restrict__ mx, T act_shift,
                                  T ratio, T thres, int nearest, int64_t n,
                                  uint8_t* __restrict__ out) {
#pragma clang fp contract(off)
  const T ex = mx[0] - mn[0], ey = mx[1] - mn[1], ez = mx[2] - mn[2];
  for (int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; p < n;
       p += (int64_t)gridDim.x * blockDim.x) {
    const T fx = world_to_index(xyz[3 * p], mn[0], ex, g.X);
    const T fy = world_to_index(xyz[3 * p + 1], mn[1], ey, g.Y);
    const T fz = world_to_index(xyz[3 * p + 2], mn[2], ez, g.Z);
    T d;
    if (nearest) {
      const int x = sat_f2i(rint(fx)), y = sat_f2i(rint(fy)), z = sat_f2i(rint(fz));
      d = in_grid<T>(x, y, z, g) ? dens[x * g.sx + y * g.sy + z * g.sz] : (T)0;
    } else {
      Tri<T> t;
      t.init(fx, fy, fz);
      d = tri_gather(dens, g, t, 0);
    }
    const T alpha = (T)1 - exp(-softplus20(d + act_shift) * ratio);
    out[p] = alpha >= thres;
  }
}

template <typename T>
__global__ void k_zero(T* p, int64_t n) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    p[i] = 0;
}

}  // namespace vx

using namespace vx;

#define ST(p) ((hipStream_t)(p))

static int make_desc(const int64_t* shape_strides, GridDesc& g) {
  // shape_strides = {C, X, Y, Z, sc, sx, sy, sz}
  g.C = (int)shape_strides[0];
  g.X = (int)shape_strides[1];
  g.Y = (int)shape_strides[2];
  g.Z = (int)shape_strides[3];
  g.sc = shape_strides[4];
  g.sx = shape_strides[5];
  g.sy = shape_strides[6];
  g.sz = shape_strides[7];
  VX_CHECK_ARG(g.C >= 1 && g.X >= 1 && g.Y >= 1 && g.Z >= 1, "grid: non-positive dimension");
  return VX_OK;
}

#define GRID_DISPATCH(dtype, ...)                                     \
  do {                                                                \
    if ((dtype) == VX_F32) {                                          \
      using scalar_t = float;                                         \
      __VA_ARGS__;                                                    \
    } else if ((dtype) == VX_F64) {                                   \
      using scalar_t = double;                                        \
      __VA_ARGS__;                                                    \
    } else {                                                          \
      vx::set_error("unsupported dtype code %d", (int)(dtype));       \
      return VX_ERR_DTYPE;                                            \
    }                                                                 \
  } while (0)

#define CP(p) ((const scalar_t*)(p))
#define MP(p) ((scalar_t*)(p))

// Channels per lane of the channels-innermost lookup: as many as one aligned load of up to 16
// bytes takes, given the channel count, the strides and the bases.
template <typename T>
static int row_vec(const GridDesc& g, const void* grid, const void* out) {
  for (int v = 16 / (int)sizeof(T); v > 1; v /= 2) {
    const uintptr_t bytes = (uintptr_t)v * sizeof(T);
    if (g.C % v == 0 && g.sx % v == 0 && g.sy % v == 0 && g.sz % v == 0 &&
        (uintptr_t)grid % bytes == 0 && (uintptr_t)out % bytes == 0)
      return v;
  }
  return 1;
}

template <typename T>
static void tri_fwd_rows(const T* grid, const GridDesc& g, const T* xyz, const T* mn, const T* mx,
                         int64_t n, T* out, hipStream_t st) {
  const int v = row_vec<T>(g, grid, out);
  const unsigned blocks = grid_for(n * (g.C / v), 256);
  if (v == 4) {
    if constexpr (sizeof(T) == 4)
      k_tri_fwd_rows<T, 4><<<blocks, 256, 0, st>>>(grid, g, xyz, mn, mx, n, out);
  } else if (v == 2) {
    k_tri_fwd_rows<T, 2><<<blocks, 256, 0, st>>>(grid, g, xyz, mn, mx, n, out);
  } else {
    k_tri_fwd_rows<T, 1><<<blocks, 256, 0, st>>>(grid, g, xyz, mn, mx, n, out);
  }
}

template <typename T>
static void tri_bwd_rows(T* grad, const GridDesc& g, const T* xyz, const T* mn, const T* mx,
                         int64_t n, const T* gout, hipStream_t st) {
#define VX_TRI_BWD(L) \
  k_tri_bwd_rows<T, L><<<grid_for(cdiv(n, 64 / L), 4), 256, 0, st>>>(grad, g, xyz, mn, mx, n, gout)
  if (g.C <= 2) VX_TRI_BWD(2);
  else if (g.C <= 4) VX_TRI_BWD(4);
  else if (g.C <= 8) VX_TRI_BWD(8);
  else if (g.C <= 16) VX_TRI_BWD(16);
  else if (g.C <= 32) VX_TRI_BWD(32);
  else VX_TRI_BWD(64);
#undef VX_TRI_BWD
}

extern "C" {

int vx_grid_sample_fwd(int dtype, const void* grid, const int64_t* geom, const void* xyz,
                       const void* xyz_min, const void* xyz_max, int64_t n, void* out,
                       void* stream) {
  GridDesc g;
  if (int st = make_desc(geom, g)) return st;
  VX_CHECK_ARG(n >= 0, "grid_sample: n < 0");
  if (n == 0) return VX_OK;
  // channels innermost: lanes over a point's channels (other orders: a lane per point)
  if (g.C > 1 && g.sc == 1) {
    GRID_DISPATCH(dtype, tri_fwd_rows<scalar_t>(CP(grid), g, CP(xyz), CP(xyz_min), CP(xyz_max), n,
                                                MP(out), ST(stream)));
    return launch_status("grid_sample_fwd");
  }
  GRID_DISPATCH(dtype, k_tri_fwd<scalar_t><<<grid_for(n, 256), 256, 0, ST(stream)>>>(
                           CP(grid), g, CP(xyz), CP(xyz_min), CP(xyz_max), n, MP(out)));
  return launch_status("grid_sample_fwd");
}

int vx_grid_sample_bwd(int dtype, void* grad, const int64_t* geom, const void* xyz,
                       const void* xyz_min, const void* xyz_max, int64_t n, const void* gout,
                       void* stream) {
  GridDesc g;
  if (int st = make_desc(geom, g)) return st;
  VX_CHECK_ARG(n >= 0, "grid_sample: n < 0");
  if (n == 0) return VX_OK;
  // channels innermost, at most a wave's lanes of them: lanes over a point's channels
  if (g.C > 1 && g.C <= 64 && g.sc == 1) {
    GRID_DISPATCH(dtype, tri_bwd_rows<scalar_t>(MP(grad), g, CP(xyz), CP(xyz_min), CP(xyz_max), n,
                                                CP(gout), ST(stream)));
    return launch_status("grid_sample_bwd");
  }
  GRID_DISPATCH(dtype, k_tri_bwd<scalar_t><<<grid_for(n, 256), 256, 0, ST(stream)>>>(
                           MP(grad), g, CP(xyz), CP(xyz_min), CP(xyz_max), n, CP(gout)));
  return launch_status("grid_sample_bwd");
}

int vx_sample_sdfs_fwd(int dtype, const void* grid, const int64_t* geom, const void* xyz,
                       const void* xyz_min, const void* xyz_max, const void* disp, int nd,
                       double voxel_size, int use_grad_norm, int64_t n, void* feat, void* grad,
                       void* stream) {
  GridDesc g;
  if (int st = make_desc(geom, g)) return st;
  VX_CHECK_ARG(g.C == 1, "sample_sdfs: the SDF grid must have one channel");
  VX_CHECK_ARG(n >= 0 && nd >= 1, "sample_sdfs: bad sizes");
  if (n == 0) return VX_OK;
  GRID_DISPATCH(dtype, k_sdfs_fwd<scalar_t><<<grid_for(n, 256), 256, 0, ST(stream)>>>(
                           CP(grid), g, CP(xyz), CP(xyz_min), CP(xyz_max), CP(disp), nd,
                           (scalar_t)voxel_size, use_grad_norm, n, MP(feat), MP(grad)));
  return launch_status("sample_sdfs_fwd");
}

int vx_sample_sdfs_bwd(int dtype, void* ggrid, const void* grid, const int64_t* geom,
                       const void* xyz, const void* xyz_min, const void* xyz_max,
                       const void* disp, int nd, double voxel_size, int use_grad_norm, int64_t n,
                       const void* gfeat, const void* ggrad, void* stream) {
  GridDesc g;
  if (int st = make_desc(geom, g)) return st;
  VX_CHECK_ARG(g.C == 1, "sample_sdfs: the SDF grid must have one channel");
  VX_CHECK_ARG(n >= 0 && nd >= 1, "sample_sdfs: bad sizes");
  if (n == 0) return VX_OK;
  GRID_DISPATCH(dtype, k_sdfs_bwd<scalar_t><<<grid_for(n, 256), 256, 0, ST(stream)>>>(
                           MP(ggrid), CP(grid), g, CP(xyz), CP(xyz_min), CP(xyz_max), CP(disp),
                           nd, (scalar_t)voxel_size, use_grad_norm, n, CP(gfeat), CP(ggrad)));
  return launch_status("sample_sdfs_bwd");
}

int vx_sdf_grad_fwd(int dtype, const void* grid, const int64_t* geom, const void* xyz,
                    const void* xyz_min, const void* xyz_max, double voxel_size, int64_t n,
                    void* sdf, void* grad, void* feat, void* stream) {
  GridDesc g;
  if (int st = make_desc(geom, g)) return st;
  VX_CHECK_ARG(g.C == 1, "sdf_grad: the SDF grid must have one channel");
  VX_CHECK_ARG(n >= 0, "sdf_grad: n < 0");
  if (n == 0) return VX_OK;
  GRID_DISPATCH(dtype, k_sdf_grad_fwd<scalar_t><<<grid_for(n, 256), 256, 0, ST(stream)>>>(
                           CP(grid), g, CP(xyz), CP(xyz_min), CP(xyz_max), (scalar_t)voxel_size,
                           n, MP(sdf), MP(grad), MP(feat)));
  return launch_status("sdf_grad_fwd");
}

int vx_sdf_grad_bwd(int dtype, void* ggrid, const int64_t* geom, const void* xyz,
                    const void* xyz_min, const void* xyz_max, double voxel_size, int64_t n,
                    const void* gsdf, const void* ggrad, const void* gfeat, void* stream) {
  GridDesc g;
  if (int st = make_desc(geom, g)) return st;
  VX_CHECK_ARG(g.C == 1, "sdf_grad: the SDF grid must have one channel");
  VX_CHECK_ARG(n >= 0, "sdf_grad: n < 0");
  if (n == 0) return VX_OK;
  // A wave takes its runs two by two, so a call of one to three waves is as long as their 32
  // turns (64 random points 12.6 us, 8.1 by themselves; 128 13.2, 10.3; 256 13.7, 16.4), and the
  // neighbour values' gradients, which the renderer never has, are the plain form's.
  if (!gfeat && n >= 256) {
    GRID_DISPATCH(dtype, k_sdf_grad_bwd_runs<scalar_t>
                  <<<grid_for(n, kScatterThreads), kScatterThreads, 0, ST(stream)>>>(
                      MP(ggrid), g, CP(xyz), CP(xyz_min), CP(xyz_max), (scalar_t)voxel_size, n,
                      CP(gsdf), CP(ggrad)));
    return launch_status("sdf_grad_bwd");
  }
  GRID_DISPATCH(dtype, k_sdf_grad_bwd<scalar_t><<<grid_for(n, 256), 256, 0, ST(stream)>>>(
                           MP(ggrid), g, CP(xyz), CP(xyz_min), CP(xyz_max), (scalar_t)voxel_size,
                           n, CP(gsdf), CP(ggrad), CP(gfeat)));
  return launch_status("sdf_grad_bwd");
}

int vx_dense_sdf_gradient_fwd(int dtype, const void* sdf, int X, int Y, int Z, double voxel_size,
                              void* out, void* stream) {
  VX_CHECK_ARG(X >= 1 && Y >= 1 && Z >= 1, "dense gradient: bad shape");
  VX_CHECK_ARG(X <= 65535 && Y <= 65535, "dense gradient: X and Y must be <= 65535");
  const dim3 grid((unsigned)cdiv(Z, 256), (unsigned)Y, (unsigned)X);
  GRID_DISPATCH(dtype, k_dense_grad_fwd<scalar_t><<<grid, 256, 0, ST(stream)>>>(
                           CP(sdf), X, Y, Z, (scalar_t)voxel_size, MP(out)));
  return launch_status("dense_sdf_gradient_fwd");
}

int vx_dense_sdf_gradient_bwd(int dtype, const void* gout, int X, int Y, int Z,
                              double voxel_size, void* gsdf, void* stream) {
  VX_CHECK_ARG(X >= 1 && Y >= 1 && Z >= 1, "dense gradient: bad shape");
  VX_CHECK_ARG(X <= 65535 && Y <= 65535, "dense gradient: X and Y must be <= 65535");
  GRID_DISPATCH(dtype, dense_grad_bwd<scalar_t>(CP(gout), X, Y, Z, (scalar_t)voxel_size, MP(gsdf),
                                                ST(stream)));
  return launch_status("dense_sdf_gradient_bwd");
}

int vx_total_variation_add_grad(int dtype, const void* param, void* grad, const int64_t* geom,
                                float wx, float wy, float wz, int dense_mode, void* stream) {
  GridDesc g;
  if (int st = make_desc(geom, g)) return st;
  const int64_t N = (int64_t)g.C * g.X * g.Y * g.Z;
  // wx /= 6; wy /= 6; wz /= 6 (total_variation_kernel.cu:76-78); the k and i axes both
  // take wz (total_variation_kernel.cu:27-32).
  wx /= 6;
  wy /= 6;
  wz /= 6;
  (void)wx;
  bool rows = false;
  GRID_DISPATCH(dtype, rows = (tv_rows<scalar_t, false>(g, CP(param), MP(grad), nullptr, wz, wy, wz,
                                                        dense_mode, ST(stream))));
  if (rows) return launch_status("total_variation_add_grad");
  GRID_DISPATCH(dtype, k_tv<scalar_t, false><<<grid_for(N, 256), 256, 0, ST(stream)>>>(
                           CP(param), MP(grad), nullptr, g, wz, wy, wz, dense_mode));
  return launch_status("total_variation_add_grad");
}

int vx_total_variation_add_grad_new(int dtype, const void* param, void* grad, const void* mask,
                                    const int64_t* geom, float wx, float wy, float wz,
                                    int dense_mode, void* stream) {
  GridDesc g;
  if (int st = make_desc(geom, g)) return st;
  const int64_t N = (int64_t)g.C * g.X * g.Y * g.Z;
  wx /= 6;
  wy /= 6;
  wz /= 6;
  bool rows = false;
  GRID_DISPATCH(dtype, rows = (tv_rows<scalar_t, true>(g, CP(param), MP(grad), CP(mask), wx, wy, wz,
                                                       dense_mode, ST(stream))));
  if (rows) return launch_status("total_variation_add_grad_new");
  GRID_DISPATCH(dtype, k_tv<scalar_t, true><<<grid_for(N, 256), 256, 0, ST(stream)>>>(
                           CP(param), MP(grad), CP(mask), g, wx, wy, wz, dense_mode));
  return launch_status("total_variation_add_grad_new");
}

int vx_sdf_query(const float* sdf, const int64_t* geom, const float* box, float voxel_size,
                 float res, const float* origin, int tile, float* out, float* normal, void* stream) {
  VX_CHECK_ARG(sdf && geom && box && origin, "sdf_query: missing argument");
  QueryArgs a;
  if (int st = make_desc(geom, a.g)) return st;
  VX_CHECK_ARG(a.g.C == 1, "sdf_query: the SDF grid must have one channel");
  VX_CHECK_ARG(tile >= 0 && tile <= 65535, "sdf_query: bad tile size");
  if (tile == 0) return VX_OK;
  VX_CHECK_ARG(out && normal, "sdf_query: missing output");
  a.sdf = sdf;
  for (int i = 0; i < 3; ++i) {
    a.mn[i] = box[i];
    a.mx[i] = box[3 + i];
    a.o[i] = origin[i];
  }
  a.voxel_size = voxel_size;
  a.step = 1.f / (res - 1.f);
  a.tile = tile;
  a.out = out;
  a.normal = normal;
  k_sdf_query<<<dim3((unsigned)cdiv(tile, 64), (unsigned)tile, (unsigned)tile), 64, 0, ST(stream)>>>(a);
  return launch_status("sdf_query");
}

int vx_maskcache_alpha(int dtype, const void* density, const int64_t* geom, const void* xyz,
                       const void* xyz_min, const void* xyz_max, double act_shift,
                       double voxel_size_ratio, double thres, int nearest, int64_t n,
                       uint8_t* out, void* stream) {
  GridDesc g;
  if (int st = make_desc(geom, g)) return st;
  VX_CHECK_ARG(g.C == 1, "maskcache: the density grid must have one channel");
  VX_CHECK_ARG(n >= 0, "maskcache: n < 0");
  if (n == 0) return VX_OK;
  GRID_DISPATCH(dtype, k_maskcache_alpha<scalar_t><<<grid_for(n, 256), 256, 0, ST(stream)>>>(
                           CP(density), g, CP(xyz), CP(xyz_min), CP(xyz_max),
                           (scalar_t)act_shift, (scalar_t)voxel_size_ratio, (scalar_t)thres,
                           nearest, n, out));
  return launch_status("maskcache_alpha");
}

int vx_zero(int dtype, void* p, int64_t n, void* stream) {
  VX_CHECK_ARG(n >= 0, "zero: n < 0");
  if (n == 0) return VX_OK;
  GRID_DISPATCH(dtype, k_zero<scalar_t><<<grid_for(n, 256), 256, 0, ST(stream)>>>(MP(p), n));
  return launch_status("zero");
}

}  // extern "C"
