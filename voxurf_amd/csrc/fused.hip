// Fused per-ray kernels of the fine training step (gfx950).
//
// The reference runs the fine forward as ~40 separate passes over materialised sample
// arrays (lib/voxurf_fine.py:620-802): sample every step of every ray, compact the
// in-box ones, gather the SDF at 7 points per sample, NeuS alpha, compact alpha > thres,
// walk the transmittance per ray, compact weight > thres, then features and colour.
// Here one wavefront owns one ray and does all of that in registers, 64 consecutive
// steps per iteration, and stops once the transmittance walk has terminated (every
// later sample has weight 0 and no gradient in the reference).  Only the samples of the
// walk range (alpha > thres, up to and including the terminating one: the only samples
// with a gradient) leave the kernel, in per-ray slots of two float4 (position and the
// transmittance before the sample; SDF gradient and SDF value).  The gather and the
// backward recompute alpha and weight from those (the same arithmetic, so the same
// bits) instead of walking the ray again.
//
// The arithmetic of every sample is the drop-in ops' own (voxel.h), and the
// transmittance walk is the reference's sequential float recurrence, so the survivor
// set, weights and alphainv_last equal those of the op-by-op pipeline.
#include "fine.h"

namespace vx {

// 64 steps of a ray in ascending order, a lane each: sample points, SDF + gradient, NeuS alpha,
// then the exact sequential transmittance walk over the active ones.
struct ChunkState {
  float q[3];
  float sdf, grad[3];
  NeusFwd<float> nf;
  float alpha, myT, w;
  bool inb, act, inrange, surv;
  bool shared;  // the sample's 7-point cells lie in the 32 voxels around its cell (sdf7)
};

__device__ __forceinline__ void run_chunk(const FusedGeom& G, const float* start, const float* dir,
                                          const float* vd, const SkipRay& sk, bool each,
                                          bool valid, int64_t s, int lane,
                                          float& T, bool& stopped, int& stop_lane,
                                          ChunkState& cs) {
  bool out = true;
  if (valid) out = sample_point<float>(start, dir, G.mn, G.mx, G.stepdist, s, cs.q[0], cs.q[1], cs.q[2]);
  cs.inb = valid && !out;
  if (G.mc && cs.inb) cs.inb = maskcache_pass(G, cs.q);
  cs.alpha = 0.f;
  cs.shared = true;
  cs.sdf = 0.f;
  cs.grad[0] = cs.grad[1] = cs.grad[2] = 0.f;
  // a sample in empty space far enough from the surface has alpha <= thres (inactive)
  // whatever its exact SDF (each: not yet known of its eight): its lookups are skipped
  const bool skip = each && cs.inb && skip_at(G, sk, s);
  if (cs.inb && !skip) {
    sdf7<float>(G.sdf, G.gs, cs.q, G.mn, G.mx, G.voxel_size, cs.sdf, cs.grad, nullptr, &cs.shared);
    cs.nf = neus_fwd<float>(vd, cs.grad, cs.sdf, G.stepdist, G.inv_s);
    cs.alpha = clip01(cs.nf.a);
  }
  cs.act = cs.inb && cs.alpha > G.thres;
  uint64_t mm = __ballot(cs.act);
  stop_lane = 64;
  cs.myT = 1.f;
  const double through = 1.0 - (double)cs.alpha;
  while (mm) {
    const int k = __ffsll((unsigned long long)mm) - 1;
    mm &= mm - 1;
    if (lane == k) cs.myT = T;
    if (walk_step(T, through, k)) {
      stopped = true;
      stop_lane = k;
      break;
    }
  }
  cs.inrange = cs.act && lane <= stop_lane;
  cs.w = cs.myT * cs.alpha;
  cs.surv = cs.inrange && cs.w > G.thres;
}

__device__ __forceinline__ void mark_page(uint32_t* pages, int64_t addr) {
  pages[addr >> kPageShift] = 1u;
}

// Flag the page(s) holding the C channels of trilinear corner `corner` (0..7, x outer,
// z inner) of t: one run of C floats when channels are innermost, C strided words
// otherwise.
__device__ __forceinline__ void mark_corner_pages(uint32_t* pages, const GridDesc& g,
                                                  const Tri<float>& t, int corner) {
  const int x = t.x0 + (corner >> 2), y = t.y0 + ((corner >> 1) & 1), z = t.z0 + (corner & 1);
  if (!in_grid<float>(x, y, z, g)) return;
  const int64_t o = x * g.sx + y * g.sy + z * g.sz;
  if (g.sc == 1) {
    mark_page(pages, o);
    mark_page(pages, o + g.C - 1);
  } else {
    for (int ch = 0; ch < g.C; ++ch) mark_page(pages, o + ch * g.sc);
  }
}

// mark_corner_pages flags the two end pages of a channels-innermost corner run, which
// must then span at most two pages.
static int check_corner_pages(const char* who, const FusedGeom& G, const void* pages) {
  VX_CHECK_ARG(!pages || G.gk.sc != 1 || G.gk.C <= kPageElems,
               "%s: page flags of a channels-innermost k0 need at most %d channels", who,
               kPageElems);
  return VX_OK;
}

// Set the page flag of every voxel within `reach` cells of q's cell (the block
// [c0 - reach, c0 + 1 + reach] per axis, clamped to the grid).  Needs z innermost and
// contiguous (sz == 1) with 2 reach + 2 <= a page: each z run of the block then lies in
// at most two pages, those of its end voxels.
__device__ __forceinline__ void mark_block_pages(uint32_t* __restrict__ pages, const GridDesc& g,
                                                 const float q[3], const float* mn,
                                                 const float* mx, int reach) {
  Tri<float> t0;
  t0.init(world_to_index(q[0], mn[0], mx[0] - mn[0], g.X),
          world_to_index(q[1], mn[1], mx[1] - mn[1], g.Y),
          world_to_index(q[2], mn[2], mx[2] - mn[2], g.Z));
  const int zl = max(t0.z0 - reach, 0), zh = min(t0.z0 + 1 + reach, g.Z - 1);
  const int xl = max(t0.x0 - reach, 0), xh = min(t0.x0 + 1 + reach, g.X - 1);
  const int yl = max(t0.y0 - reach, 0), yh = min(t0.y0 + 1 + reach, g.Y - 1);
  if (zl > zh || xl > xh || yl > yh) return;
  for (int x = xl; x <= xh; ++x)
    for (int y = yl; y <= yh; ++y) {
      const int64_t row = x * g.sx + y * g.sy;
      pages[(row + zl) >> kPageShift] = 1u;
      pages[(row + zh) >> kPageShift] = 1u;
    }
}

// What bounds it is the issue of its vector instructions (83% of the time at 131,072 rays):
// 4,440 a ray when every 64 steps were sampled and tested for empty space by themselves and
// the steps around the surface spread over two or three of them, 2,245 with empty space told
// by eights and the rest taken 64 together (1162 -> 671 us; 50 -> 35 at 1000 rays).
//
// Forward.  Outputs per ray: cnt (survivors), last (alphainv_last), stats
// {m0 in the box up to the end of the 64 steps that the walk ended in, m1 in the walk range
// (= slots used), m0 of the whole ray (if count_all)};
// per walk-range sample k of ray r at slot r*cap + k: s4 = (x, y, z, T before the
// sample), g4 = (gx, gy, gz, sdf).
__global__ void __launch_bounds__(256, 3) k_fused_fwd(
    FusedGeom G, const float* __restrict__ rays_o, const float* __restrict__ rays_d,
    const float* __restrict__ viewdirs, int64_t n_rays, int cap, float4* __restrict__ s4,
    float4* __restrict__ g4, int64_t* __restrict__ cnt_out, float* __restrict__ last_out,
    int* __restrict__ stats, int count_all, int* __restrict__ overflow,
    unsigned long long* __restrict__ walk_total, uint32_t* __restrict__ k0_pages,
    uint32_t* __restrict__ sdf_pages, int hier_reach) {
  const int lane = threadIdx.x & 63;
  const int64_t waves = (int64_t)gridDim.x * (blockDim.x >> 6);
  // walk-range samples of this wave's rays (lane 0), summed per block at the end: one
  // atomic per block on walk_total instead of one per ray
  __shared__ unsigned long long wave_m1[256 / 64];
  unsigned long long my_m1 = 0;
  for (int64_t r = blockIdx.x * (int64_t)(blockDim.x >> 6) + (threadIdx.x >> 6); r < n_rays;
       r += waves) {
    float start[3], dir[3];
    int64_t n;
    ray_setup(G, rays_o + 3 * r, rays_d + 3 * r, start, dir, n);
    const float* vd = viewdirs + 3 * r;
    SkipRay sk;
    skip_ray(G, start, dir, vd, sk);
    // (a mask cache's samples are counted one by one)
    const bool grouped = sk.eights && !G.mc;
    float T = 1.f;
    bool stopped = false;
    int cnt = 0, m0 = 0, m1 = 0, stop_lane = 64;
    int64_t base = 0, window = 0, s = 0;
    uint64_t live = 0;  // eights of the window (of 512 steps) that are not empty space
    while (!stopped) {
      bool valid;
      if (grouped) {
        // the next eight such eights, wherever they are, side by side
        while (!live && base < n) {
          const int64_t s0 = base + kSkipGroup * lane;
          live = __ballot(s0 < n && !skip_at(G, sk, s0 + kSkipGroup / 2));
          window = base;
          base += 64 * kSkipGroup;
        }
        if (!live) break;
        const int rank = __popcll(live & lanemask_lt(lane));
        const bool mine = live >> lane & 1;
        // rank k's lane number to lane k (the others' to a lane that is not read)
        const int at = __builtin_amdgcn_ds_permute(4 * (mine && rank < 8 ? rank : 63), lane);
        const int g = __shfl(at, lane >> 3, 64);
        s = window + kSkipGroup * g + (lane & 7);
        valid = (lane >> 3) < __popcll(live) && s < n;
        live = __ballot(mine && rank >= 8);
      } else {
        if (base >= n) break;
        s = base + lane;
        valid = s < n;
        base += 64;
      }
      ChunkState cs;
      run_chunk(G, start, dir, vd, sk, sk.on && !grouped, valid, s, lane, T, stopped, stop_lane, cs);
      if (!grouped) m0 += __popcll(__ballot(cs.inb));
      const uint64_t im = __ballot(cs.inrange);
      if (cs.inrange) {
        const int k = m1 + __popcll(im & lanemask_lt(lane));
        if (k < cap) {
          const int64_t slot = r * cap + k;
          s4[slot] = make_float4(cs.q[0], cs.q[1], cs.q[2], cs.myT);
          g4[slot] = make_float4(cs.grad[0], cs.grad[1], cs.grad[2], cs.sdf);
        }
      }
      m1 += __popcll(im);
      // every SDF-gradient page the backward's stencil scatter of this walk-range sample
      // can write
      if (sdf_pages && cs.inrange) sdf7_mark_pages<float>(sdf_pages, G.gs, cs.q, G.mn, G.mx, cs.shared);
      // the displaced-sample stencils of the survivors' rgbnet rows (sample_sdfs)
      if (sdf_pages && hier_reach > 0 && cs.surv) mark_block_pages(sdf_pages, G.gs, cs.q, G.mn, G.mx, hier_reach);
      cnt += __popcll(__ballot(cs.surv));
      if (k0_pages && cs.surv) {
        // every k0_grad page the feature scatter of this survivor can write
        Tri<float> t;
        t.init(world_to_index(cs.q[0], G.mn[0], G.mx[0] - G.mn[0], G.gk.X),
               world_to_index(cs.q[1], G.mn[1], G.mx[1] - G.mn[1], G.gk.Y),
               world_to_index(cs.q[2], G.mn[2], G.mx[2] - G.mn[2], G.gk.Z));
        for (int corner = 0; corner < 8; ++corner) mark_corner_pages(k0_pages, G.gk, t, corner);
      }
    }
    if (grouped) {
      // samples in the box: along each axis a step's coordinate never turns back (rounding is
      // monotonic), so they are one run of steps, and its ends are among the first and last 64
      auto in_box = [&](int64_t t) {
        float q[3];
        return t >= 0 && t < n &&
               !sample_point<float>(start, dir, G.mn, G.mx, G.stepdist, t, q[0], q[1], q[2]);
      };
      const int64_t s_stop = __shfl(s, stop_lane & 63, 64);
      const int64_t upto = stopped ? ((s_stop >> 6) + 1) << 6 : n;
      const uint64_t first = __ballot(in_box(lane)), last = __ballot(in_box(n - 64 + lane));
      if (first && last) {
        const int64_t lo = __ffsll((unsigned long long)first) - 1;
        const int64_t hi = n - 1 - __clzll((long long)last);
        m0 = (int)((hi < upto ? hi + 1 : upto) - lo);
      } else {
        for (int64_t t = 0; t < upto; t += 64) m0 += __popcll(__ballot(t + lane < upto && in_box(t + lane)));
      }
      base = upto;
    }
    int m0_all = m0;
    if (count_all) {
      // in-box samples after termination (bbox tests only), for sample statistics
      for (; base < n; base += 64) {
        const int64_t s = base + lane;
        float q[3];
        bool out = true;
        if (s < n) out = sample_point<float>(start, dir, G.mn, G.mx, G.stepdist, s, q[0], q[1], q[2]);
        m0_all += __popcll(__ballot(s < n && !out));
      }
    }
    if (lane == 0) {
      if (m1 > cap) {
        atomicOr(overflow, 1);
        m1 = cap;
      }
      my_m1 += (unsigned long long)m1;
      cnt_out[r] = cnt;
      last_out[r] = T;
      stats[3 * r + 0] = m0;
      stats[3 * r + 1] = m1;
      stats[3 * r + 2] = m0_all;
    }
  }
  if (walk_total) {
    if (lane == 0) wave_m1[threadIdx.x >> 6] = my_m1;
    __syncthreads();
    if (threadIdx.x == 0) {
      unsigned long long t = 0;
      for (int w = 0; w < (int)(blockDim.x >> 6); ++w) t += wave_m1[w];
      if (t) atomicAdd(walk_total, t);
    }
  }
}

// Survivors (w > thres) of the walk-range slots: (x, y, z, w), (gradient, sdf) and the ray at
// rows off[r] .. off[r] + cnt[r], sixteen lanes a ray.  What a row needs beyond that is built
// by kernels over whole tiles of rows (k_fused_rows, k_voxurf_rows).  Both in one kernel, a
// wavefront per ray, was bound by the instructions of half-empty wavefronts: a view embedding
// per ray in sixteen of 64 lanes, both branches of sinf and cosf four columns deep (462 us of
// a 131,072-ray render with 1.4 M rows, 41 at 1000 rays); in two: 29 + 140 us, and 4 + 7.
__global__ void __launch_bounds__(256) k_survivors(
    FusedGeom G, const float* __restrict__ viewdirs, int64_t n_rays, int cap,
    const float4* __restrict__ s4, const float4* __restrict__ g4, const int* __restrict__ stats,
    const int64_t* __restrict__ cnt, const int64_t* __restrict__ off_incl, int64_t max_rows,
    float4* __restrict__ P4, float4* __restrict__ G4, int* __restrict__ rid,
    uint32_t* __restrict__ pages) {
  const int l = threadIdx.x & 15, sub = (threadIdx.x & 63) >> 4;
  const int64_t r = blockIdx.x * (int64_t)(blockDim.x >> 4) + (threadIdx.x >> 4);
  int64_t c = 0, o = 0;
  int c1 = 0;
  float vd[3] = {0.f, 0.f, 0.f};
  if (r < n_rays) {
    c = cnt[r];
    c1 = stats[3 * r + 1];
    o = off_incl[r] - c;
    for (int e = 0; e < 3; ++e) vd[e] = viewdirs[3 * r + e];
    // past the output capacity nothing is written
    if (c == 0 || (o >= max_rows && !pages)) c1 = 0;
  }
  int64_t ks = 0;
  for (int base = 0; __any(base < c1 && ks < c); base += 16) {
    const int k = base + l;
    float4 a = make_float4(0.f, 0.f, 0.f, 0.f), b = a;
    bool surv = false;
    if (k < c1) {
      a = s4[r * cap + k];
      b = g4[r * cap + k];
      SlotSample ss;
      load_slot(G, vd, a, b, ss);
      surv = ss.w > G.thres;
      a.w = ss.w;
    }
    const uint32_t sm = (uint32_t)(__ballot(surv) >> (16 * sub)) & 0xffffu;
    // rows past the forward's survivor count are never written (they cannot occur: the
    // recomputed weights are the forward's)
    const int64_t j = ks + __popc(sm & ((1u << l) - 1u));
    if (surv && j < c) {
      if (o + j < max_rows) {
        P4[o + j] = a;
        G4[o + j] = b;
        rid[o + j] = (int)r;
      }
      if (pages) {
        Tri<float> t;
        t.init(world_to_index(a.x, G.mn[0], G.mx[0] - G.mn[0], G.gk.X),
               world_to_index(a.y, G.mn[1], G.mx[1] - G.mn[1], G.gk.Y),
               world_to_index(a.z, G.mn[2], G.mx[2] - G.mn[2], G.gk.Z));
        for (int corner = 0; corner < 8; ++corner) mark_corner_pages(pages, G.gk, t, corner);
      }
    }
    ks += __popc(sm);
  }
}

void launch_survivors(const FusedGeom& G, const float* viewdirs, int64_t n_rays, int cap,
                      const void* s4, const void* g4, const int* stats, const int64_t* cnt,
                      const int64_t* off_incl, int64_t max_rows, void* P4, void* G4, int* rid,
                      uint32_t* pages, hipStream_t st) {
  k_survivors<<<(unsigned)cdiv(n_rays, 16), 256, 0, st>>>(
      G, viewdirs, n_rays, cap, (const float4*)s4, (const float4*)g4, stats, cnt, off_incl,
      max_rows, (float4*)P4, (float4*)G4, rid, pages);
}

// rgbnet rows X = [k0 (C) | normal (3) | view PE (3 + 6 nf) | 0 pad], 64 of the survivors a
// workgroup and pass: k0 with a lane per row and four channels (or channel), the embedding
// once for each ray among them (their rows are neighbours) with a lane per sine and cosine,
// then the columns past C with sixteen lanes a row.
// normal = grad / (|grad| + 1e-5) (lib/voxurf_fine.py:766 with the 1e-5 of :810);
// view PE = [v, sin(v_i f_j), cos(v_i f_j)] with f_j = 2^j (lib/voxurf_fine.py:694-695).
constexpr int kRowTile = 64;

__global__ void __launch_bounds__(256) k_fused_rows(
    FusedGeom G, const float* __restrict__ viewdirs, int64_t n_rays, int n_freq,
    const int64_t* __restrict__ off_incl, int xstride, int64_t max_rows, float* __restrict__ X,
    const float4* __restrict__ P4, const float4* __restrict__ G4, const int* __restrict__ rid) {
  __shared__ float4 pos[kRowTile], nrml[kRowTile];  // nrml.w: the slot of the row's ray
  __shared__ int ray[kRowTile];                     // [slot]
  __shared__ int n_slots;
  __shared__ float4 tail[kRowTile][16];             // [slot]: embeddings at column - (C & ~3)
  const int tid = threadIdx.x;
  const int C = G.gk.C, c0 = C & ~3;
  const int npe = 3 + 6 * n_freq, half = 3 * n_freq;
  // channels innermost with 16-byte aligned corner rows: four channels per load
  const bool vec4 = G.gk.sc == 1 && (C & 3) == 0 && ((G.gk.sx | G.gk.sy | G.gk.sz) & 3) == 0 &&
                    (reinterpret_cast<uintptr_t>(G.k0) & 15) == 0;
  const int64_t total = off_incl[n_rays - 1];
  const int64_t rows = total < max_rows ? total : max_rows;
  for (int64_t row0 = blockIdx.x * (int64_t)kRowTile; row0 < rows; row0 += gridDim.x * (int64_t)kRowTile) {
    const int m = (int)(rows - row0 < kRowTile ? rows - row0 : kRowTile);
    if (tid < kRowTile) {
      const int64_t j = row0 + (tid < m ? tid : m - 1);
      const float4 a = P4[j], b = G4[j];
      const int rr = rid[j];
      const int before = __shfl_up(rr, 1, 64);
      const uint64_t heads = __ballot(tid == 0 || rr != before);
      const int slot = __popcll(heads & (lanemask_lt(tid) | (1ull << tid))) - 1;
      const float nrm = sqrtf(b.x * b.x + b.y * b.y + b.z * b.z) + 1e-5f;
      pos[tid] = a;
      nrml[tid] = make_float4(b.x / nrm, b.y / nrm, b.z / nrm, __int_as_float(slot));
      if (heads >> tid & 1) ray[slot] = min(max(rr, 0), (int)n_rays - 1);
      if (tid == 0) n_slots = __popcll(heads);
    }
    __syncthreads();
    const int nch = vec4 ? C >> 2 : C;
    for (int i = tid; i < m * nch; i += 256) {
      const int row = (int)((unsigned)i / (unsigned)nch), ch = i - row * nch;
      const float4 q = pos[row];
      Tri<float> t;
      t.init(world_to_index(q.x, G.mn[0], G.mx[0] - G.mn[0], G.gk.X),
             world_to_index(q.y, G.mn[1], G.mx[1] - G.mn[1], G.gk.Y),
             world_to_index(q.z, G.mn[2], G.mx[2] - G.mn[2], G.gk.Z));
      float* x = X + (row0 + row) * xstride;
      if (vec4) *reinterpret_cast<float4*>(x + 4 * ch) = tri_gather4(G.k0, G.gk, t, 4 * ch);
      else x[ch] = tri_gather(G.k0, G.gk, t, ch);
    }
    const int npt = half + 3, nt = n_slots * npt;
    for (int i = 255 - tid; i < nt; i += 256) {
      const int slot = (int)((unsigned)i / (unsigned)npt), k = i - slot * npt;
      const float* vd = viewdirs + 3 * (int64_t)ray[slot];
      float* pe = reinterpret_cast<float*>(tail[slot]) + (C + 3 - c0);
      if (k < 3) {
        pe[k] = vd[k];
      } else {
        const int q = k - 3;  // (component, freq) in component-major order
        const int comp = q / n_freq, f = q % n_freq;
        const float arg = vd[comp] * (float)(1 << f);
        pe[3 + q] = sinf(arg);
        pe[3 + half + q] = cosf(arg);
      }
    }
    __syncthreads();
    // the columns past C
    for (int row = tid >> 4; row < m; row += 16) {
      const float4 n4 = nrml[row];
      const float4* tl = tail[__float_as_int(n4.w)];
      float* x = X + (row0 + row) * xstride;
      auto value = [&](int col, float pe) {
        if (col < C + 3) return col == C ? n4.x : (col == C + 1 ? n4.y : n4.z);
        return col < C + 3 + npe ? pe : 0.f;
      };
      if ((C & 3) == 0) {
        const int col = C + 4 * (tid & 15);
        if (col < xstride) {
          const float4 pe = tl[tid & 15];
          *reinterpret_cast<float4*>(x + col) = make_float4(
              value(col, pe.x), value(col + 1, pe.y), value(col + 2, pe.z), value(col + 3, pe.w));
        }
      } else {
        for (int col = C + (tid & 15); col < xstride; col += 16)
          x[col] = value(col, reinterpret_cast<const float*>(tl)[col - c0]);
      }
    }
    __syncthreads();
  }
}

// Compositing, loss and the colour-side adjoints, one thread per ray:
//   rgb_marched = sum_j w_j sigmoid(logit_j) + last * bg          (lib/voxurf_fine.py:761-763)
//   loss_r = sum_c (rgb_marched - target)^2,  g = 2 (rgb_marched - target) / (3 N)
//   dlogit_j = (w_j g) * rgb (1 - rgb);  gw_j = <g, rgb_j>;  glast = <g, bg>;
//   S_r = sum_j gw_j w_j  (total of the transmittance adjoint's suffix sums)
__global__ void __launch_bounds__(256) k_fused_composite(
    int64_t n_rays, const int64_t* __restrict__ cnt, const int64_t* __restrict__ off_incl,
    const float* __restrict__ logits, int lstride, const float4* __restrict__ P4,
    const float* __restrict__ last, const float* __restrict__ target, float bg, float inv_count,
    float* __restrict__ rgb_out, float* __restrict__ dlogit, float* __restrict__ gw,
    float* __restrict__ glast, float* __restrict__ S, float* __restrict__ loss_r,
    int64_t max_rows) {
  // sixteen lanes per ray (four rays per wavefront): lane sl takes the ray's rows
  // sl, sl + 16, ...; the per-ray sums close with 16-lane butterflies
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
    // a ray whose rows run past the buffers' capacity is left out (the caller repeats
    // the step with larger buffers)
    const int64_t c = ok && off_incl[r] <= max_rows ? cnt[r] : 0;
    const int64_t o = ok ? off_incl[r] - cnt[r] : 0;
    float acc[3] = {0.f, 0.f, 0.f};
    for (int64_t j = o + sl; j < o + c; j += SEG) {
      const float w = P4[j].w;
      for (int ch = 0; ch < 3; ++ch) {
        const float rgb = 1.f / (1.f + expf(-logits[j * lstride + ch]));
        acc[ch] += w * rgb;
      }
    }
    for (int ch = 0; ch < 3; ++ch) acc[ch] = seg_sum(acc[ch]);
    if (!ok) continue;
    const float lr = last[r];
    if (!target) {  // rendering only
      if (sl == 0)
        for (int ch = 0; ch < 3; ++ch) rgb_out[3 * r + ch] = acc[ch] + lr * bg;
      continue;
    }
    float g[3], l = 0.f;
    for (int ch = 0; ch < 3; ++ch) {
      const float v = acc[ch] + lr * bg;
      if (sl == 0) rgb_out[3 * r + ch] = v;
      const float d = v - target[3 * r + ch];
      l += d * d;
      g[ch] = 2.f * d * inv_count;
    }
    if (sl == 0) {
      loss_r[r] = l;
      glast[r] = (g[0] + g[1] + g[2]) * bg;
    }
    float s = 0.f;
    for (int64_t j = o + sl; j < o + c; j += SEG) {
      const float w = P4[j].w;
      float gwj = 0.f;
      for (int ch = 0; ch < 3; ++ch) {
        const float rgb = 1.f / (1.f + expf(-logits[j * lstride + ch]));
        gwj += g[ch] * rgb;
        dlogit[j * 3 + ch] = (w * g[ch]) * (rgb * (1.f - rgb));
      }
      gw[j] = gwj;
      s += gwj * w;
    }
    s = seg_sum(s);
    if (sl == 0) S[r] = s;
  }
}

// Feature-side adjoint per survivor: dX[:, 0:C] -> k0 grad (trilinear scatter);
// dX[:, C:C+3] (normal) -> d grad through n = g / (|g| + 1e-5); result stored in dgf.

__global__ void __launch_bounds__(256) k_fused_feat_bwd(
    FusedGeom G, int64_t m, const int64_t* __restrict__ m_dev, const float* __restrict__ dX,
    int dxs, const float4* __restrict__ P4, const float4* __restrict__ G4,
    float* __restrict__ k0_grad, float* __restrict__ dgf, uint32_t* __restrict__ pages) {
  if (m_dev) m = *m_dev < m ? *m_dev : m;  // the device row count, within the capacity
  const int C = G.gk.C;
  const int lane = threadIdx.x & 63, grp = lane >> 4, cl = lane & 15;
  const int64_t nwaves = (int64_t)gridDim.x * (blockDim.x >> 6);
  for (int64_t base = ((int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) * 64; base < m;
       base += nwaves * 64) {
    // Trilinear scatter of the feature adjoint: four samples per pass, sixteen lanes
    // per sample, lane cl taking channels cl, cl + 16, ...  With channels innermost the
    // lanes of one atomic instruction hit one or two cache lines per sample instead of
    // one line per lane.  The four samples are consecutive rows (survivors of a ray in
    // depth order): those in the same cell sum their corner terms first, and the first
    // of them issues the atomics.
    for (int i = 0; i < 16; ++i) {
      if (base + 4 * i >= m) break;  // uniform over the wavefront
      const int64_t j = base + 4 * i + grp;
      const bool valid = j < m;
      const float4 a = P4[valid ? j : m - 1];
      Tri<float> t;
      t.init(world_to_index(a.x, G.mn[0], G.mx[0] - G.mn[0], G.gk.X),
             world_to_index(a.y, G.mn[1], G.mx[1] - G.mn[1], G.gk.Y),
             world_to_index(a.z, G.mn[2], G.mx[2] - G.mn[2], G.gk.Z));
      if (!valid) t.x0 = -2 - grp;  // matches no cell
      const int px = __shfl(t.x0, (lane - 16) & 63, 64), py = __shfl(t.y0, (lane - 16) & 63, 64),
                pz = __shfl(t.z0, (lane - 16) & 63, 64);
      const bool head = grp == 0 || px != t.x0 || py != t.y0 || pz != t.z0;
      const uint64_t hb = __ballot(head);
      // run index of this sample among the four (head flags of groups 0..grp)
      int rid = 0;
#pragma unroll
      for (int q = 0; q < 4; ++q) rid += q <= grp && ((hb >> (16 * q)) & 1ull) ? 1 : 0;
      for (int ch0 = 0; ch0 < C; ch0 += 16) {
        const int ch = ch0 + cl;
        const float go = valid && ch < C ? dX[j * dxs + ch] : 0.f;
        float v[8];
#pragma unroll
        for (int b = 0; b < 8; ++b) v[b] = t.w(b >> 2, (b >> 1) & 1, b & 1) * go;
#pragma unroll
        for (int off = 16; off < 64; off <<= 1) {
          const int orid = __shfl_down(rid, off, 64);
          const bool same = grp + off / 16 < 4 && orid == rid;
#pragma unroll
          for (int b = 0; b < 8; ++b) {
            const float o = __shfl_down(v[b], off, 64);
            if (same) v[b] += o;
          }
        }
        if (valid && head && ch < C) {
#pragma unroll
          for (int b = 0; b < 8; ++b) {
            const int x = t.x0 + (b >> 2), y = t.y0 + ((b >> 1) & 1), z = t.z0 + (b & 1);
            if (v[b] != 0.f && in_grid<float>(x, y, z, G.gk))
              atomic_add(&k0_grad[ch * G.gk.sc + x * G.gk.sx + y * G.gk.sy + z * G.gk.sz], v[b]);
          }
        }
      }
      if (valid && pages && cl < 8) mark_corner_pages(pages, G.gk, t, cl);
    }
    // adjoint of the normal n = g / (|g| + 1e-5): one sample per lane
    const int64_t j = base + lane;
    if (j < m) {
      const float4 b = G4[j];
      const float gvec[3] = {b.x, b.y, b.z};
      const float dn[3] = {dX[j * dxs + C], dX[j * dxs + C + 1], dX[j * dxs + C + 2]};
      const float nr = sqrtf(gvec[0] * gvec[0] + gvec[1] * gvec[1] + gvec[2] * gvec[2]);
      const float den = nr + 1e-5f;
      const float dot = gvec[0] * dn[0] + gvec[1] * dn[1] + gvec[2] * dn[2];
      const float k = nr > 0.f ? dot / (nr * den) : 0.f;
      for (int q = 0; q < 3; ++q) dgf[3 * j + q] = (dn[q] - gvec[q] * k) / den;
    }
  }
}

// The SDF backward in five passes (brick-binned, LDS-staged scatter), in two phases: the
// first needs only the compositing's adjoints and can run beside the rgbnet backward,
// the second adds the survivors' adjoints from the colour side and scatters.
//
// The grid is cut into 16^3-voxel bricks, each owned by one workgroup of the last pass.
// Phase 1 (vx_fused_fine_bwd_alpha):
// 1. k_bwd_alpha, over each ray's stored walk-range samples, kBwdSeg lanes per ray
//    (kBwdSeg samples per pass; a ray holds about a dozen walk-range samples, so a whole
//    wave per ray would leave most lanes idle):
//      dalpha_i = gw_i T_i - back_i / (1 - alpha_i + 1e-10)   on the walk range,
//      back_i = glast * last + S_r - sum_{survivors j <= i} gw_j w_j
//    (render_utils_kernel.cu:654-677 with the suffix sum written as total - prefix), then
//    the NeuS adjoint: the sample's adjoints of its centre SDF value and of its gradient
//    replace g4[slot] (gx, gy, gz, sdf) by (ggx, ggy, ggz, gsdf).  The voxels its 7-point
//    stencil reaches span one or two bricks per axis; the first brick and the three
//    "spans the next brick" bits, with a survivor bit, replace s4[slot].w (T, no longer
//    needed), and the sample is counted in each of its (1 to 8) bricks, one atomic per
//    brick and run of consecutive samples with the same bricks.
// 2. k_brick_alloc: a segment of the slot-index list per non-empty brick (atomic
//    allocation: the bricks' order in the list does not matter) and the brick list.
// 3. k_bwd_bin: each sample's slot index into the segment of each of its bricks.
// Phase 2 (vx_fused_fine_bwd_grid):
// 4. k_bwd_stencil: the survivors' colour-side adjoints (normal, and centre SDF for the
//    reference fine model) added, then the stencil's adjoints: g4[slot] = (gd_z, gd_y,
//    gd_x, gsdf), gd = dL/dgrad_c / (clamped difference) / voxel_size for the cells
//    displaced by -+1 along zyx axis ax, and a bound on every corner term of the call.
// 5. k_bwd_bricks, one workgroup per non-empty brick: every sample binned to the brick
//    adds those of the 56 corner terms of its stencil (sdf7_scatter's terms) that fall in
//    the brick into a 16^3 LDS tile, then the tile's nonzero voxels are added to the SDF
//    gradient with plain loads and stores: each voxel belongs to one brick, so no other
//    workgroup writes it, and no atomics are left.
constexpr int kBrickShift = 4;
constexpr int kBrick = 1 << kBrickShift;
constexpr int kBrick3 = kBrick * kBrick * kBrick;

struct BrickGrid {
  int bx, by, bz;  // bricks per axis
};

// First brick and spans of a sample's stencil: bits 0-23 the brick (x major), bit 24 + a
// set when the stencil also reaches the next brick along world axis a (x, y, z); ind
// receives the sample's zyx index.
__device__ __forceinline__ uint32_t stencil_bricks(const FusedGeom& G, const BrickGrid& B,
                                                   const float q[3], float ind[3]) {
#pragma clang fp contract(off)
  const GridDesc& g = G.gs;
  Tri<float> t0;
  t0.init(world_to_index(q[0], G.mn[0], G.mx[0] - G.mn[0], g.X),
          world_to_index(q[1], G.mn[1], G.mx[1] - G.mn[1], g.Y),
          world_to_index(q[2], G.mn[2], G.mx[2] - G.mn[2], g.Z));
  int lo[3] = {t0.x0, t0.y0, t0.z0}, hi[3] = {t0.x0 + 1, t0.y0 + 1, t0.z0 + 1};
  zyx_index(q, G.mn, G.mx, g, ind);
#pragma unroll
  for (int ax = 0; ax < 3; ++ax)
#pragma unroll
    for (int side = 0; side < 2; ++side) {
      Tri<float> td;
      displaced_cell(g, ind, ax, side ? 1.f : -1.f, td);
      const int c[3] = {td.x0, td.y0, td.z0};
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        lo[k] = min(lo[k], c[k]);
        hi[k] = max(hi[k], c[k] + 1);
      }
    }
  const int nb[3] = {B.bx, B.by, B.bz};
  int b0[3];
  uint32_t span = 0u;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const int l = max(lo[k], 0) >> kBrickShift;
    const int h = min(max(hi[k], 0) >> kBrickShift, nb[k] - 1);
    b0[k] = min(l, nb[k] - 1);
    if (h > b0[k]) span |= 1u << (24 + k);
  }
  return (uint32_t)((b0[0] * B.by + b0[1]) * B.bz + b0[2]) | span;
}

// The k-th (0..7) brick of a code from stencil_bricks, or -1 when the code spans fewer.
__device__ __forceinline__ int code_brick(const BrickGrid& B, uint32_t code, int k) {
  const int dx = k >> 2, dy = (k >> 1) & 1, dz = k & 1;
  if ((dx && !(code >> 24 & 1u)) || (dy && !(code >> 25 & 1u)) || (dz && !(code >> 26 & 1u)))
    return -1;
  const int b = (int)(code & 0xFFFFFFu);
  return b + (dx * B.by + dy) * B.bz + dz;
}

// Bit 31 of a walk-range slot's brick code marks a survivor (weight > thres).
constexpr uint32_t kSurvivorBit = 0x80000000u;

// Lanes per ray (SEG) of the backward's two per-ray passes: a walk range holds about 13
// samples at 256^3, so 32 lanes take most rays in one pass, and two rays per wavefront
// give twice the wavefronts of sixteen lanes to hide the passes' memory round trips.
constexpr int kBwdSeg = 32;

template <int SEG>
__global__ void __launch_bounds__(256) k_bwd_alpha(
    FusedGeom G, BrickGrid B, const float* __restrict__ viewdirs, int64_t n_rays, int cap,
    float4* __restrict__ s4, float4* __restrict__ g4, const int* __restrict__ stats,
    const int64_t* __restrict__ cnt, const int64_t* __restrict__ off_incl,
    const float* __restrict__ last, const float* __restrict__ gw, const float* __restrict__ glast,
    const float* __restrict__ S, int* __restrict__ brick_cnt, int64_t max_rows) {
  const int lane = threadIdx.x & 63, grp = lane / SEG, sl = lane % SEG;
  const uint64_t seg_lt = sl ? ((1ull << sl) - 1ull) : 0ull;
  const uint64_t seg_mask = SEG == 64 ? ~0ull : ((1ull << (SEG & 63)) - 1ull);
  const int64_t groups = (int64_t)gridDim.x * (blockDim.x >> 6) * (64 / SEG);
  for (int64_t r0 = ((int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) * (64 / SEG);
       r0 < n_rays; r0 += groups) {
    const int64_t r = r0 + grp;
    // (a ray whose rows run past the buffers' capacity is left out, as in the composite)
    const bool ray_ok = r < n_rays && off_incl[r] <= max_rows;
    const float* vd = viewdirs + 3 * (ray_ok ? r : 0);
    const int c1 = ray_ok ? stats[3 * r + 1] : 0;
    const int64_t c_r = ray_ok ? cnt[r] : 0;
    const int64_t o = ray_ok ? off_incl[r] - c_r : 0;
    const float base_back = ray_ok ? glast[r] * last[r] + S[r] : 0.f;
    // every lane runs the same number of passes (the largest c1 of the four rays) so the
    // segment shuffles below always see their whole segment active
    int passes = (c1 + SEG - 1) / SEG;
#pragma unroll
    for (int off = SEG; off < 64; off <<= 1) {
      const int t = __shfl_xor(passes, off, 64);
      passes = t > passes ? t : passes;
    }
    float prefix = 0.f;
    int k_surv = 0;
    for (int ps = 0; ps < passes; ++ps) {
      const int k = ps * SEG + sl;
      const bool valid = k < c1;
      SlotSample ss;
      bool surv = false;
      if (valid) {
        load_slot(G, vd, s4[r * cap + k], g4[r * cap + k], ss);
        surv = ss.w > G.thres;
      } else {
        ss.w = 0.f;
      }
      const uint64_t sm = (__ballot(surv) >> (grp * SEG)) & seg_mask;
      float gwl = 0.f;
      const int64_t kk = k_surv + __popcll(sm & seg_lt);
      if (surv && kk < c_r) gwl = gw[o + kk];
      k_surv += __popcll(sm);
      // inclusive prefix of gw*w over the survivors of this pass
      const float c = gwl * ss.w;
      float incl = c;
#pragma unroll
      for (int off = 1; off < SEG; off <<= 1) {
        const float u = __shfl_up(incl, off, SEG);
        if (sl >= off) incl += u;
      }
      const float back = base_back - (prefix + incl);
      prefix += __shfl(incl, SEG - 1, SEG);
      uint32_t code = 0xFFFFFFFFu;
      if (valid) {
        const double den = (double)(1.f - ss.alpha) + 1e-10;
        const float da = (float)((double)(gwl * ss.myT) - (double)back / den);
        float gsdf, gg[3];
        neus_bwd<float>(vd, ss.nf, G.stepdist, G.inv_s, da, gsdf, gg);
        g4[r * cap + k] = make_float4(gg[0], gg[1], gg[2], gsdf);
        float ind[3];
        code = stencil_bricks(G, B, ss.q, ind);
        s4[r * cap + k].w = __uint_as_float(code | (surv ? kSurvivorBit : 0u));
      }
      // count the samples per brick: one atomic per brick and run of lanes with the
      // same bricks
      const uint32_t pc = __shfl_up(code, 1, SEG);
      const bool head = valid && (sl == 0 || pc != code);
      const uint64_t hm = (__ballot(head) >> (grp * SEG)) & seg_mask;
      const uint64_t vm = (__ballot(valid) >> (grp * SEG)) & seg_mask;
      if (head) {
        const uint64_t later = hm & ~((2ull << sl) - 1ull);
        const int end = later ? __ffsll((unsigned long long)later) - 1 : 64 - __clzll(vm);
        for (int q = 0; q < 8; ++q) {
          const int bq = code_brick(B, code, q);
          if (bq >= 0) atomicAdd(&brick_cnt[bq], end - sl);
        }
      }
    }
  }
}

// The colour side's adjoints of the survivors (dgf: of their gradient, dsf: of their
// centre SDF value) added to the alpha adjoints in g4, then the stencil's adjoints
// (gd_z, gd_y, gd_x, gsdf) and the largest |corner term| bound of the call; SEG lanes
// per ray as k_bwd_alpha, survivors from the code's survivor bit.
template <int SEG>
__global__ void __launch_bounds__(256) k_bwd_stencil(
    FusedGeom G, int64_t n_rays, int cap, const float4* __restrict__ s4, float4* __restrict__ g4,
    const int* __restrict__ stats, const int64_t* __restrict__ cnt,
    const int64_t* __restrict__ off_incl, const float* __restrict__ dgf,
    const float* __restrict__ dsf, uint32_t* __restrict__ term_max, int64_t max_rows) {
  const int lane = threadIdx.x & 63, grp = lane / SEG, sl = lane % SEG;
  const uint64_t seg_lt = sl ? ((1ull << sl) - 1ull) : 0ull;
  const uint64_t seg_mask = SEG == 64 ? ~0ull : ((1ull << (SEG & 63)) - 1ull);
  const int64_t groups = (int64_t)gridDim.x * (blockDim.x >> 6) * (64 / SEG);
  // largest |corner term| bound of this wave's samples (infinite if any is not finite)
  float tmax = 0.f;
  for (int64_t r0 = ((int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) * (64 / SEG);
       r0 < n_rays; r0 += groups) {
    const int64_t r = r0 + grp;
    const bool ray_ok = r < n_rays && off_incl[r] <= max_rows;
    const int c1 = ray_ok ? stats[3 * r + 1] : 0;
    const int64_t c_r = ray_ok ? cnt[r] : 0;
    const int64_t o = ray_ok ? off_incl[r] - c_r : 0;
    int passes = (c1 + SEG - 1) / SEG;
#pragma unroll
    for (int off = SEG; off < 64; off <<= 1) {
      const int t = __shfl_xor(passes, off, 64);
      passes = t > passes ? t : passes;
    }
    int k_surv = 0;
    for (int ps = 0; ps < passes; ++ps) {
#pragma clang fp contract(off)
      const int k = ps * SEG + sl;
      const bool valid = k < c1;
      float4 a = make_float4(0.f, 0.f, 0.f, 0.f), t = a;
      bool surv = false;
      if (valid) {
        a = s4[r * cap + k];
        t = g4[r * cap + k];
        surv = (__float_as_uint(a.w) & kSurvivorBit) != 0u;
      }
      const uint64_t sm = (__ballot(surv) >> (grp * SEG)) & seg_mask;
      float dg[3] = {0.f, 0.f, 0.f}, dsd = 0.f;
      const int64_t kk = k_surv + __popcll(sm & seg_lt);
      if (surv && kk < c_r) {
        const int64_t j = o + kk;
        dg[0] = dgf[3 * j];
        dg[1] = dgf[3 * j + 1];
        dg[2] = dgf[3 * j + 2];
        if (dsf) dsd = dsf[j];
      }
      k_surv += __popcll(sm);
      if (valid) {
        const float gsdf = t.w + dsd;
        const float gg[3] = {t.x + dg[0], t.y + dg[1], t.z + dg[2]};
        const float q[3] = {a.x, a.y, a.z};
        float ind[3];
        zyx_index(q, G.mn, G.mx, G.gs, ind);
        // the stencil's adjoints: gsdf on the centre cell, +-gd[ax] on the cells displaced
        // along zyx axis ax (gd = d/dgrad of the central difference); every corner term
        // is a trilinear weight in [0, 1] times one of them
        float gd[3];
        bool fin = isfinite(gsdf);
        float m = fabsf(gsdf);
#pragma unroll
        for (int ax = 0; ax < 3; ++ax) {
          const float df = clamped_diff(ind, ax, 1.f, G.gs);
          gd[ax] = (gg[2 - ax] / df) / G.voxel_size;
          fin = fin && isfinite(gd[ax]);
          m = fmaxf(m, fabsf(gd[ax]));
        }
        g4[r * cap + k] = make_float4(gd[0], gd[1], gd[2], gsdf);
        tmax = fmaxf(tmax, fin ? m : INFINITY);
      }
    }
  }
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) tmax = fmaxf(tmax, __shfl_xor(tmax, off, 64));
  // one atomic per block: the waves' bounds meet in LDS first (a non-negative float's
  // bits order as its value)
  __shared__ float wave_max[256 / 64];
  if (lane == 0) wave_max[threadIdx.x >> 6] = tmax;
  __syncthreads();
  if (threadIdx.x == 0) {
    float m = 0.f;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) m = fmaxf(m, wave_max[w]);
    if (m > 0.f) atomicMax(term_max, __float_as_uint(m));
  }
}

// A segment of the slot-index list per non-empty brick (atomic allocation), cursors at
// the segments' starts, and the list of non-empty bricks with its length.  A brick whose
// segment would end past the list's capacity (a workspace sized for fewer walk-range
// samples than the walk holds) is left out: its cursor starts at the capacity, so
// k_bwd_bin writes none of its entries.
__global__ void k_brick_alloc(const int* __restrict__ brick_cnt, int nb, int* __restrict__ off,
                              int* __restrict__ cur, int* __restrict__ list, int* __restrict__ nlist,
                              int* __restrict__ total, int order_cap) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= nb) return;
  const int c = brick_cnt[b];
  if (c == 0) return;
  const int o = atomicAdd(total, c);
  off[b] = o;
  const bool fits = (int64_t)o + c <= order_cap;
  cur[b] = fits ? o : order_cap;
  if (fits) list[atomicAdd(nlist, 1)] = b;
}

// Each walk-range slot into the segment of each of its bricks (one atomic per brick and
// run of lanes with the same bricks).
__global__ void __launch_bounds__(256) k_bwd_bin(
    BrickGrid B, int64_t n_rays, int cap, const float4* __restrict__ s4,
    const int* __restrict__ stats, const int64_t* __restrict__ off_incl, int* __restrict__ cur,
    int* __restrict__ order, int order_cap, int64_t max_rows) {
  const int lane = threadIdx.x & 63;
  const int64_t waves = (int64_t)gridDim.x * (blockDim.x >> 6);
  for (int64_t r = blockIdx.x * (int64_t)(blockDim.x >> 6) + (threadIdx.x >> 6); r < n_rays;
       r += waves) {
    if (off_incl[r] > max_rows) continue;
    const int c1 = stats[3 * r + 1];
    for (int base = 0; base < c1; base += 64) {
      const int k = base + lane;
      const bool valid = k < c1;
      const uint32_t code =
          valid ? (__float_as_uint(s4[r * cap + k].w) & ~kSurvivorBit) : 0xFFFFFFFFu;
      const uint32_t pc = __shfl_up(code, 1, 64);
      const bool head = valid && (lane == 0 || pc != code);
      const uint64_t hm = __ballot(head), vm = __ballot(valid);
      // the run's head lane: the nearest head at or below this lane
      const int hl = 63 - __clzll(hm & ((2ull << lane) - 1ull));
      int end = 0;
      if (head) {
        const uint64_t later = hm & ~((2ull << lane) - 1ull);
        end = later ? __ffsll((unsigned long long)later) - 1 : 64 - __clzll(vm);
      }
      for (int q = 0; q < 8; ++q) {
        int pos = 0;
        const int bq = valid ? code_brick(B, code, q) : -1;
        if (head && bq >= 0) pos = atomicAdd(&cur[bq], end - lane);
        const int p = __shfl(pos, hl, 64) + lane - hl;
        if (valid && bq >= 0 && p < order_cap) order[p] = (int)(r * cap + k);
      }
    }
  }
}

// Workgroups of 8 wavefronts stride over the listed bricks (a fixed grid of four per
// CU: a launch of one workgroup per possible brick would spend its time starting
// workgroups that find no brick).  A brick's segment holds runs of consecutive samples
// of one ray, whose stencils overlap; lane l of wave w takes entry e0 + 8 l + w, so the
// 64 lanes of an LDS atomic are 8 entries apart (mostly on other rays) and rarely add
// to the same voxel.
//
// The tile sums in 64-bit fixed point: every term is a multiple of 2^-f with
// f = 35 - floor(log2 T), T the largest |term| bound of the call (k_bwd_stencil), so that
// each term is below 2^36 units and a voxel holds up to 2^27 terms without overflow.
// Integer LDS atomics run at the rate of plain LDS stores, float ones far slower; the
// sum is also independent of the order of the adds (each term is rounded once, to
// 2^-37 T, and the voxel's total once more, to float).  When a term is not finite the
// tile sums in float instead (the sums then carry the reference's inf / nan).
// 512 threads per workgroup: up to four fit a CU beside each other, so every listed
// brick of a 256^3 step starts at once (1,024-thread workgroups went in two rounds, the
// last starting ~25 us after the first)
// x rounded to the nearest integer, ties to even, for |x| < 2^51 (the same integer as
// __double2ll_rn there): the sum x + 1.5 * 2^52 lies in [2^52, 2^53), whose spacing is
// 1, so the addition rounds x at the units place and the sum's bit pattern is that of
// 1.5 * 2^52 plus the integer.  Three FP64 operations and a 64-bit subtraction against
// eight FP64 operations of the general conversion.
__device__ __forceinline__ long long rne_i64(double x) {
  const double y = x + 6755399441055744.0;
  return __double_as_longlong(y) - 0x4338000000000000LL;
}

constexpr int kBrickThreads = 512;
constexpr int kBrickBlocks = 1024;
constexpr int kFixedBits = 35;

__global__ void __launch_bounds__(kBrickThreads) k_bwd_bricks(
    FusedGeom G, BrickGrid B, const float4* __restrict__ s4, const float4* __restrict__ g4,
    const int* __restrict__ off, const int* __restrict__ brick_cnt, const int* __restrict__ list,
    const int* __restrict__ nlist, const uint32_t* __restrict__ term_max,
    const int* __restrict__ order, float* __restrict__ sdf_grad) {
  __shared__ unsigned long long tile[kBrick3];
  float* tile_f = reinterpret_cast<float*>(tile);  // the float sums (non-finite terms)
  // the term bound, the list length and this workgroup's first list entry in one round
  // trip (the launch has at most as many workgroups as the list has entries; the entry
  // is used only if it is inside the list)
  const uint32_t tb = *term_max;
  const int nl = *nlist;
  const int b_first = list[blockIdx.x];
  if (tb == 0u) return;  // every term is zero
  const bool fixed = tb < 0x7f800000u;
  const int lg = fixed ? ilogbf(__uint_as_float(tb)) : 0;
  const double scale = ldexp(1.0, kFixedBits - lg), unscale = ldexp(1.0, lg - kFixedBits);
  const GridDesc& g = G.gs;
  const int spread = (threadIdx.x & 63) * (kBrickThreads / 64) + (threadIdx.x >> 6);
  for (int bi = blockIdx.x; bi < nl; bi += gridDim.x) {
    const int b = bi == (int)blockIdx.x ? b_first : list[bi];
    const int iz = b % B.bz, iy = (b / B.bz) % B.by, ix = b / (B.bz * B.by);
    const int ox = ix * kBrick, oy = iy * kBrick, oz = iz * kBrick;
    for (int i = threadIdx.x; i < kBrick3; i += kBrickThreads) tile[i] = 0ull;
    __syncthreads();
    auto add_cell = [&](const Tri<float>& t, float go) {
#pragma clang fp contract(off)
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        const int x = t.x0 + (c >> 2) - ox, y = t.y0 + ((c >> 1) & 1) - oy,
                  z = t.z0 + (c & 1) - oz;
        if ((unsigned)x >= (unsigned)kBrick || (unsigned)y >= (unsigned)kBrick ||
            (unsigned)z >= (unsigned)kBrick)
          continue;
        const float w = t.w(c >> 2, (c >> 1) & 1, c & 1) * go;
        const int v = (x * kBrick + y) * kBrick + z;
        if (fixed) {
          if (w != 0.f) atomicAdd(&tile[v], (unsigned long long)rne_i64((double)w * scale));
        } else {
          atomicAdd(&tile_f[v], w);
        }
      }
    };
    const int beg = off[b], n = brick_cnt[b];
    for (int e0 = 0; e0 < n; e0 += kBrickThreads) {
#pragma clang fp contract(off)
      const int e = e0 + spread;
      if (e >= n) continue;
      const int slot = order[beg + e];
      const float4 a = s4[slot], tm = g4[slot];
      const float q[3] = {a.x, a.y, a.z};
      Tri<float> t0;
      t0.init(world_to_index(q[0], G.mn[0], G.mx[0] - G.mn[0], g.X),
              world_to_index(q[1], G.mn[1], G.mx[1] - G.mn[1], g.Y),
              world_to_index(q[2], G.mn[2], G.mx[2] - G.mn[2], g.Z));
      if (tm.w != 0.f) add_cell(t0, tm.w);
      float ind[3];
      zyx_index(q, G.mn, G.mx, g, ind);
      const float gds[3] = {tm.x, tm.y, tm.z};
#pragma unroll
      for (int ax = 0; ax < 3; ++ax) {
        const float gd = gds[ax];
        if (gd == 0.f) continue;
#pragma unroll
        for (int side = 0; side < 2; ++side) {
          Tri<float> td;
          displaced_cell(g, ind, ax, side ? 1.f : -1.f, td);
          add_cell(td, side ? gd : -gd);
        }
      }
    }
    __syncthreads();
    // the brick's voxels, z fastest: each is owned by this workgroup alone.  A thread's
    // kPer voxels load their gradient words together (one round trip), then add
    constexpr int kPer = kBrick3 / kBrickThreads;
    static_assert(kBrick3 % kBrickThreads == 0, "whole voxels per thread");
    float vals[kPer];
    float* ptrs[kPer];
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const int i = threadIdx.x + u * kBrickThreads;
      const float v = fixed ? (float)((double)(long long)tile[i] * unscale) : tile_f[i];
      const int x = ox + i / (kBrick * kBrick), y = oy + (i / kBrick) % kBrick,
                z = oz + i % kBrick;
      ptrs[u] = (v != 0.f && in_grid<float>(x, y, z, g))
                    ? sdf_grad + x * g.sx + y * g.sy + z * g.sz
                    : nullptr;
      vals[u] = v;
    }
    float cur[kPer];
#pragma unroll
    for (int u = 0; u < kPer; ++u) cur[u] = ptrs[u] ? *ptrs[u] : 0.f;
#pragma unroll
    for (int u = 0; u < kPer; ++u)
      if (ptrs[u]) *ptrs[u] = cur[u] + vals[u];
    // the tile is cleared for the next brick only after every thread has read it
    __syncthreads();
  }
}

__global__ void k_zero_i32(int* __restrict__ p, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

static inline BrickGrid brick_grid(const GridDesc& g) {
  BrickGrid B;
  B.bx = (int)cdiv(g.X, kBrick);
  B.by = (int)cdiv(g.Y, kBrick);
  B.bz = (int)cdiv(g.Z, kBrick);
  return B;
}

// ---- empty-space bounds (vx_sdf_skip_bounds) ---------------------------------------
// Pass 1: per 8^3 block of lattice voxels, the block's smallest SDF value and, per axis,
// the largest |s(v + e_a) - s(v)| over its voxels v whose neighbour v + e_a is in the
// grid (the neighbour may lie in the next block).  A workgroup of 8 wavefronts takes the
// 8 x 8 columns of one (x, y) block pair over one run of 64 z values, lane l at
// z = 64 c + l (coalesced rows): wave w takes x = 8 bx + w and the 8 y of the block, all
// its loads issued together; the eight lanes of a z block then reduce with shuffles and
// the eight waves through LDS.
__global__ void __launch_bounds__(512) k_sdf_block_stats(const float* __restrict__ sdf,
                                                         GridDesc g, int skx, int sky, int skz,
                                                         float4* __restrict__ stats) {
  const int bx = blockIdx.x / sky, by = blockIdx.x % sky, zc = blockIdx.y;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  __shared__ float4 part[8][8];
  const int z = zc * 64 + lane, x = (bx << kSkipShift) + wave;
  float mn = INFINITY, dx = 0.f, dy = 0.f, dz = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int y = (by << kSkipShift) + i;
    if (x < g.X && y < g.Y && z < g.Z) {
      const int64_t o = x * g.sx + y * g.sy + z * g.sz;
      const float v = sdf[o];
      mn = fminf(mn, v);
      if (x + 1 < g.X) dx = fmaxf(dx, fabsf(sdf[o + g.sx] - v));
      if (y + 1 < g.Y) dy = fmaxf(dy, fabsf(sdf[o + g.sy] - v));
      if (z + 1 < g.Z) dz = fmaxf(dz, fabsf(sdf[o + g.sz] - v));
    }
  }
#pragma unroll
  for (int off = 1; off < 8; off <<= 1) {
    mn = fminf(mn, __shfl_xor(mn, off, 64));
    dx = fmaxf(dx, __shfl_xor(dx, off, 64));
    dy = fmaxf(dy, __shfl_xor(dy, off, 64));
    dz = fmaxf(dz, __shfl_xor(dz, off, 64));
  }
  if ((lane & 7) == 0) part[wave][lane >> 3] = make_float4(mn, dx, dy, dz);
  __syncthreads();
  if (threadIdx.x < 8) {
    const int j = threadIdx.x, bz = zc * 8 + j;
    float4 r = part[0][j];
    for (int w = 1; w < 8; ++w) {
      r.x = fminf(r.x, part[w][j].x);
      r.y = fmaxf(r.y, part[w][j].y);
      r.z = fmaxf(r.z, part[w][j].z);
      r.w = fmaxf(r.w, part[w][j].w);
    }
    if (bz < skz) stats[((int64_t)bx * sky + by) * skz + bz] = r;
  }
}

// The same over a z-contiguous grid whose rows are float4-aligned (sz == 1, Z % 4 == 0,
// 16-byte aligned): a workgroup of 4 wavefronts takes one column block's 64 rows over a
// run of 64 z values as 16 float4 per row, thread t the float4 t % 16 of rows
// 4 (t / 16) .. + 3, with the rows x + 1 and y + 1 loaded as float4 beside them and the
// z neighbour of each float4's last element taken from the next lane.
__global__ void __launch_bounds__(256) k_sdf_block_stats4(const float* __restrict__ sdf,
                                                          GridDesc g, int skx, int sky, int skz,
                                                          float4* __restrict__ stats) {
  const int bx = blockIdx.x / sky, by = blockIdx.x % sky, zc = blockIdx.y;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, zq = t & 15, rg = t >> 4;
  const int z0 = zc * 64 + 4 * zq;
  __shared__ float4 part[4][8];
  float mn = INFINITY, dx = 0.f, dy = 0.f, dz = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = 4 * rg + i;
    const int x = (bx << kSkipShift) + (r >> 3), y = (by << kSkipShift) + (r & 7);
    const bool ok = x < g.X && y < g.Y && z0 < g.Z;
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f), vx = v, vy = v;
    float vn = 0.f;
    const int64_t o = (int64_t)x * g.sx + (int64_t)y * g.sy + z0;
    if (ok) {
      v = *reinterpret_cast<const float4*>(sdf + o);
      if (x + 1 < g.X) vx = *reinterpret_cast<const float4*>(sdf + o + g.sx);
      if (y + 1 < g.Y) vy = *reinterpret_cast<const float4*>(sdf + o + g.sy);
    }
    // the z neighbour of the last element: the next float4 (the next lane of this row,
    // or a load at the end of the run)
    const float nxt = __shfl_down(v.x, 1, 16);
    if (ok && z0 + 4 < g.Z) vn = zq < 15 ? nxt : sdf[o + 4];
    if (ok) {
      mn = fminf(mn, fminf(fminf(v.x, v.y), fminf(v.z, v.w)));
      if (x + 1 < g.X)
        dx = fmaxf(dx, fmaxf(fmaxf(fabsf(vx.x - v.x), fabsf(vx.y - v.y)),
                             fmaxf(fabsf(vx.z - v.z), fabsf(vx.w - v.w))));
      if (y + 1 < g.Y)
        dy = fmaxf(dy, fmaxf(fmaxf(fabsf(vy.x - v.x), fabsf(vy.y - v.y)),
                             fmaxf(fabsf(vy.z - v.z), fabsf(vy.w - v.w))));
      dz = fmaxf(dz, fmaxf(fmaxf(fabsf(v.y - v.x), fabsf(v.z - v.y)), fabsf(v.w - v.z)));
      if (z0 + 4 < g.Z) dz = fmaxf(dz, fabsf(vn - v.w));
    }
  }
  // z block j = zq / 2: combine the lane pair, then the wave's four row groups
#pragma unroll
  for (int off : {1, 16, 32}) {
    mn = fminf(mn, __shfl_xor(mn, off, 64));
    dx = fmaxf(dx, __shfl_xor(dx, off, 64));
    dy = fmaxf(dy, __shfl_xor(dy, off, 64));
    dz = fmaxf(dz, __shfl_xor(dz, off, 64));
  }
  if (lane < 16 && (lane & 1) == 0) part[wave][lane >> 1] = make_float4(mn, dx, dy, dz);
  __syncthreads();
  if (t < 8) {
    const int bz = zc * 8 + t;
    float4 r = part[0][t];
    for (int w = 1; w < 4; ++w) {
      r.x = fminf(r.x, part[w][t].x);
      r.y = fmaxf(r.y, part[w][t].y);
      r.z = fmaxf(r.z, part[w][t].z);
      r.w = fmaxf(r.w, part[w][t].w);
    }
    if (bz < skz) stats[((int64_t)bx * sky + by) * skz + bz] = r;
  }
}

// Pass 2, per brick: over the 3x3x3 blocks around it (the 7-point stencil of a sample in
// the brick reads voxels at most 2 below and 3 above its cell, and the central
// differences of those lookups are bounded by the one-step differences there), the
// smallest SDF value and sqrt(sum_a D_a^2) / voxel_size, an upper bound on the gradient
// length (with a margin for float rounding).
__global__ void k_sdf_skip_bounds(const float4* __restrict__ stats, int skx, int sky, int skz,
                                  float voxel_size, float margin, float4* __restrict__ bounds) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= skx * sky * skz) return;
  const int bz = b % skz, by = (b / skz) % sky, bx = b / (skz * sky);
  float mn = INFINITY, dx = 0.f, dy = 0.f, dz = 0.f;
  for (int i = max(bx - 1, 0); i <= min(bx + 1, skx - 1); ++i)
    for (int j = max(by - 1, 0); j <= min(by + 1, sky - 1); ++j)
      for (int k = max(bz - 1, 0); k <= min(bz + 1, skz - 1); ++k) {
        const float4 st = stats[((int64_t)i * sky + j) * skz + k];
        mn = fminf(mn, st.x);
        dx = fmaxf(dx, st.y);
        dy = fmaxf(dy, st.z);
        dz = fmaxf(dz, st.w);
      }
  // a grid that may still change by up to `margin` per voxel: its values by -margin, its
  // one-step differences by up to 2 margin
  mn -= margin;
  dx += 2.f * margin;
  dy += 2.f * margin;
  dz += 2.f * margin;
  const float gmax = sqrtf(dx * dx + dy * dy + dz * dz) / voxel_size * (1.f + 1e-4f);
  bounds[b] = make_float4(mn, gmax, 0.f, 0.f);
}

// out[0] = scale * sum x[0..n): one block, fixed summation order (deterministic).
__global__ void __launch_bounds__(1024) k_sum_f32(const float* __restrict__ x, int64_t n, float scale,
                                                  float* __restrict__ out) {
  __shared__ float part[16];
  float s = 0.f;
  for (int64_t i = threadIdx.x; i < n; i += blockDim.x) s += x[i];
  s = wave_sum_f32(s);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    float t = 0.f;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) t += part[w];
    out[0] = t * scale;
  }
}

}  // namespace vx

using namespace vx;

extern "C" {

int vx_fused_fine_fwd(const float* sdf, const int64_t* sdf_geom, const float* box,
                      const float* params, const float* mc, const int64_t* mc_geom,
                      const float* mc_params, const float* rays_o, const float* rays_d,
                      const float* viewdirs, int64_t n_rays, int cap, void* s4, void* g4,
                      int64_t* cnt, float* last, int* stats, int count_all, int* overflow,
                      int64_t* walk_total, const int64_t* k0_geom, uint32_t* k0_pages,
                      uint32_t* sdf_pages, int hier_reach, const void* skip_bounds,
                      void* stream) {
  FusedGeom G;
  VX_CHECK_ARG(!k0_pages || k0_geom, "fused_fine_fwd: k0_pages needs k0_geom");
  if (int st = fused_geom(G, sdf, sdf_geom, nullptr, k0_geom, box, params)) return st;
  if (int st = fused_maskcache(G, mc, mc_geom, mc_params)) return st;
  fused_skip(G, skip_bounds);
  if (int st = check_corner_pages("fused_fine_fwd", G, k0_pages)) return st;
  VX_CHECK_ARG(n_rays >= 0 && cap >= 1, "fused_fine_fwd: bad sizes");
  VX_CHECK_ARG(hier_reach >= 0 && 2 * hier_reach + 2 <= kPageElems &&
                   (hier_reach == 0 || G.gs.sz == 1),
               "fused_fine_fwd: hier_reach needs a z-contiguous SDF grid and a block within a page");
  if (n_rays == 0) return VX_OK;
  k_fused_fwd<<<grid_for(n_rays, 4, 1 << 16), 256, 0, (hipStream_t)stream>>>(
      G, rays_o, rays_d, viewdirs, n_rays, cap, (float4*)s4, (float4*)g4, cnt, last, stats,
      count_all, overflow, reinterpret_cast<unsigned long long*>(walk_total), k0_pages,
      sdf_pages, hier_reach);
  return launch_status("fused_fine_fwd");
}

int vx_fused_fine_gather(const float* k0, const int64_t* k0_geom, const int64_t* sdf_geom,
                         const float* box, const float* params, const float* viewdirs,
                         int64_t n_rays, int cap, int n_freq, const void* s4, const void* g4,
                         const int* stats, const int64_t* cnt, const int64_t* off_incl,
                         int xstride, int64_t max_rows, float* X, void* P4, void* G4, int* rid,
                         uint32_t* k0_pages, void* stream) {
  FusedGeom G;
  if (int st = fused_geom(G, nullptr, sdf_geom, k0, k0_geom, box, params)) return st;
  VX_CHECK_ARG(G.gk.C + 3 + 3 + 6 * n_freq <= xstride && xstride <= 64 && xstride % 4 == 0,
               "fused_fine_gather: feature row does not fit xstride (a multiple of 4, <= 64)");
  VX_CHECK_ARG(cap >= 1, "fused_fine_gather: cap < 1");
  if (int st = check_corner_pages("fused_fine_gather", G, k0_pages)) return st;
  if (n_rays == 0) return VX_OK;
  hipStream_t st = (hipStream_t)stream;
  launch_survivors(G, viewdirs, n_rays, cap, s4, g4, stats, cnt, off_incl, max_rows, P4, G4, rid,
                   k0_pages, st);
  // max_rows may be a capacity far past the survivors: a few passes for a full one
  if (max_rows > 0)
    k_fused_rows<<<grid_for(max_rows, kRowTile, 1 << 12), 256, 0, st>>>(
        G, viewdirs, n_rays, n_freq, off_incl, xstride, max_rows, X, (const float4*)P4,
        (const float4*)G4, rid);
  return launch_status("fused_fine_gather");
}

int vx_fused_fine_composite(int64_t n_rays, const int64_t* cnt, const int64_t* off_incl,
                            const float* logits, int lstride, const void* P4, const float* last,
                            const float* target, float bg, float* rgb, float* dlogit, float* gw,
                            float* glast, float* S, float* loss_r, int64_t max_rows,
                            void* stream) {
  VX_CHECK_ARG(n_rays >= 0, "fused_fine_composite: n_rays < 0");
  if (n_rays == 0) return VX_OK;
  const float inv_count = 1.f / (3.f * (float)n_rays);
  k_fused_composite<<<grid_for(n_rays, 16, 1 << 16), 256, 0, (hipStream_t)stream>>>(
      n_rays, cnt, off_incl, logits, lstride, (const float4*)P4, last, target, bg, inv_count, rgb,
      dlogit, gw, glast, S, loss_r, max_rows);
  return launch_status("fused_fine_composite");
}

int vx_fused_fine_feat_bwd(const int64_t* k0_geom, const int64_t* sdf_geom, const float* box,
                           const float* params, int64_t m, const float* dX, int dxs,
                           const void* P4, const void* G4, float* k0_grad, float* dgf,
                           uint32_t* k0_pages, const int64_t* m_dev, void* stream) {
  FusedGeom G;
  if (int st = fused_geom(G, nullptr, sdf_geom, nullptr, k0_geom, box, params)) return st;
  if (int st = check_corner_pages("fused_fine_feat_bwd", G, k0_pages)) return st;
  if (m == 0) return VX_OK;
  k_fused_feat_bwd<<<grid_for(m, 256, 1 << 16), 256, 0, (hipStream_t)stream>>>(
      G, m, m_dev, dX, dxs, (const float4*)P4, (const float4*)G4, k0_grad, dgf, k0_pages);
  return launch_status("fused_fine_feat_bwd");
}

int64_t vx_fused_bwd_workspace_bytes(int64_t walk_total, int X, int Y, int Z) {
  if (walk_total < 0 || X < 1 || Y < 1 || Z < 1) return -1;
  const int64_t nb = cdiv(X, kBrick) * cdiv(Y, kBrick) * cdiv(Z, kBrick);
  // nlist, total, term bound, brick_cnt, off, cur, list (nb each), order (up to 8 bricks
  // per walk-range sample)
  return 4 * (4 * nb + 3 + 8 * walk_total);
}

// The workspace of the SDF backward: nlist, total, the term bound and brick_cnt first
// (cleared together), then off, cur, list, order.
struct BwdWs {
  int *nlist, *total, *brick_cnt, *off, *cur, *list, *order;
  uint32_t* term_max;
  int order_cap;  // entries of the slot-index list
};

static int bwd_setup(const char* who, FusedGeom& G, BrickGrid& B, BwdWs& W, const float* sdf,
                     const int64_t* sdf_geom, const float* box, const float* params,
                     int64_t n_rays, int cap, void* ws, int64_t ws_bytes) {
  if (int st = fused_geom(G, sdf, sdf_geom, nullptr, nullptr, box, params)) return st;
  VX_CHECK_ARG(cap >= 1 && n_rays >= 0, "%s: cap < 1 or n_rays < 0", who);
  B = brick_grid(G.gs);
  const int64_t nb = (int64_t)B.bx * B.by * B.bz;
  const int64_t head = vx_fused_bwd_workspace_bytes(0, G.gs.X, G.gs.Y, G.gs.Z);
  VX_CHECK_ARG(ws && ws_bytes >= head, "%s: workspace of %lld bytes, at least %lld needed", who,
               (long long)ws_bytes, (long long)head);
  VX_CHECK_ARG(8 * n_rays * (int64_t)cap < ((int64_t)1 << 31) && nb < ((int64_t)1 << 24),
               "%s: more than 2^28 slots or 2^24 bricks", who);
  const int64_t ocap = (ws_bytes - head) / 4;
  W.order_cap = (int)(ocap < ((int64_t)1 << 31) - 1 ? ocap : ((int64_t)1 << 31) - 1);
  W.nlist = static_cast<int*>(ws);
  W.total = W.nlist + 1;
  W.term_max = reinterpret_cast<uint32_t*>(W.total + 1);
  W.brick_cnt = W.total + 2;
  W.off = W.brick_cnt + nb;
  W.cur = W.off + nb;
  W.list = W.cur + nb;
  W.order = W.list + nb;
  return VX_OK;
}

int vx_fused_fine_bwd_alpha(const float* sdf, const int64_t* sdf_geom, const float* box,
                            const float* params, const float* viewdirs, int64_t n_rays, int cap,
                            void* s4, void* g4, const int* stats, const int64_t* cnt,
                            const int64_t* off_incl, const float* last, const float* gw,
                            const float* glast, const float* S, int64_t max_rows, void* ws,
                            int64_t ws_bytes, void* stream) {
  FusedGeom G;
  BrickGrid B;
  BwdWs W;
  if (int st = bwd_setup("fused_fine_bwd_alpha", G, B, W, sdf, sdf_geom, box, params, n_rays,
                         cap, ws, ws_bytes))
    return st;
  const int64_t nb = (int64_t)B.bx * B.by * B.bz;
  hipStream_t st = (hipStream_t)stream;
  k_zero_i32<<<grid_for(nb + 3, 256), 256, 0, st>>>(W.nlist, nb + 3);
  if (n_rays > 0) {
    k_bwd_alpha<kBwdSeg><<<grid_for(n_rays, 4 * (64 / kBwdSeg), 1 << 16), 256, 0, st>>>(
        G, B, viewdirs, n_rays, cap, (float4*)s4, (float4*)g4, stats, cnt, off_incl, last, gw,
        glast, S, W.brick_cnt, max_rows);
    k_brick_alloc<<<grid_for(nb, 256), 256, 0, st>>>(W.brick_cnt, (int)nb, W.off, W.cur, W.list,
                                                     W.nlist, W.total, W.order_cap);
    k_bwd_bin<<<grid_for(n_rays, 4, 1 << 16), 256, 0, st>>>(
        B, n_rays, cap, (const float4*)s4, stats, off_incl, W.cur, W.order, W.order_cap,
        max_rows);
  }
  return launch_status("fused_fine_bwd_alpha");
}

int vx_fused_fine_bwd_grid(const float* sdf, const int64_t* sdf_geom, const float* box,
                           const float* params, int64_t n_rays, int cap, const void* s4, void* g4,
                           const int* stats, const int64_t* cnt, const int64_t* off_incl,
                           const float* dgf, const float* dsf, float* sdf_grad, int64_t max_rows,
                           void* ws, int64_t ws_bytes, void* stream) {
  FusedGeom G;
  BrickGrid B;
  BwdWs W;
  if (int st = bwd_setup("fused_fine_bwd_grid", G, B, W, sdf, sdf_geom, box, params, n_rays,
                         cap, ws, ws_bytes))
    return st;
  if (n_rays == 0) return VX_OK;
  const int64_t nb = (int64_t)B.bx * B.by * B.bz;
  hipStream_t st = (hipStream_t)stream;
  k_bwd_stencil<kBwdSeg><<<grid_for(n_rays, 4 * (64 / kBwdSeg), 1 << 16), 256, 0, st>>>(
      G, n_rays, cap, (const float4*)s4, (float4*)g4, stats, cnt, off_incl, dgf, dsf, W.term_max,
      max_rows);
  k_bwd_bricks<<<(unsigned)(nb < kBrickBlocks ? nb : kBrickBlocks), kBrickThreads, 0, st>>>(
      G, B, (const float4*)s4, (const float4*)g4, W.off, W.brick_cnt, W.list, W.nlist, W.term_max,
      W.order, sdf_grad);
  return launch_status("fused_fine_bwd_grid");
}

int vx_fused_fine_bwd(const float* sdf, const int64_t* sdf_geom, const float* box,
                      const float* params, const float* viewdirs, int64_t n_rays, int cap,
                      void* s4, void* g4, const int* stats, const int64_t* cnt,
                      const int64_t* off_incl, const float* last, const float* gw,
                      const float* glast, const float* S, const float* dgf, const float* dsf,
                      float* sdf_grad, int64_t max_rows, void* ws, int64_t ws_bytes,
                      void* stream) {
  if (int st = vx_fused_fine_bwd_alpha(sdf, sdf_geom, box, params, viewdirs, n_rays, cap, s4, g4,
                                       stats, cnt, off_incl, last, gw, glast, S, max_rows, ws,
                                       ws_bytes, stream))
    return st;
  return vx_fused_fine_bwd_grid(sdf, sdf_geom, box, params, n_rays, cap, s4, g4, stats, cnt,
                                off_incl, dgf, dsf, sdf_grad, max_rows, ws, ws_bytes, stream);
}

int64_t vx_sdf_skip_bricks(const int64_t* sdf_geom) {
  if (!sdf_geom || sdf_geom[1] < 1 || sdf_geom[2] < 1 || sdf_geom[3] < 1) return -1;
  const int64_t b = (int64_t)1 << kSkipShift;
  return ((sdf_geom[1] + b - 1) / b) * ((sdf_geom[2] + b - 1) / b) * ((sdf_geom[3] + b - 1) / b);
}

int vx_sdf_skip_bounds(const float* sdf, const int64_t* sdf_geom, float voxel_size,
                       float margin, void* bounds, void* ws, void* stream) {
  VX_CHECK_ARG(sdf && sdf_geom && bounds && ws, "sdf_skip_bounds: null pointer");
  VX_CHECK_ARG(sdf_geom[0] == 1, "sdf_skip_bounds: the SDF grid must have one channel");
  VX_CHECK_ARG(voxel_size > 0.f, "sdf_skip_bounds: voxel_size <= 0");
  VX_CHECK_ARG(margin >= 0.f, "sdf_skip_bounds: margin < 0");
  const int64_t nb = vx_sdf_skip_bricks(sdf_geom);
  VX_CHECK_ARG(nb > 0 && nb < ((int64_t)1 << 31), "sdf_skip_bounds: bad grid size");
  GridDesc g;
  g.C = 1;
  g.X = (int)sdf_geom[1];
  g.Y = (int)sdf_geom[2];
  g.Z = (int)sdf_geom[3];
  g.sc = sdf_geom[4];
  g.sx = sdf_geom[5];
  g.sy = sdf_geom[6];
  g.sz = sdf_geom[7];
  const int b = 1 << kSkipShift;
  const int skx = (g.X + b - 1) / b, sky = (g.Y + b - 1) / b, skz = (g.Z + b - 1) / b;
  hipStream_t st = (hipStream_t)stream;
  const dim3 grid((unsigned)(skx * sky), (unsigned)((g.Z + 63) / 64));
  if (g.sz == 1 && g.Z % 4 == 0 && g.sy % 4 == 0 && g.sx % 4 == 0 &&
      reinterpret_cast<uintptr_t>(sdf) % 16 == 0)
    k_sdf_block_stats4<<<grid, 256, 0, st>>>(sdf, g, skx, sky, skz, static_cast<float4*>(ws));
  else
    k_sdf_block_stats<<<grid, 512, 0, st>>>(sdf, g, skx, sky, skz, static_cast<float4*>(ws));
  k_sdf_skip_bounds<<<grid_for(nb, 256), 256, 0, st>>>(static_cast<const float4*>(ws), skx, sky,
                                                       skz, voxel_size, margin,
                                                       static_cast<float4*>(bounds));
  return launch_status("sdf_skip_bounds");
}

int vx_sum_f32(const float* x, int64_t n, float scale, float* out, void* stream) {
  VX_CHECK_ARG(n >= 0, "sum: n < 0");
  k_sum_f32<<<1, 1024, 0, (hipStream_t)stream>>>(x, n, scale, out);
  return launch_status("sum");
}

}  // extern "C"
