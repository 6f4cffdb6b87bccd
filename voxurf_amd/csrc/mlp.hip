// rgbnet on the matrix cores (gfx950): Linear(+ReLU) layers of width 192 for the colour
// MLP of lib/voxurf_fine.py:132-149, forward and backward, FP32 (v_mfma_f32_32x32x2f32)
// and BF16 inputs with FP32 accumulation (v_mfma_f32_32x32x16_bf16).
//
// Layout.  A 32x32 MFMA leaves output element (row i, col j) in lane
// j + 32*((i % 8) / 4), register (i % 4) + 4*(i / 8).  The layers compute
// H_out^T = W * H_in^T: the sample index is the MFMA column and the feature index the
// row, so a lane pair holds one sample.  The B operand of reduction step s in lane half
// h is input feature dfeat(s / 16, s % 16, h) of that lane's sample (four consecutive
// features per float4 load), and the weights are packed once per call in exactly that
// order and in lane order, so every LDS read of the A operand is one conflict-free
// ds_read_b128 per four MFMAs.
//
// Per 32-sample tile and layer: 6 output tiles x 96 reduction steps = 576 MFMAs (FP32)
// or 6 x 12 = 72 (BF16).  Weight gradients dW = dY^T X are a separate split-M GEMM
// (FP32 MFMAs, BF16 inputs, or three-way BF16 splits) whose partial sums are reduced in
// two deterministic passes.
#include "common.h"

namespace vx {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kWidth = 192;

// feature held by accumulator register v of output tile t in lane half h
__host__ __device__ constexpr int dfeat(int t, int v, int h) {
  return 32 * t + 8 * (v >> 2) + 4 * h + (v & 3);
}

// ---- weight packing --------------------------------------------------------------
// Packed A operand, FP32: element ((to * S/4 + s/4) * 64 + lane) * 4 + s%4 holds
//   fwd: A[i = 32 to + lane%32][k = dfeat(s/16, s%16, lane/32)] = Wt[i][k]
//   bwd: A[i = 32 to + lane%32][k = ...] = Wt[k][i]        (W transposed)
// with zero outside [0, n_out) x [0, k_in).  S = 16 * KT reduction steps.
__device__ __forceinline__ float pack_f32_value(const float* __restrict__ Wt, int n_out, int k_in,
                                                int KT, int transpose, int64_t idx, int64_t& dst) {
  const int S = 16 * KT;
  const int lane = (int)(idx & 63), s = (int)((idx >> 6) % S), to = (int)((idx >> 6) / S);
  const int i = 32 * to + (lane & 31);
  const int k = dfeat(s >> 4, s & 15, lane >> 5);
  float v = 0.f;
  if (!transpose) {
    if (i < n_out && k < k_in) v = Wt[i * k_in + k];
  } else {
    // A[i][k] = Wt[k][i]: i indexes the layer's inputs (< k_in), k its outputs (< n_out)
    if (k < n_out && i < k_in) v = Wt[k * k_in + i];
  }
  dst = (((int64_t)to * (S / 4) + (s >> 2)) * 64 + lane) * 4 + (s & 3);
  return v;
}

__global__ void k_pack_f32(const float* __restrict__ Wt, int n_out, int k_in, int KT, int NTO,
                           int transpose, float* __restrict__ out) {
  const int64_t total = (int64_t)NTO * 16 * KT * 64;
  for (int64_t idx = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; idx < total;
       idx += (int64_t)gridDim.x * blockDim.x) {
    int64_t dst;
    const float v = pack_f32_value(Wt, n_out, k_in, KT, transpose, idx, dst);
    out[dst] = v;
  }
}

// Packed A operand, BF16 (K = 16 per MFMA, 8 values per lane): element
// ((to * S + s) * 64 + lane) * 8 + e holds A[i = 32 to + lane%32][k] with
// k = dfeat(s / 2, 8 (s % 2) + e, lane / 32), S = 2 * KT steps.
__device__ __forceinline__ float pack_bf16_value(const float* __restrict__ Wt, int n_out, int k_in,
                                                 int KT, int transpose, int64_t idx) {
  const int S = 2 * KT;
  const int e = (int)(idx & 7), lane = (int)((idx >> 3) & 63), s = (int)((idx >> 9) % S),
            to = (int)((idx >> 9) / S);
  const int i = 32 * to + (lane & 31);
  const int k = dfeat(s >> 1, 8 * (s & 1) + e, lane >> 5);
  (void)e;
  float v = 0.f;
  if (!transpose) {
    if (i < n_out && k < k_in) v = Wt[i * k_in + k];
  } else {
    if (k < n_out && i < k_in) v = Wt[k * k_in + i];
  }
  return v;
}

// ---- FP32 through three-way BF16 splits --------------------------------------------
// A float32 x is the exact sum of three bfloat16 values: x0 = bf16(x) (round to nearest
// even), x1 = bf16(x - x0), x2 = x - x0 - x1 (each difference is exact in float32 by
// Sterbenz's lemma, and x2 has at most 8 significant bits).  A product x w is then the
// sum of the nine x_i w_j; the six with i + j <= 2 are computed (BF16 MFMAs, each
// product exact in the FP32 accumulator) and the three dropped terms are below
// 2^-23 |x w| together.  One 16-deep reduction step takes six 32x32x16 BF16 MFMAs
// (6 x 32 cycles) against eight 32x32x2 FP32 MFMAs (8 x 64 cycles).
__device__ __forceinline__ void split3(float x, __bf16& p0, __bf16& p1, __bf16& p2) {
  p0 = (__bf16)x;
  const float r1 = x - (float)p0;
  p1 = (__bf16)r1;
  p2 = (__bf16)(r1 - (float)p1);
}

__device__ __forceinline__ void split8(const float4& a, const float4& b, bf16x8& p0, bf16x8& p1,
                                       bf16x8& p2) {
  const float x[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    __bf16 q0, q1, q2;
    split3(x[e], q0, q1, q2);
    p0[e] = q0;
    p1[e] = q1;
    p2[e] = q2;
  }
}

// Packed A operand, split: the BF16 operand order (pack_bf16_value) with the three
// parts of each step side by side: bf16x8 vector ((to * S + s) * 3 + part) * 64 + lane.
template <typename Seg>
__device__ __forceinline__ void pack_split_store(const Seg& sg, int64_t idx, __bf16* out) {
  const float v = pack_bf16_value(sg.W, sg.n_out, sg.k_in, sg.kt, sg.transpose, idx);
  const int64_t e = idx & 7, lane = (idx >> 3) & 63, ts = idx >> 9;  // ts = to * S + s
  __bf16 q0, q1, q2;
  split3(v, q0, q1, q2);
  __bf16* o = out + 3 * sg.offset + ((ts * 3) * 64 + lane) * 8 + e;
  o[0] = q0;
  o[64 * 8] = q1;
  o[2 * 64 * 8] = q2;
}

__global__ void k_pack_bf16(const float* __restrict__ Wt, int n_out, int k_in, int KT, int NTO,
                            int transpose, __bf16* __restrict__ out) {
  const int64_t total = (int64_t)NTO * 2 * KT * 64 * 8;
  for (int64_t idx = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; idx < total;
       idx += (int64_t)gridDim.x * blockDim.x)
    out[idx] = (__bf16)pack_bf16_value(Wt, n_out, k_in, KT, transpose, idx);
}

// Every packed operand of a network in one launch: segment blockIdx.y.
struct PackSeg {
  const float* W;
  int64_t offset;  // elements into the output
  int n_out, k_in, kt, nto, transpose;
};
constexpr int kMaxPackSegs = 8;
struct PackNet {
  PackSeg seg[kMaxPackSegs];
};

// PREC 0: FP32 operands; 1: BF16; 2: three BF16 parts per value (pack_split_store).
template <int PREC>
__global__ void k_pack_net(PackNet net, void* __restrict__ out) {
  const PackSeg sg = net.seg[blockIdx.y];
  const int64_t total = (int64_t)sg.nto * 16 * sg.kt * 64;  // same count in every layout
  for (int64_t idx = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; idx < total;
       idx += (int64_t)gridDim.x * blockDim.x) {
    if constexpr (PREC == 2) {
      pack_split_store(sg, idx, reinterpret_cast<__bf16*>(out));
    } else if constexpr (PREC == 1) {
      reinterpret_cast<__bf16*>(out)[sg.offset + idx] =
          (__bf16)pack_bf16_value(sg.W, sg.n_out, sg.k_in, sg.kt, sg.transpose, idx);
    } else {
      int64_t dst;
      const float v = pack_f32_value(sg.W, sg.n_out, sg.k_in, sg.kt, sg.transpose, idx, dst);
      reinterpret_cast<float*>(out)[sg.offset + dst] = v;
    }
  }
}

// Rows to process: M, or the device count *Md (clamped to M, the buffers' capacity) when
// given, so that a launch can be queued before the count is known on the host.
__device__ __forceinline__ int64_t eff_rows(int64_t M, const int64_t* Md) {
  if (!Md) return M;
  const int64_t m = *Md;
  return m < M ? (m > 0 ? m : 0) : M;
}

// ---- one layer over all rows -------------------------------------------------------
// MODE 0: out = relu(W x + b)            (hidden layer, forward)
// MODE 2: out = (W^T dy) * [mask > 0]    (backward data through a ReLU layer)
// MODE 3: out = W^T dy                   (backward data to the network input)
// Input rows: `in` [M, in_stride], read at the permuted feature order: activations
// (MODE 0) in the layer's element type, gradients (MODE 2/3) float32.  Output rows
// [M, out_stride]: activations in the element type (bfloat16 when BF), gradients
// float32.  Persistent: each wave walks 32-row tiles; weights stay in LDS.
constexpr int kLayerThreads = 512;

// One 32-row tile of a layer, output column tiles [to_lo, to_hi) of the NTO (FULL: all).
template <int KT, int NTO, int MODE, bool BF, bool FULL>
__device__ __forceinline__ void layer_tile(const void* __restrict__ in_, int in_stride, int64_t M,
                                           const unsigned char* lds_raw, const float* lb,
                                           const void* __restrict__ mask_, int mask_stride,
                                           void* __restrict__ out_, int out_stride, int64_t tile,
                                           int to_lo, int to_hi) {
  constexpr int S = BF ? 2 * KT : 16 * KT;     // reduction steps
  const int lane = threadIdx.x & 63, h = lane >> 5, rl = lane & 31;
  const int64_t row = tile * 32 + rl;
  const bool valid = row < M;
  f32x16 acc[NTO];
#pragma unroll
  for (int t = 0; t < NTO; ++t)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[t][v] = 0.f;
  // rows past M read row M-1 (in bounds); their results are never stored
  const int64_t rrow = valid ? row : M - 1;
  if constexpr (!BF) {
    // The B operand of reduction step s = 16 t + 4 u + w is input feature
    // 32 t + 8 u + 4 h + w of this lane's row: one float4 per (t, u).  The 16 values
    // of input tile t + 1 are loaded while tile t's 16 * NTO MFMAs run, so at most two
    // tiles of operands are live beside the NTO accumulators.
    const float* rp = reinterpret_cast<const float*>(in_) + rrow * in_stride + 4 * h;
    const float4* lw = reinterpret_cast<const float4*>(lds_raw);
    float4 cur[4], nxt[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) cur[u] = *reinterpret_cast<const float4*>(rp + 8 * u);
#pragma unroll 1
    for (int t = 0; t < KT; ++t) {
      if (t + 1 < KT) {
#pragma unroll
        for (int u = 0; u < 4; ++u)
          nxt[u] = *reinterpret_cast<const float4*>(rp + 32 * (t + 1) + 8 * u);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int sq = 4 * t + u;
#pragma unroll
        for (int to = 0; to < NTO; ++to) {
          if (!FULL && (to < to_lo || to >= to_hi)) continue;
          const float4 a = lw[(to * (S / 4) + sq) * 64 + lane];
          acc[to] = __builtin_amdgcn_mfma_f32_32x32x2f32(a.x, cur[u].x, acc[to], 0, 0, 0);
          acc[to] = __builtin_amdgcn_mfma_f32_32x32x2f32(a.y, cur[u].y, acc[to], 0, 0, 0);
          acc[to] = __builtin_amdgcn_mfma_f32_32x32x2f32(a.z, cur[u].z, acc[to], 0, 0, 0);
          acc[to] = __builtin_amdgcn_mfma_f32_32x32x2f32(a.w, cur[u].w, acc[to], 0, 0, 0);
        }
      }
      if (t + 1 < KT) {
#pragma unroll
        for (int u = 0; u < 4; ++u) cur[u] = nxt[u];
      }
    }
  } else {
    // BF16: step s takes the 8 features dfeat(s/2, 8 (s%2) + e, h), e = 0..7, which
    // are 8 consecutive registers of the producing layer's output.  Input tile t
    // (steps 2t, 2t+1) is loaded while tile t-1's MFMAs run.
    const bf16x8* lw = reinterpret_cast<const bf16x8*>(lds_raw);
    bf16x8 cur[2], nxt[2];
    auto load_tile = [&](bf16x8* dst, int t) {
      if constexpr (MODE == 0) {
        // features 32 t + 8 u + 4 h + w for u = 0..3, w = 0..3, stored as bfloat16
        const __bf16* in = reinterpret_cast<const __bf16*>(in_) + rrow * in_stride + 4 * h + 32 * t;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const uint2 lo = *reinterpret_cast<const uint2*>(in + 16 * q);
          const uint2 hi = *reinterpret_cast<const uint2*>(in + 16 * q + 8);
          uint4 v = make_uint4(lo.x, lo.y, hi.x, hi.y);
          dst[q] = *reinterpret_cast<bf16x8*>(&v);
        }
      } else {
        // backward: the incoming gradient rows are float32; rounded to bf16 here
        const float* in = reinterpret_cast<const float*>(in_) + rrow * in_stride + 4 * h + 32 * t;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const float4 lo = *reinterpret_cast<const float4*>(in + 16 * q);
          const float4 hi = *reinterpret_cast<const float4*>(in + 16 * q + 8);
          dst[q][0] = (__bf16)lo.x;
          dst[q][1] = (__bf16)lo.y;
          dst[q][2] = (__bf16)lo.z;
          dst[q][3] = (__bf16)lo.w;
          dst[q][4] = (__bf16)hi.x;
          dst[q][5] = (__bf16)hi.y;
          dst[q][6] = (__bf16)hi.z;
          dst[q][7] = (__bf16)hi.w;
        }
      }
    };
    load_tile(cur, 0);
#pragma unroll 1
    for (int t = 0; t < KT; ++t) {
      if (t + 1 < KT) load_tile(nxt, t + 1);
#pragma unroll
      for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int to = 0; to < NTO; ++to)
          if (FULL || (to >= to_lo && to < to_hi))
            acc[to] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(lw[(to * S + 2 * t + q) * 64 + lane],
                                                               cur[q], acc[to], 0, 0, 0);
      if (t + 1 < KT) {
        cur[0] = nxt[0];
        cur[1] = nxt[1];
      }
    }
  }
  // ---- epilogue ----
  const int64_t obase = rrow * out_stride + 4 * h;
  const int64_t mbase = rrow * mask_stride + 4 * h;
#pragma unroll
  for (int to = 0; to < NTO; ++to) {
    if (!FULL && (to < to_lo || to >= to_hi)) continue;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      float v4[4];
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const int v = 4 * u + w;
        float x = acc[to][v];
        if (MODE == 0) {
          x += lb[dfeat(to, v, h)];
          x = x > 0.f ? x : 0.f;
        }
        v4[w] = x;
      }
      const int cofs = 32 * to + 8 * u;          // compile-time column offset
      const int col = cofs + 4 * h;
      if (MODE == 2 && valid) {
        if constexpr (BF) {
          const __bf16* mk = reinterpret_cast<const __bf16*>(mask_) + mbase + cofs;
#pragma unroll
          for (int w = 0; w < 4; ++w) v4[w] = (float)mk[w] > 0.f ? v4[w] : 0.f;
        } else {
          const float4 mk = *reinterpret_cast<const float4*>(reinterpret_cast<const float*>(mask_) +
                                                            mbase + cofs);
          v4[0] = mk.x > 0.f ? v4[0] : 0.f;
          v4[1] = mk.y > 0.f ? v4[1] : 0.f;
          v4[2] = mk.z > 0.f ? v4[2] : 0.f;
          v4[3] = mk.w > 0.f ? v4[3] : 0.f;
        }
      }
      if (valid) {
        if (BF && MODE == 0) {
          __bf16* o = reinterpret_cast<__bf16*>(out_) + obase + cofs;
          __bf16 q[4] = {(__bf16)v4[0], (__bf16)v4[1], (__bf16)v4[2], (__bf16)v4[3]};
          *reinterpret_cast<uint2*>(o) = *reinterpret_cast<uint2*>(q);
        } else {
          float* o = reinterpret_cast<float*>(out_) + obase + cofs;
          *reinterpret_cast<float4*>(o) = make_float4(v4[0], v4[1], v4[2], v4[3]);
        }
      }
    }
  }
}

template <int KT, int NTO, int MODE, bool BF>
__global__ void __launch_bounds__(kLayerThreads) k_mlp_layer(
    const void* __restrict__ in_, int in_stride, int64_t M, const int64_t* __restrict__ Md,
    const void* __restrict__ wpk, const float* __restrict__ bias, const void* __restrict__ mask_,
    int mask_stride, void* __restrict__ out_, int out_stride) {
  constexpr int S = BF ? 2 * KT : 16 * KT;     // reduction steps
  constexpr int WELEMS = NTO * S * 64 * (BF ? 8 : 1);
  __shared__ __attribute__((aligned(16))) unsigned char lds_raw[WELEMS * (BF ? 2 : 4)];
  __shared__ float lb[NTO * 32];
  const int tid = threadIdx.x;
  {
    // weights into LDS: every load of a thread in flight before its first store (a
    // load-store loop one vector at a time serialises on the L2 latency)
    const float4* src = reinterpret_cast<const float4*>(wpk);
    float4* dst = reinterpret_cast<float4*>(lds_raw);
    constexpr int n4 = WELEMS * (BF ? 2 : 4) / 16;
    constexpr int P = (n4 + kLayerThreads - 1) / kLayerThreads;  // vectors per thread
    float4 v[P];
#pragma unroll
    for (int b = 0; b < P; ++b) {
      const int i = tid + b * kLayerThreads;
      v[b] = i < n4 ? src[i] : make_float4(0.f, 0.f, 0.f, 0.f);
    }
#pragma unroll
    for (int b = 0; b < P; ++b) {
      const int i = tid + b * kLayerThreads;
      if (i < n4) dst[i] = v[b];
    }
    if (MODE == 0)
      for (int i = tid; i < NTO * 32; i += blockDim.x) lb[i] = bias[i];
  }
  __syncthreads();
  // Stream-K split: the ntiles x NTO (32 x 32 output block) units are divided evenly
  // over the grid's waves, so every SIMD gets the same MFMA work; a wave's first and last
  // tiles may be partial (a subset of the output column tiles).
  const int wave = tid >> 6;
  M = eff_rows(M, Md);
  const int64_t ntiles = (M + 31) / 32;
  const int64_t nw = (int64_t)gridDim.x * (blockDim.x >> 6);
  const int64_t gw = (int64_t)blockIdx.x * (blockDim.x >> 6) + wave;
  const int64_t total = ntiles * NTO;
  int64_t u = total * gw / nw;
  const int64_t u1 = total * (gw + 1) / nw;
  while (u < u1) {
    const int64_t tile = u / NTO;
    const int lo = (int)(u - tile * NTO);
    const int hi = (u1 - u) < (int64_t)(NTO - lo) ? lo + (int)(u1 - u) : NTO;
    if (lo == 0 && hi == NTO)
      layer_tile<KT, NTO, MODE, BF, true>(in_, in_stride, M, lds_raw, lb, mask_, mask_stride, out_,
                                          out_stride, tile, 0, NTO);
    else
      layer_tile<KT, NTO, MODE, BF, false>(in_, in_stride, M, lds_raw, lb, mask_, mask_stride, out_,
                                           out_stride, tile, lo, hi);
    u += hi - lo;
  }
}

// ---- one layer, FP32 through BF16 splits --------------------------------------------
// The modes of k_mlp_layer with float32 inputs, outputs and masks, the inputs split into
// three BF16 parts as they are loaded and the weights packed in three parts
// (pack_split_store).  The block's weights cover NTL of the layer's NTL * NCG output
// column tiles: with NCG = 2 (192 outputs, 110.6 KB of weights in LDS) block b serves
// column group (b / 8) % 2, so blocks b and b + 8, which run on the same XCD, read the
// same input rows and the second read is an L2 hit; the blocks of a group split its
// ntiles x NTL output blocks evenly over their waves (stream-K).
//
// A 32-feature slab of a lane's row is four float4 loads; one slab feeds 2 * 6 * NTL
// MFMAs, about a microsecond, less than a loaded HBM round trip, so slabs are loaded two
// ahead (three in registers), and the last two slabs of a tile prefetch the first two of
// the wave's next tile.

// The first QN (of two) 16-deep reduction steps of slab t (features 32 t + 16 q + 4 h +
// {0..3} and the same + 8 for step 2 t + q) into the accumulators of output tiles
// [to_lo, to_hi).  QN = 1 leaves out features 32 t + 16 .. 32 t + 31, for weights whose
// columns there are zero (their products add nothing).
template <int KT, int NTL, bool FULL, int QN = 2>
__device__ __forceinline__ void split_slab(f32x16 (&acc)[NTL], const bf16x8* lw, int lane,
                                           const float4 (&x)[4], int t, int to_lo, int to_hi) {
  constexpr int S = 2 * KT;
#pragma unroll
  for (int q = 0; q < QN; ++q) {
    bf16x8 b0, b1, b2;
    split8(x[2 * q], x[2 * q + 1], b0, b1, b2);
    bf16x8 a0[NTL], a1[NTL], a2[NTL];
#pragma unroll
    for (int to = 0; to < NTL; ++to) {
      if (!FULL && (to < to_lo || to >= to_hi)) continue;
      const bf16x8* a = lw + ((to * S + 2 * t + q) * 3) * 64 + lane;
      a0[to] = a[0];
      a1[to] = a[64];
      a2[to] = a[128];
    }
    // smallest terms first; independent accumulators interleaved
#define SPLIT_MFMA(A, B)                                                              \
  _Pragma("unroll") for (int to = 0; to < NTL; ++to) {                                \
    if (!FULL && (to < to_lo || to >= to_hi)) continue;                               \
    acc[to] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A[to], B, acc[to], 0, 0, 0);    \
  }
    SPLIT_MFMA(a2, b0)
    SPLIT_MFMA(a1, b1)
    SPLIT_MFMA(a0, b2)
    SPLIT_MFMA(a1, b0)
    SPLIT_MFMA(a0, b1)
    SPLIT_MFMA(a0, b0)
#undef SPLIT_MFMA
  }
}

__device__ __forceinline__ void load_slab(float4 (&x)[4], const float* __restrict__ in,
                                          int in_stride, int64_t row, int t, int h) {
  const float* rp = in + row * in_stride + 32 * t + 4 * h;
#pragma unroll
  for (int u = 0; u < 4; ++u) x[u] = *reinterpret_cast<const float4*>(rp + 8 * u);
}

// Epilogue of k_mlp_layer's modes on float32 rows: bias and ReLU (MODE 0), the ReLU mask
// (MODE 2), or the plain product (MODE 3); columns col0 + 32 to + ...  bits (may be
// NULL): the ReLU masks as bits, six words per 192-column row (bit k of word w: column
// 32 w + k positive) -- written by MODE 0, read by MODE 2 instead of the float mask.
template <int NTL, int MODE, bool FULL>
__device__ __forceinline__ void split_store(const f32x16 (&acc)[NTL], const float* lb,
                                            const float* __restrict__ mask, int mask_stride,
                                            uint32_t* __restrict__ bits,
                                            float* __restrict__ out, int out_stride, int64_t row,
                                            int h, int to_lo, int to_hi, int col0) {
  const int64_t obase = row * out_stride + 4 * h;
  const int64_t mbase = row * mask_stride + 4 * h;
  uint32_t* brow = bits ? bits + row * (kWidth / 32) + (col0 >> 5) : nullptr;
#pragma unroll
  for (int to = 0; to < NTL; ++to) {
    if (!FULL && (to < to_lo || to >= to_hi)) continue;
    uint32_t word = 0u;
    if (MODE == 2 && brow) word = brow[to];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      float v4[4];
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const int v = 4 * u + w;
        float x = acc[to][v];
        if (MODE == 0) {
          x += lb[dfeat(to, v, h)];
          x = x > 0.f ? x : 0.f;
        }
        v4[w] = x;
      }
      const int cofs = col0 + 32 * to + 8 * u;
      const int bit0 = 8 * u + 4 * h;  // bit of column cofs + 4 h in the word
      if (MODE == 0 && brow) {
#pragma unroll
        for (int w = 0; w < 4; ++w) word |= (v4[w] > 0.f ? 1u : 0u) << (bit0 + w);
      }
      if (MODE == 2) {
        if (brow) {
#pragma unroll
          for (int w = 0; w < 4; ++w) v4[w] = (word >> (bit0 + w)) & 1u ? v4[w] : 0.f;
        } else {
          const float4 mk = *reinterpret_cast<const float4*>(mask + mbase + cofs);
          v4[0] = mk.x > 0.f ? v4[0] : 0.f;
          v4[1] = mk.y > 0.f ? v4[1] : 0.f;
          v4[2] = mk.z > 0.f ? v4[2] : 0.f;
          v4[3] = mk.w > 0.f ? v4[3] : 0.f;
        }
      }
      *reinterpret_cast<float4*>(out + obase + cofs) = make_float4(v4[0], v4[1], v4[2], v4[3]);
    }
    if (MODE == 0 && brow) {
      // the two lane halves hold the two halves of the row's 32 columns
      word |= (uint32_t)__shfl_xor((int)word, 32, 64);
      if (h == 0) brow[to] = word;
    }
  }
}

// One 32-row tile, output tiles [to_lo, to_hi).  On entry ring[0] and ring[1] hold (or
// are loading) slabs 0 and 1 of this tile; slab t + 2 goes into ring[(t + 2) % 3] while
// slab t is multiplied, from the next tile (next_row: this lane's row in it) once t + 2
// passes the end.  KT % 3 == 0 keeps the ring positions the same for every tile.
template <int KT, int NTL, int MODE, bool FULL, int KQ>
__device__ __forceinline__ void split_tile(float4 (&ring)[3][4], const float* __restrict__ in,
                                           int in_stride, int64_t M, const bf16x8* lw,
                                           const float* lb, const float* __restrict__ mask,
                                           int mask_stride, uint32_t* __restrict__ bits,
                                           float* __restrict__ out, int out_stride, int64_t tile,
                                           int64_t next_row, int to_lo, int to_hi, int col0) {
  static_assert(KT % 3 == 0, "ring of three slabs");
  const int lane = threadIdx.x & 63, h = lane >> 5, rl = lane & 31;
  const int64_t row = tile * 32 + rl;
  const int64_t rrow = row < M ? row : M - 1;
  f32x16 acc[NTL];
#pragma unroll
  for (int t = 0; t < NTL; ++t)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[t][v] = 0.f;
#pragma unroll
  for (int t = 0; t < KT; ++t) {
    if (t + 2 < KT) load_slab(ring[(t + 2) % 3], in, in_stride, rrow, t + 2, h);
    else if (next_row >= 0) load_slab(ring[(t + 2) % 3], in, in_stride, next_row, t + 2 - KT, h);
    if (t < KT - 1 || KQ == 2 * KT)
      split_slab<KT, NTL, FULL>(acc, lw, lane, ring[t % 3], t, to_lo, to_hi);
    else
      split_slab<KT, NTL, FULL, 1>(acc, lw, lane, ring[t % 3], t, to_lo, to_hi);
  }
  if (row < M)
    split_store<NTL, MODE, FULL>(acc, lb, mask, mask_stride, bits, out, out_stride, row, h, to_lo,
                                 to_hi, col0);
}

// The same for KT = 2 (the 64-wide first layer): both slabs of the next tile load while
// this tile's are multiplied (ring[2..3] <- next tile, then swapped).
template <int NTL, int MODE, bool FULL, int KQ>
__device__ __forceinline__ void split_tile2(float4 (&ring)[4][4], const float* __restrict__ in,
                                            int in_stride, int64_t M, const bf16x8* lw,
                                            const float* lb, const float* __restrict__ mask,
                                            int mask_stride, uint32_t* __restrict__ bits,
                                            float* __restrict__ out, int out_stride, int64_t tile,
                                            int64_t next_row, int to_lo, int to_hi, int col0) {
  const int lane = threadIdx.x & 63, h = lane >> 5, rl = lane & 31;
  const int64_t row = tile * 32 + rl;
  f32x16 acc[NTL];
#pragma unroll
  for (int t = 0; t < NTL; ++t)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[t][v] = 0.f;
  if (next_row >= 0) {
    load_slab(ring[2], in, in_stride, next_row, 0, h);
    load_slab(ring[3], in, in_stride, next_row, 1, h);
  }
  split_slab<2, NTL, FULL>(acc, lw, lane, ring[0], 0, to_lo, to_hi);
  if (KQ == 4)
    split_slab<2, NTL, FULL>(acc, lw, lane, ring[1], 1, to_lo, to_hi);
  else
    split_slab<2, NTL, FULL, 1>(acc, lw, lane, ring[1], 1, to_lo, to_hi);
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    ring[0][u] = ring[2][u];
    ring[1][u] = ring[3][u];
  }
  if (row < M)
    split_store<NTL, MODE, FULL>(acc, lb, mask, mask_stride, bits, out, out_stride, row, h, to_lo,
                                 to_hi, col0);
}

// KQ: the 16-deep reduction steps to run, 2 KT, or 2 KT - 1 when the weights' last 16
// input columns are zero (the padding of a first layer's packed weights).
template <int KT, int NTL, int NCG, int MODE, int KQ = 2 * KT>
__global__ void __launch_bounds__(kLayerThreads) k_mlp_layer_split(
    const float* __restrict__ in, int in_stride, int64_t M, const int64_t* __restrict__ Md,
    const bf16x8* __restrict__ wpk, const float* __restrict__ bias,
    const float* __restrict__ mask, int mask_stride, float* __restrict__ out, int out_stride,
    uint32_t* __restrict__ bits) {
  static_assert(KT == 2 || KT % 3 == 0, "input width 64, 96 or 192");
  static_assert(KQ == 2 * KT || KQ == 2 * KT - 1, "whole slabs, or all but the last 16");
  constexpr int S = 2 * KT;
  constexpr int WV = NTL * S * 3 * 64;   // bf16x8 vectors of one column group
  __shared__ bf16x8 lw[WV];
  __shared__ float lb[NTL * 32];
  const int tid = threadIdx.x;
  const int cg = NCG == 1 ? 0 : (int)((blockIdx.x >> 3) % NCG);
  const int64_t bw = NCG == 1 ? (int64_t)blockIdx.x
                              : (int64_t)((blockIdx.x >> 3) / NCG) * 8 + (blockIdx.x & 7);
  const int64_t nb = gridDim.x / NCG;
  // the wave index is uniform: the tile and column choices below stay scalar
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, h = lane >> 5, rl = lane & 31;
  M = eff_rows(M, Md);
  const int64_t ntiles = (M + 31) / 32;
  const int64_t nw = nb * (blockDim.x >> 6);
  const int64_t gw = bw * (blockDim.x >> 6) + wave;
  const int64_t total = ntiles * NTL;
  // the wave's share [u, u1) of the output blocks; in 32 bits when the products fit
  // (the 64-bit divisions are long scalar sequences at the start of every wave)
  int64_t u, u1;
  if ((uint64_t)total * (uint64_t)nw < (1ull << 32)) {
    const uint32_t t32 = (uint32_t)total, n32 = (uint32_t)nw, g32 = (uint32_t)gw;
    u = t32 * g32 / n32;
    u1 = t32 * (g32 + 1u) / n32;
  } else {
    u = total * gw / nw;
    u1 = total * (gw + 1) / nw;
  }
  const int col0 = cg * NTL * 32;
  // this lane's row of a tile, clamped into [0, M) (rows past M are computed, not stored)
  auto lane_row = [&](int64_t tile) {
    const int64_t r = tile * 32 + rl;
    return r < M ? r : M - 1;
  };
  constexpr int R = KT == 2 ? 4 : 3;
  float4 ring[R][4];
  // the wave's first two input slabs load while the workgroup stages the weights
  if (u < u1) {
    load_slab(ring[0], in, in_stride, lane_row(u / NTL), 0, h);
    load_slab(ring[1], in, in_stride, lane_row(u / NTL), 1, h);
  }
  {
    const uint4* src = reinterpret_cast<const uint4*>(wpk) + (int64_t)cg * WV;
    uint4* dst = reinterpret_cast<uint4*>(lw);
    constexpr int P = (WV + kLayerThreads - 1) / kLayerThreads;
    uint4 v[P];
#pragma unroll
    for (int b = 0; b < P; ++b) {
      const int i = tid + b * kLayerThreads;
      v[b] = i < WV ? src[i] : make_uint4(0u, 0u, 0u, 0u);
    }
#pragma unroll
    for (int b = 0; b < P; ++b) {
      const int i = tid + b * kLayerThreads;
      if (i < WV) dst[i] = v[b];
    }
    if (MODE == 0)
      for (int i = tid; i < NTL * 32; i += blockDim.x) lb[i] = bias[cg * NTL * 32 + i];
  }
  __syncthreads();
  while (u < u1) {
    const int64_t tile = u / NTL;
    const int lo = (int)(u - tile * NTL);
    const int hi = (u1 - u) < (int64_t)(NTL - lo) ? lo + (int)(u1 - u) : NTL;
    const int64_t un = u + (hi - lo);
    const int64_t next_row = un < u1 ? lane_row(un / NTL) : -1;
    if constexpr (KT == 2) {
      if (lo == 0 && hi == NTL)
        split_tile2<NTL, MODE, true, KQ>(ring, in, in_stride, M, lw, lb, mask, mask_stride, bits, out,
                                     out_stride, tile, next_row, 0, NTL, col0);
      else
        split_tile2<NTL, MODE, false, KQ>(ring, in, in_stride, M, lw, lb, mask, mask_stride, bits, out,
                                      out_stride, tile, next_row, lo, hi, col0);
    } else {
      if (lo == 0 && hi == NTL)
        split_tile<KT, NTL, MODE, true, KQ>(ring, in, in_stride, M, lw, lb, mask, mask_stride, bits, out,
                                        out_stride, tile, next_row, 0, NTL, col0);
      else
        split_tile<KT, NTL, MODE, false, KQ>(ring, in, in_stride, M, lw, lb, mask, mask_stride, bits, out,
                                         out_stride, tile, next_row, lo, hi, col0);
    }
    u = un;
  }
}

// ---- the whole network in one pass, FP32 through BF16 splits ------------------------------
// A layer at a time, every activation row goes to HBM and back between the layers: at 1.4 M
// rows a 131,072-ray render spent 2.3 ms on 4.3 GB of them.  For a forward whose activations
// nobody reads afterwards (no backward to come) a wave keeps a tile of 32 rows in registers
// through all the layers: a layer's accumulators (row = feature, column = sample) hold, after
// bias and ReLU, exactly the next layer's B operands.  What moves is the weights: a layer's
// 32-feature slab (all 192 outputs, three parts, 36.9 KB) is staged in one of three LDS
// buffers, loaded from L2 two slabs ahead, and the eight waves of a workgroup (two per SIMD,
// 256 registers each) multiply it together, one barrier a slab.  Every output element's MFMAs,
// bias, ReLU and logit sums are those of k_mlp_layer_split and k_mlp_logits in the same order,
// so the logits are theirs bit for bit, with a gradient to follow or without.
//
// Bound by the matrix cores: 1.4 M rows of 42 columns in 1,186 us, 1,175 TFLOP/s of BF16
// products where a large product reaches 1,212 (the layers' passes: 2,300 us).  Up to 256 rows
// a CU (65,536) it is one round of 14 slabs, 45 us from one row on.  Three products of two
// FP16 parts with a scale a row took 803 us, but kept 22 bits of an operand instead of 24, and
// fewer of entries far below their row's largest (beside one of 1e8 with zero weights: 6e-6
// off float64 where this is 4e-7), so the parts are the layers' three.
constexpr int kNetMaxHidden = 4;
constexpr int kNetWaves = 8;                // two per SIMD
constexpr int kNetRuns = 36;                // 1 KB runs of a slab: [tile][step][part]
constexpr int kNetStage = (kNetRuns + kNetWaves - 1) / kNetWaves;
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

struct NetArgs {
  const float* in;
  int in_stride, n_hidden;
  int64_t M;
  const int64_t* Md;
  const bf16x8* w[kNetMaxHidden];
  const float* b[kNetMaxHidden];
  const float* w3;
  const float* b3;
  float* logits;
};

// Slab (step pair t) of a layer with `steps` 16-deep steps: runs of 64 vectors, six an output
// tile, run wave + kNetWaves k in each wave's k-th register (a run past the slab reads its
// last one and is not stored).
__device__ __forceinline__ void net_load(u32x4 (&v)[kNetStage], const bf16x8* __restrict__ w,
                                         int steps, int t, int wave, int lane) {
#pragma unroll
  for (int k = 0; k < kNetStage; ++k) {
    const int run = min(wave + kNetWaves * k, kNetRuns - 1), to = run / 6;
    v[k] = reinterpret_cast<const u32x4*>(w)[(to * steps + 2 * t) * 192 + (run - 6 * to) * 64 + lane];
  }
}

__device__ __forceinline__ void net_store(const u32x4 (&v)[kNetStage], bf16x8* lw, int wave, int lane) {
#pragma unroll
  for (int k = 0; k < kNetStage; ++k) {
    const int run = wave + kNetWaves * k;
    if (run < kNetRuns) reinterpret_cast<u32x4*>(lw)[run * 64 + lane] = v[k];
  }
}

// One slab into the accumulators: acc[to] += W slab x x (the 16 features of the slab a lane
// holds of its row).  QN as in split_slab.  Two output tiles at a time: their independent
// MFMAs alternate.
template <int QN>
__device__ __forceinline__ void net_slab(f32x16 (&acc)[6], const f32x16& x, const bf16x8* lw,
                                         int lane) {
#pragma unroll
  for (int q = 0; q < QN; ++q) {
    bf16x8 b0, b1, b2;
    split8(make_float4(x[8 * q], x[8 * q + 1], x[8 * q + 2], x[8 * q + 3]),
           make_float4(x[8 * q + 4], x[8 * q + 5], x[8 * q + 6], x[8 * q + 7]), b0, b1, b2);
    constexpr int P = 2;
#pragma unroll
    for (int to = 0; to < 6; to += P) {
      bf16x8 a0[P], a1[P], a2[P];
#pragma unroll
      for (int i = 0; i < P; ++i) {
        const bf16x8* a = lw + (((to + i) * 2 + q) * 3) * 64 + lane;
        a0[i] = a[0];
        a1[i] = a[64];
        a2[i] = a[128];
      }
      // smallest terms first, as split_slab
#define NET_MFMA(A, B)                                                                    \
  _Pragma("unroll") for (int i = 0; i < P; ++i)                                           \
    acc[to + i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A[i], B, acc[to + i], 0, 0, 0);
      NET_MFMA(a2, b0)
      NET_MFMA(a1, b1)
      NET_MFMA(a0, b2)
      NET_MFMA(a1, b0)
      NET_MFMA(a0, b1)
      NET_MFMA(a0, b0)
#undef NET_MFMA
    }
  }
}

__device__ __forceinline__ void net_zero(f32x16 (&acc)[6]) {
#pragma unroll
  for (int to = 0; to < 6; ++to)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[to][v] = 0.f;
}

// The slab after next on its way while this one is multiplied, then into the buffer that the
// slab before this one has left.
#define NET_STEP(T, QN)                                                                  \
  {                                                                                       \
    load();                                                                               \
    net_slab<QN>(acc, x[T], lw[cur], lane);                                               \
    net_store(stage, lw[cur == 0 ? 2 : cur - 1], wave, lane);                             \
    cur = cur == 2 ? 0 : cur + 1;                                                         \
    __syncthreads();                                                                      \
  }

// Logits of X without keeping the activations.  KT0: 32-feature slabs of the input (its
// packed width), KQ0: its 16-deep steps with weights that are not all zero.
template <int KT0, int KQ0>
__global__ void __launch_bounds__(64 * kNetWaves) k_mlp_net_fwd(NetArgs a) {
  __shared__ bf16x8 lw[3][kNetRuns * 64];
  __shared__ float lb[kNetMaxHidden][kWidth];
  __shared__ float l3[3 * kWidth + 4];
  const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, rl = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t M = eff_rows(a.M, a.Md);
  constexpr int kRows = 32 * kNetWaves;
  const int64_t rounds = (M + kRows - 1) / kRows;
  if ((int64_t)blockIdx.x >= rounds) return;
  for (int li = 0; li < a.n_hidden; ++li)
    if (tid < kWidth) lb[li][tid] = a.b[li][tid];
  for (int i = tid; i < 3 * kWidth + 3; i += 64 * kNetWaves)
    l3[i] = i < 3 * kWidth ? a.w3[i] : a.b3[i - 3 * kWidth];
  // the slab to load next: its layer and step pair
  int nli = 0, nts = 0;
  u32x4 stage[kNetStage];
  auto load = [&]() __attribute__((always_inline)) {
    net_load(stage, a.w[nli], nli == 0 ? 2 * KT0 : 12, nts, wave, lane);
    if (++nts == (nli == 0 ? KT0 : 6)) {
      nts = 0;
      if (++nli == a.n_hidden) nli = 0;
    }
  };
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    load();
    net_store(stage, lw[i], wave, lane);
  }
  int cur = 0;
  f32x16 x[6];    // the layer's input, slab by slab
  f32x16 acc[6];
  __syncthreads();
  for (int64_t round = blockIdx.x; round < rounds; round += gridDim.x) {
    const int64_t r = round * kRows + wave * 32 + rl;
    {
      const float* rp = a.in + (r < M ? r : M - 1) * a.in_stride + 4 * h;
#pragma unroll
      for (int t = 0; t < KT0; ++t)
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const float4 v = *reinterpret_cast<const float4*>(rp + 32 * t + 8 * u);
          x[t][4 * u] = v.x;
          x[t][4 * u + 1] = v.y;
          x[t][4 * u + 2] = v.z;
          x[t][4 * u + 3] = v.w;
        }
    }
    // bias and ReLU: the next layer's input (and the logits' at the end)
    auto finish = [&](int li) __attribute__((always_inline)) {
#pragma unroll
      for (int to = 0; to < 6; ++to) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const float4 b4 = *reinterpret_cast<const float4*>(&lb[li][32 * to + 8 * u + 4 * h]);
          const float bv[4] = {b4.x, b4.y, b4.z, b4.w};
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float v = acc[to][4 * u + e] + bv[e];
            x[to][4 * u + e] = v > 0.f ? v : 0.f;
          }
        }
        __builtin_amdgcn_sched_barrier(0);  // (or the reads of all tiles come first, and spill)
      }
    };
    net_zero(acc);
#pragma unroll
    for (int t = 0; t < KT0; ++t) {
      if (t < KT0 - 1 || KQ0 == 2 * KT0) NET_STEP(t, 2)
      else NET_STEP(t, 1)
    }
    finish(0);
    for (int li = 1; li < a.n_hidden; ++li) {
      net_zero(acc);
#pragma unroll
      for (int t = 0; t < 6; ++t) NET_STEP(t, 2)
      finish(li);
    }
    // logits: the features 64 q + 4 sl .. + 3 summed over q for each of sixteen sl (this half
    // holds sl = 8 (t % 2) + 2 u + h), then those sums pairwise, as k_mlp_logits does
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      float p[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        float t = 0.f;
#pragma unroll
        for (int q = 0; q < 3; ++q) {
          const int tt = 2 * q + (j >> 2), u = j & 3;
          const float4 w = *reinterpret_cast<const float4*>(&l3[c * kWidth + 32 * tt + 8 * u + 4 * h]);
          t += x[tt][4 * u] * w.x + x[tt][4 * u + 1] * w.y + x[tt][4 * u + 2] * w.z +
               x[tt][4 * u + 3] * w.w;
        }
        p[j] = t;
      }
      __builtin_amdgcn_sched_barrier(0);
      const float s = ((p[0] + p[4]) + (p[2] + p[6])) + ((p[1] + p[5]) + (p[3] + p[7]));
      const float res = s + __shfl_xor(s, 32, 64) + l3[3 * kWidth + c];
      if (r < M && h == 0) a.logits[3 * r + c] = res;
    }
  }
}

#undef NET_STEP

// logits [M, 3] = H W3^T + b3 from the stored activations (bfloat16 when BF).  Sixteen
// lanes per row (three float4 of features each, 256 contiguous bytes per load across the
// group), four rows per wave and two such row sets in flight per iteration; the partial
// dot products are summed over the 16-lane group.
template <bool BF>
__global__ void __launch_bounds__(256) k_mlp_logits(const void* __restrict__ H_, int hs,
                                                    int64_t M, const int64_t* __restrict__ Md,
                                                    const float* __restrict__ w3,
                                                    const float* __restrict__ b3,
                                                    float* __restrict__ logits) {
  constexpr int U = 2;
  M = eff_rows(M, Md);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, rg = lane >> 4, sl = lane & 15;
  float4 w[3][3];
#pragma unroll
  for (int c = 0; c < 3; ++c)
#pragma unroll
    for (int q = 0; q < 3; ++q)
      w[c][q] = *reinterpret_cast<const float4*>(w3 + c * kWidth + 64 * q + 4 * sl);
  const float c0 = b3[0], c1 = b3[1], c2 = b3[2];
  const int64_t waves = (int64_t)gridDim.x * (blockDim.x >> 6);
  for (int64_t r0 = ((int64_t)blockIdx.x * (blockDim.x >> 6) + wave) * 4 * U; r0 < M;
       r0 += waves * 4 * U) {
    float4 x[U][3];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t r = r0 + 4 * u + rg;
      const int64_t rr = r < M ? r : M - 1;
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        const int f = 64 * q + 4 * sl;
        if constexpr (BF) {
          const uint2 v = *reinterpret_cast<const uint2*>(reinterpret_cast<const __bf16*>(H_) + rr * hs + f);
          const __bf16* b = reinterpret_cast<const __bf16*>(&v);
          x[u][q] = make_float4((float)b[0], (float)b[1], (float)b[2], (float)b[3]);
        } else {
          x[u][q] = *reinterpret_cast<const float4*>(reinterpret_cast<const float*>(H_) + rr * hs + f);
        }
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      float p[3];
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        float t = 0.f;
#pragma unroll
        for (int q = 0; q < 3; ++q)
          t += x[u][q].x * w[c][q].x + x[u][q].y * w[c][q].y + x[u][q].z * w[c][q].z +
               x[u][q].w * w[c][q].w;
#pragma unroll
        for (int off = 8; off >= 1; off >>= 1) t += __shfl_xor(t, off, 64);
        p[c] = t;
      }
      const int64_t r = r0 + 4 * u + rg;
      if (sl == 0 && r < M) {
        logits[3 * r] = p[0] + c0;
        logits[3 * r + 1] = p[1] + c1;
        logits[3 * r + 2] = p[2] + c2;
      }
    }
  }
}

// Backward through the 3-output layer, one pass over H:
//   dH [M, 192] = (dlogit W3) * [H > 0]   (DH true),
//   part3[blk][c * 192 + f] = sum over the block's rows of dlogit[r][c] H[r][f],
//   partb3[blk][c]          = sum over the block's rows of dlogit[r][c].
template <bool BF, bool DH>
__global__ void __launch_bounds__(192) k_mlp_last_bwd(const float* __restrict__ dlogit,
                                                      const void* __restrict__ H_, int hs,
                                                      int64_t M, const int64_t* __restrict__ Md,
                                                      const float* __restrict__ w3,
                                                      float* __restrict__ dH, int dhs,
                                                      float* __restrict__ part3,
                                                      float* __restrict__ partb3) {
  const int f = threadIdx.x;
  const float w0 = DH ? w3[f] : 0.f, w1 = DH ? w3[kWidth + f] : 0.f;
  const float w2 = DH ? w3[2 * kWidth + f] : 0.f;
  M = eff_rows(M, Md);
  const int64_t rows_per_block = (M + gridDim.x - 1) / gridDim.x;
  const int64_t r_begin = blockIdx.x * rows_per_block;
  const int64_t r_end = (r_begin + rows_per_block < M) ? r_begin + rows_per_block : M;
  float a0 = 0.f, a1 = 0.f, a2 = 0.f, c0 = 0.f, c1 = 0.f, c2 = 0.f;
#pragma unroll 4
  for (int64_t r = r_begin; r < r_end; ++r) {
    const float hv = BF ? (float)reinterpret_cast<const __bf16*>(H_)[r * hs + f]
                        : reinterpret_cast<const float*>(H_)[r * hs + f];
    const float g0 = dlogit[3 * r], g1 = dlogit[3 * r + 1], g2 = dlogit[3 * r + 2];
    if (DH) {
      const float g = g0 * w0 + g1 * w1 + g2 * w2;
      dH[r * dhs + f] = hv > 0.f ? g : 0.f;
    }
    a0 += g0 * hv;
    a1 += g1 * hv;
    a2 += g2 * hv;
    c0 += g0;
    c1 += g1;
    c2 += g2;
  }
  float* pb = part3 + (int64_t)blockIdx.x * 3 * kWidth;
  pb[f] = a0;
  pb[kWidth + f] = a1;
  pb[2 * kWidth + f] = a2;
  if (f == 0) {
    partb3[3 * blockIdx.x] = c0;
    partb3[3 * blockIdx.x + 1] = c1;
    partb3[3 * blockIdx.x + 2] = c2;
  }
}

// dH [M, 192] = (dlogit W3) * mask from the last hidden layer's ReLU mask bits (bit
// f % 32 of word f / 32 of a row's six words is column f's).  A thread owns four columns
// 4 q .. 4 q + 3 of a row (48 threads a row, four rows a block) and keeps their twelve
// W3 entries in registers; blocks stride over the rows.
__global__ void __launch_bounds__(192) k_mlp_last_dgrad(const float* __restrict__ dlogit,
                                                        const uint32_t* __restrict__ bits,
                                                        int64_t M, const int64_t* __restrict__ Md,
                                                        const float* __restrict__ w3,
                                                        float* __restrict__ dH, int dhs) {
  constexpr int Q = kWidth / 4;
  const int q = threadIdx.x % Q, rb = threadIdx.x / Q;
  float w[3][4];
#pragma unroll
  for (int c = 0; c < 3; ++c)
#pragma unroll
    for (int e = 0; e < 4; ++e) w[c][e] = w3[c * kWidth + 4 * q + e];
  M = eff_rows(M, Md);
  const int shift = 4 * (q % 8);
  for (int64_t r = (int64_t)blockIdx.x * 4 + rb; r < M; r += (int64_t)gridDim.x * 4) {
    const float g0 = dlogit[3 * r], g1 = dlogit[3 * r + 1], g2 = dlogit[3 * r + 2];
    const uint32_t word = bits[r * (kWidth / 32) + q / 8] >> shift;
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float g = g0 * w[0][e] + g1 * w[1][e] + g2 * w[2][e];
      v[e] = (word >> e) & 1u ? g : 0.f;
    }
    *reinterpret_cast<float4*>(dH + r * dhs + 4 * q) = make_float4(v[0], v[1], v[2], v[3]);
  }
}

// ---- weight gradients: part[blk] = dY[rows]^T X[rows], partb[blk] = sum dY[rows] --------
// dY [M, 192] float32, X [M, 32*KT] (float32 or bfloat16).  A block takes a contiguous
// range of rows and streams it through LDS in chunks of 32 rows (double buffered: the
// next chunk's global loads are in flight while the current chunk's MFMAs run).  Wave w
// owns output tiles n in [TNW (w % NWN), +TNW) x k in [TKW (w / NWN), +TKW) of the
// [192, 32 KT] slice.  One MFMA step reduces over two rows: lane half h takes row
// 2 s + h of the chunk, lane l % 32 the column.
template <int KT>
struct WgradShape {
  // KT = 6: 4 waves of 3x3 tiles; KT = 3: 3 waves of 2x3; KT = 2: 4 waves of 3x1
  static constexpr int TNW = KT == 3 ? 2 : 3;
  static constexpr int TKW = KT == 2 ? 1 : 3;
  static constexpr int NWN = 6 / TNW;
  static constexpr int NWK = KT / TKW;
  static constexpr int WAVES = NWN * NWK;
};
constexpr int kWgradChunk = 32;

template <int KT, bool BF>
__global__ void __launch_bounds__(256) k_mlp_wgrad(const float* __restrict__ dY, int dys,
                                                   const void* __restrict__ X_, int xs, int64_t M,
                                                   const int64_t* __restrict__ Md,
                                                   float* __restrict__ part,
                                                   float* __restrict__ partb) {
  using Sh = WgradShape<KT>;
  constexpr int K = 32 * KT, TNW = Sh::TNW, TKW = Sh::TKW, NWN = Sh::NWN;
  constexpr int NT = 64 * Sh::WAVES;
  constexpr int CH = kWgradChunk;
  constexpr int NY4 = CH * kWidth / 4 / NT;  // float4 of dY per thread per chunk
  constexpr int NX4 = CH * K / 4 / NT;       // 4-element groups of X per thread per chunk
  static_assert(CH * kWidth / 4 % NT == 0 && CH * K / 4 % NT == 0, "chunk split");
  __shared__ __attribute__((aligned(16))) float sY[2][CH][kWidth];
  __shared__ __attribute__((aligned(16))) float sX[2][CH][K];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, h = lane >> 5, rl = lane & 31;
  const int tn0 = TNW * (wave % NWN), tk0 = TKW * (wave / NWN);
  M = eff_rows(M, Md);
  // contiguous row ranges of whole chunks, one per block
  const int64_t rows_per_block = ((M + gridDim.x - 1) / gridDim.x + CH - 1) / CH * CH;
  const int64_t r_begin = blockIdx.x * rows_per_block;
  const int64_t r_end = (r_begin + rows_per_block < M) ? r_begin + rows_per_block : M;

  float4 ry[NY4], rx[NX4];
  auto load = [&](int64_t r0) {
#pragma unroll
    for (int q = 0; q < NY4; ++q) {
      const int e = tid + q * NT, row = e / (kWidth / 4), c4 = e % (kWidth / 4);
      const int64_t r = r0 + row;
      ry[q] = r < r_end ? *reinterpret_cast<const float4*>(dY + r * dys + 4 * c4)
                        : make_float4(0.f, 0.f, 0.f, 0.f);
    }
#pragma unroll
    for (int q = 0; q < NX4; ++q) {
      const int e = tid + q * NT, row = e / (K / 4), c4 = e % (K / 4);
      const int64_t r = r0 + row;
      float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
      if (r < r_end) {
        if constexpr (BF) {
          const uint2 u = *reinterpret_cast<const uint2*>(reinterpret_cast<const __bf16*>(X_) + r * xs + 4 * c4);
          const __bf16* b = reinterpret_cast<const __bf16*>(&u);
          v = make_float4((float)b[0], (float)b[1], (float)b[2], (float)b[3]);
        } else {
          v = *reinterpret_cast<const float4*>(reinterpret_cast<const float*>(X_) + r * xs + 4 * c4);
        }
      }
      rx[q] = v;
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int q = 0; q < NY4; ++q) {
      const int e = tid + q * NT;
      *reinterpret_cast<float4*>(&sY[buf][e / (kWidth / 4)][4 * (e % (kWidth / 4))]) = ry[q];
    }
#pragma unroll
    for (int q = 0; q < NX4; ++q) {
      const int e = tid + q * NT;
      *reinterpret_cast<float4*>(&sX[buf][e / (K / 4)][4 * (e % (K / 4))]) = rx[q];
    }
  };

  f32x16 acc[TNW][TKW];
#pragma unroll
  for (int i = 0; i < TNW; ++i)
#pragma unroll
    for (int j = 0; j < TKW; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
  float bs[TNW];
#pragma unroll
  for (int i = 0; i < TNW; ++i) bs[i] = 0.f;

  const int64_t nch = r_end > r_begin ? (r_end - r_begin + CH - 1) / CH : 0;
  if (nch > 0) {
    load(r_begin);
    store(0);
  }
  __syncthreads();
  for (int64_t c = 0; c < nch; ++c) {
    const int buf = (int)(c & 1);
    if (c + 1 < nch) load(r_begin + (c + 1) * CH);
#pragma unroll
    for (int st = 0; st < CH / 2; ++st) {
      float a[TNW], b[TKW];
#pragma unroll
      for (int i = 0; i < TNW; ++i) {
        a[i] = sY[buf][2 * st + h][32 * (tn0 + i) + rl];
        bs[i] += a[i];
      }
#pragma unroll
      for (int j = 0; j < TKW; ++j) b[j] = sX[buf][2 * st + h][32 * (tk0 + j) + rl];
#pragma unroll
      for (int i = 0; i < TNW; ++i)
#pragma unroll
        for (int j = 0; j < TKW; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], b[j], acc[i][j], 0, 0, 0);
    }
    if (c + 1 < nch) store(buf ^ 1);
    __syncthreads();
  }
  float* pb = part + (int64_t)blockIdx.x * kWidth * K;
#pragma unroll
  for (int i = 0; i < TNW; ++i)
#pragma unroll
    for (int j = 0; j < TKW; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int n = dfeat(tn0 + i, v, h);
        pb[n * K + 32 * (tk0 + j) + rl] = acc[i][j][v];
      }
  if (wave < NWN) {
#pragma unroll
    for (int i = 0; i < TNW; ++i) {
      const float t = bs[i] + __shfl_xor(bs[i], 32, 64);
      if (h == 0) partb[(int64_t)blockIdx.x * kWidth + 32 * (tn0 + i) + rl] = t;
    }
  }
}

// ---- weight gradients from three-way BF16 splits (PREC_F32_SPLIT) --------------------
// The same product as k_mlp_wgrad with FP32 accuracy: each element of dY and X is split
// once, when its 32-row chunk is staged in LDS, into three BF16 parts (split3), and each
// 16-deep reduction step of an output tile is six 32x32x16 BF16 MFMAs (the products
// x_i w_j with i + j <= 2) instead of eight 32x32x2 FP32 MFMAs.  The LDS holds, per part,
// row group g (rows 8 g .. 8 g + 7 of the chunk) and column c as one bf16x8 vector, so a
// lane's operand (lane half h: row group 2 s + h in reduction step s, lane % 32: the
// column) is one ds_read_b128.  A thread stages fixed (row group, column) units: unit
// u = tid + q * threads, dY's 4 x 192 units first, then X's 4 x K; its eight loads (one
// per row) are coalesced across the lanes, which take consecutive columns.  The next
// chunk's loads are issued before the current chunk's MFMAs.  The bias gradient sum dY
// comes from the staged FP32 values of the dY units (fixed per thread, so summed in
// registers).
constexpr int kWsChunk = 32;
constexpr int kWsGroups = kWsChunk / 8;

template <int KT>
__global__ void __launch_bounds__(256) k_mlp_wgrad_split(const float* __restrict__ dY, int dys,
                                                         const float* __restrict__ X, int xs,
                                                         int64_t M, const int64_t* __restrict__ Md,
                                                         float* __restrict__ part,
                                                         float* __restrict__ partb,
                                                         unsigned long long* __restrict__ stamps) {
  if (stamps && threadIdx.x == 0) atomicMin(&stamps[0], (unsigned long long)wall_clock64());
  using Sh = WgradShape<KT>;
  constexpr int K = 32 * KT, TNW = Sh::TNW, TKW = Sh::TKW, NWN = Sh::NWN;
  constexpr int NT = 64 * Sh::WAVES;
  constexpr int UY = kWsGroups * kWidth, UX = kWsGroups * K, U = UY + UX;
  constexpr int NU = (U + NT - 1) / NT;
  __shared__ bf16x8 sY[3][kWsGroups][kWidth];
  __shared__ bf16x8 sX[3][kWsGroups][K];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, h = lane >> 5, rl = lane & 31;
  const int tn0 = TNW * (wave % NWN), tk0 = TKW * (wave / NWN);
  M = eff_rows(M, Md);
  const int64_t rows_per_block =
      ((M + gridDim.x - 1) / gridDim.x + kWsChunk - 1) / kWsChunk * kWsChunk;
  const int64_t r_begin = blockIdx.x * rows_per_block;
  const int64_t r_end = (r_begin + rows_per_block < M) ? r_begin + rows_per_block : M;
  const int64_t nch = r_end > r_begin ? (r_end - r_begin + kWsChunk - 1) / kWsChunk : 0;

  // per unit: its first row's address in the block's first chunk, its row group (row
  // offset 8 g in a chunk) and the row stride; idle units (u >= U) load nothing
  const float* ubase[NU];
  int ugrp[NU], ustride[NU];
#pragma unroll
  for (int q = 0; q < NU; ++q) {
    const int u = tid + q * NT;
    int g = 0, c = 0, st = 0;
    const float* src = dY;
    if (u < UY) {
      g = u / kWidth;
      c = u % kWidth;
      st = dys;
    } else if (u < U) {
      g = (u - UY) / K;
      c = (u - UY) % K;
      src = X;
      st = xs;
    }
    ugrp[q] = g;
    ustride[q] = st;
    ubase[q] = src + (r_begin + 8 * g) * (int64_t)st + c;
  }
  float v[NU][8];
  float bsum[NU];
#pragma unroll
  for (int q = 0; q < NU; ++q) bsum[q] = 0.f;
  // rows r0 + 8 g + e of every unit, zero past r_end (the address is clamped to the
  // unit's last valid row, or its first row when it has none, so every load is in bounds)
  auto load = [&](int64_t ch) {
    const int64_t r0 = r_begin + ch * kWsChunk;
    if (r0 + kWsChunk <= r_end) {
      // a whole chunk (every chunk but a block's last): no row checks
#pragma unroll
      for (int q = 0; q < NU; ++q) {
        const float* p = ubase[q] + ch * kWsChunk * (int64_t)ustride[q];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          v[q][e] = *p;
          p += ustride[q];
        }
      }
      return;
    }
#pragma unroll
    for (int q = 0; q < NU; ++q) {
      const int64_t avail = r_end - (r0 + 8 * ugrp[q]);
      const int n = tid + q * NT < U ? (avail < 0 ? 0 : (avail > 8 ? 8 : (int)avail)) : 0;
      const float* p = ubase[q] + ch * kWsChunk * (int64_t)ustride[q];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int ee = e < n ? e : (n > 0 ? n - 1 : 0);
        const float x = p[(n > 0 ? ee : -8 * ugrp[q] - ch * kWsChunk) * (int64_t)ustride[q]];
        v[q][e] = e < n ? x : 0.f;
      }
    }
  };
  auto store = [&]() {
#pragma unroll
    for (int q = 0; q < NU; ++q) {
      const int u = tid + q * NT;
      if (u >= U) continue;
      bf16x8 p0, p1, p2;
      split8(make_float4(v[q][0], v[q][1], v[q][2], v[q][3]),
             make_float4(v[q][4], v[q][5], v[q][6], v[q][7]), p0, p1, p2);
      if (u < UY) {
        const int g = u / kWidth, c = u % kWidth;
        sY[0][g][c] = p0;
        sY[1][g][c] = p1;
        sY[2][g][c] = p2;
#pragma unroll
        for (int e = 0; e < 8; ++e) bsum[q] += v[q][e];
      } else {
        const int g = (u - UY) / K, c = (u - UY) % K;
        sX[0][g][c] = p0;
        sX[1][g][c] = p1;
        sX[2][g][c] = p2;
      }
    }
  };

  f32x16 acc[TNW][TKW];
#pragma unroll
  for (int i = 0; i < TNW; ++i)
#pragma unroll
    for (int j = 0; j < TKW; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  if (nch > 0) {
    load(0);
    store();
  }
  __syncthreads();
  for (int64_t c = 0; c < nch; ++c) {
    if (c + 1 < nch) load(c + 1);
#pragma unroll
    for (int s2 = 0; s2 < kWsGroups / 2; ++s2) {
      const int g = 2 * s2 + h;
      bf16x8 a[TNW][3], b[TKW][3];
#pragma unroll
      for (int i = 0; i < TNW; ++i)
#pragma unroll
        for (int pp = 0; pp < 3; ++pp) a[i][pp] = sY[pp][g][32 * (tn0 + i) + rl];
#pragma unroll
      for (int j = 0; j < TKW; ++j)
#pragma unroll
        for (int pp = 0; pp < 3; ++pp) b[j][pp] = sX[pp][g][32 * (tk0 + j) + rl];
      // smallest terms first; independent accumulators interleaved
#define WS_MFMA(PA, PB)                                                                   \
  _Pragma("unroll") for (int i = 0; i < TNW; ++i)                                         \
  _Pragma("unroll") for (int j = 0; j < TKW; ++j)                                         \
    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i][PA], b[j][PB], acc[i][j], 0, 0, 0);
      WS_MFMA(2, 0)
      WS_MFMA(1, 1)
      WS_MFMA(0, 2)
      WS_MFMA(1, 0)
      WS_MFMA(0, 1)
      WS_MFMA(0, 0)
#undef WS_MFMA
    }
    if (c + 1 < nch) {
      __syncthreads();  // every wave has read the chunk before it is overwritten
      store();
    }
    __syncthreads();
  }
  float* pb = part + (int64_t)blockIdx.x * kWidth * K;
#pragma unroll
  for (int i = 0; i < TNW; ++i)
#pragma unroll
    for (int j = 0; j < TKW; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int n = dfeat(tn0 + i, e, h);
        pb[n * K + 32 * (tk0 + j) + rl] = acc[i][j][e];
      }
  // bias: the row groups' sums of each column, through LDS (the staging buffers are free
  // after the loop's last barrier)
  float* bl = reinterpret_cast<float*>(&sX[0][0][0]);
#pragma unroll
  for (int q = 0; q < NU; ++q) {
    const int u = tid + q * NT;
    if (u < UY) bl[u] = bsum[q];
  }
  __syncthreads();
  for (int n = tid; n < kWidth; n += NT) {
    float t = 0.f;
#pragma unroll
    for (int g = 0; g < kWsGroups; ++g) t += bl[g * kWidth + n];
    partb[(int64_t)blockIdx.x * kWidth + n] = t;
  }
  if (stamps) {
    __syncthreads();
    if (threadIdx.x == 0) atomicMax(&stamps[1], (unsigned long long)wall_clock64());
  }
}

// Deterministic two-pass sum of nblk partial slices of n floats each:
//   pass 1: red[g][i] = sum of part[b][i] over b in group g (kReduceGroups groups),
//   pass 2: out[r * k_real + c] = sum over g of red[g][r * k_pad + c], c < k_real.
constexpr int kReduceGroups = 16;

// Two independent reductions (a weight slice and its bias slice) in the same two
// launches: blockIdx.z selects the job.
struct RedJob {
  const float* part;
  float* red;
  float* out;
  int n, rows, k_pad, k_real;
};

__global__ void k_reduce2_pass1(RedJob ja, RedJob jb, int nblk) {
  const RedJob& j = blockIdx.z ? jb : ja;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int g = blockIdx.y;
  if (i >= j.n) return;
  const int b0 = (int)((int64_t)nblk * g / kReduceGroups);
  const int b1 = (int)((int64_t)nblk * (g + 1) / kReduceGroups);
  float s0 = 0.f, s1 = 0.f, s2 = 0.f, s3 = 0.f;
  int b = b0;
  for (; b + 4 <= b1; b += 4) {
    s0 += j.part[(int64_t)b * j.n + i];
    s1 += j.part[(int64_t)(b + 1) * j.n + i];
    s2 += j.part[(int64_t)(b + 2) * j.n + i];
    s3 += j.part[(int64_t)(b + 3) * j.n + i];
  }
  for (; b < b1; ++b) s0 += j.part[(int64_t)b * j.n + i];
  j.red[(int64_t)g * j.n + i] = (s0 + s1) + (s2 + s3);
}

__global__ void k_reduce2_pass2(RedJob ja, RedJob jb) {
  const RedJob& j = blockIdx.z ? jb : ja;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= j.rows * j.k_real) return;
  const int r = i / j.k_real, c = i % j.k_real;
  float s = 0.f;
#pragma unroll
  for (int g = 0; g < kReduceGroups; ++g) s += j.red[(int64_t)g * j.n + r * j.k_pad + c];
  j.out[i] = s;
}

// out_a [rows_a, k_real_a] and out_b from nblk slices each; each job's `red` holds
// kReduceGroups slices.
static void reduce_two(const RedJob& a, const RedJob& b, int nblk, hipStream_t st) {
  const int n = a.n > b.n ? a.n : b.n;
  const int o = a.rows * a.k_real > b.rows * b.k_real ? a.rows * a.k_real : b.rows * b.k_real;
  k_reduce2_pass1<<<dim3((unsigned)cdiv(n, 256), kReduceGroups, 2), 256, 0, st>>>(a, b, nblk);
  k_reduce2_pass2<<<dim3((unsigned)cdiv(o, 256), 1, 2), 256, 0, st>>>(a, b);
}

__global__ void k_f32_to_bf16(const float* __restrict__ x, int64_t n, __bf16* __restrict__ y) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    y[i] = (__bf16)x[i];
}

static int num_cus() {
  static int cus = 0;
  if (!cus) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) dev = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
      cus = 256;
  }
  return cus;
}

template <int KT, int NTO, int MODE, bool BF>
static void launch_layer(const void* in, int in_stride, int64_t M, const int64_t* Md,
                         const void* wpk, const float* bias, const void* mask, int mask_stride,
                         void* out, int out_stride, hipStream_t st) {
  // about two 32 x 32 output blocks per wave at least (the stream-K split evens out the
  // rest), at most one block per CU (the weights fill its LDS)
  const int64_t tiles = (M + 31) / 32;
  int64_t blocks = (tiles * NTO + 15) / 16;
  const int64_t cap = num_cus();
  if (blocks > cap) blocks = cap;
  if (blocks < 1) blocks = 1;
  k_mlp_layer<KT, NTO, MODE, BF><<<(unsigned)blocks, kLayerThreads, 0, st>>>(
      in, in_stride, M, Md, wpk, bias, mask, mask_stride, out, out_stride);
}

template <int KT, int NTL, int NCG, int MODE, int KQ = 2 * KT>
static void launch_layer_split(const void* in, int in_stride, int64_t M, const int64_t* Md,
                               const void* wpk, const float* bias, const void* mask,
                               int mask_stride, void* out, int out_stride, uint32_t* bits,
                               hipStream_t st) {
  // per column group: about two 32 x 32 output blocks per wave at least, at most one
  // block per CU over all groups (the weights fill the LDS); with two groups the group
  // size is a multiple of 8 (the block -> group map pairs blocks 8 apart)
  const int64_t tiles = (M + 31) / 32;
  int64_t b = (tiles * NTL + 15) / 16;
  const int64_t cap = (int64_t)num_cus() / NCG;
  if (b > cap) b = cap;
  if (b < 1) b = 1;
  if (NCG > 1) b = (b + 7) / 8 * 8;
  k_mlp_layer_split<KT, NTL, NCG, MODE, KQ><<<(unsigned)(b * NCG), kLayerThreads, 0, st>>>(
      reinterpret_cast<const float*>(in), in_stride, M, Md, reinterpret_cast<const bf16x8*>(wpk),
      bias, reinterpret_cast<const float*>(mask), mask_stride, reinterpret_cast<float*>(out),
      out_stride, bits);
}

// A workgroup per CU at most (the slabs and registers fill it).
static unsigned net_blocks(int64_t M) {
  const int64_t rounds = cdiv(M, 32 * kNetWaves), cus = num_cus();
  return (unsigned)(rounds < cus ? rounds : cus);
}

// Row blocks of the weight-gradient kernel: at least one chunk of rows per block, at
// most one block per CU (each holds two row chunks, up to 96 KB of LDS), or max_blocks
// when that is smaller and positive.
static int wgrad_blocks(int64_t M, int kt, int max_blocks = 0) {
  (void)kt;
  int64_t b = cdiv(M, kWgradChunk);
  const int64_t cap = max_blocks > 0 && max_blocks < num_cus() ? max_blocks : num_cus();
  if (b > cap) b = cap;
  return (int)(b < 1 ? 1 : b);
}

static int last_blocks(int64_t M) {
  int64_t b = cdiv(M, 64);
  const int64_t cap = 4 * (int64_t)num_cus();
  if (b > cap) b = cap;
  return (int)(b < 1 ? 1 : b);
}

}  // namespace vx

using namespace vx;

extern "C" {

int vx_mlp_pack(int prec, const float* W, int n_out, int k_in, int kt, int nto, int transpose,
                void* out, void* stream) {
  VX_CHECK_ARG(prec >= 0 && prec <= 2, "mlp_pack: prec must be 0, 1 or 2");
  VX_CHECK_ARG(kt >= 1 && nto >= 1 && n_out >= 1 && k_in >= 1, "mlp_pack: bad sizes");
  hipStream_t st = (hipStream_t)stream;
  if (prec == 2) {
    PackNet net{};
    net.seg[0] = PackSeg{W, 0, n_out, k_in, kt, nto, transpose};
    k_pack_net<2><<<dim3(grid_for((int64_t)nto * kt * 16 * 64, 256), 1), 256, 0, st>>>(net, out);
  } else if (prec == 1)
    k_pack_bf16<<<grid_for((int64_t)nto * kt * 2 * 64 * 8, 256), 256, 0, st>>>(
        W, n_out, k_in, kt, nto, transpose, (__bf16*)out);
  else
    k_pack_f32<<<grid_for((int64_t)nto * kt * 16 * 64, 256), 256, 0, st>>>(W, n_out, k_in, kt,
                                                                             nto, transpose,
                                                                             (float*)out);
  return launch_status("mlp_pack");
}

int64_t vx_mlp_pack_elems(int kt, int nto) { return (int64_t)nto * kt * 16 * 64; }

static int pack_net_segments(int n_hidden, int k_in0, const int64_t* w_ptrs, PackNet* net,
                             int64_t* total) {
  const int kt0 = k_in0 <= 64 ? 2 : 3;
  int64_t off = 0;
  for (int li = 0; li < n_hidden; ++li) {
    const int kt = li == 0 ? kt0 : 6;
    const int k_in = li == 0 ? k_in0 : kWidth;
    for (int dir = 0; dir < 2; ++dir) {
      PackSeg sg;
      sg.W = w_ptrs ? reinterpret_cast<const float*>(w_ptrs[li]) : nullptr;
      sg.offset = off;
      sg.n_out = kWidth;
      sg.k_in = k_in;
      sg.kt = dir == 0 ? kt : 6;
      sg.nto = dir == 0 ? 6 : kt;
      sg.transpose = dir;
      if (net) net->seg[2 * li + dir] = sg;
      off += vx_mlp_pack_elems(sg.kt, sg.nto);
    }
  }
  *total = off;
  return VX_OK;
}

int64_t vx_mlp_pack_net_elems(int n_hidden, int k_in0) {
  if (n_hidden < 1 || 2 * n_hidden > kMaxPackSegs || k_in0 < 1 || k_in0 > 96) return -1;
  int64_t total = 0;
  pack_net_segments(n_hidden, k_in0, nullptr, nullptr, &total);
  return total;
}

int vx_mlp_pack_net(int prec, int n_hidden, const int64_t* w_ptrs, int k_in0, void* out,
                    void* stream) {
  VX_CHECK_ARG(prec >= 0 && prec <= 2, "mlp_pack_net: prec must be 0, 1 or 2");
  VX_CHECK_ARG(n_hidden >= 1 && 2 * n_hidden <= kMaxPackSegs, "mlp_pack_net: 1..%d hidden layers",
               kMaxPackSegs / 2);
  VX_CHECK_ARG(k_in0 >= 1 && k_in0 <= 96, "mlp_pack_net: input width must be 1..96");
  PackNet net;
  int64_t total = 0;
  pack_net_segments(n_hidden, k_in0, w_ptrs, &net, &total);
  int64_t biggest = 0;
  for (int i = 0; i < 2 * n_hidden; ++i) {
    const int64_t e = vx_mlp_pack_elems(net.seg[i].kt, net.seg[i].nto);
    if (e > biggest) biggest = e;
  }
  dim3 grid(grid_for(biggest, 256), 2 * n_hidden);
  hipStream_t st = (hipStream_t)stream;
  if (prec == 2) k_pack_net<2><<<grid, 256, 0, st>>>(net, out);
  else if (prec == 1) k_pack_net<1><<<grid, 256, 0, st>>>(net, out);
  else k_pack_net<0><<<grid, 256, 0, st>>>(net, out);
  return launch_status("mlp_pack_net");
}

int vx_mlp_layer_fwd(int prec, int kt, int k_in, int last, const void* in, int in_stride,
                     int64_t M, const void* wpk, const float* bias, void* out, int out_stride,
                     const float* w3, const float* b3, float* logits, const int64_t* M_dev,
                     uint32_t* mask_bits, void* stream) {
  VX_CHECK_ARG(prec >= 0 && prec <= 2, "mlp_layer_fwd: prec must be 0, 1 or 2");
  VX_CHECK_ARG(!mask_bits || prec == 2, "mlp_layer_fwd: mask bits need prec 2");
  const int bf16 = prec == 1;
  VX_CHECK_ARG(M >= 0, "mlp_layer_fwd: M < 0");
  VX_CHECK_ARG(kt == 2 || kt == 3 || kt == 6, "mlp_layer_fwd: input width must be 64, 96 or 192");
  VX_CHECK_ARG(k_in >= 0 && k_in <= 32 * kt, "mlp_layer_fwd: k_in outside [0, 32 kt]");
  // the weights' last 16 columns zero: those reduction steps are left out (prec 2)
  const bool tail = k_in > 0 && k_in <= 32 * kt - 16;
  if (M == 0) return VX_OK;
  VX_CHECK_ARG(!last || (w3 && b3 && logits), "mlp_layer_fwd: last layer needs w3, b3, logits");
  hipStream_t st = (hipStream_t)stream;
#define L(KT, BF) launch_layer<KT, 6, 0, BF>(in, in_stride, M, M_dev, wpk, bias, nullptr, 0, out, out_stride, st)
#define LS(KT, NTL, NCG) launch_layer_split<KT, NTL, NCG, 0>(in, in_stride, M, M_dev, wpk, bias, nullptr, 0, out, out_stride, mask_bits, st)
  if (prec == 2) {
    if (kt == 2 && tail) launch_layer_split<2, 3, 2, 0, 3>(in, in_stride, M, M_dev, wpk, bias, nullptr, 0, out, out_stride, mask_bits, st);
    else if (kt == 2) LS(2, 3, 2);
    else if (kt == 3 && tail) launch_layer_split<3, 3, 2, 0, 5>(in, in_stride, M, M_dev, wpk, bias, nullptr, 0, out, out_stride, mask_bits, st);
    else if (kt == 3) LS(3, 3, 2);
    else LS(6, 3, 2);
  } else if (!bf16) {
    if (kt == 2) L(2, false);
    else if (kt == 3) L(3, false);
    else L(6, false);
  } else {
    if (kt == 2) L(2, true);
    else if (kt == 3) L(3, true);
    else L(6, true);
  }
#undef L
#undef LS
  if (last) {
    const unsigned g = grid_for(M, 32, 8 * (int64_t)num_cus());
    if (bf16) k_mlp_logits<true><<<g, 256, 0, st>>>(out, out_stride, M, M_dev, w3, b3, logits);
    else k_mlp_logits<false><<<g, 256, 0, st>>>(out, out_stride, M, M_dev, w3, b3, logits);
  }
  return launch_status("mlp_layer_fwd");
}

int vx_mlp_net_fwd(int n_hidden, int k_in0, const float* X, int xs, int64_t M, const void* packed,
                   const int64_t* biases, const float* w3, const float* b3, float* logits,
                   const int64_t* M_dev, void* stream) {
  VX_CHECK_ARG(n_hidden >= 1 && n_hidden <= kNetMaxHidden, "mlp_net_fwd: 1..%d hidden layers",
               kNetMaxHidden);
  VX_CHECK_ARG(k_in0 >= 1 && k_in0 <= 96, "mlp_net_fwd: input width must be 1..96");
  const int kt0 = k_in0 <= 64 ? 2 : 3;
  VX_CHECK_ARG(M >= 0, "mlp_net_fwd: M < 0");
  VX_CHECK_ARG(xs >= 32 * kt0 && xs % 4 == 0, "mlp_net_fwd: rows must be padded to 64 or 96");
  if (M == 0) return VX_OK;
  VX_CHECK_ARG(X && packed && biases && w3 && b3 && logits, "mlp_net_fwd: null pointer");
  PackNet net;
  int64_t total = 0;
  pack_net_segments(n_hidden, k_in0, nullptr, &net, &total);
  NetArgs a{};
  a.in = X;
  a.in_stride = xs;
  a.n_hidden = n_hidden;
  a.M = M;
  a.Md = M_dev;
  a.w3 = w3;
  a.b3 = b3;
  a.logits = logits;
  for (int li = 0; li < n_hidden; ++li) {
    a.w[li] = (const bf16x8*)((const __bf16*)packed + 3 * net.seg[2 * li].offset);
    a.b[li] = (const float*)biases[li];
  }
  const bool tail = k_in0 <= 32 * kt0 - 16;  // the last 16-deep step's weights are zero
  const unsigned blocks = net_blocks(M);
  hipStream_t st = (hipStream_t)stream;
#define NF(KT, KQ) k_mlp_net_fwd<KT, KQ><<<blocks, 64 * kNetWaves, 0, st>>>(a)
  if (kt0 == 2) { if (tail) NF(2, 3); else NF(2, 4); }
  else { if (tail) NF(3, 5); else NF(3, 6); }
#undef NF
  return launch_status("mlp_net_fwd");
}

int vx_mlp_logits(int prec, const void* H, int hs, int64_t M, const float* w3, const float* b3,
                  float* logits, const int64_t* M_dev, void* stream) {
  VX_CHECK_ARG(prec >= 0 && prec <= 2, "mlp_logits: prec must be 0, 1 or 2");
  VX_CHECK_ARG(M >= 0, "mlp_logits: M < 0");
  if (M == 0) return VX_OK;
  VX_CHECK_ARG(H && w3 && b3 && logits && hs >= kWidth, "mlp_logits: bad arguments");
  hipStream_t st = (hipStream_t)stream;
  const unsigned g = grid_for(M, 32, 8 * (int64_t)num_cus());
  if (prec == 1) k_mlp_logits<true><<<g, 256, 0, st>>>(H, hs, M, M_dev, w3, b3, logits);
  else k_mlp_logits<false><<<g, 256, 0, st>>>(H, hs, M, M_dev, w3, b3, logits);
  return launch_status("mlp_logits");
}

int vx_mlp_layer_bwd(int prec, int nto, const float* dy, int dy_stride, int64_t M,
                     const void* wpk_t, const void* mask, int mask_stride, float* dx,
                     int dx_stride, const int64_t* M_dev, const uint32_t* mask_bits,
                     void* stream) {
  VX_CHECK_ARG(prec >= 0 && prec <= 2, "mlp_layer_bwd: prec must be 0, 1 or 2");
  VX_CHECK_ARG(!mask_bits || (prec == 2 && mask && nto == 6),
               "mlp_layer_bwd: mask bits need prec 2 and a masked 192-wide layer");
  const int bf16 = prec == 1;
  VX_CHECK_ARG(M >= 0, "mlp_layer_bwd: M < 0");
  VX_CHECK_ARG(nto == 2 || nto == 3 || nto == 6 || (nto == 1 && prec == 2 && !mask),
               "mlp_layer_bwd: output width must be 64, 96 or 192 (32 only for prec 2 "
               "without a mask)");
  if (M == 0) return VX_OK;
  hipStream_t st = (hipStream_t)stream;
#define L(NTO, MODE, BF) launch_layer<6, NTO, MODE, BF>(dy, dy_stride, M, M_dev, wpk_t, nullptr, mask, mask_stride, dx, dx_stride, st)
#define LS(NTL, NCG, MODE) launch_layer_split<6, NTL, NCG, MODE>(dy, dy_stride, M, M_dev, wpk_t, nullptr, mask, mask_stride, dx, dx_stride, const_cast<uint32_t*>(mask_bits), st)
  if (prec == 2) {
    if (nto == 6) { if (mask) LS(3, 2, 2); else LS(3, 2, 3); }
    else if (nto == 3) LS(3, 1, 3);
    else if (nto == 2) LS(1, 2, 3);
    else LS(1, 1, 3);  // the first 32 columns of an operand packed for 64
  } else if (!bf16) {
    if (nto == 6) { if (mask) L(6, 2, false); else L(6, 3, false); }
    else if (nto == 3) L(3, 3, false);
    else L(2, 3, false);
  } else {
    if (nto == 6) { if (mask) L(6, 2, true); else L(6, 3, true); }
    else if (nto == 3) L(3, 3, true);
    else L(2, 3, true);
  }
#undef L
#undef LS
  return launch_status("mlp_layer_bwd");
}

int64_t vx_mlp_wgrad_part_elems(int64_t M) {
  int64_t need = 0;
  for (int kt : {2, 3, 6}) {
    const int64_t e = ((int64_t)wgrad_blocks(M, kt) + kReduceGroups) * kWidth * 32 * kt;
    if (e > need) need = e;
  }
  const int64_t e3 = ((int64_t)last_blocks(M) + kReduceGroups) * 3 * kWidth;
  return need > e3 ? need : e3;
}

int64_t vx_mlp_wgrad_partb_elems(int64_t M) {
  int64_t nb = last_blocks(M);
  for (int kt : {2, 3, 6})
    if (wgrad_blocks(M, kt) > nb) nb = wgrad_blocks(M, kt);
  return (nb + kReduceGroups) * kWidth;
}

int64_t vx_wall_clock_khz(void) {
  int dev = 0, khz = 0;
  if (hipGetDevice(&dev) != hipSuccess) return -1;
  if (hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev) != hipSuccess) return -1;
  return khz;
}

int vx_mlp_wgrad_partials(int prec, int kt, const float* dY, int dys, const void* X, int xs,
                          int64_t M, float* part, float* partb, const int64_t* M_dev,
                          int max_blocks, uint64_t* stamps, void* stream) {
  VX_CHECK_ARG(!stamps || prec == 2, "mlp_wgrad_partials: stamps need prec 2");
  VX_CHECK_ARG(prec >= 0 && prec <= 2, "mlp_wgrad: prec must be 0, 1 or 2");
  const int bf16 = prec == 1;
  VX_CHECK_ARG(kt == 2 || kt == 3 || kt == 6, "mlp_wgrad: input width must be 64, 96 or 192");
  VX_CHECK_ARG(M >= 0, "mlp_wgrad: M < 0");
  VX_CHECK_ARG(max_blocks >= 0, "mlp_wgrad: max_blocks < 0");
  hipStream_t st = (hipStream_t)stream;
  const int nblk = wgrad_blocks(M, kt, max_blocks);
#define L(KT, BF) k_mlp_wgrad<KT, BF><<<nblk, 64 * WgradShape<KT>::WAVES, 0, st>>>(dY, dys, X, xs, M, M_dev, part, partb)
#define LS(KT) k_mlp_wgrad_split<KT><<<nblk, 64 * WgradShape<KT>::WAVES, 0, st>>>(dY, dys, static_cast<const float*>(X), xs, M, M_dev, part, partb, reinterpret_cast<unsigned long long*>(stamps))
  if (prec == 2) {
    if (kt == 2) LS(2);
    else if (kt == 3) LS(3);
    else LS(6);
  } else if (kt == 2) { if (bf16) L(2, true); else L(2, false); }
  else if (kt == 3) { if (bf16) L(3, true); else L(3, false); }
  else { if (bf16) L(6, true); else L(6, false); }
#undef LS
#undef L
  return launch_status("mlp_wgrad_partials");
}

int vx_mlp_wgrad_reduce(int kt, int k_real, int64_t M, float* part, float* partb,
                        float* dW, float* db, int max_blocks, void* stream) {
  VX_CHECK_ARG(kt == 2 || kt == 3 || kt == 6, "mlp_wgrad: input width must be 64, 96 or 192");
  VX_CHECK_ARG(k_real >= 1 && k_real <= 32 * kt, "mlp_wgrad: k_real out of range");
  VX_CHECK_ARG(M >= 0 && max_blocks >= 0, "mlp_wgrad: M < 0 or max_blocks < 0");
  const int nblk = wgrad_blocks(M, kt, max_blocks);
  const int K = 32 * kt;
  // the reduction's group sums go to the workspaces past the nblk partial slices
  const RedJob jw{part, part + (int64_t)nblk * kWidth * K, dW, kWidth * K, kWidth, K, k_real};
  const RedJob jb{partb, partb + (int64_t)nblk * kWidth, db, kWidth, 1, kWidth, kWidth};
  reduce_two(jw, jb, nblk, (hipStream_t)stream);
  return launch_status("mlp_wgrad_reduce");
}

int vx_mlp_wgrad(int prec, int kt, int k_real, const float* dY, int dys, const void* X, int xs,
                 int64_t M, float* part, float* partb, float* dW, float* db, const int64_t* M_dev,
                 int max_blocks, void* stream) {
  VX_CHECK_ARG(k_real >= 1 && k_real <= 32 * kt, "mlp_wgrad: k_real out of range");
  if (int rc = vx_mlp_wgrad_partials(prec, kt, dY, dys, X, xs, M, part, partb, M_dev,
                                     max_blocks, nullptr, stream))
    return rc;
  return vx_mlp_wgrad_reduce(kt, k_real, M, part, partb, dW, db, max_blocks, stream);
}

int vx_mlp_last_bwd(int prec, const float* dlogit, const void* H, int hs, int64_t M,
                    const float* w3, float* dH, int dhs, float* part, float* partb, float* dW3,
                    float* db3, const int64_t* M_dev, void* stream) {
  VX_CHECK_ARG(prec >= 0 && prec <= 2, "mlp_last_bwd: prec must be 0, 1 or 2");
  const int bf16 = prec == 1;
  VX_CHECK_ARG(M >= 0, "mlp_last_bwd: M < 0");
  hipStream_t st = (hipStream_t)stream;
  const int nblk = last_blocks(M);
  if (bf16) k_mlp_last_bwd<true, true><<<nblk, kWidth, 0, st>>>(dlogit, H, hs, M, M_dev, w3, dH, dhs, part, partb);
  else k_mlp_last_bwd<false, true><<<nblk, kWidth, 0, st>>>(dlogit, H, hs, M, M_dev, w3, dH, dhs, part, partb);
  const RedJob jw{part, part + (int64_t)nblk * 3 * kWidth, dW3, 3 * kWidth, 3, kWidth, kWidth};
  const RedJob jb{partb, partb + (int64_t)nblk * 3, db3, 3, 1, 3, 3};
  reduce_two(jw, jb, nblk, st);
  return launch_status("mlp_last_bwd");
}

int vx_mlp_last_dgrad(const float* dlogit, const uint32_t* mask_bits, int64_t M, const float* w3,
                      float* dH, int dhs, const int64_t* M_dev, void* stream) {
  VX_CHECK_ARG(M >= 0, "mlp_last_dgrad: M < 0");
  VX_CHECK_ARG(dhs >= kWidth && dhs % 4 == 0, "mlp_last_dgrad: dH stride must be >= 192, a multiple of 4");
  if (M == 0) return VX_OK;
  VX_CHECK_ARG(dlogit && mask_bits && w3 && dH, "mlp_last_dgrad: null pointer");
  const int64_t cap = 16 * (int64_t)num_cus();
  const int64_t b = cdiv(M, 4);
  k_mlp_last_dgrad<<<(unsigned)(b < cap ? b : cap), kWidth, 0, (hipStream_t)stream>>>(
      dlogit, mask_bits, M, M_dev, w3, dH, dhs);
  return launch_status("mlp_last_dgrad");
}

int vx_mlp_last_wgrad(int prec, const float* dlogit, const void* H, int hs, int64_t M,
                      float* part, float* partb, float* dW3, float* db3, const int64_t* M_dev,
                      void* stream) {
  VX_CHECK_ARG(prec >= 0 && prec <= 2, "mlp_last_wgrad: prec must be 0, 1 or 2");
  VX_CHECK_ARG(M >= 0, "mlp_last_wgrad: M < 0");
  hipStream_t st = (hipStream_t)stream;
  const int nblk = last_blocks(M);
  if (prec == 1) k_mlp_last_bwd<true, false><<<nblk, kWidth, 0, st>>>(dlogit, H, hs, M, M_dev, nullptr, nullptr, 0, part, partb);
  else k_mlp_last_bwd<false, false><<<nblk, kWidth, 0, st>>>(dlogit, H, hs, M, M_dev, nullptr, nullptr, 0, part, partb);
  const RedJob jw{part, part + (int64_t)nblk * 3 * kWidth, dW3, 3 * kWidth, 3, kWidth, kWidth};
  const RedJob jb{partb, partb + (int64_t)nblk * 3, db3, 3, 1, 3, 3};
  reduce_two(jw, jb, nblk, st);
  return launch_status("mlp_last_wgrad");
}

int vx_f32_to_bf16(const float* x, int64_t n, void* y, void* stream) {
  if (n == 0) return VX_OK;
  k_f32_to_bf16<<<grid_for(n, 256), 256, 0, (hipStream_t)stream>>>(x, n, (__bf16*)y);
  return launch_status("f32_to_bf16");
}

}  // extern "C"
