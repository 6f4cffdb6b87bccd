// Boolean row selection of several arrays at once (gfx950): the compactions between the stages
// of the op-by-op forward, x[mask] for four or five arrays under one mask.  Taken apart into
// index operations each array finds the selected rows by itself (a scan, a partition, a host
// synchronisation) and its backward sorts the indices before it adds: 350 of the 1,300 us of
// kernels in a coarse step over 1.6 M samples, most of it in launches of a few microseconds.
// Here the rows are counted once, every array is copied in one launch, and the adjoint is a
// dense pass (the selected rows are distinct: nothing to add up): 26 us a selection of three
// arrays, 11 its adjoint, and the step 1,470 -> 1,031 us.  Bound by the bytes moved.
#include "common.h"

namespace vx {

constexpr int kSelBlock = 4096;  // mask elements per workgroup, sixteen a thread
constexpr int kSelMax = 8;       // arrays per launch

struct SelArrays {
  const uint32_t* src[kSelMax];
  uint32_t* dst[kSelMax];
  int words[kSelMax];  // 32-bit words a row
  int n;
};

// Selection bits of the thread's sixteen elements.
__device__ __forceinline__ uint32_t sel_bits(const uint8_t* __restrict__ mask, int64_t n) {
  const int64_t i0 = blockIdx.x * (int64_t)kSelBlock + 16 * threadIdx.x;
  uint32_t bits = 0;
  if (i0 + 16 <= n && (reinterpret_cast<uintptr_t>(mask) & 15) == 0) {
    const uint4 v = *reinterpret_cast<const uint4*>(mask + i0);
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int k = 0; k < 16; ++k) bits |= ((w[k >> 2] >> (8 * (k & 3)) & 255u) ? 1u : 0u) << k;
  } else {
    for (int k = 0; k < 16; ++k)
      if (i0 + k < n && mask[i0 + k]) bits |= 1u << k;
  }
  return bits;
}

// Exclusive prefix of v over the workgroup's 256 threads; total: the sum.
__device__ __forceinline__ int block_prefix(int v, int& total) {
  __shared__ int part[4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int s = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int o = __shfl_up(s, off, 64);
    if (lane >= off) s += o;
  }
  if (lane == 63) part[wave] = s;
  __syncthreads();
  int before = 0;
  total = 0;
  for (int w = 0; w < 4; ++w) {
    if (w < wave) before += part[w];
    total += part[w];
  }
  return before + s - v;
}

__global__ void __launch_bounds__(256) k_sel_count(const uint8_t* __restrict__ mask, int64_t n,
                                                   int* __restrict__ counts) {
  int total;
  block_prefix(__popc(sel_bits(mask, n)), total);
  if (threadIdx.x == 0) counts[blockIdx.x] = total;
}

// counts -> exclusive offsets, in place; the sum.
__global__ void __launch_bounds__(256) k_sel_scan(int* __restrict__ counts, int64_t nb,
                                                  int64_t* __restrict__ sum) {
  int carry = 0;
  for (int64_t b0 = 0; b0 < nb; b0 += 256) {
    const int64_t b = b0 + threadIdx.x;
    const int c = b < nb ? counts[b] : 0;
    int total;
    const int p = block_prefix(c, total);
    if (b < nb) counts[b] = carry + p;
    carry += total;
    __syncthreads();
  }
  if (threadIdx.x == 0) *sum = carry;
}

// dst rows = the selected src rows, in order: the block's selected elements listed in LDS, then
// every array's words of them in one run.
template <int W>
__device__ __forceinline__ void sel_copy(const uint32_t* __restrict__ src, uint32_t* __restrict__ dst,
                                         const uint16_t* list, int total, int words) {
  if (W) words = W;
  for (int i = threadIdx.x; i < total * words; i += 256) {
    const int r = (int)((unsigned)i / (unsigned)words);
    dst[i] = src[(int64_t)list[r] * words + (i - r * words)];
  }
}

__global__ void __launch_bounds__(256) k_sel_rows(const uint8_t* __restrict__ mask, int64_t n,
                                                  const int* __restrict__ offsets, SelArrays a) {
  __shared__ uint16_t list[kSelBlock];
  uint32_t bits = sel_bits(mask, n);
  int total;
  int p = block_prefix(__popc(bits), total);
  while (bits) {
    list[p++] = (uint16_t)(16 * threadIdx.x + __ffs(bits) - 1);
    bits &= bits - 1;
  }
  __syncthreads();
  const int64_t base = blockIdx.x * (int64_t)kSelBlock, out = offsets[blockIdx.x];
  for (int k = 0; k < a.n; ++k) {
    const int w = a.words[k];
    const uint32_t* src = a.src[k] + base * w;
    uint32_t* dst = a.dst[k] + out * w;
    if (w == 1) sel_copy<1>(src, dst, list, total, w);
    else if (w == 2) sel_copy<2>(src, dst, list, total, w);
    else if (w == 3) sel_copy<3>(src, dst, list, total, w);
    else sel_copy<0>(src, dst, list, total, w);
  }
}

// The adjoint: dst rows = the src row of each selected element in order, zero elsewhere.
template <int W>
__device__ __forceinline__ void sel_spread(const uint32_t* __restrict__ src, uint32_t* __restrict__ dst,
                                           const uint16_t* rank, int m, int words) {
  if (W) words = W;
  for (int i = threadIdx.x; i < m * words; i += 256) {
    const int e = (int)((unsigned)i / (unsigned)words);
    const int r = rank[e];
    dst[i] = r != 0xffff ? src[(int64_t)r * words + (i - e * words)] : 0u;
  }
}

__global__ void __launch_bounds__(256) k_sel_rows_bwd(const uint8_t* __restrict__ mask, int64_t n,
                                                      const int* __restrict__ offsets, SelArrays a) {
  __shared__ uint16_t rank[kSelBlock];
  const uint32_t bits = sel_bits(mask, n);
  int total;
  int p = block_prefix(__popc(bits), total);
  for (int k = 0; k < 16; ++k) rank[16 * threadIdx.x + k] = (bits >> k & 1u) ? (uint16_t)p++ : 0xffff;
  __syncthreads();
  const int64_t base = blockIdx.x * (int64_t)kSelBlock, in = offsets[blockIdx.x];
  const int m = (int)(n - base < kSelBlock ? n - base : kSelBlock);
  for (int k = 0; k < a.n; ++k) {
    const int w = a.words[k];
    const uint32_t* src = a.src[k] + in * w;
    uint32_t* dst = a.dst[k] + base * w;
    if (w == 1) sel_spread<1>(src, dst, rank, m, w);
    else if (w == 2) sel_spread<2>(src, dst, rank, m, w);
    else if (w == 3) sel_spread<3>(src, dst, rank, m, w);
    else sel_spread<0>(src, dst, rank, m, w);
  }
}

static int sel_arrays(SelArrays& a, int count, const int64_t* src, const int64_t* dst, const int* words) {
  VX_CHECK_ARG(count >= 1 && count <= kSelMax, "select_rows: 1 to %d arrays", kSelMax);
  VX_CHECK_ARG(src && dst && words, "select_rows: missing argument");
  a.n = count;
  for (int k = 0; k < count; ++k) {
    VX_CHECK_ARG(words[k] >= 1 && words[k] <= 4096, "select_rows: rows of 1 to 4096 words");
    a.src[k] = (const uint32_t*)src[k];
    a.dst[k] = (uint32_t*)dst[k];
    a.words[k] = words[k];
  }
  return VX_OK;
}

}  // namespace vx

using namespace vx;

extern "C" {

int64_t vx_select_blocks(int64_t n) { return cdiv(n, kSelBlock); }

int vx_select_count(const uint8_t* mask, int64_t n, int* offsets, int64_t* total, void* stream) {
  VX_CHECK_ARG(n >= 1 && n < ((int64_t)1 << 31), "select_count: 1 to 2^31 - 1 elements");
  VX_CHECK_ARG(mask && offsets && total, "select_count: missing argument");
  const int64_t nb = cdiv(n, kSelBlock);
  hipStream_t st = (hipStream_t)stream;
  k_sel_count<<<(unsigned)nb, 256, 0, st>>>(mask, n, offsets);
  k_sel_scan<<<1, 256, 0, st>>>(offsets, nb, total);
  return launch_status("select_count");
}

int vx_select_rows(const uint8_t* mask, int64_t n, const int* offsets, int count,
                   const int64_t* src, const int64_t* dst, const int* words, int transpose,
                   void* stream) {
  VX_CHECK_ARG(n >= 1 && n < ((int64_t)1 << 31), "select_rows: 1 to 2^31 - 1 elements");
  VX_CHECK_ARG(mask && offsets, "select_rows: missing argument");
  SelArrays a;
  if (int e = sel_arrays(a, count, src, dst, words)) return e;
  const unsigned nb = (unsigned)cdiv(n, kSelBlock);
  hipStream_t st = (hipStream_t)stream;
  if (transpose) k_sel_rows_bwd<<<nb, 256, 0, st>>>(mask, n, offsets, a);
  else k_sel_rows<<<nb, 256, 0, st>>>(mask, n, offsets, a);
  return launch_status("select_rows");
}

}  // extern "C"
