// Lattice SDF query and marching cubes (gfx950): the mesh extraction of
// Voxurf.extract_geometry (lib/voxurf_fine.py:894-910 -> lib/dvgo_ori.py:679-703), whose
// reference runs the SDF query chunk by chunk through grid_sample, copies the field to
// the host and calls PyMCubes on the CPU.
//
// Here the field stays on the device: vx_extract_fields evaluates the trilinear SDF at
// the lattice points (torch.linspace's arithmetic), and marching cubes counts (crossing
// edges owned by each point, triangles of the cube at each point), scans and writes
// (vertices on the owned edges, triangles by table): vx_mc_classify / vx_mc_write on
// bit rows of the lattice, vx_mc_count / vx_mc_emit with per-point counts and a scan of the
// caller's between them.  Every vertex sits on exactly one lattice edge and is
// shared by all triangles that use that edge, so the mesh is indexed without a hash.
//
// The triangle table is generated here (vx_mc_tables), not transcribed: for each of the
// 256 corner configurations the isosurface crosses each cube face in one segment, or in
// two on a face whose below-threshold corners are diagonal (these are separated, a rule
// that depends only on the face, so neighbouring cubes agree and the mesh is closed);
// segments are oriented so that triangles face the below-threshold side, linked into
// loops around the cube, and each loop is triangulated as a fan.
#include "voxel.h"

#include <string.h>

namespace vx {

// Corner c of a cube: offsets (c & 1, c >> 1 & 1, c >> 2 & 1) along (x, y, z).
// Edge e = 4 * axis + (b0 | b1 << 1): along `axis`, at offsets b0, b1 on the other two
// axes in increasing axis order; it starts at the corner with offset 0 along `axis`.
constexpr int kMcMaxTris = 8;

struct McTables {
  int8_t count[256];
  int8_t edges[256][3 * kMcMaxTris];
};

static void edge_corners(int e, int& c0, int& c1) {
  const int axis = e >> 2, b0 = e & 1, b1 = e >> 1 & 1;
  const int o0 = axis == 0 ? 1 : 0, o1 = axis == 2 ? 1 : 2;  // the other two axes
  c0 = (b0 << o0) | (b1 << o1);
  c1 = c0 | (1 << axis);
}

static int edge_between(int ca, int cb) {
  const int d = ca ^ cb;
  const int axis = d == 1 ? 0 : (d == 2 ? 1 : 2);
  const int base = ca & ~d;
  const int o0 = axis == 0 ? 1 : 0, o1 = axis == 2 ? 1 : 2;
  return 4 * axis + ((base >> o0 & 1) | (base >> o1 & 1) << 1);
}

static void edge_mid(int e, double p[3]) {
  int c0, c1;
  edge_corners(e, c0, c1);
  for (int a = 0; a < 3; ++a) p[a] = 0.5 * ((c0 >> a & 1) + (c1 >> a & 1));
}

// Bit (2 * axis + side) is set for each cube face the edge lies on.
static int edge_faces(int e) {
  const int axis = e >> 2, o0 = axis == 0 ? 1 : 0, o1 = axis == 2 ? 1 : 2;
  return 1 << (2 * o0 + (e & 1)) | 1 << (2 * o1 + (e >> 1 & 1));
}

static bool same_face(int a, int b, int c) { return (edge_faces(a) & edge_faces(b) & edge_faces(c)) != 0; }

static void build_tables(McTables& t) {
  memset(&t, 0, sizeof(t));
  for (int cfg = 0; cfg < 256; ++cfg) {
    int seg_from[12], seg_to_of[12];  // segment starting at edge e ends at seg_to_of[e]
    for (int e = 0; e < 12; ++e) seg_from[e] = seg_to_of[e] = -1;
    for (int axis = 0; axis < 3; ++axis) {
      const int u = axis == 0 ? 1 : 0, v = axis == 2 ? 1 : 2;
      for (int side = 0; side < 2; ++side) {
        // face corners in cyclic order (u, v) = (0,0), (1,0), (1,1), (0,1)
        int fc[4];
        const int uv[4][2] = {{0, 0}, {1, 0}, {1, 1}, {0, 1}};
        for (int q = 0; q < 4; ++q) fc[q] = (side << axis) | (uv[q][0] << u) | (uv[q][1] << v);
        bool below[4];
        for (int q = 0; q < 4; ++q) below[q] = cfg >> fc[q] & 1;
        int cross[4], nc = 0;
        for (int q = 0; q < 4; ++q)
          if (below[q] != below[(q + 1) & 3]) cross[nc++] = q;  // edge fc[q] - fc[q+1]
        if (nc == 0) continue;
        // segments as pairs of face-edge slots, with the below corner each cuts off
        int segs[2][2], cut[2], ns = 0;
        if (nc == 2) {
          segs[0][0] = cross[0];
          segs[0][1] = cross[1];
          int qb = -1;
          for (int q = 0; q < 4; ++q)
            if (below[q]) qb = q;
          cut[0] = qb;
          ns = 1;
        } else {
          // diagonal below corners: each is cut off by the segment of its two edges
          for (int q = 0; q < 4; ++q) {
            if (!below[q]) continue;
            segs[ns][0] = (q + 3) & 3;  // edge fc[q-1] - fc[q]
            segs[ns][1] = q;            // edge fc[q] - fc[q+1]
            cut[ns] = q;
            ++ns;
          }
        }
        double n[3] = {0, 0, 0};
        n[axis] = side ? 1.0 : -1.0;  // outward face normal
        for (int s = 0; s < ns; ++s) {
          int ea = edge_between(fc[segs[s][0]], fc[(segs[s][0] + 1) & 3]);
          int eb = edge_between(fc[segs[s][1]], fc[(segs[s][1] + 1) & 3]);
          double pa[3], pb[3], q[3];
          edge_mid(ea, pa);
          edge_mid(eb, pb);
          for (int a = 0; a < 3; ++a) q[a] = fc[cut[s]] >> a & 1;
          const double d[3] = {pb[0] - pa[0], pb[1] - pa[1], pb[2] - pa[2]};
          const double w[3] = {d[1] * n[2] - d[2] * n[1], d[2] * n[0] - d[0] * n[2],
                               d[0] * n[1] - d[1] * n[0]};
          const double side_q = w[0] * (q[0] - pa[0]) + w[1] * (q[1] - pa[1]) + w[2] * (q[2] - pa[2]);
          if (side_q > 0) {  // (b - a) x n must point away from the below corner
            const int tmp = ea;
            ea = eb;
            eb = tmp;
          }
          seg_from[ea] = ea;
          seg_to_of[ea] = eb;
        }
      }
    }
    // link segments into loops and fan-triangulate each
    bool used[12] = {false};
    int nt = 0;
    for (int e0 = 0; e0 < 12; ++e0) {
      if (seg_from[e0] < 0 || used[e0]) continue;
      int loop[12], nl = 0, e = e0;
      do {
        used[e] = true;
        loop[nl++] = e;
        e = seg_to_of[e];
      } while (e != e0 && e >= 0 && nl < 12);
      // fan from the first apex whose triangles all cut through the cube (no triangle
      // with its three vertices on one cube face, which a neighbouring cube could
      // duplicate in the shared face)
      int apex = 0;
      for (int a = 0; a < nl; ++a) {
        bool ok = true;
        for (int k = 1; k + 1 < nl && ok; ++k)
          ok = !same_face(loop[a], loop[(a + k) % nl], loop[(a + k + 1) % nl]);
        if (ok) {
          apex = a;
          break;
        }
      }
      for (int k = 1; k + 1 < nl; ++k) {
        t.edges[cfg][3 * nt + 0] = (int8_t)loop[apex];
        t.edges[cfg][3 * nt + 1] = (int8_t)loop[(apex + k) % nl];
        t.edges[cfg][3 * nt + 2] = (int8_t)loop[(apex + k + 1) % nl];
        ++nt;
      }
    }
    t.count[cfg] = (int8_t)nt;
  }
}

static const McTables& tables() {
  static const McTables t = [] {
    McTables x;
    build_tables(x);
    return x;
  }();
  return t;
}

// ---- lattice SDF query (lib/dvgo_ori.py:679-693 with Voxurf.grid_sampler) ------------

// torch.linspace(start, end, n)[i] in float: start + step * i for the first half,
// end - step * (n - 1 - i) for the rest, step = (end - start) / (n - 1), each value
// with one rounding (a fused multiply-add, as torch's vectorised kernel computes it).
__device__ __forceinline__ float linspace_at(float start, float end, int n, int i) {
#pragma clang fp contract(off)
  if (n == 1) return start;
  const float step = (end - start) / (float)(n - 1);
  return i < n / 2 ? fmaf(step, (float)i, start) : fmaf(-step, (float)(n - 1 - i), end);
}

struct FieldArgs {
  const float* sdf;
  GridDesc g;
  float mn[3], mx[3];   // grid box
  float bmin[3], bmax[3];
  int n[3];             // lattice points per axis
  float scale;          // -1: the field of -sdf (Voxurf.extract_geometry)
  float* u;             // [n0, n1, n2]
};

// One axis of the lattice: the cell and the weights of its points, as the drop-in
// grid_sample's Tri::init has them, with the in-grid bits of the cell's two lattice lines.
struct FieldAxis {
  int off0, off1;    // element offsets of the two (clamped) lattice lines
  float w0, w1;
  int x0;            // cell (unclamped)
  unsigned in;
};

__device__ __forceinline__ FieldAxis field_axis(const FieldArgs& a, int ax, int i, int size,
                                                int64_t stride) {
#pragma clang fp contract(off)
  const float p = linspace_at(a.bmin[ax], a.bmax[ax], a.n[ax], i);
  const float f = world_to_index(p, a.mn[ax], a.mx[ax] - a.mn[ax], size);
  const float ff = floorf(f);
  FieldAxis r;
  r.x0 = sat_f2i(ff);
  r.w0 = (ff + 1.f) - f;
  r.w1 = f - ff;
  r.off0 = (int)(clamp_index(r.x0, size) * stride);
  r.off1 = (int)(clamp_index(r.x0 + 1, size) * stride);
  r.in = ((unsigned)r.x0 < (unsigned)size ? 1u : 0u) |
         ((unsigned)(r.x0 + 1) < (unsigned)size ? 2u : 0u);
  return r;
}

// The lattice field, a thread's z of kFieldRows consecutive rows (3-D grid: z chunks of 256,
// row groups, x).  Bound by instruction issue: with one point per thread the three axes'
// divisions and 64-bit addresses of every point took 735 us for a 512^3 lattice of a 256^3
// grid (537 MB written).  Here the x axis is made once per thread, the z axis once per
// thread, the y axis once per row in the lanes of the block that hold it (LDS), and a
// row whose cell is the previous row's keeps its eight corner values (the lattice is
// finer than the grid).  Each point's value is the drop-in grid_sample's, bit for bit.
constexpr int kFieldRows = 8;
__global__ void __launch_bounds__(256) k_extract_fields(FieldArgs a) {
  __shared__ FieldAxis ys[kFieldRows];
  const int k = blockIdx.x * blockDim.x + threadIdx.x, i = blockIdx.z;
  const int j0 = blockIdx.y * kFieldRows;
  const int rows = min(kFieldRows, a.n[1] - j0);
  if ((int)threadIdx.x < rows)
    ys[threadIdx.x] = field_axis(a, 1, j0 + threadIdx.x, a.g.Y, a.g.sy);
  const FieldAxis x = field_axis(a, 0, i, a.g.X, a.g.sx);
  const FieldAxis z = field_axis(a, 2, min(k, a.n[2] - 1), a.g.Z, a.g.sz);
  __syncthreads();
  if (k >= a.n[2]) return;
  float* out = a.u + ((int64_t)i * a.n[1] + j0) * a.n[2] + k;
  // cells wholly in the grid (every wave's but the border's) sum without the selections
  const bool zx = __all((x.in & z.in) == 3u);
  float v[8];
  int cell = 0;
  for (int r = 0; r < rows; ++r) {
    const FieldAxis y = ys[r];
    const int yc = __builtin_amdgcn_readfirstlane(y.x0);
    if (r == 0 || yc != cell) {
      cell = yc;
#pragma unroll
      for (int c = 0; c < 8; ++c)
        v[c] = a.sdf[(c >> 2 ? x.off1 : x.off0) + (c >> 1 & 1 ? y.off1 : y.off0) +
                     (c & 1 ? z.off1 : z.off0)];
    }
    float acc = 0.f;
    auto add = [&](int c) {
#pragma clang fp contract(off)
      const int bx = c >> 2, by = c >> 1 & 1, bz = c & 1;
      const float w = ((bz ? z.w1 : z.w0) * (by ? y.w1 : y.w0)) * (bx ? x.w1 : x.w0);
      return acc + v[c] * w;
    };
    if (zx && __builtin_amdgcn_readfirstlane((int)y.in) == 3) {
#pragma unroll
      for (int c = 0; c < 8; ++c) acc = add(c);
    } else {
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        const float t = add(c);
        acc = (x.in >> (c >> 2) & y.in >> (c >> 1 & 1) & z.in >> (c & 1) & 1u) ? t : acc;
      }
    }
    out[(int64_t)r * a.n[2]] = a.scale * acc;
  }
}

// The same, one point per thread (3-D grid: z chunks of 256, y, x), for grids whose element
// offsets pass 32 bits.
__global__ void __launch_bounds__(256) k_extract_fields_wide(FieldArgs a) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y, i = blockIdx.z;
  if (k >= a.n[2]) return;
  const float px = linspace_at(a.bmin[0], a.bmax[0], a.n[0], i);
  const float py = linspace_at(a.bmin[1], a.bmax[1], a.n[1], j);
  const float pz = linspace_at(a.bmin[2], a.bmax[2], a.n[2], k);
  // the trilinear lookup of the drop-in grid_sample (voxel.h), zero outside the grid
  Tri<float> t;
  t.init(world_to_index(px, a.mn[0], a.mx[0] - a.mn[0], a.g.X),
         world_to_index(py, a.mn[1], a.mx[1] - a.mn[1], a.g.Y),
         world_to_index(pz, a.mn[2], a.mx[2] - a.mn[2], a.g.Z));
  const float v = tri_gather(a.sdf, a.g, t, 0);
  a.u[((int64_t)i * a.n[1] + j) * a.n[2] + k] = a.scale * v;
}

// ---- marching cubes, per-point counts ------------------------------------------------------

struct McArgs {
  const float* u;
  int nx, ny, nz;
  float iso;
  const int8_t* count;  // [256] device copy of the table
  const int8_t* edges;  // [256][3 * kMcMaxTris]
};

__device__ __forceinline__ bool below(const McArgs& a, int64_t p) { return a.u[p] < a.iso; }

// Crossing bits (x, y, z) of the three lattice edges starting at point (i, j, k).
__device__ __forceinline__ int owned_bits(const McArgs& a, int i, int j, int k, int64_t p) {
  const int64_t sx = (int64_t)a.ny * a.nz, sy = a.nz;
  const bool b = below(a, p);
  int bits = 0;
  if (i + 1 < a.nx && below(a, p + sx) != b) bits |= 1;
  if (j + 1 < a.ny && below(a, p + sy) != b) bits |= 2;
  if (k + 1 < a.nz && below(a, p + 1) != b) bits |= 4;
  return bits;
}

__device__ __forceinline__ int cube_index(const McArgs& a, int64_t p) {
  const int64_t sx = (int64_t)a.ny * a.nz, sy = a.nz;
  int idx = 0;
  for (int c = 0; c < 8; ++c)
    if (below(a, p + (c & 1) * sx + (c >> 1 & 1) * sy + (c >> 2 & 1))) idx |= 1 << c;
  return idx;
}

// Pass 1: vertices owned and triangles of the cube at each lattice point.
__global__ void __launch_bounds__(256) k_mc_count(McArgs a, int64_t* __restrict__ vcnt,
                                                  int64_t* __restrict__ tcnt) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y, i = blockIdx.z;
  if (k >= a.nz) return;
  const int64_t p = ((int64_t)i * a.ny + j) * a.nz + k;
  vcnt[p] = __popc(owned_bits(a, i, j, k, p));
  tcnt[p] = (i + 1 < a.nx && j + 1 < a.ny && k + 1 < a.nz) ? a.count[cube_index(a, p)] : 0;
}

// Pass 2: vertices (index space, or world space when bmin/bmax are given) and faces.
__global__ void __launch_bounds__(256) k_mc_emit(McArgs a, const int64_t* __restrict__ vincl,
                                                 const int64_t* __restrict__ tincl, int world,
                                                 double b0, double b1, double b2, double e0,
                                                 double e1, double e2, double* __restrict__ verts,
                                                 int64_t* __restrict__ faces) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y, i = blockIdx.z;
  if (k >= a.nz) return;
  const int64_t sx = (int64_t)a.ny * a.nz, sy = a.nz;
  const int64_t p = (i * sx + j * sy) + k;
  const int bits = owned_bits(a, i, j, k, p);
  if (bits) {
    int64_t vid = p ? vincl[p - 1] : 0;
    const double f1 = a.u[p];
    const int64_t step[3] = {sx, sy, 1};
    const double bmin[3] = {b0, b1, b2}, ext[3] = {e0, e1, e2};
    const int nn[3] = {a.nx, a.ny, a.nz};
    for (int ax = 0; ax < 3; ++ax) {
      if (!(bits >> ax & 1)) continue;
      const double f2 = a.u[p + step[ax]];
      double v[3] = {(double)i, (double)j, (double)k};
      v[ax] += ((double)a.iso - f1) / (f2 - f1);
      for (int c = 0; c < 3; ++c) {
        double w = v[c];
        if (world) w = w / (double)(nn[c] - 1) * ext[c] + bmin[c];
        verts[3 * vid + c] = w;
      }
      ++vid;
    }
  }
  if (i + 1 < a.nx && j + 1 < a.ny && k + 1 < a.nz) {
    const int ci = cube_index(a, p);
    const int nt = a.count[ci];
    int64_t t = p ? tincl[p - 1] : 0;
    for (int q = 0; q < nt; ++q, ++t) {
      for (int r = 0; r < 3; ++r) {
        const int e = a.edges[ci * 3 * kMcMaxTris + 3 * q + r];
        const int ax = e >> 2, o0 = ax == 0 ? 1 : 0, o1 = ax == 2 ? 1 : 2;
        int off[3] = {0, 0, 0};
        off[o0] = e & 1;
        off[o1] = e >> 1 & 1;
        const int qi = i + off[0], qj = j + off[1], qk = k + off[2];
        const int64_t qp = (qi * sx + qj * sy) + qk;
        const int qb = owned_bits(a, qi, qj, qk, qp);
        faces[3 * t + r] = (qp ? vincl[qp - 1] : 0) + __popc(qb & ((1 << ax) - 1));
      }
    }
  }
}

// ---- marching cubes on bit rows ----------------------------------------------------------
// The passes above keep two int64 per lattice point and scan them: 2 GiB written, and read
// and written three times more, for a 512^3 lattice of which one point in a hundred touches
// the surface (5.1 ms).  Here a point's side of the threshold is one bit: 64 consecutive
// points of a z row make a 64-bit word (a row's last word is padded), and every later
// question is asked of words -- which of a group's edges cross, which of its cubes are cut,
// how many vertices come before a point.  Three passes:
//   k_mc_below   the field once, 64 points per ballot (bound by the read);
//   k_mc_groups  per group (word) the vertices its points own and the triangles of its
//                cubes, with their prefix over the block's groups (bits from L2);
//   k_mc_write   the points that own a vertex or a cut cube, a lane each: a vertex number is
//                its group's offset plus the popcounts below the point's bit.
// Vertices and triangles come in the order of the passes above: by point, then by axis or
// by the table.
constexpr int kMcThreads = 128;   // groups per block

struct McGroups {
  int64_t words;      // words of a z row
  int64_t total;      // groups: nx * ny * words
  uint64_t* bits;     // [total] u < iso
  uint64_t* pre;      // [total] vertices | triangles << 32 of the block's earlier groups
  int64_t* blk;       // [2 * blocks] per block: vertices, triangles (then their offsets)
};

// Row of group q (32-bit division where the groups' numbers fit: the 64-bit one is a long
// sequence).
__device__ __forceinline__ int64_t mc_row(const McGroups& g, int64_t q) {
  if (g.total <= 0x7fffffff) return (int64_t)((uint32_t)q / (uint32_t)g.words);
  return q / g.words;
}

__global__ void __launch_bounds__(256) k_mc_below(const float* __restrict__ u, int nz, float iso,
                                                  McGroups g) {
  constexpr int U = 8;  // words per wave and round: their loads are all in flight together
  const int lane = threadIdx.x & 63;
  const int64_t waves = (int64_t)gridDim.x * (blockDim.x >> 6);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int64_t q0 = ((int64_t)blockIdx.x * (blockDim.x >> 6) + wave) * U;
  for (; q0 < g.total; q0 += waves * U) {
    float v[U];
    bool in[U];
    int64_t row = mc_row(g, q0);
    int w = (int)(q0 - row * g.words);
#pragma unroll
    for (int e = 0; e < U; ++e) {
      const int z = 64 * w + lane;
      in[e] = q0 + e < g.total && z < nz;
      v[e] = in[e] ? u[row * nz + z] : 0.f;
      if (++w == g.words) {
        w = 0;
        ++row;
      }
    }
#pragma unroll
    for (int e = 0; e < U; ++e) {
      const uint64_t b = __ballot(in[e] && v[e] < iso);
      if (lane == 0 && q0 + e < g.total) g.bits[q0 + e] = b;
    }
  }
}

// The words of a group's neighbourhood: b[di][dj] the word at (i + di, j + dj, w), n[di][dj]
// the row's next word (0 past the row), as far as they lie in the lattice (else 0).
template <int D>
struct McWords {
  uint64_t b[D][D], n[D][D];
  int nzw;         // points of this word (64, or fewer in a row's last)
  bool ix, jy;     // i + 1, j + 1 in the lattice
  bool more;       // the row goes on past this word
};

template <int D>
__device__ __forceinline__ void mc_words(const McArgs& a, const McGroups& g, int i, int j, int w,
                                         McWords<D>& m) {
  m.nzw = min(64, a.nz - 64 * w);
  m.ix = i + 1 < a.nx;
  m.jy = j + 1 < a.ny;
  m.more = w + 1 < g.words;
#pragma unroll
  for (int di = 0; di < D; ++di)
#pragma unroll
    for (int dj = 0; dj < D; ++dj) {
      const bool in = i + di < a.nx && j + dj < a.ny;
      const int64_t q = ((int64_t)min(i + di, a.nx - 1) * a.ny + min(j + dj, a.ny - 1)) * g.words + w;
      m.b[di][dj] = in ? g.bits[q] : 0;
      m.n[di][dj] = in && m.more ? g.bits[q + 1] : 0;
    }
}

__device__ __forceinline__ uint64_t low_bits(int n) { return n >= 64 ? ~0ull : (1ull << n) - 1; }

// Word of the points one further along z, and the bits of the word's points that have one.
__device__ __forceinline__ uint64_t mc_up(uint64_t b, uint64_t next) { return b >> 1 | next << 63; }
template <int D>
__device__ __forceinline__ uint64_t mc_zmask(const McWords<D>& m) {
  return low_bits(m.more ? 64 : m.nzw - 1);
}

// Crossing edges along x, y and z owned by the points of the word at (di, dj).
template <int D>
__device__ __forceinline__ void mc_edges(const McArgs& a, const McWords<D>& m, int i, int j, int di,
                                         int dj, uint64_t e[3]) {
  const uint64_t b = m.b[di][dj], in = low_bits(m.nzw);
  e[0] = i + di + 1 < a.nx ? (b ^ m.b[di + 1][dj]) & in : 0;
  e[1] = j + dj + 1 < a.ny ? (b ^ m.b[di][dj + 1]) & in : 0;
  e[2] = (b ^ mc_up(b, m.n[di][dj])) & mc_zmask(m);
}

// Configuration words of the word's cubes (bit k of word c: corner c of cube k is below) and
// the cubes that are cut.
template <int D>
__device__ __forceinline__ uint64_t mc_cubes(const McWords<D>& m, uint64_t c[8]) {
  uint64_t all = ~0ull, any = 0;
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const uint64_t b = m.b[q & 1][q >> 1 & 1];
    c[q] = q >> 2 ? mc_up(b, m.n[q & 1][q >> 1 & 1]) : b;
    all &= c[q];
    any |= c[q];
  }
  return m.ix && m.jy ? any & ~all & mc_zmask(m) : 0;
}

__device__ __forceinline__ int mc_config(const uint64_t c[8], int k) {
  int cfg = 0;
#pragma unroll
  for (int q = 0; q < 8; ++q) cfg |= (int)(c[q] >> k & 1) << q;
  return cfg;
}

__global__ void __launch_bounds__(kMcThreads) k_mc_groups(McArgs a, McGroups g) {
  __shared__ int8_t count[256];
  __shared__ uint64_t wave_sum[kMcThreads / 64];
  for (int i = threadIdx.x; i < 256; i += kMcThreads) count[i] = a.count[i];
  __syncthreads();
  const int64_t q = (int64_t)blockIdx.x * kMcThreads + threadIdx.x;
  uint32_t nv = 0, nt = 0;
  if (q < g.total) {
    const int64_t row = mc_row(g, q);
    const int w = (int)(q - row * g.words), i = (int)(row / a.ny), j = (int)(row - (int64_t)i * a.ny);
    McWords<2> m;
    mc_words(a, g, i, j, w, m);
    uint64_t e[3], c[8];
    mc_edges(a, m, i, j, 0, 0, e);
    nv = (uint32_t)(__popcll(e[0]) + __popcll(e[1]) + __popcll(e[2]));
    for (uint64_t cut = mc_cubes(m, c); cut; cut &= cut - 1)
      nt += count[mc_config(c, __ffsll((unsigned long long)cut) - 1)];
  }
  // block-wide exclusive prefix of both counts (at most 192 and 320 per group)
  const uint64_t own = (uint64_t)nt << 32 | nv;
  const uint64_t inc = (uint64_t)wave_incl_scan_i64((int64_t)own);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 63) wave_sum[wave] = inc;
  __syncthreads();
  uint64_t before = 0, total = 0;
#pragma unroll
  for (int k = 0; k < kMcThreads / 64; ++k) {
    if (k < wave) before += wave_sum[k];
    total += wave_sum[k];
  }
  if (q < g.total) g.pre[q] = before + inc - own;
  if (threadIdx.x == 0) {
    g.blk[2 * blockIdx.x] = (int64_t)(total & 0xffffffffull);
    g.blk[2 * blockIdx.x + 1] = (int64_t)(total >> 32);
  }
}

// Exclusive scan of the blocks' counts in place by one workgroup, sixteen blocks per thread
// and round, their 16-byte loads in flight together; totals[0] and [1] receive the numbers of vertices and triangles.
__global__ void __launch_bounds__(1024) k_mc_scan(int64_t* __restrict__ blk, int64_t blocks,
                                                  int64_t* __restrict__ totals) {
  constexpr int U = 16;
  __shared__ int64_t lds[2][16];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int64_t carry[2] = {0, 0};
  for (int64_t base = 0; base < blocks; base += 1024 * U) {
    const int64_t b0 = base + (int64_t)threadIdx.x * U;
    int64_t v[U][2], s[2] = {0, 0}, inc[2];
#pragma unroll
    for (int e = 0; e < U; ++e) {
      const longlong2 p = b0 + e < blocks ? reinterpret_cast<const longlong2*>(blk)[b0 + e]
                                          : make_longlong2(0, 0);
      s[0] += v[e][0] = p.x;
      s[1] += v[e][1] = p.y;
    }
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      inc[c] = wave_incl_scan_i64(s[c]);
      if (lane == 63) lds[c][wave] = inc[c];
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      int64_t off = carry[c] + inc[c] - s[c];
      for (int k = 0; k < 16; ++k) {
        if (k < wave) off += lds[c][k];
        carry[c] += lds[c][k];
      }
#pragma unroll
      for (int e = 0; e < U; ++e) {
        if (b0 + e < blocks) blk[2 * (b0 + e) + c] = off;
        off += v[e][c];
      }
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    totals[0] = carry[0];
    totals[1] = carry[1];
  }
}

struct McWorld {
  int on;
  double bmin[3], ext[3];
};

// A block's groups once more: their points that own a vertex or whose cube is cut are listed
// in LDS in point order (a group is a row's 64 points, of which the surface takes one or two),
// then a lane takes a point each.  With a wave per group and a lane per point of it the waves
// ran nearly empty: 797 us for the 381 k vertices of a 512^3 mesh, 172 so.
__global__ void __launch_bounds__(kMcThreads) k_mc_write(McArgs a, McGroups g, McWorld wd,
                                                         double* __restrict__ verts,
                                                         int64_t* __restrict__ faces) {
  // per listed point: its bit (6), its group in the block (7), its cube's configuration (8),
  // the triangles of the group's earlier cubes (9)
  __shared__ uint32_t list[kMcThreads * 64];
  __shared__ int8_t count[256];
  __shared__ int wave_sum[kMcThreads / 64];
  for (int i = threadIdx.x; i < 256; i += kMcThreads) count[i] = a.count[i];
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t first = (int64_t)blockIdx.x * kMcThreads;
  uint64_t act = 0, cut = 0, c[8];
  {
    const int64_t q = first + threadIdx.x;
    if (q < g.total) {
      const int64_t row = mc_row(g, q);
      const int w = (int)(q - row * g.words), i = (int)(row / a.ny), j = (int)(row - (int64_t)i * a.ny);
      McWords<2> m;
      mc_words(a, g, i, j, w, m);
      uint64_t e[3];
      mc_edges(a, m, i, j, 0, 0, e);
      cut = mc_cubes(m, c);
      act = e[0] | e[1] | e[2] | cut;
    }
  }
  const int n = __popcll(act);
  const int inc = (int)wave_incl_scan_i64(n);
  if (lane == 63) wave_sum[wave] = inc;
  __syncthreads();
  int at = inc - n, total = 0;
#pragma unroll
  for (int k = 0; k < kMcThreads / 64; ++k) {
    if (k < wave) at += wave_sum[k];
    total += wave_sum[k];
  }
  uint32_t tris = 0;
  for (; act; act &= act - 1) {
    const int k = __ffsll((unsigned long long)act) - 1;
    const int cfg = cut >> k & 1 ? mc_config(c, k) : 0;
    list[at++] = (uint32_t)k | threadIdx.x << 6 | (uint32_t)cfg << 13 | tris << 21;
    tris += count[cfg];
  }
  __syncthreads();
  const int64_t sx = (int64_t)a.ny * a.nz, sy = a.nz;
  const int nn[3] = {a.nx, a.ny, a.nz};
  for (int p = blockIdx.y * kMcThreads + threadIdx.x; p < total; p += gridDim.y * kMcThreads) {
    const uint32_t en = list[p];
    const int bit = en & 63, cfg = en >> 13 & 255;
    const int64_t q = first + (en >> 6 & 127);
    const int64_t row = mc_row(g, q);
    const int w = (int)(q - row * g.words), i = (int)(row / a.ny), j = (int)(row - (int64_t)i * a.ny);
    const int k = 64 * w + bit;
    McWords<3> m;
    mc_words(a, g, i, j, w, m);
    auto first_vertex = [&](int64_t gq) {
      return g.blk[2 * (gq / kMcThreads)] + (int64_t)(g.pre[gq] & 0xffffffffull);
    };
    // the number of the vertex on edge `ax` of the point at (i + di, j + dj, k + dk)
    auto vertex = [&](int di, int dj, int dk, int ax) {
      uint64_t e[3], nb = 0, ni = 0;
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y)
          if (di == x && dj == y) {
            mc_edges(a, m, i, j, x, y, e);
            nb = m.n[x][y];
            ni = m.n[x + 1][y];
          }
      const int64_t gq = ((int64_t)(i + di) * a.ny + (j + dj)) * g.words + w;
      if (bit + dk < 64) {
        const uint64_t lt = low_bits(bit + dk);
        int64_t v = first_vertex(gq) + __popcll(e[0] & lt) + __popcll(e[1] & lt) + __popcll(e[2] & lt);
        if (ax > 0) v += e[0] >> (bit + dk) & 1;
        if (ax > 1) v += e[1] >> (bit + dk) & 1;
        return v;
      }
      // the first point of the row's next word: no point of its group comes before it
      int64_t v = first_vertex(gq + 1);
      // (nor a z edge: those of this cube start in its own word)
      if (ax > 0 && i + di + 1 < a.nx) v += (nb ^ ni) & 1;
      return v;
    };
    uint64_t own[3];
    mc_edges(a, m, i, j, 0, 0, own);
    if ((own[0] | own[1] | own[2]) >> bit & 1) {
      const int64_t at0 = (i * sx + j * sy) + k;
      const int64_t step[3] = {sx, sy, 1};
      int64_t vid = vertex(0, 0, 0, 0);
      const double f1 = a.u[at0];
#pragma unroll
      for (int ax = 0; ax < 3; ++ax) {
        if (!(own[ax] >> bit & 1)) continue;
        const double f2 = a.u[at0 + step[ax]];
        double v[3] = {(double)i, (double)j, (double)k};
        v[ax] += ((double)a.iso - f1) / (f2 - f1);
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          double o = v[d];
          if (wd.on) o = o / (double)(nn[d] - 1) * wd.ext[d] + wd.bmin[d];
          verts[3 * vid + d] = o;
        }
        ++vid;
      }
    }
    const int nt = count[cfg];   // configuration 0 (not cut) has none
    if (nt == 0) continue;
    int64_t t = g.blk[2 * blockIdx.x + 1] + (int64_t)(g.pre[q] >> 32) + (en >> 21);
    for (int s = 0; s < nt; ++s, ++t)
#pragma unroll
      for (int r = 0; r < 3; ++r) {
        const int e = a.edges[cfg * 3 * kMcMaxTris + 3 * s + r];
        const int ax = e >> 2, e0 = e & 1, e1 = e >> 1 & 1;
        // the owning point: offset 0 along the edge, (e0, e1) on the other two axes
        faces[3 * t + r] = vertex(ax == 0 ? 0 : e0, ax == 0 ? e0 : (ax == 1 ? 0 : e1),
                                  ax == 2 ? 0 : e1, ax);
      }
  }
}

}  // namespace vx

using namespace vx;

extern "C" {

int vx_mc_tables(int8_t* count, int8_t* edges) {
  VX_CHECK_ARG(count && edges, "mc_tables: missing output");
  const McTables& t = tables();
  memcpy(count, t.count, sizeof(t.count));
  memcpy(edges, t.edges, sizeof(t.edges));
  return VX_OK;
}

int vx_mc_max_tris(void) { return kMcMaxTris; }

int vx_extract_fields(const float* sdf, const int64_t* geom, const float* box, const float* bounds,
                      int n0, int n1, int n2, float scale, float* u, void* stream) {
  VX_CHECK_ARG(sdf && geom && box && bounds && u, "extract_fields: missing argument");
  VX_CHECK_ARG(geom[0] == 1, "extract_fields: the SDF grid must have one channel");
  VX_CHECK_ARG(n0 >= 1 && n1 >= 1 && n2 >= 1 && n0 <= 65535 && n1 <= 65535,
               "extract_fields: bad lattice size");
  FieldArgs a;
  a.sdf = sdf;
  a.g.C = 1;
  a.g.X = (int)geom[1];
  a.g.Y = (int)geom[2];
  a.g.Z = (int)geom[3];
  a.g.sc = geom[4];
  a.g.sx = geom[5];
  a.g.sy = geom[6];
  a.g.sz = geom[7];
  for (int i = 0; i < 3; ++i) {
    a.mn[i] = box[i];
    a.mx[i] = box[3 + i];
    a.bmin[i] = bounds[i];
    a.bmax[i] = bounds[3 + i];
  }
  a.n[0] = n0;
  a.n[1] = n1;
  a.n[2] = n2;
  a.scale = scale;
  a.u = u;
  const int64_t last = (int64_t)(a.g.X - 1) * a.g.sx + (int64_t)(a.g.Y - 1) * a.g.sy +
                       (int64_t)(a.g.Z - 1) * a.g.sz;
  if (last < ((int64_t)1 << 31))
    k_extract_fields<<<dim3((unsigned)cdiv(n2, 256), (unsigned)cdiv(n1, kFieldRows), (unsigned)n0),
                       256, 0, (hipStream_t)stream>>>(a);
  else
    k_extract_fields_wide<<<dim3((unsigned)cdiv(n2, 256), (unsigned)n1, (unsigned)n0), 256, 0,
                            (hipStream_t)stream>>>(a);
  return launch_status("extract_fields");
}

// count: device copy of the [256] table counts, edges: [256 * 3 * vx_mc_max_tris()].
int vx_mc_count(const float* u, int nx, int ny, int nz, float iso, const int8_t* count,
                const int8_t* edges, int64_t* vcnt, int64_t* tcnt, void* stream) {
  VX_CHECK_ARG(u && count && edges && vcnt && tcnt, "mc_count: missing argument");
  VX_CHECK_ARG(nx >= 1 && ny >= 1 && nz >= 1 && nx <= 65535 && ny <= 65535, "mc_count: bad size");
  McArgs a{u, nx, ny, nz, iso, count, edges};
  const dim3 grid((unsigned)cdiv(nz, 256), (unsigned)ny, (unsigned)nx);
  k_mc_count<<<grid, 256, 0, (hipStream_t)stream>>>(a, vcnt, tcnt);
  return launch_status("mc_count");
}

int vx_mc_emit(const float* u, int nx, int ny, int nz, float iso, const int8_t* count,
               const int8_t* edges, const int64_t* vincl, const int64_t* tincl,
               const double* bounds, double* verts, int64_t* faces, void* stream) {
  VX_CHECK_ARG(u && count && edges && vincl && tincl, "mc_emit: missing argument");
  VX_CHECK_ARG(nx >= 1 && ny >= 1 && nz >= 1 && nx <= 65535 && ny <= 65535, "mc_emit: bad size");
  McArgs a{u, nx, ny, nz, iso, count, edges};
  double b[3] = {0, 0, 0}, e[3] = {0, 0, 0};
  // float32 bounds, their difference taken in float32 (lib/dvgo_ori.py:699-702 scales
  // float64 vertices by float32 numpy arrays)
  if (bounds)
    for (int i = 0; i < 3; ++i) {
      b[i] = (double)(float)bounds[i];
      e[i] = (double)((float)bounds[3 + i] - (float)bounds[i]);
    }
  const dim3 grid((unsigned)cdiv(nz, 256), (unsigned)ny, (unsigned)nx);
  k_mc_emit<<<grid, 256, 0, (hipStream_t)stream>>>(a, vincl, tincl, bounds ? 1 : 0, b[0], b[1],
                                                   b[2], e[0], e[1], e[2], verts, faces);
  return launch_status("mc_emit");
}

// Workspace of vx_mc_classify: the lattice's bit words, the groups' prefixes and the blocks'
// counts.
static int mc_groups(int64_t nx, int64_t ny, int64_t nz, void* ws, McGroups& g, int64_t& blocks) {
  VX_CHECK_ARG(nx >= 1 && ny >= 1 && nz >= 1 && nx <= 65535 && ny <= 65535,
               "marching cubes: bad size");
  g.words = cdiv(nz, 64);
  g.total = nx * ny * g.words;
  blocks = cdiv(g.total, kMcThreads);
  VX_CHECK_ARG(blocks <= 0x7fffffff, "marching cubes: field too large");
  g.bits = (uint64_t*)ws;
  g.pre = g.bits + g.total;
  g.blk = (int64_t*)(g.pre + g.total);  // 16-byte aligned: after an even number of words
  return VX_OK;
}

int64_t vx_mc_workspace_bytes(int nx, int ny, int nz) {
  McGroups g;
  int64_t blocks;
  if (mc_groups(nx, ny, nz, nullptr, g, blocks)) return -1;
  return 8 * (2 * g.total + 2 * blocks);
}

int vx_mc_classify(const float* u, int nx, int ny, int nz, float iso, const int8_t* count,
                   void* ws, int64_t* totals, void* stream) {
  VX_CHECK_ARG(u && count && ws && totals, "mc_classify: missing argument");
  VX_CHECK_ARG(((uintptr_t)ws & 15) == 0, "mc_classify: the workspace must be 16-byte aligned");
  McGroups g;
  int64_t blocks;
  if (int e = mc_groups(nx, ny, nz, ws, g, blocks)) return e;
  hipStream_t st = (hipStream_t)stream;
  McArgs a{u, nx, ny, nz, iso, count, nullptr};
  k_mc_below<<<grid_for(g.total, 32, 8192), 256, 0, st>>>(u, nz, iso, g);
  k_mc_groups<<<(unsigned)blocks, kMcThreads, 0, st>>>(a, g);
  k_mc_scan<<<1, 1024, 0, st>>>(g.blk, blocks, totals);
  return launch_status("mc_classify");
}

int vx_mc_write(const float* u, int nx, int ny, int nz, float iso, const int8_t* count,
                const int8_t* edges, void* ws, int64_t n_verts, int64_t n_faces,
                const double* bounds, double* verts, int64_t* faces, void* stream) {
  VX_CHECK_ARG(u && count && edges && ws && verts && faces, "mc_write: missing argument");
  VX_CHECK_ARG(n_verts >= 0 && n_faces >= 0, "mc_write: negative size");
  if (n_verts == 0) return VX_OK;
  McGroups g;
  int64_t blocks;
  if (int e = mc_groups(nx, ny, nz, ws, g, blocks)) return e;
  McArgs a{u, nx, ny, nz, iso, count, edges};
  McWorld wd{};
  wd.on = bounds != nullptr;
  // float32 bounds, their difference taken in float32, as vx_mc_emit
  if (bounds)
    for (int i = 0; i < 3; ++i) {
      wd.bmin[i] = (double)(float)bounds[i];
      wd.ext[i] = (double)((float)bounds[3 + i] - (float)bounds[i]);
    }
  // about n_faces / 2 points are listed, which workgroups share where that is more than a pass
  // of them each: with one a list, a 64^3 lattice of noise ran in 32 (535 us the call, 79 with
  // 32 shares, 92 with 16; 128^3, in 256: 584, 305 and 284).  Each makes the whole list.
  const int64_t passes = cdiv(n_faces, 2 * blocks * kMcThreads), most = blocks < 64 ? 32 : 16;
  const unsigned shares = (unsigned)(passes < 1 ? 1 : (passes > most ? most : passes));
  k_mc_write<<<dim3((unsigned)blocks, shares), kMcThreads, 0, (hipStream_t)stream>>>(a, g, wd, verts,
                                                                                    faces);
  return launch_status("mc_write");
}

}  // extern "C"
