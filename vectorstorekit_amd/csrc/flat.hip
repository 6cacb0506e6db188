// flat.hip -- flat (brute-force) k-NN: query x row distances on fp32 MFMA
// (L2^2 / L2 / cosine / normalised cosine / dot) or on the VALU (Manhattan),
// fused with the filter/append stage of the progressive top-k, so no
// query x row distance matrix is written to HBM.
//
// Reference: the batched distance kernels batchEuclideanDistance /
// batchCosineDistance / batchManhattanDistance / batchDotProduct
// (Acceleration/Metal/Shaders/DistanceShaders.metal:248-379, one thread per
// (query, row) pair) and their host side
// MetalAccelerationEngine.batchComputeDistancesGPU
// (Acceleration/MetalAccelerationEngine.swift:377-478), which reads back the
// full matrix and sorts each row on the CPU.
//
// MFMA kernel: a workgroup owns 64 queries and a contiguous slice of rows,
// walks the slice in tiles of 128 rows; each of its 4 waves computes a
// 32-row x 64-query block as 2x4 v_mfma_f32_16x16x4f32 tiles, with both
// operands staged through LDS in 32-dim stages.  Distances follow from the
// dot product and precomputed norms:
//   L2^2 = |q|^2 + |x|^2 - 2 q.x       cosine = 1 - q.x / (|q||x| + 1e-8)
//   normalised cosine = 1 - q.x        dot = -q.x
#include <cstring>

#include "flat.hpp"

namespace vsk {

typedef float f4 __attribute__((ext_vector_type(4)));

constexpr int FB_N = 128;  // rows per tile
constexpr int FB_Q = 64;   // queries per workgroup
constexpr int FB_K = 32;   // dims per LDS stage
constexpr int FS = FB_K + 2;  // LDS row stride (floats): conflict-free MFMA reads

// the metric is a template parameter: the epilogue has no runtime switch
template <int METRIC>
__device__ inline float metric_from_dot(float dot, float qa, float xa) {
  if constexpr (METRIC == VSK_METRIC_L2SQ || METRIC == VSK_METRIC_L2)
    return fmaxf(qa + xa - 2.0f * dot, 0.0f);
  else if constexpr (METRIC == VSK_METRIC_COSINE)
    return 1.0f - dot / (qa * xa + 1e-8f);
  else if constexpr (METRIC == VSK_METRIC_COSINE_NORMALIZED)
    return 1.0f - dot;
  else
    return -dot;
}

// one (query, row, distance) result of a tile
template <int MODE, int METRIC>
__device__ inline void emit(const FlatArgs &a, int64_t qi, int64_t row,
                            float dist, uint64_t th) {
  if constexpr (MODE == MODE_MATRIX) {
    a.mat[qi * a.ldm + row] = METRIC == VSK_METRIC_L2 ? sqrtf(dist) : dist;
  } else {
    if (MODE == MODE_DENSE && a.words) {
      a.words[qi * a.cap + (row - a.r0)] = vsk_f2ord(dist);
      return;
    }
    uint64_t key = vsk_key(dist, (uint32_t)row);
    if constexpr (MODE == MODE_DENSE) {
      a.cand[qi * a.cap + (row - a.r0)] = key;
    } else if (key <= th) {
      int slot = atomicAdd(&a.counts[qi], 1);
      if (slot < a.cap) a.cand[qi * a.cap + slot] = key;
    }
  }
}

template <int MODE, int METRIC>
__global__ __launch_bounds__(256) void k_flat_mfma(FlatArgs a) {
  __shared__ float xs[FB_N * FS];
  __shared__ float qs[FB_Q * FS];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int64_t q0 = (int64_t)blockIdx.x * FB_Q;
  const int64_t s0 = a.r0 + (int64_t)blockIdx.y * a.rows_per_split;
  int64_t s1 = s0 + a.rows_per_split;
  if (s1 > a.r1) s1 = a.r1;
  if (s0 >= s1) return;

  // the 4 queries this lane's accumulators belong to
  int64_t qi[4];
  bool qok[4];
  uint64_t th[4];
  float qa[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    qi[j] = q0 + j * 16 + (lane & 15);
    qok[j] = qi[j] < a.nq && (!a.active || a.active[qi[j]]);
    th[j] = (MODE == MODE_FILTER && qok[j]) ? a.thresh[qi[j]] : 0;
    qa[j] = (a.qaux && qi[j] < a.nq) ? a.qaux[qi[j]] : 0.f;
  }
  // global->LDS copy assignment: 8 threads per 32-float row segment
  const int crow = tid >> 3, ccol = (tid & 7) * 4;

  for (int64_t t0 = s0; t0 < s1; t0 += FB_N) {
    f4 acc[2][4];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = f4{0.f, 0.f, 0.f, 0.f};

    f4 xr[4], qr[2];
    auto gload = [&](int k0) {
      const bool kin = k0 + ccol < a.kdim;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        int64_t grow = t0 + u * 32 + crow;
        xr[u] = (kin && grow < s1)
                    ? *reinterpret_cast<const f4 *>(a.X + grow * a.ldx + k0 +
                                                    ccol)
                    : f4{0.f, 0.f, 0.f, 0.f};
      }
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        int64_t gq = q0 + u * 32 + crow;
        qr[u] = (kin && gq < a.nq)
                    ? *reinterpret_cast<const f4 *>(a.Q + gq * a.ldq + k0 +
                                                    ccol)
                    : f4{0.f, 0.f, 0.f, 0.f};
      }
    };
    gload(0);
    for (int k0 = 0; k0 < a.kdim; k0 += FB_K) {
      __syncthreads();
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        float *p = xs + (u * 32 + crow) * FS + ccol;
        p[0] = xr[u].x;
        p[1] = xr[u].y;
        p[2] = xr[u].z;
        p[3] = xr[u].w;
      }
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        float *p = qs + (u * 32 + crow) * FS + ccol;
        p[0] = qr[u].x;
        p[1] = qr[u].y;
        p[2] = qr[u].z;
        p[3] = qr[u].w;
      }
      __syncthreads();
      if (k0 + FB_K < a.kdim) gload(k0 + FB_K);
#pragma unroll
      for (int kk = 0; kk < FB_K; kk += 4) {
        float af[2], bf[4];
#pragma unroll
        for (int i = 0; i < 2; ++i)
          af[i] = xs[(w * 32 + i * 16 + (lane & 15)) * FS + kk + (lane >> 4)];
#pragma unroll
        for (int j = 0; j < 4; ++j)
          bf[j] = qs[(j * 16 + (lane & 15)) * FS + kk + (lane >> 4)];
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(af[i], bf[j],
                                                             acc[i][j], 0, 0,
                                                             0);
      }
    }
    // epilogue: D[row = 4*(lane/16) + r][query = lane%16] of each tile
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t row = t0 + w * 32 + i * 16 + 4 * (lane >> 4) + r;
        if (row >= s1) continue;
        const float xa = a.xaux ? a.xaux[row] : 0.f;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if (!qok[j]) continue;
          float dist = metric_from_dot<METRIC>(acc[i][j][r], qa[j], xa);
          emit<MODE, METRIC>(a, qi[j], row, dist, th[j]);
        }
      }
    }
  }
}

// Exact VALU distances, every term added in dimension order:
//  OP_L1    sum |q-x|   (the order of the reference's per-candidate vDSP
//           loop, Acceleration/AccelerateOptimizer.swift:322-360)
//  OP_L2SEQ sqrt(sum (q-x)^2) with separate multiply and add (no FMA), as
//           IVFIndex.computeDistance (Indexes/IVFIndex.swift:542-549)
// so the distances are bit-identical to a sequential fp32 loop.  Thread
// (tid) owns rows (tid%32)+32u, u<4, and queries (tid/32)+8v, v<8.
// MODE_ARGMIN keeps, per query, the smallest (distance, row) key over all
// rows, i.e. the first minimum under strict '<' (findNearestCentroid,
// Indexes/IVFIndex.swift:514-527), and writes the row index to argmin[q]
// (and its distance to a.amin[q] when a.amin is set).
constexpr int LS = FB_K + 1;  // odd stride: conflict-free column reads
// sequential (dimension-order, no FMA) terms and final transforms of the
// exact VALU kernel, one per metric of the CPU reference
//  OP_COSSEQ 1 - (sum q x)/(|q| |x| + 1e-8) with the norms the reference
//           computes (AccelerateOptimizer.swift:285-320, sums sequential)
enum { OP_L1 = 0, OP_L2SEQ = 1, OP_L2SQSEQ = 2, OP_CNSEQ = 3, OP_DOTSEQ = 4, OP_HAM = 5,
       OP_COSSEQ = 6 };

__device__ inline uint64_t shfl_xor_u64(uint64_t v, int m) {
  uint32_t lo = __shfl_xor((uint32_t)v, m);
  uint32_t hi = __shfl_xor((uint32_t)(v >> 32), m);
  return ((uint64_t)hi << 32) | lo;
}

template <int OP>
__device__ inline float valu_term(float q, float x) {
#pragma clang fp contract(off)
  if constexpr (OP == OP_L1) {
    return fabsf(q - x);
  } else if constexpr (OP == OP_HAM) {
    // hammingDistance: count += 1 where the components differ
    // (Core/Distance/UnifiedDistanceComputation.swift:249-261; NaN differs)
    return q != x ? 1.0f : 0.0f;
  } else if constexpr (OP == OP_L2SEQ || OP == OP_L2SQSEQ) {
    float t = q - x;
    return t * t;
  } else {
    return q * x;
  }
}

template <int OP>
__device__ inline float valu_final(float s) {
  if constexpr (OP == OP_L2SEQ) return sqrtf(s);
  else if constexpr (OP == OP_CNSEQ) return 1.0f - s;
  else if constexpr (OP == OP_DOTSEQ) return -s;
  else return s;
}

template <int MODE, int OP, int U, int V>
__global__ __launch_bounds__(256) void k_flat_valu(FlatArgs a, int32_t *argmin) {
#pragma clang fp contract(off)
  // a tile of 32 U rows x 8 V queries; thread (rsub, qsub) owns rows
  // rsub + 32 u and queries qsub + 8 v
  static_assert(V % 4 == 0, "queries are staged 32 at a time");
  __shared__ float xs[32 * U * LS];
  __shared__ float qs[8 * V * LS];
  const int tid = threadIdx.x;
  const int64_t q0 = (int64_t)blockIdx.x * (8 * V);
  const int64_t s0 = a.r0 + (int64_t)blockIdx.y * a.rows_per_split;
  int64_t s1 = s0 + a.rows_per_split;
  if (s1 > a.r1) s1 = a.r1;
  if (s0 >= s1) return;
  const int rsub = tid & 31, qsub = tid >> 5;
  int64_t qi[V];
  bool qok[V];
  uint64_t th[V];
  uint64_t best[V];
  float qn[V];  // OP_COSSEQ: the queries' norms
#pragma unroll
  for (int v = 0; v < V; ++v) {
    qi[v] = q0 + qsub + 8 * v;
    qok[v] = qi[v] < a.nq && (!a.active || a.active[qi[v]]);
    qn[v] = (OP == OP_COSSEQ && qi[v] < a.nq) ? a.qaux[qi[v]] : 0.f;
    th[v] = (MODE == MODE_FILTER && qok[v]) ? a.thresh[qi[v]] : 0;
    best[v] = VSK_KEY_NONE;
  }
  const int crow = tid >> 3, ccol = (tid & 7) * 4;
  for (int64_t t0 = s0; t0 < s1; t0 += 32 * U) {
    float acc[U][V];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int v = 0; v < V; ++v) acc[u][v] = 0.f;
    for (int k0 = 0; k0 < a.kdim; k0 += FB_K) {
      const bool kin = k0 + ccol < a.kdim;
      __syncthreads();
#pragma unroll
      for (int u = 0; u < U; ++u) {
        int64_t grow = t0 + u * 32 + crow;
        f4 v = (kin && grow < s1)
                   ? *reinterpret_cast<const f4 *>(a.X + grow * a.ldx + k0 +
                                                   ccol)
                   : f4{0.f, 0.f, 0.f, 0.f};
        float *p = xs + (u * 32 + crow) * LS + ccol;
        p[0] = v.x;
        p[1] = v.y;
        p[2] = v.z;
        p[3] = v.w;
      }
#pragma unroll
      for (int u = 0; u < V / 4; ++u) {
        int64_t gq = q0 + u * 32 + crow;
        f4 v = (kin && gq < a.nq)
                   ? *reinterpret_cast<const f4 *>(a.Q + gq * a.ldq + k0 +
                                                   ccol)
                   : f4{0.f, 0.f, 0.f, 0.f};
        float *p = qs + (u * 32 + crow) * LS + ccol;
        p[0] = v.x;
        p[1] = v.y;
        p[2] = v.z;
        p[3] = v.w;
      }
      __syncthreads();
      const int kend = a.kdim - k0 < FB_K ? a.kdim - k0 : FB_K;
      for (int kk = 0; kk < kend; ++kk) {
        float xv[U], qv[V];
#pragma unroll
        for (int u = 0; u < U; ++u) xv[u] = xs[(rsub + 32 * u) * LS + kk];
#pragma unroll
        for (int v = 0; v < V; ++v) qv[v] = qs[(qsub + 8 * v) * LS + kk];
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int v = 0; v < V; ++v) acc[u][v] += valu_term<OP>(qv[v], xv[u]);
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t row = t0 + rsub + 32 * u;
      if (row >= s1) continue;
      const float xn = OP == OP_COSSEQ ? a.xaux[row] : 0.f;
#pragma unroll
      for (int v = 0; v < V; ++v) {
        if (!qok[v]) continue;
        const float dist = OP == OP_COSSEQ ? 1.0f - acc[u][v] / (qn[v] * xn + 1e-8f)
                                           : valu_final<OP>(acc[u][v]);
        if constexpr (MODE == MODE_ARGMIN) {
          uint64_t key = vsk_key(dist, (uint32_t)row);
          best[v] = key < best[v] ? key : best[v];
        } else {
          // the keys/matrix carry the final distance already
          emit<MODE, VSK_METRIC_L1>(a, qi[v], row, dist, th[v]);
        }
      }
    }
  }
  if constexpr (MODE == MODE_ARGMIN) {
    // the 32 lanes with equal qsub hold disjoint rows of the same queries
#pragma unroll
    for (int v = 0; v < V; ++v) {
      uint64_t b = best[v];
#pragma unroll
      for (int m = 16; m > 0; m >>= 1) {
        uint64_t o = shfl_xor_u64(b, m);
        b = o < b ? o : b;
      }
      if (rsub == 0 && qok[v]) {
        argmin[qi[v]] = (int32_t)(uint32_t)b;
        if (a.amin) a.amin[qi[v]] = vsk_ord2f((uint32_t)(b >> 32));
      }
    }
  }
}

// The same distances as a stream over the rows, for launches of few queries
// or few tiles.  A wave owns 64 rows and V queries: it gathers C columns of
// its rows in whole 4 C-byte segments into its own LDS tile, the next C
// columns' loads in flight meanwhile, and each lane adds its row's terms in
// dimension order for every query.  The queries' columns are staged beside
// them and read as broadcasts (scalar loads of them made every 16 columns
// wait for the scalar cache: 1.5 x slower at V = 4).  No barrier: the waves
// are independent, and 9 (C = 64) or 17 (C = 32) of them share a CU.  Query
// groups of the same rows run next to each other on one XCD, whose L2 then
// serves all but the first.
//
// Bound: HBM up to about 4 queries, then the VALU (2 or 3 operations a term).
// Measured against the 64 x 32 tiles of k_flat_valu (dot product): 100,000 x
// 768, 1 query 49 against 163 us (6.3 TB/s), 4 queries 53 against 165, 16
// queries 95 against 167, 32 queries 159 against 173; 10,000 x 128, 1 query
// 4.7 against 16 us, 100 queries about 15 against 18.
template <int MODE, int OP, int V, int C>
__global__ __launch_bounds__(64) void k_flat_stream(FlatArgs a, int32_t groups, int32_t few) {
#pragma clang fp contract(off)
  constexpr int NL = C / 4;      // row loads a chunk, 16 bytes a lane
  constexpr int LD = C + 4;      // LDS row stride (floats): conflict-free 16-byte reads
  constexpr int LPR = C / 4;     // lanes a row segment
  constexpr int RPI = 64 / LPR;  // rows a load instruction
  constexpr int QN = (V + RPI - 1) / RPI;  // query loads a chunk
  __shared__ __attribute__((aligned(16))) float tile[64 * LD];
  __shared__ __attribute__((aligned(16))) float qt[V * C];
  const int lane = threadIdx.x;
  // block L runs on XCD L % 8: there, groups of one row tile in turn; with
  // few row tiles (their number, else 0) all tiles of a group in turn
  const uint32_t l = few ? blockIdx.x : blockIdx.x >> 3;
  const uint32_t g = few ? l / (uint32_t)few : l % (uint32_t)groups;
  const uint32_t t = few ? l - g * (uint32_t)few
                         : l / (uint32_t)groups * 8 + (blockIdx.x & 7);
  const int64_t q0 = (int64_t)g * V;
  const int64_t row0 = a.r0 + (int64_t)t * 64;
  if (row0 >= a.r1) return;
  const int seg = lane % LPR, sub = lane / LPR;
  const int64_t last = a.r1 - 1 - row0;  // rows past the end read the last one
  const float *src[NL];
#pragma unroll
  for (int i = 0; i < NL; ++i) {
    const int64_t r = sub + RPI * i;
    src[i] = a.X + (row0 + (r < last ? r : last)) * a.ldx;
  }
  const float *qsrc[QN];  // (queries past the last read the last one)
#pragma unroll
  for (int u = 0; u < QN; ++u) {
    const int64_t q = q0 + RPI * u + sub;
    qsrc[u] = a.Q + (q < a.nq ? q : a.nq - 1) * a.ldq;
  }
  const int32_t cmax = a.kdim - 4;  // a segment past the row end is clamped
  f4 buf[NL], qbuf[QN];
  auto load = [&](int32_t c0) {
    const int32_t col = c0 + 4 * seg < cmax ? c0 + 4 * seg : cmax;
#pragma unroll
    for (int u = 0; u < QN; ++u) qbuf[u] = *reinterpret_cast<const f4 *>(qsrc[u] + col);
#pragma unroll
    for (int i = 0; i < NL; ++i) buf[i] = *reinterpret_cast<const f4 *>(src[i] + col);
  };
  float acc[V];
#pragma unroll
  for (int v = 0; v < V; ++v) acc[v] = 0.f;
  // one query a wave: its cosine norm is summed here too (the wave waits on
  // memory), which saves a launch before the scan
  float qsum = 0.f;
  load(0);
  for (int32_t k0 = 0; k0 < a.kdim; k0 += C) {
#pragma unroll
    for (int i = 0; i < NL; ++i)
      *reinterpret_cast<f4 *>(tile + (sub + RPI * i) * LD + 4 * seg) = buf[i];
#pragma unroll
    for (int u = 0; u < QN; ++u)
      if (RPI * u + sub < V)
        *reinterpret_cast<f4 *>(qt + (RPI * u + sub) * C + 4 * seg) = qbuf[u];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if (k0 + C < a.kdim) load(k0 + C);
    const float *xr = tile + lane * LD;
    const int32_t kn = a.kdim - k0 < C ? a.kdim - k0 : C;
#pragma unroll 4
    for (int32_t k = 0; k < kn; k += 4) {
      const f4 xv = *reinterpret_cast<const f4 *>(xr + k);
#pragma unroll
      for (int v = 0; v < V; ++v) {
        const f4 qv = *reinterpret_cast<const f4 *>(qt + v * C + k);
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[v] += valu_term<OP>(qv[c], xv[c]);
        if constexpr (OP == OP_COSSEQ && V == 1) {
#pragma unroll
          for (int c = 0; c < 4; ++c) qsum += qv[c] * qv[c];
        }
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
  if (lane > last) return;
  const int64_t row = row0 + lane;
  const float xn = OP == OP_COSSEQ ? a.xaux[row] : 0.f;
#pragma unroll
  for (int v = 0; v < V; ++v) {
    if (q0 + v >= a.nq) break;
    if (a.active && !a.active[q0 + v]) continue;
    const float qn = OP != OP_COSSEQ ? 0.f : V == 1 ? sqrtf(qsum) : a.qaux[q0 + v];
    const float dist = OP == OP_COSSEQ ? 1.0f - acc[v] / (qn * xn + 1e-8f)
                                       : valu_final<OP>(acc[v]);
    emit<MODE, VSK_METRIC_L1>(a, q0 + v, row, dist,
                              MODE == MODE_FILTER ? a.thresh[q0 + v] : 0);
  }
}

template <int OP, int V, int C>
static void launch_stream_v(vsk_ctx *ctx, const FlatArgs &a, int mode) {
  const int64_t groups = ceil_div(a.nq, V);
  // A tile of its own XCD leaves up to seven XCDs of eight without work where
  // the tiles are few (an index's centroids: 111 rows x 32, 1,798 queries used
  // two of them: 10.5 us, now 5.6), and up to 1/8 of them at 64 tiles.
  int64_t tiles = ceil_div(a.r1 - a.r0, 64);
  const int32_t few = tiles < 64 ? (int32_t)tiles : 0;
  if (!few) tiles = ceil_div(tiles, 8) * 8;
  const dim3 grid((unsigned)(groups * tiles));
  const int32_t g = (int32_t)groups;
  if (mode == MODE_DENSE)
    k_flat_stream<MODE_DENSE, OP, V, C><<<grid, 64, 0, ctx->stream>>>(a, g, few);
  else if (mode == MODE_FILTER)
    k_flat_stream<MODE_FILTER, OP, V, C><<<grid, 64, 0, ctx->stream>>>(a, g, few);
  else
    k_flat_stream<MODE_MATRIX, OP, V, C><<<grid, 64, 0, ctx->stream>>>(a, g, few);
}

// Queries a wave: as few as leave the launch about one round of resident
// waves (9 or so a CU), since a small launch takes one wave's time; eight
// when there is more to do, which reads the rows least often.  (10,000 x 128:
// 8 queries one a wave 6.4, four a wave 7.4 us; 16 queries 9.6 and 8.1; 64
// queries four a wave 15.3, eight 16.0; 128 queries 23.5 and 20.4.)  Rows of
// at most 32 columns are one chunk of 32: with 64, the loads of the absent
// half and nine waves a CU instead of 17 made 10,000 queries over 40 rows x 32
// take 8.1 us (in tiles 7.9), now 6.1; of 8 columns 7.0 (5.0), now 4.9.
template <int OP>
static void launch_stream(vsk_ctx *ctx, const FlatArgs &a, int mode) {
  const int64_t tiles = ceil_div(a.r1 - a.r0, 64), cus = ctx->cu_count;
  const bool narrow = a.kdim <= 32;  // (one chunk of 32 columns: half the loads and LDS)
  if (a.nq == 1 || tiles * a.nq <= 8 * cus) {
    if (narrow)
      launch_stream_v<OP, 1, 32>(ctx, a, mode);
    else
      launch_stream_v<OP, 1, 64>(ctx, a, mode);
  } else if (tiles * ceil_div(a.nq, 4) <= 10 * cus) {
    if (narrow)
      launch_stream_v<OP, 4, 32>(ctx, a, mode);
    else
      launch_stream_v<OP, 4, 64>(ctx, a, mode);
  } else {
    launch_stream_v<OP, 8, 32>(ctx, a, mode);
  }
}

template <int METRIC>
static void launch_mfma(vsk_ctx *ctx, dim3 grid, const FlatArgs &a, int mode) {
  if (mode == MODE_DENSE)
    k_flat_mfma<MODE_DENSE, METRIC><<<grid, 256, 0, ctx->stream>>>(a);
  else if (mode == MODE_FILTER)
    k_flat_mfma<MODE_FILTER, METRIC><<<grid, 256, 0, ctx->stream>>>(a);
  else
    k_flat_mfma<MODE_MATRIX, METRIC><<<grid, 256, 0, ctx->stream>>>(a);
}

// the exact VALU scan in tiles of 32 U rows x 8 V queries (argmin: 128 x 64)
template <int OP, int U, int V>
static void launch_valu_tiles(vsk_ctx *ctx, dim3 grid, const FlatArgs &a, int mode,
                              int32_t *argmin) {
  if (mode == MODE_DENSE)
    k_flat_valu<MODE_DENSE, OP, U, V><<<grid, 256, 0, ctx->stream>>>(a, argmin);
  else if (mode == MODE_FILTER)
    k_flat_valu<MODE_FILTER, OP, U, V><<<grid, 256, 0, ctx->stream>>>(a, argmin);
  else if (mode == MODE_MATRIX)
    k_flat_valu<MODE_MATRIX, OP, U, V><<<grid, 256, 0, ctx->stream>>>(a, argmin);
  else if constexpr (V == 8)
    k_flat_valu<MODE_ARGMIN, OP, U, V><<<grid, 256, 0, ctx->stream>>>(a, argmin);
}

// metrics of the exact VALU scan
static bool metric_is_valu(int32_t metric) {
  return metric == VSK_METRIC_L1 || metric == VSK_METRIC_HAMMING || metric >= METRIC_L2_EXACT;
}

template <int OP>
static void launch_exact(vsk_ctx *ctx, dim3 grid, const FlatArgs &a, int mode,
                         int32_t *argmin, bool stream, bool small) {
  if (stream)
    launch_stream<OP>(ctx, a, mode);
  else if (small)
    launch_valu_tiles<OP, 2, 4>(ctx, grid, a, mode, argmin);
  else
    launch_valu_tiles<OP, 4, 8>(ctx, grid, a, mode, argmin);
}

// grid: query tiles x row splits, enough workgroups to fill 256 CUs (argmin
// keeps every row of a query in one workgroup)
void launch_flat(vsk_ctx *ctx, FlatArgs a, int mode, int32_t *argmin) {
  const int64_t rows = a.r1 - a.r0;
  if (rows <= 0 || a.nq <= 0) return;
  const bool valu = metric_is_valu(a.metric);
  int64_t tq = FB_Q, tn = FB_N, qt, splits;
  auto split = [&] {
    qt = ceil_div(a.nq, tq);
    splits = mode == MODE_ARGMIN ? 1 : ceil_div(4096, qt);
    const int64_t max_splits = ceil_div(rows, tn);
    if (splits > max_splits) splits = max_splits;
    if (splits > 65535) splits = 65535;
    if (splits < 1) splits = 1;
    a.rows_per_split = ceil_div(ceil_div(rows, splits), tn) * tn;
    splits = ceil_div(rows, a.rows_per_split);
  };
  split();
  // few 128 x 64 tiles and more than 64 queries: from some ten waves of the
  // stream a CU on, short rows are faster in tiles of 64 x 32, which read a
  // row half as often (us, tiles and stream: 2,048 x 32, 1,000 queries 15.9
  // and 13.1, 4,000 queries 28.8 and 34.3; 10,000 x 128, 256 queries 33.6 and
  // 35.3; of 512 columns, 1,800 queries x 4,096 rows, 281 and 269)
  const bool few = valu && mode != MODE_ARGMIN && qt * splits < 4 * (int64_t)ctx->cu_count;
  // (of at most 32 columns also fewer queries, where they nearly fill a tile:
  // 100,000 x 32, the distances of 32 queries 13.4 and 14.5, 40 21.8 and 16.4,
  // 64 22.2 and 24.9)
  const bool narrow = a.kdim <= 32;
  const int64_t pairs = a.nq * rows;
  const bool small = few && a.kdim <= 128 &&
                     ((a.nq > 64 && pairs >= 10000 * (int64_t)ctx->cu_count) ||
                      (narrow && (a.nq > 40 || (a.nq > 16 && a.nq <= 32)) &&
                       pairs >= 9000 * (int64_t)ctx->cu_count));
  if (small) {
    tq = 32;
    tn = 64;
    split();
  }
  if (qt > 0x7FFFFFFF) fail(VSK_ERR_INVALID_BUFFER_SIZE, "too many queries");
  dim3 grid((unsigned)qt, (unsigned)splits);
  static const char *names[2][4] = {
      {"flat_mfma_dense", "flat_mfma_filter", "flat_mfma_matrix", "flat_mfma_argmin"},
      {"flat_valu_dense", "flat_valu_filter", "flat_valu_matrix", "flat_valu_argmin"}};
  const char *name = names[valu ? 1 : 0][mode];
  KernelTimer t(ctx, name, (double)a.nq * (double)rows);
  if (valu) {
    // up to 48 queries, or fewer than 4 tiles a CU: the stream over the rows,
    // whose waves all wait on the VALU from there on, where a tile of 64
    // queries reads a row once (us, tiles and stream; 854,462 x 768,
    // Manhattan: 40 queries 2,000 and 1,510, 48 1,930 and 1,800, 49 1,940 and
    // 2,060, 64 1,930 and 2,310; the dot products of 300,000 x 128: 48 115 and
    // 107, 49 115 and 123, 64 119 and 139; of 854,462 x 32: 40 89 and 86, 48
    // 103 and 108; 100,000 x 768 in few tiles: 56 285 and 244, 64 290 and 294)
    // (a grid of at most 2^25 waves)
    const bool stream = mode != MODE_ARGMIN && !small &&
                        (a.nq <= (narrow ? 40 : 48) || few) &&
                        ceil_div(rows, 64) * ceil_div(a.nq, 8) <= 1 << 25;
    switch (a.metric) {
    case VSK_METRIC_L1: launch_exact<OP_L1>(ctx, grid, a, mode, argmin, stream, small); break;
    case VSK_METRIC_HAMMING: launch_exact<OP_HAM>(ctx, grid, a, mode, argmin, stream, small); break;
    case METRIC_L2_EXACT: launch_exact<OP_L2SEQ>(ctx, grid, a, mode, argmin, stream, small); break;
    case METRIC_L2SQ_EXACT: launch_exact<OP_L2SQSEQ>(ctx, grid, a, mode, argmin, stream, small); break;
    case METRIC_CN_EXACT: launch_exact<OP_CNSEQ>(ctx, grid, a, mode, argmin, stream, small); break;
    case METRIC_DOT_EXACT: launch_exact<OP_DOTSEQ>(ctx, grid, a, mode, argmin, stream, small); break;
    case METRIC_COS_EXACT: launch_exact<OP_COSSEQ>(ctx, grid, a, mode, argmin, stream, small); break;
    default: fail(VSK_ERR_INVALID_ARGUMENT, "no exact kernel for this metric");
    }
  } else {
    if (mode == MODE_ARGMIN)
      fail(VSK_ERR_UNSUPPORTED, "argmin needs an exact VALU metric");
    switch (a.metric) {
    case VSK_METRIC_L2SQ: launch_mfma<VSK_METRIC_L2SQ>(ctx, grid, a, mode); break;
    case VSK_METRIC_L2: launch_mfma<VSK_METRIC_L2>(ctx, grid, a, mode); break;
    case VSK_METRIC_COSINE: launch_mfma<VSK_METRIC_COSINE>(ctx, grid, a, mode); break;
    case VSK_METRIC_COSINE_NORMALIZED:
      launch_mfma<VSK_METRIC_COSINE_NORMALIZED>(ctx, grid, a, mode);
      break;
    default: launch_mfma<VSK_METRIC_DOT>(ctx, grid, a, mode); break;
    }
  }
  check_launch(name);
}

const float *x_aux(const vsk_db *db, int32_t metric) {
  if (metric == VSK_METRIC_L2SQ || metric == VSK_METRIC_L2)
    return db->sqnorm.as<float>();
  if (metric == VSK_METRIC_COSINE) return db->norm.as<float>();
  if (metric == METRIC_COS_EXACT) {
    if (!db->seqnorm.p) fail(VSK_ERR_EXECUTION_FAILED, "exact cosine norms not made");
    return db->seqnorm.as<float>();
  }
  return nullptr;
}

void ensure_seq_norms(vsk_ctx *ctx, const vsk_db *db) {
  if (db->seqnorm.p) return;
  DevBuf norms;
  norms.reserve(sizeof(float) * (size_t)db->n);
  seq_norms(ctx, db->x.as<float>(), db->n, db->d, db->ld, norms.as<float>());
  db->seqnorm.swap(norms);
}

float *q_aux(vsk_ctx *ctx, const float *dq, int64_t nq, int32_t d, int32_t ld,
             int32_t metric) {
  if (metric != VSK_METRIC_L2SQ && metric != VSK_METRIC_L2 &&
      metric != VSK_METRIC_COSINE && metric != METRIC_COS_EXACT)
    return nullptr;
  float *aux = static_cast<float *>(ctx->scratch_ptr("flat.qaux", 4 * nq));
  if (metric == METRIC_COS_EXACT)
    seq_norms(ctx, dq, nq, d, ld, aux);
  else if (metric == VSK_METRIC_COSINE)
    row_norms(ctx, dq, nq, d, ld, nullptr, aux);
  else
    row_norms(ctx, dq, nq, d, ld, aux, nullptr);
  return aux;
}

static bool use_bf16x3(const vsk_ctx *ctx, int32_t metric) {
  return !ctx->flat_fp32 && !metric_is_valu(metric);
}

SplitPtrs make_split(vsk_ctx *ctx, const vsk_db *db, const float *dq,
                     int64_t nq, bool qlo, float *qnh, float *qnr) {
  // whole 64-dimension stages of the screen (zero padding)
  const int32_t ldb = (db->d + 63) & ~63;
  if (!db->split.p) {
    // the hi plane (all the IVF probe's screen reads) and the maxima of its
    // bound (the database gets it when both are whole: a plane whose maxima
    // were never read would pass for exact)
    DevBuf hi;
    hi.reserve(sizeof(uint16_t) * (size_t)db->n * ldb);
    uint32_t *mb =
        static_cast<uint32_t *>(ctx->scratch_ptr("flat.splitmax", 2 * sizeof(uint32_t)));
    fill_i32(ctx, reinterpret_cast<int32_t *>(mb), 2, 0);
    split_bf16(ctx, db->x.as<float>(), db->n, db->d, db->ld, hi.as<uint16_t>(), nullptr, ldb,
               nullptr, nullptr, mb);
    uint32_t hb[2];
    VSK_HIP(hipMemcpyAsync(hb, mb, sizeof(hb), hipMemcpyDeviceToHost, ctx->stream));
    stream_sync(ctx);
    std::memcpy(&db->split_max_hi, &hb[0], sizeof(float));
    std::memcpy(&db->split_max_res, &hb[1], sizeof(float));
    db->ldb = ldb;
    db->split.swap(hi);
  }
  if (qlo && !db->split_lo.p) {
    // the lo plane only for the bf16x3 kernel (hi is written again, the
    // same values)
    DevBuf lo;
    lo.reserve(sizeof(uint16_t) * (size_t)db->n * ldb);
    split_bf16(ctx, db->x.as<float>(), db->n, db->d, db->ld, db->split.as<uint16_t>(),
               lo.as<uint16_t>(), ldb, nullptr, nullptr, nullptr);
    db->split_lo.swap(lo);
  }
  uint16_t *qs = static_cast<uint16_t *>(ctx->scratch_ptr(
      "flat.qsplit", sizeof(uint16_t) * (qlo ? 2 : 1) * (size_t)nq * ldb));
  split_bf16(ctx, dq, nq, db->d, db->ld, qs, qlo ? qs + (size_t)nq * ldb : nullptr,
             ldb, qnh, qnr, nullptr);
  SplitPtrs s;
  s.xh = db->split.as<uint16_t>();
  s.xl = db->split_lo.as<uint16_t>();  // (null until a bf16x3 call made it)
  s.qh = qs;
  s.ql = qlo ? qs + (size_t)nq * ldb : nullptr;
  s.ldxb = ldb;
  s.ldqb = ldb;
  s.kb = ldb;
  return s;
}

// whether the screen can read the rows for this metric: their plane, made by
// the first search that asks for it.  Without memory for one more plane (each
// family of metrics has its own: L2, L2^2 and dot; cosine; normalised cosine)
// the answer is no, and the exact scan serves the search.
static bool screen_plane_ok(vsk_ctx *ctx, const vsk_db *db, int32_t metric) {
  try {
    if (metric == VSK_METRIC_COSINE) return cosine_screen_ok(ctx, db);
    const bool bf16 = metric == VSK_METRIC_COSINE_NORMALIZED;
    auto &pl = db->plane[bf16 ? 1 : 0];
    if (pl.h.p) return true;
    const int32_t ldb = (db->d + 63) & ~63;
    pl.state.reserve(4 * sizeof(uint32_t));
    DevBuf h;  // (the database gets it with its maxima, as in make_split)
    h.reserve(plane_bytes(db->n, ldb));
    uint32_t *st = pl.state.as<uint32_t>();
    half_rows(ctx, bf16 ? PLANE_BF16 : PLANE_HALF, db->x.as<float>(), db->sqnorm.as<float>(),
              nullptr, db->n, db->d, db->ld, h.as<uint16_t>(), ldb, nullptr, st);
    uint32_t hb[2];
    VSK_HIP(hipMemcpyAsync(hb, st, sizeof(hb), hipMemcpyDeviceToHost, ctx->stream));
    stream_sync(ctx);
    std::memcpy(&pl.max_hi, &hb[0], sizeof(float));
    std::memcpy(&pl.max_res, &hb[1], sizeof(float));
    pl.h.swap(h);
    return true;
  } catch (const Error &e) {
    if (e.code != VSK_ERR_OUT_OF_MEMORY) throw;
    return false;
  }
}

// the screen's planes: the database's (screen_plane_ok) and the query batch's
static SplitPtrs make_half(vsk_ctx *ctx, const vsk_db *db, const float *dq, int64_t nq,
                           int32_t metric, float *qnh, float *qnr) {
  // whole 64-dimension stages of the screen (zero padding)
  const int32_t ldb = (db->d + 63) & ~63;
  const bool cosine = metric == VSK_METRIC_COSINE;
  const bool bf16 = metric == VSK_METRIC_COSINE_NORMALIZED;
  const auto &pl = db->plane[bf16 ? 1 : 0];
  uint16_t *qh = static_cast<uint16_t *>(
      ctx->scratch_ptr("flat.qhalf", sizeof(uint16_t) * (size_t)nq * ldb));
  SplitPtrs s{};
  s.xh = cosine ? db->cos_half.as<uint16_t>() : pl.h.as<uint16_t>();
  s.qh = qh;
  s.ldxb = ldb;
  s.ldqb = ldb;
  s.kb = ldb;
  if (bf16) {
    split_bf16(ctx, dq, nq, db->d, db->ld, qh, nullptr, ldb, qnh, qnr, nullptr);
    return s;
  }
  float *qsc = static_cast<float *>(ctx->scratch_ptr("flat.qscale", sizeof(float) * (size_t)nq));
  half_queries(ctx, dq, nq, db->d, db->ld, qh, ldb, qsc, qnh, qnr);
  s.qsc = qsc;
  s.xmax = cosine ? nullptr : pl.state.as<uint32_t>() + 3;
  return s;
}

// top-k over a resident database for queries already on the device
bool flat_topk_device(vsk_ctx *ctx, const vsk_db *db, const float *dq,
                      int64_t nq, int32_t k, int32_t metric, uint64_t *best,
                      ScreenDeferred *defer) {
  // a small problem (at most 2^28 query x row x dimension terms, some 20 us
  // of exact VALU work) is cheaper by the exact sequential scan alone than
  // by the screen's fixed chain of launches and its check read-back
  const bool screen = !ctx->flat_no_screen && screen_applies(metric, k);
  if (screen && !ctx->flat_force_screen &&
      (ctx->exact_only || (double)nq * (double)db->n * (double)db->d <= 268435456.0)) {
    approx_topk(ctx, db, dq, nq, k, exact_metric(metric), best, 3);
    return true;
  }
  if (screen && screen_plane_ok(ctx, db, metric)) {
    screen_topk(ctx, db, dq, nq, k, metric, best, defer);
    return true;
  }
  if (screen) {
    // cosine over rows whose norms the screen's bound cannot cover, or no
    // memory for the plane: the exact scan
    approx_topk(ctx, db, dq, nq, k, exact_metric(metric), best, 3);
    return true;
  }
  approx_topk(ctx, db, dq, nq, k, metric, best, 3);
  return false;
}

void approx_topk(vsk_ctx *ctx, const vsk_db *db, const float *dq, int64_t nq,
                 int32_t k, int32_t metric, uint64_t *best, int passes,
                 float *qnh, float *qnr, int64_t max_growth) {
  int64_t cap = passes == 1 ? screen_cap(k) : default_cap(k);
  // The screen at up to 1,024 queries: four times the slots its chunks are
  // expected to fill.  With screen_cap's two times, a launch of few query
  // tiles spreads a query's slots over some 56 workgroups, about 18
  // candidates in 36 slots each, and of 333 queries one or two overflowed:
  // the call ran again, its chunks re-scanned (200,003 x 384, k = 50:
  // 1.52 ms a call, with room 0.37, and 0.28 since no workgroups are launched
  // for absent query tiles).
  if (passes == 1 && nq <= 1024 && ctx->max_tile_bytes <= 0) {
    // (whole row tiles, so that every chunk starts on one)
    cap = std::max<int64_t>(cap, std::min<int64_t>(ceil_div(32 * (int64_t)k, 256) * 256, 16384));
  }
  // few queries by the exact scan: every row's key in one dense chunk, which
  // saves a second scan and selection (a first chunk of cap rows fills a
  // fraction of the chip: 100,000 x 768, one query, 93 of 253 us went there);
  // where the keys, written and read, are no more traffic than the rows, and
  // up to 32 MB of them, so that they stay in the memory-side cache
  if (passes != 1 && metric_is_valu(metric) && k <= VSK_SPLIT_K && cap < db->n &&
      4 * nq <= db->ld && nq * db->n <= (int64_t)1 << 22 &&
      (ctx->max_tile_bytes <= 0 || nq * db->n * 8 <= ctx->max_tile_bytes))
    cap = db->n;
  const int64_t qb = query_batch(ctx, nq, cap);
  for (int64_t b0 = 0; b0 < nq; b0 += qb) {
    const int64_t nb = nq - b0 < qb ? nq - b0 : qb;
    const float *qbat = dq + b0 * db->ld;
    if (metric == METRIC_COS_EXACT) ensure_seq_norms(ctx, db);
    // (a single query's cosine norm is summed by its scan)
    float *qa = metric == METRIC_COS_EXACT && nb == 1
                    ? nullptr
                    : q_aux(ctx, qbat, nb, db->d, db->ld, metric);
    FlatArgs base{};
    base.X = db->x.as<float>();
    base.ldx = db->ld;
    base.Q = qbat;
    base.ldq = db->ld;
    base.xaux = x_aux(db, metric);
    base.qaux = qa;
    base.kdim = db->ld;
    base.nq = (int32_t)nb;
    base.metric = metric;
    const bool x3 = use_bf16x3(ctx, metric);
    SplitPtrs sp{};
    if (x3 && passes == 1) {
      sp = make_half(ctx, db, qbat, nb, metric, qnh + b0, qnr + b0);
      if (metric == VSK_METRIC_COSINE) base.xaux = db->cos_inv.as<float>();
    } else if (x3) {
      sp = make_split(ctx, db, qbat, nb, true, nullptr, nullptr);
    }
    ScanFn scan = [&](const ScanRequest &r) {
      FlatArgs a = base;
      a.r0 = r.r0;
      a.r1 = r.r1;
      a.thresh = r.thresh;
      a.active = r.active;
      a.cand = r.cand;
      a.words = r.cand32;
      a.cap = r.cap;
      a.counts = r.counts;
      if (x3 && passes == 1) {
        a.seg_n = r.dense ? nullptr : r.seg_n;
        launch_flat_screen(ctx, a, sp, r.dense ? MODE_DENSE : MODE_FILTER, r.seg_nseg,
                           r.seg_stride);
      }
      else if (x3)
        launch_flat_bf16x3(ctx, a, sp, r.dense ? MODE_DENSE : MODE_FILTER, passes);
      else
        launch_flat(ctx, a, r.dense ? MODE_DENSE : MODE_FILTER, nullptr);
    };
    progressive_topk(ctx, nb, db->n, k, cap, scan, best + b0 * k,
                     "flat_select", max_growth, nullptr, passes == 1 || metric_is_valu(metric));
  }
}

// a row filter's rows as a database of their own: row t = rows[t] of db,
// with its norms (the same values, so the filtered search ranks as the
// whole database does)
__global__ void k_gather_db_rows(const float *X, const float *sq, const float *nrm, int32_t ld,
                                 const int32_t *rows, int64_t m, float *out, float *osq,
                                 float *onrm) {
  const int lane = threadIdx.x & 63;
  for (int64_t t = blockIdx.x * 4 + (threadIdx.x >> 6); t < m; t += (int64_t)gridDim.x * 4) {
    const int64_t r = rows[t];
    for (int j = lane; j < ld; j += 64) out[t * ld + j] = X[r * ld + j];
    if (lane == 0) {
      osq[t] = sq[r];
      onrm[t] = nrm[r];
    }
  }
}

}  // namespace vsk

using namespace vsk;

extern "C" {

static vsk_status search_flat_filtered_body(vsk_ctx *ctx, const vsk_db *db, const float *q,
                                    int64_t nq, int32_t k, int32_t metric,
                                    const uint32_t *allow, int64_t allow_bits,
                                    float *out_dist, int64_t *out_ids) {
  if (!allow && allow_bits == 0)
    return vsk_search_flat(ctx, db, q, nq, k, metric, out_dist, out_ids);
  VSK_API_BEGIN(ctx);
  VSK_REQUIRE(db, VSK_ERR_INVALID_ARGUMENT, "db is null");
  VSK_REQUIRE(metric_valid(metric), VSK_ERR_INVALID_ARGUMENT, "unknown metric");
  VSK_REQUIRE(nq > 0, VSK_ERR_EMPTY_INPUT, "no queries");
  VSK_REQUIRE(q && out_dist && out_ids, VSK_ERR_INVALID_ARGUMENT, "null buffer");
  VSK_REQUIRE(k >= 1, VSK_ERR_INVALID_ARGUMENT, "k must be >= 1");
  VSK_REQUIRE(k <= VSK_MAX_K, VSK_ERR_INVALID_BUFFER_SIZE, "k exceeds VSK_MAX_K");
  VSK_REQUIRE(nq <= 0x7FFFFFFFll, VSK_ERR_INVALID_BUFFER_SIZE, "too many queries");
  VSK_REQUIRE(allow && allow_bits >= 0, VSK_ERR_INVALID_ARGUMENT,
              "row filter: null bitmap or negative size");
  CallScope cs(ctx);
  for (auto &rec : ctx->screen_redo) rec.clear();
  // the rows the filter keeps, ascending (so ties still go to the lower row)
  const int64_t nbits = allow_bits < db->n ? allow_bits : db->n;
  std::vector<uint32_t> bits((size_t)ceil_div(nbits, 32));
  if (!bits.empty()) {
    VSK_HIP(hipMemcpyAsync(bits.data(), allow, sizeof(uint32_t) * bits.size(), hipMemcpyDefault,
                           ctx->stream));
    stream_sync(ctx);
  }
  std::vector<int32_t> rows;
  for (int64_t r = 0; r < nbits; ++r)
    if ((bits[(size_t)(r >> 5)] >> (r & 31)) & 1u) rows.push_back((int32_t)r);
  const int64_t m = (int64_t)rows.size();
  OutputStage od(ctx, out_dist, sizeof(float) * (size_t)nq * k, "out.dist");
  OutputStage oi(ctx, out_ids, sizeof(int64_t) * (size_t)nq * k, "out.ids");
  uint64_t *best = static_cast<uint64_t *>(
      ctx->scratch_ptr("flat.best", sizeof(uint64_t) * (size_t)nq * k));
  vsk_db sub;  // (freed after the call's synchronisation below)
  bool final_keys = true;
  int64_t *id_map = nullptr;
  if (m == 0) {
    fill_u64(ctx, best, nq * (int64_t)k, VSK_KEY_NONE);  // nothing passes
  } else {
    sub.n = m;
    sub.d = db->d;
    sub.ld = db->ld;
    sub.x.reserve(sizeof(float) * (size_t)m * db->ld);
    sub.sqnorm.reserve(sizeof(float) * (size_t)m);
    sub.norm.reserve(sizeof(float) * (size_t)m);
    int32_t *drows = static_cast<int32_t *>(
        ctx->scratch_ptr("flat.frows", sizeof(int32_t) * (size_t)m));
    id_map = static_cast<int64_t *>(ctx->scratch_ptr("flat.fmap", sizeof(int64_t) * (size_t)m));
    std::vector<int64_t> map(rows.begin(), rows.end());
    VSK_HIP(hipMemcpyAsync(drows, rows.data(), sizeof(int32_t) * (size_t)m,
                           hipMemcpyHostToDevice, ctx->stream));
    VSK_HIP(hipMemcpyAsync(id_map, map.data(), sizeof(int64_t) * (size_t)m,
                           hipMemcpyHostToDevice, ctx->stream));
    {
      KernelTimer t(ctx, "flat_filter_gather");
      const int64_t g = ceil_div(m, 4);
      k_gather_db_rows<<<(unsigned)(g < 65535 * 16 ? g : 65535 * 16), 256, 0, ctx->stream>>>(
          db->x.as<float>(), db->sqnorm.as<float>(), db->norm.as<float>(), db->ld, drows, m,
          sub.x.as<float>(), sub.sqnorm.as<float>(), sub.norm.as<float>());
      check_launch("flat_filter_gather");
    }
    const float *dq = rows_to_device_padded(ctx, q, nq, db->d, db->ld, "flat.q");
    final_keys = flat_topk_device(ctx, &sub, dq, nq, k, metric, best);
    // (the host vectors above must outlive their copies)
    stream_sync(ctx);
  }
  decode_keys(ctx, best, nq * (int64_t)k, metric == VSK_METRIC_L2 && !final_keys, id_map,
              od.ptr<float>(), oi.ptr<int64_t>());
  od.copy_back();
  oi.copy_back();
  cs.finish();
  VSK_API_END(ctx);
}

// top-k overflow is checked at the call's end (topk_call)
vsk_status vsk_search_flat_filtered(vsk_ctx *ctx, const vsk_db *db, const float *q,
                                    int64_t nq, int32_t k, int32_t metric,
                                    const uint32_t *allow, int64_t allow_bits,
                                    float *out_dist, int64_t *out_ids) {
  return topk_call(ctx, [&] { return search_flat_filtered_body(ctx, db, q, nq, k, metric, allow, allow_bits, out_dist, out_ids); });
}

static vsk_status search_flat_body(vsk_ctx *ctx, const vsk_db *db, const float *q,
                           int64_t nq, int32_t k, int32_t metric,
                           float *out_dist, int64_t *out_ids) {
  VSK_API_BEGIN(ctx);
  VSK_REQUIRE(db, VSK_ERR_INVALID_ARGUMENT, "db is null");
  VSK_REQUIRE(metric_valid(metric), VSK_ERR_INVALID_ARGUMENT,
              "unknown metric");
  VSK_REQUIRE(nq > 0, VSK_ERR_EMPTY_INPUT, "no queries");
  VSK_REQUIRE(q && out_dist && out_ids, VSK_ERR_INVALID_ARGUMENT,
              "null buffer");
  VSK_REQUIRE(k >= 1, VSK_ERR_INVALID_ARGUMENT, "k must be >= 1");
  VSK_REQUIRE(k <= VSK_MAX_K, VSK_ERR_INVALID_BUFFER_SIZE,
              "k exceeds VSK_MAX_K");
  VSK_REQUIRE(nq <= 0x7FFFFFFFll, VSK_ERR_INVALID_BUFFER_SIZE,
              "too many queries");
  CallScope cs(ctx);
  for (auto &rec : ctx->screen_redo) rec.clear();
  const float *dq = rows_to_device_padded(ctx, q, nq, db->d, db->ld, "flat.q");
  uint64_t *best = static_cast<uint64_t *>(
      ctx->scratch_ptr("flat.best", sizeof(uint64_t) * (size_t)nq * k));
  // the screen's bound check is read with the call's synchronisation
  ScreenDeferred defer;
  const bool final_keys = flat_topk_device(ctx, db, dq, nq, k, metric, best, &defer);
  OutputStage od(ctx, out_dist, sizeof(float) * (size_t)nq * k, "out.dist");
  OutputStage oi(ctx, out_ids, sizeof(int64_t) * (size_t)nq * k, "out.ids");
  decode_keys(ctx, best, nq * (int64_t)k, metric == VSK_METRIC_L2 && !final_keys,
              nullptr, od.ptr<float>(), oi.ptr<int64_t>());
  od.copy_back();
  oi.copy_back();
  cs.finish();
  // queries that failed the bound (near ties) are redone now and the
  // results written again; an overflowed top-k reruns the whole call
  if (!ctx->topk_overflowed && screen_finish(ctx, db, dq, k, metric, best, defer)) {
    decode_keys(ctx, best, nq * (int64_t)k, false, nullptr, od.ptr<float>(),
                oi.ptr<int64_t>());
    od.copy_back();
    oi.copy_back();
    cs.finish();
  }
  VSK_API_END(ctx);
}

// top-k overflow is checked at the call's end (topk_call)
vsk_status vsk_search_flat(vsk_ctx *ctx, const vsk_db *db, const float *q,
                           int64_t nq, int32_t k, int32_t metric,
                           float *out_dist, int64_t *out_ids) {
  return topk_call(ctx, [&] { return search_flat_body(ctx, db, q, nq, k, metric, out_dist, out_ids); });
}

vsk_status vsk_distances(vsk_ctx *ctx, const vsk_db *db, const float *q,
                         int64_t nq, int32_t metric, float *out) {
  VSK_API_BEGIN(ctx);
  VSK_REQUIRE(db, VSK_ERR_INVALID_ARGUMENT, "db is null");
  VSK_REQUIRE(metric_valid(metric), VSK_ERR_INVALID_ARGUMENT,
              "unknown metric");
  VSK_REQUIRE(nq > 0, VSK_ERR_EMPTY_INPUT, "no queries");
  VSK_REQUIRE(q && out, VSK_ERR_INVALID_ARGUMENT, "null buffer");
  VSK_REQUIRE(nq <= 0x7FFFFFFFll, VSK_ERR_INVALID_BUFFER_SIZE,
              "too many queries");
  CallScope cs(ctx);
  const float *dq = rows_to_device_padded(ctx, q, nq, db->d, db->ld, "flat.q");
  OutputStage om(ctx, out, sizeof(float) * (size_t)nq * db->n, "out.matrix");
  FlatArgs a{};
  a.X = db->x.as<float>();
  a.ldx = db->ld;
  a.Q = dq;
  a.ldq = db->ld;
  a.kdim = db->ld;
  a.nq = (int32_t)nq;
  a.r0 = 0;
  a.r1 = db->n;
  a.metric = metric;
  a.mat = om.ptr<float>();
  a.ldm = db->n;
  // Every metric of the reference's CPU path is evaluated as it evaluates
  // it, on the exact VALU kernel: L2 and L2^2 sum (q - x)^2 in dimension
  // order (the norm expansion |q|^2 + |x|^2 - 2 q.x of an MFMA path cancels
  // for close pairs: a duplicate row would get sqrt of the rounding error,
  // not 0); cosine, normalised cosine and dot sum q.x in dimension order,
  // cosine with the sequential norms.  The matrix is then the reference's
  // bit for bit, and exactly symmetric when the rows are the queries.
  if (exact_metric(metric) >= 0) {
    a.metric = exact_metric(metric);
    if (metric == VSK_METRIC_COSINE) {
      ensure_seq_norms(ctx, db);
      a.xaux = x_aux(db, METRIC_COS_EXACT);
      if (nq > 1) a.qaux = q_aux(ctx, dq, nq, db->d, db->ld, METRIC_COS_EXACT);
    }
  } else {
    a.xaux = x_aux(db, metric);
    a.qaux = q_aux(ctx, dq, nq, db->d, db->ld, metric);
  }
  if (use_bf16x3(ctx, a.metric))
    launch_flat_bf16x3(ctx, a, make_split(ctx, db, dq, nq, true, nullptr, nullptr),
                       MODE_MATRIX);
  else
    launch_flat(ctx, a, MODE_MATRIX, nullptr);
  om.copy_back();
  cs.finish();
  VSK_API_END(ctx);
}

}  // extern "C"
