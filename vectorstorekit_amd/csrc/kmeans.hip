// kmeans.hip -- k-means on the GPU as KMeansClustering.cluster runs it
// (Clustering/KMeansClustering.swift:48-113): the trainer of IVF coarse
// centroids (Indexes/IVFIndex.swift:397-446) and of PQ codebooks
// (Quantization/ProductQuantizer.swift:270-324).
//
// One Lloyd iteration is
//   assignment  each row's nearest centroid under the sequential sqrt-L2 of
//               :421-428 (strict '<', :271-295) and its distance: the bf16
//               screen with a proven bound and an exact recomputation of the
//               winner (flat_screen.hip, screen_argmin) when the problem is
//               large, else the exact VALU argmin scan (flat.hip);
//   inertia     distances.reduce(0, +) (:97): one wave adds the distances in
//               row order, so the fp32 rounding is the reference's;
//   grouping    a stable LSD radix pass per 4-bit digit of the cluster id
//               lists the rows of every cluster in row order;
//   update      one wave per (cluster, 64 columns) adds its rows' values in
//               that order, x * weight then +=, and divides by the fp32
//               count (:342-380), so every centroid is bit-identical to the
//               reference's sequential loop.
// Empty clusters are refilled on the device from a seeded draw (the
// reference's draw, :374, is unseeded).  The inertia is summed on a second
// stream while the next iteration already runs; the host reads it back
// (pinned memory) and tests convergence (|inertia - previous| < tolerance,
// :98).  An iteration started past convergence writes only the other halves
// of the double-buffered centroids, assignments and distances, and is
// dropped.
//
// k-means++ (:209-259) picks each next centroid with probability
// proportional to D(x)^2, D the distance to the nearest chosen centroid.  The
// reference's weights are D^2 / sum(D) (:237), which is not a distribution,
// and its cumulative fp32 sum is sequential over all rows per pick.  Here the
// weights are D^2 as 32-bit fixed point of D^2 / max D^2 (exact integer
// sums, so any summation order gives the same draw) and the draw is
// Int.random(in: 0..<total) from one SeedableRNG(seed) stream that also drew
// the first row.  (The reference reseeds each pick with seed + picks so far,
// :241; an LCG's first output is affine in its seed, which correlates those
// draws from pick to pick.)  All k picks run on the device.
#include <unordered_map>
#include <vector>

#include "flat.hpp"

namespace vsk {

// ---------------------------------------------------------------------------
// SeedableRNG (:480-491) and Swift's bounded draw (RandomNumberGenerator.
// next(upperBound:), Lemire's nearly-divisionless method, arXiv:1805.10941)
// ---------------------------------------------------------------------------
__host__ __device__ inline uint64_t swift_lcg(uint64_t &s) {
  s = s * 2862933555777941757ull + 3037000493ull;
  return s;
}
__host__ __device__ inline uint64_t mul_hi64(uint64_t a, uint64_t b) {
#ifdef __HIP_DEVICE_COMPILE__
  return __umul64hi(a, b);
#else
  return (uint64_t)(((unsigned __int128)a * b) >> 64);
#endif
}
__host__ __device__ inline uint64_t swift_bounded(uint64_t &s, uint64_t bound) {
  uint64_t r = swift_lcg(s);
  uint64_t lo = r * bound;
  if (lo < bound) {
    const uint64_t t = (0 - bound) % bound;
    while (lo < t) {
      r = swift_lcg(s);
      lo = r * bound;
    }
  }
  return mul_hi64(r, bound);
}

// ---------------------------------------------------------------------------
// inertia: the fp32 sum of n values in index order, by one wave.  The wave
// copies blocks of 4096 values into LDS with coalesced loads (the next
// block's loads in flight meanwhile), and lane 0 adds each block in order
// from 16-byte LDS reads: the adds form one dependent chain with no
// cross-lane moves in it.  v must be 16-byte aligned.
// ---------------------------------------------------------------------------
constexpr int SS_BLOCK = 4096;  // values per LDS block (16 KB)
typedef float ss_f4 __attribute__((ext_vector_type(4)));
__global__ __launch_bounds__(64) void k_seq_sum(const float *v, int64_t n,
                                                float *out) {
  __shared__ ss_f4 buf[SS_BLOCK / 4];
  const int lane = threadIdx.x;
  const int64_t nb = n / SS_BLOCK;  // whole blocks
  const ss_f4 *src = reinterpret_cast<const ss_f4 *>(v);
  ss_f4 r[SS_BLOCK / 256];
  if (nb > 0) {
#pragma unroll
    for (int u = 0; u < SS_BLOCK / 256; ++u) r[u] = src[u * 64 + lane];
  }
  float s = 0.f;
  for (int64_t b = 0; b < nb; ++b) {
#pragma unroll
    for (int u = 0; u < SS_BLOCK / 256; ++u) buf[u * 64 + lane] = r[u];
    __syncthreads();
    if (b + 1 < nb) {
      const ss_f4 *nx = src + (b + 1) * (SS_BLOCK / 4);
#pragma unroll
      for (int u = 0; u < SS_BLOCK / 256; ++u) r[u] = nx[u * 64 + lane];
    }
    if (lane == 0) {
      for (int i = 0; i < SS_BLOCK / 4; ++i) {
        const ss_f4 t = buf[i];
        s = s + t.x;
        s = s + t.y;
        s = s + t.z;
        s = s + t.w;
      }
    }
    __syncthreads();
  }
  if (lane == 0) {
    for (int64_t i = nb * SS_BLOCK; i < n; ++i) s = s + v[i];
    out[0] = s;
  }
}

// ---------------------------------------------------------------------------
// grouping: stable LSD radix sort of (cluster, row) by cluster, 4-bit digits.
// A block owns GR_B consecutive rows, GR_PER consecutive ones per thread, so
// the order inside a digit is thread order then row order: the row order.
// ---------------------------------------------------------------------------
constexpr int GR_T = 256, GR_PER = 8, GR_B = GR_T * GR_PER;

// cnt[g][t] = rows of thread t in this block with digit g
__device__ inline void grp_count(const int32_t *keys, int64_t n, int shift,
                                 int32_t (*cnt)[GR_T]) {
  const int t = threadIdx.x;
#pragma unroll
  for (int g = 0; g < 16; ++g) cnt[g][t] = 0;
  const int64_t r0 = (int64_t)blockIdx.x * GR_B + (int64_t)t * GR_PER;
#pragma unroll
  for (int j = 0; j < GR_PER; ++j) {
    const int64_t r = r0 + j;
    if (r < n) cnt[(keys[r] >> shift) & 15][t] += 1;
  }
}

// hist[g * nb + b] = rows of block b with digit g
__global__ __launch_bounds__(GR_T) void k_grp_hist(const int32_t *keys, int64_t n,
                                                   int shift, int32_t *hist) {
  __shared__ int32_t cnt[16][GR_T];
  grp_count(keys, n, shift, cnt);
  __syncthreads();
  // thread t sums 16 entries of digit t/16; the 16 threads of a digit share
  // one wave quarter and reduce by shuffles
  const int t = threadIdx.x, g = t >> 4, part = t & 15;
  int32_t s = 0;
#pragma unroll
  for (int i = 0; i < 16; ++i) s += cnt[g][part * 16 + i];
#pragma unroll
  for (int m = 8; m > 0; m >>= 1) s += __shfl_xor(s, m, 16);
  if (part == 0) hist[(int64_t)g * gridDim.x + blockIdx.x] = s;
}

// in-place exclusive scan of m int32 values by one block of 1024 threads
__global__ __launch_bounds__(1024) void k_scan_excl(int32_t *h, int64_t m) {
  __shared__ int32_t wsum[16];
  __shared__ int32_t carry_s;
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  if (t == 0) carry_s = 0;
  __syncthreads();
  for (int64_t base = 0; base < m; base += 1024) {
    const int64_t i = base + t;
    const int32_t v = i < m ? h[i] : 0;
    int32_t incl = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int32_t u = __shfl_up(incl, o);
      if (lane >= o) incl += u;
    }
    if (lane == 63) wsum[w] = incl;
    __syncthreads();
    int32_t before = carry_s;
    for (int j = 0; j < w; ++j) before += wsum[j];
    if (i < m) h[i] = before + incl - v;
    __syncthreads();
    if (t == 1023) carry_s = before + incl;
    __syncthreads();
  }
}

// scatter rows to hist-scanned positions, stable within the block
__global__ __launch_bounds__(GR_T) void k_grp_scatter(
    const int32_t *keys, const int32_t *vals, int64_t n, int shift,
    const int32_t *hist, int32_t *keys_out, int32_t *vals_out) {
  __shared__ int32_t cnt[16][GR_T];
  __shared__ int32_t wtot[16][GR_T / 64];
  grp_count(keys, n, shift, cnt);
  __syncthreads();
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  // exclusive prefix of cnt[g][.] over the threads, plus the block's base
  int32_t incl[16];
#pragma unroll
  for (int g = 0; g < 16; ++g) {
    int32_t x = cnt[g][t];
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int32_t u = __shfl_up(x, o);
      if (lane >= o) x += u;
    }
    incl[g] = x;
    if (lane == 63) wtot[g][w] = x;
  }
  __syncthreads();
#pragma unroll
  for (int g = 0; g < 16; ++g) {
    int32_t before = hist[(int64_t)g * gridDim.x + blockIdx.x];
    for (int j = 0; j < w; ++j) before += wtot[g][j];
    cnt[g][t] = before + incl[g] - cnt[g][t];  // this thread's next slot
  }
  // (each thread reads and writes only its own column of cnt)
  const int64_t r0 = (int64_t)blockIdx.x * GR_B + (int64_t)t * GR_PER;
#pragma unroll
  for (int j = 0; j < GR_PER; ++j) {
    const int64_t r = r0 + j;
    if (r < n) {
      const int32_t key = keys[r];
      const int g = (key >> shift) & 15;
      const int32_t pos = cnt[g][t];
      cnt[g][t] = pos + 1;
      keys_out[pos] = key;
      vals_out[pos] = vals ? vals[r] : (int32_t)r;
    }
  }
}

__global__ void k_count_clusters(const int32_t *assign, int64_t n, int32_t *counts) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    atomicAdd(&counts[assign[i]], 1);
}

// ---------------------------------------------------------------------------
// update: one wave per (cluster c = blockIdx.x, columns 64 * blockIdx.y ..).
// The members' row numbers are read 64 at a time; rows are loaded 16 ahead
// of the sequential adds.  cent[c][j] = sum / count for j < d, 0 in the
// padding; cntf[c] = the fp32 count (or weight sum) the reference divides
// by.  A cluster whose count is not > 0 keeps zeros (the host refills it).
// ---------------------------------------------------------------------------
constexpr int MU = 16;
__global__ __launch_bounds__(64) void k_cluster_means(
    const float *x, int64_t ld, int32_t d, const int32_t *order,
    const int32_t *off, const int32_t *counts, const float *weights,
    float *cent, float *cntf) {
#pragma clang fp contract(off)
  const int lane = threadIdx.x;
  const int64_t c = blockIdx.x;
  const int64_t col = (int64_t)blockIdx.y * 64 + lane;
  const bool colok = col < ld;
  const int32_t m = counts[c], o = off[c];
  float s = 0.f, cw = 0.f;
  for (int32_t p0 = 0; p0 < m; p0 += 64) {
    const int32_t idx = p0 + lane < m ? order[o + p0 + lane] : 0;
    const float wl = weights ? weights[idx] : 1.f;
    const int32_t mm = m - p0 < 64 ? m - p0 : 64;
    for (int32_t j = 0; j < mm; j += MU) {
      float v[MU];
      float wv[MU];
#pragma unroll
      for (int u = 0; u < MU; ++u) {
        // rows past mm load row idx of lane 0's slot (in bounds), unused
        const int32_t row = __builtin_amdgcn_readlane(idx, (j + u) & 63);
        v[u] = colok ? x[(int64_t)row * ld + col] : 0.f;
        wv[u] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(wl), (j + u) & 63));
      }
#pragma unroll
      for (int u = 0; u < MU; ++u) {
        if (j + u < mm) {
          if (weights) {
            s = s + v[u] * wv[u];
            cw = cw + wv[u];
          } else {
            s = s + v[u];
          }
        }
      }
    }
  }
  // fp32 count += 1 saturates at 2^24 (2^24 + 1 rounds back to it)
  const float cnt = weights ? cw : (m > (1 << 24) ? 16777216.f : (float)m);
  if (colok) cent[c * ld + col] = (col < d && cnt > 0.f) ? s / cnt : 0.f;
  if (blockIdx.y == 0 && lane == 0) cntf[c] = cnt;
}

// empty clusters (fp32 count not > 0) in ascending order each take row
// Int.random(in: 0..<n) of the SeedableRNG stream whose state is *rng: one
// wave, every lane draws the same sequence, the lanes copy the row
__global__ __launch_bounds__(64) void k_refill_empty(const float *cntf, int32_t k,
                                                     const float *x, int64_t ld, int32_t d,
                                                     int64_t n, uint64_t *rng, float *cent) {
  const int lane = threadIdx.x;
  uint64_t st = *rng;
  for (int32_t c0 = 0; c0 < k; c0 += 64) {
    const int32_t c = c0 + lane;
    const bool empty = c < k && !(cntf[c] > 0.f);
    uint64_t mask = __builtin_amdgcn_ballot_w64(empty);
    while (mask) {
      const int b = __builtin_ctzll(mask);
      mask &= mask - 1;
      const int64_t r = (int64_t)swift_bounded(st, (uint64_t)n);
      const float *src = x + r * ld;
      float *dst = cent + (int64_t)(c0 + b) * ld;
      for (int32_t j = lane; j < d; j += 64) dst[j] = src[j];
    }
  }
  if (lane == 0) *rng = st;
}

__global__ void k_gather_rows_i64(const float *src, int64_t ld, const int64_t *rows,
                                  int64_t m, float *dst) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < m * ld;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t r = i / ld, c = i - r * ld;
    dst[i] = src[rows[r] * ld + c];
  }
}

// ---------------------------------------------------------------------------
// k-means++ on the device
// ---------------------------------------------------------------------------
constexpr int KP_T = 256;       // threads of a block, rows of an update block
constexpr int KP_B = 4 * KP_T;  // rows of a weight-sum chunk
constexpr int KP_BLOCKS = 512;  // weight-sum blocks at most
constexpr int KP_SLOTS = 64;    // max slots per pick (a power of two, one wave's lanes)
constexpr int KP_TILE = 33 * KP_T;  // floats of the update's row tile
// From these bytes of codes or rows on, the triangle test first
// (k_kpp_update_queued).  us a pick, without and with it: 1M x 768 (732 MB of
// codes), 4,096 picks of 256 clusters 182 and 79, 512 of 512 194 and 192; 4M x
// 128, 2,048 of 128 137 and 75; 1.5M x 32, 512 of 64 55 and 49, 512 of 512 54
// and 55; 350,000 x 768 (257 MB), 1,024 of 64 81 and 69, 1,024 of 1,024 77 and
// 83; but 1M x 128, 4,096 of 4,096 46 and 58; 100,000 x 128 16 and 23.
constexpr size_t KP_NEAR = (size_t)256 << 20;
constexpr int64_t KP_NEAR_ROWS = 5 << 18;
// rows of 64 that make the int8 screen of k_kpp_update_queued worth its wait
constexpr int KP_FEW = 16;

// The rows as int8 for the update's screen: x_i = s_i q_i + residual, s_i =
// max |x_ij| / 127, q_ij the nearest integer; par[i] = (s_i, |s_i q_i|^2, a
// bound e_i on the residual's norm, 0).  A row with a component that is not
// finite has e_i = +inf, which the screen never decides.  Codes: 16-byte
// chunk ch of row i at dword 4 ((i / 64 * nch + ch) * 64 + i % 64), so that
// 64 rows' loads of one chunk are one kilobyte.  One wave per row.
__global__ __launch_bounds__(KP_T) void k_kpp_codes(const float *x, int64_t ld, int32_t d,
                                                    int64_t n, int32_t nch, uint32_t *codes,
                                                    float4 *par) {
  const int lane = threadIdx.x & 63;
  for (int64_t i = (int64_t)blockIdx.x * (KP_T / 64) + (threadIdx.x >> 6); i < n;
       i += (int64_t)gridDim.x * (KP_T / 64)) {
    const float *xi = x + i * ld;
    float mx = 0.f;
    bool bad = false;
    for (int32_t j = lane; j < d; j += 64) {
      const float v = fabsf(xi[j]);
      bad |= !(v <= 0x1.fffffep127f);
      mx = fmaxf(mx, v);
    }
  #pragma unroll
    for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
    bad = __ballot(bad) != 0;
    const float sc = bad ? 0.f : mx * (1.0f / 127.0f);
    const float inv = sc > 0.f ? 1.0f / sc : 0.f;  // (inf for a tiny sc: codes clamp)
    uint32_t qq = 0;  // (exact: at most 127^2 2^17)
    float rr = 0.f;
    uint32_t *out = codes + 4 * ((i >> 6) * nch * 64 + (i & 63));
    for (int32_t w = lane; w < 4 * nch; w += 64) {
      uint32_t pack = 0;
  #pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int32_t j = 4 * w + u;
        const float v = j < d ? xi[j] : 0.f;
        float c = bad ? 0.f : rintf(v * inv);
        c = fminf(fmaxf(c, -127.f), 127.f);  // (NaN of 0 * inf: -127, a larger residual)
        const float res = __builtin_fmaf(-sc, c, v);  // one rounding
        qq += (uint32_t)((int32_t)c * (int32_t)c);
        rr += res * res;
        pack |= ((uint32_t)(int32_t)c & 255u) << (8 * u);
      }
      out[256 * (w >> 2) + (w & 3)] = pack;
    }
  #pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      qq += __shfl_xor(qq, o);
      rr += __shfl_xor(rr, o);
    }
    if (lane == 0) {
      // e: the sums' and residuals' roundings are far below 2^-10 of it and
      // 2^-20 of the row's norm; an underflowed square adds at most 2^-60
      const float nx = sc * sqrtf((float)qq);
      const float e = sqrtf(rr) * (1.f + 0x1p-10f) + nx * 0x1p-20f + 0x1p-60f * sqrtf((float)d);
      par[i] = make_float4(sc, sc * sc * (float)qq, bad || !(e < 0x1p60f) ? __int_as_float(0x7f800000) : e,
                           0.f);
    }
  }
}

// cc[a] = |x_c - x_{chosen[a]}| for the picks a < r, c = chosen[r]: one
// wave per a, lanes over the coordinates.  Only the triangle test of
// k_kpp_update reads it, so any summation order with a small relative error
// serves (this one's is under (d / 64 + 11) 2^-25).
__global__ __launch_bounds__(256) void k_kpp_cc(const float *x, int64_t ld, int32_t d,
                                                const int64_t *chosen, int r, float *cc) {
#pragma clang fp contract(off)
  const int64_t c = chosen[r];
  if (c < 0) return;
  const int a = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (a >= r) return;  // wave-uniform
  const float *xc = x + c * ld, *xa = x + chosen[a] * ld;
  float s = 0.f;
  for (int32_t j = lane; j < d; j += 64) {
    const float t = xc[j] - xa[j];
    s = s + t * t;
  }
#pragma unroll
  for (int m = 32; m > 0; m >>= 1) s = s + __shfl_xor(s, m);
  if (lane == 0) cc[a] = sqrtf(s);
}

// Whether row i (distance dm to its nearest pick) may come nearer to row c:
// the int8 screen of k_kpp_update's comment
__device__ inline bool kpp_may_move(const uint4 *__restrict__ codes,
                                    const float4 *__restrict__ par, int64_t i, int64_t c,
                                    int32_t nch, float dm, float skipm) {
#pragma clang fp contract(off)
  const float4 pi = par[i], pc = par[c];
  const uint4 *qi = codes + (i >> 6) * nch * 64 + (i & 63);
  const uint4 *qc = codes + (c >> 6) * nch * 64 + (c & 63);
  int32_t dot = 0;
#pragma unroll 8
  for (int ch = 0; ch < nch; ++ch) {
    const uint4 a = qi[64 * ch], o = qc[64 * ch];
    dot = __builtin_amdgcn_sdot4((int)a.x, (int)o.x, dot, false);
    dot = __builtin_amdgcn_sdot4((int)a.y, (int)o.y, dot, false);
    dot = __builtin_amdgcn_sdot4((int)a.z, (int)o.z, dot, false);
    dot = __builtin_amdgcn_sdot4((int)a.w, (int)o.w, dot, false);
  }
  const float t = pi.y + pc.y;
  const float sq = (t - 2.0f * (pi.x * pc.x) * (float)dot) - 0x1p-20f * t;
  const float lb = (sqrtf(fmaxf(sq, 0.f)) - (pi.z + pc.z)) * (1.f - 0x1p-20f);
  return !(dm >= 0x1p-40f && dm <= 0x1p60f && t <= 0x1p100f && lb >= dm * skipm);
}

// D[i] = min(D[i], |x_i - x_c|) with c = chosen[r] (sequential sqrt-L2, as
// computeMinDistances, :401-419); the max over rows of D^2 lands in
// maxbits[(r + 1) * KP_SLOTS + s] for the KP_SLOTS slots s (non-negative
// floats order as their bits; spread so the atomics do not queue on one
// address).
//
// A block owns 256 rows, a thread one of them.  Most rows keep their D, and
// the int8 rows show it: |x_i - x_c| >= |s_i q_i - s_c q_c| - e_i - e_c, and
// the first term's square is |s_i q_i|^2 + |s_c q_c|^2 - 2 s_i s_c (q_i.q_c),
// the dot product exact in integers, the rest within 2^-20 of the two norms'
// sum.  A row whose bound is at least D skipm, skipm = 1 + (d + 4) 2^-22, is
// left alone: the sequential fp32 distance is within (d + 4) 2^-25 of the
// real one, so it would not be below D.  (Only for 2^-40 <= D <= 2^60 and
// norms below 2^100, where nothing under- or overflows enough to matter.)
// The screen reads d bytes a row where the distance reads 4 d, and 100,000
// rows' codes at 128 dims stay in the XCDs' L2s from pick to pick.  Measured
// at 100,000 x 128, 1,024 picks: 8.9 us a pick, against 30.7 us (and 3.7 us
// for the distances between the picks) with a triangle test against the
// nearest pick, which an uncovered cluster's rows never pass.
//
// The m rows that do need the distance are compacted in LDS and staged there
// in column chunks (coalesced), one lane then summing each row in coordinate
// order.  Late rounds leave a block a handful of rows and the kernel is a
// chain of memory latencies, so the chunk is as wide as the tile allows: 32
// columns for 256 rows up to 512 for 16 (a 128-dim row then takes one pass
// where 32-column chunks took four), the next chunk's loads in flight while
// one is summed.
__global__ __launch_bounds__(KP_T) void k_kpp_update(const float *__restrict__ x, int64_t ld,
                                                     int32_t d, int64_t n,
                                                     const int64_t *__restrict__ chosen, int r,
                                                     const uint4 *__restrict__ codes,
                                                     const float4 *__restrict__ par,
                                                     int32_t nch, float skipm,
                                                     float *__restrict__ D,
                                                     uint32_t *__restrict__ maxbits) {
#pragma clang fp contract(off)
  __shared__ float tile[KP_TILE];
  __shared__ float s_xc[512];
  __shared__ int32_t l_row[KP_T];
  __shared__ float l_dm[KP_T];
  __shared__ int32_t s_cnt[KP_T / 64];
  __shared__ uint32_t s_max[KP_T / 64];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int64_t row0 = (int64_t)blockIdx.x * KP_T;
  const int64_t c = chosen[r];
  const bool live = row0 + tid < n;
  const float dm = live ? D[row0 + tid] : 0.f;
  if (c < 0) return;  // an earlier pick found degenerate data
  const float *__restrict__ xc = x + c * ld;
  uint32_t b = 0;  // max D^2 bits seen by this thread
  const bool need = live && kpp_may_move(codes, par, row0 + tid, c, nch, dm, skipm);
  if (live && !need) b = __float_as_uint(dm * dm);
  const uint64_t mask = __ballot(need);
  if (lane == 0) s_cnt[w] = __popcll(mask);
  __syncthreads();
  int base = 0, m = 0;
#pragma unroll
  for (int j = 0; j < KP_T / 64; ++j) {
    if (j < w) base += s_cnt[j];
    m += s_cnt[j];
  }
  if (m > 0) {  // block-uniform
    if (need) {
      const int pos = base + (int)__builtin_amdgcn_mbcnt_hi(
                                 (uint32_t)(mask >> 32),
                                 __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
      l_row[pos] = tid;
      l_dm[pos] = dm;
    }
    // columns per chunk: rows rounded up to a power of two x columns = 8192
    const int sh = m <= 16 ? 9 : m <= 32 ? 8 : m <= 64 ? 7 : m <= 128 ? 6 : 5;
    const int cw = 1 << sh, stride = cw + 1;  // (odd: a lane per row reads without conflicts)
    __syncthreads();
    constexpr int NV = 8192 / KP_T;
    float v[NV];
    auto load = [&](int32_t j0) {
#pragma unroll
      for (int u = 0; u < NV; ++u) {
        const int e = u * KP_T + tid;
        const int rr = e >> sh, col = j0 + (e & (cw - 1));
        v[u] = rr < m && col < d ? x[(row0 + l_row[rr]) * ld + col] : 0.f;
      }
    };
    load(0);
    float s = 0.f;
    for (int32_t j0 = 0; j0 < d; j0 += cw) {
      if (j0 > 0) __syncthreads();  // the previous chunk has been read
#pragma unroll
      for (int u = 0; u < NV; ++u) {
        const int e = u * KP_T + tid;
        tile[(e >> sh) * stride + (e & (cw - 1))] = v[u];
      }
      for (int j = tid; j < cw && j0 + j < d; j += KP_T) s_xc[j] = xc[j0 + j];
      __syncthreads();
      if (j0 + cw < d) load(j0 + cw);
      if (tid < m) {
        const int jn = d - j0 < cw ? d - j0 : cw;
        const float *t = tile + tid * stride;
#pragma unroll 8
        for (int j = 0; j < jn; ++j) {
          const float e = t[j] - s_xc[j];
          s = s + e * e;
        }
      }
    }
    if (tid < m) {
      float old = l_dm[tid];
      const float dist = sqrtf(s);
      if (dist < old) {
        old = dist;
        D[row0 + l_row[tid]] = dist;
      }
      const uint32_t bw = __float_as_uint(old * old);
      b = bw > b ? bw : b;
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const uint32_t v = __shfl_xor(b, o);
    b = v > b ? v : b;
  }
  if (lane == 0) s_max[w] = b;
  __syncthreads();
  if (tid == 0) {
#pragma unroll
    for (int j = 0; j < KP_T / 64; ++j) b = s_max[j] > b ? s_max[j] : b;
    atomicMax(&maxbits[(r + 1) * KP_SLOTS + blockIdx.x % KP_SLOTS], b);
  }
}

// The same for codes that do not stay in the caches, which would be read
// from HBM on every pick long after most rows are covered: the triangle test
// comes first.  near[i] is the pick a that set D[i], and a row with
// |x_c - x_a| >= 2 D skipm is left alone, its code unread.  The exact distance
// is at least |x_c - x_a| - |x_i - x_a|, and (d + 4) 2^-22 exceeds the
// relative errors of the three computed distances taken together (a
// sequential one: under (d + 4) 2^-25; k_kpp_cc's: under (d / 64 + 11) 2^-25,
// counted twice), so the computed distance would not be below D (for 2^-60 <=
// D <= 2^60, where no sum under- or overflows enough to break the relative
// bounds).  Without codes (null) the triangle test stands alone.
//
// One wave a block strides over groups of 64 rows: few rows of a group need
// anything, so those that need the distance queue in LDS across the groups.
// 64 of them, or what is left at the end, are staged in column chunks as wide
// as the tile allows (32 columns for 64 rows, 512 for up to 4), the next
// chunk's loads in flight, and every lane sums its own row in order.
__global__ __launch_bounds__(64) void k_kpp_update_queued(
    const float *__restrict__ x, int64_t ld, int32_t d, int64_t n,
    const int64_t *__restrict__ chosen, int r, const uint4 *__restrict__ codes,
    const float4 *__restrict__ par, int32_t nch, float skipm, const float *__restrict__ cc,
    int32_t *__restrict__ near, float *__restrict__ D, uint32_t *__restrict__ maxbits) {
#pragma clang fp contract(off)
  constexpr int E = 2048;  // floats of a chunk
  __shared__ float tile[E + 64];
  __shared__ int64_t l_row[128];
  __shared__ float l_dm[128];
  const int64_t c = chosen[r];
  if (c < 0) return;  // an earlier pick found degenerate data
  const int lane = threadIdx.x;
  const float *__restrict__ xc = x + c * ld;
  uint32_t b = 0;  // max D^2 bits seen by this lane
  // the distances of the first m <= 64 queued rows
  auto run = [&](int m) {
    const int sh = m <= 4 ? 9 : m <= 8 ? 8 : m <= 16 ? 7 : m <= 32 ? 6 : 5;
    const int cw = 1 << sh, stride = cw + 1;
    float v[E / 64];
    auto load = [&](int32_t j0) {
#pragma unroll
      for (int u = 0; u < E / 64; ++u) {
        const int e = u * 64 + lane, rr = e >> sh, col = j0 + (e & (cw - 1));
        v[u] = rr < m && col < d ? x[l_row[rr] * ld + col] : 0.f;
      }
    };
    load(0);
    float s = 0.f;
    for (int32_t j0 = 0; j0 < d; j0 += cw) {
      if (j0 > 0) __syncthreads();  // the previous chunk has been read
#pragma unroll
      for (int u = 0; u < E / 64; ++u) {
        const int e = u * 64 + lane;
        tile[(e >> sh) * stride + (e & (cw - 1))] = v[u];
      }
      __syncthreads();
      if (j0 + cw < d) load(j0 + cw);
      if (lane < m) {
        const int jn = d - j0 < cw ? d - j0 : cw;
        const float *t = tile + lane * stride;
#pragma unroll 8
        for (int j = 0; j < jn; ++j) {
          const float e = t[j] - xc[j0 + j];
          s = s + e * e;
        }
      }
    }
    if (lane < m) {
      float dm = l_dm[lane];
      const float dist = sqrtf(s);
      if (dist < dm) {
        dm = dist;
        const int64_t i = l_row[lane];
        D[i] = dm;
        near[i] = r;
      }
      const uint32_t bw = __float_as_uint(dm * dm);
      b = bw > b ? bw : b;
    }
  };
  int cnt = 0;  // queued rows (wave-uniform)
  for (int64_t row0 = (int64_t)blockIdx.x * 64; row0 < n; row0 += (int64_t)gridDim.x * 64) {
    const int64_t i = row0 + lane;
    bool need = false;
    float dm = 0.f;
    if (i < n) {
      dm = D[i];
      const int32_t a = near[i];
      need = !(a >= 0 && dm >= 0x1p-60f && dm <= 0x1p60f && cc[a] >= 2.0f * dm * skipm);
    }
    // (a wait for a few rows' codes costs more than their distances: 10M x 32,
    // 512 picks of 64 clusters, late ones 133 us with it and 70 without)
    if (codes && __popcll(__ballot(need)) >= KP_FEW && need)
      need = kpp_may_move(codes, par, i, c, nch, dm, skipm);
    if (i < n && !need) {
      const uint32_t bw = __float_as_uint(dm * dm);
      b = bw > b ? bw : b;
    }
    const uint64_t mask = __ballot(need);
    if (need) {
      const int pos = cnt + (int)__builtin_amdgcn_mbcnt_hi(
                                (uint32_t)(mask >> 32),
                                __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
      l_row[pos] = i;
      l_dm[pos] = dm;
    }
    cnt += __popcll(mask);
    if (cnt >= 64) {
      __syncthreads();
      run(64);
      __syncthreads();
      if (lane < cnt - 64) {
        l_row[lane] = l_row[64 + lane];
        l_dm[lane] = l_dm[64 + lane];
      }
      cnt -= 64;
    }
  }
  if (cnt > 0) {
    __syncthreads();
    run(cnt);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const uint32_t v = __shfl_xor(b, o);
    b = v > b ? v : b;
  }
  if (lane == 0) atomicMax(&maxbits[(r + 1) * KP_SLOTS + blockIdx.x % KP_SLOTS], b);
}

// the max of pick r + 1's KP_SLOTS slots, through LDS to the whole block
__device__ inline float kpp_maxw(const uint32_t *maxbits, int r, uint32_t *sm) {
  if (threadIdx.x < 64) {
    uint32_t b = maxbits[(r + 1) * KP_SLOTS + threadIdx.x];
#pragma unroll
    for (int m = 32; m > 0; m >>= 1) {
      const uint32_t o = __shfl_xor(b, m);
      b = o > b ? o : b;
    }
    if (threadIdx.x == 0) *sm = b;
  }
  __syncthreads();
  return __uint_as_float(*sm);
}

// the 32-bit fixed-point weight of D^2 (exact: one correctly rounded
// division, an exact scaling, truncation)
__device__ inline uint64_t kpp_fixed(float dm, float maxw) {
  if (!(maxw > 0.f)) return 0;
  const float w = dm * dm;
  return (uint64_t)((double)w / (double)maxw * 4294967296.0);
}

__device__ inline uint64_t shfl_up_u64(uint64_t v, int o) {
  const uint32_t lo = __shfl_up((uint32_t)v, o), hi = __shfl_up((uint32_t)(v >> 32), o);
  return ((uint64_t)hi << 32) | lo;
}

// exclusive prefix over the block's threads of one uint64 per thread;
// *total receives the block's sum
__device__ uint64_t block_excl_u64(uint64_t v, uint64_t *wsum, uint64_t *total) {
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  uint64_t incl = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint64_t u = shfl_up_u64(incl, o);
    if (lane >= o) incl += u;
  }
  __syncthreads();
  if (lane == 63) wsum[w] = incl;
  __syncthreads();
  uint64_t before = 0, all = 0;
  for (int j = 0; j < (int)(blockDim.x >> 6); ++j) {
    if (j < w) before += wsum[j];
    all += wsum[j];
  }
  *total = all;
  return before + incl - v;
}

// pick r + 1: u = Int.random(in: 0..<total) from the SeedableRNG stream
// whose state is *rng; the chosen row is the first whose inclusive
// fixed-weight prefix exceeds u.  total = 0 (every row on a chosen centroid)
// is the reference's degenerateData (:235-237): chosen[r + 1] = -1.
//
// Every block sums the fixed weights of its m chunks of 1024 rows; the block
// that counts itself last in *done has them all and picks: one launch of 7.2
// us at 100,000 rows instead of a sum and a pick launch of 4.4 and 6.6 us.  m
// keeps the blocks to KP_BLOCKS, since their counts queue on one address: 4M
// rows with m = 1 took 55 us, now 20 (39 as two launches).  No
// fence is needed, and none is used (an agent-scope release writes back the
// XCD's whole L2): a block's sum goes out by a returning exchange at agent
// scope, its arrival is counted only after that returned, and the last block
// reads the sums by agent-scope loads.  No block waits for another.
__global__ __launch_bounds__(KP_T) void k_kpp_pick(uint64_t *bsum, int64_t nb, int32_t m,
                                                   const float *D, int64_t n,
                                                   const uint32_t *maxbits,
                                                   uint64_t *rng, int r, int64_t *chosen,
                                                   uint32_t *done) {
  __shared__ uint64_t wsum[KP_T / 64];
  __shared__ uint64_t s_base;
  __shared__ int64_t s_blk, s_row;
  __shared__ uint32_t s_mx;
  __shared__ bool s_last;
  const int t = threadIdx.x;
  const int64_t i0 = (int64_t)blockIdx.x * m * KP_B;
  float dv[KP_B / KP_T];
  auto load = [&](int64_t c0) {
#pragma unroll
    for (int u = 0; u < KP_B / KP_T; ++u) {
      const int64_t i = c0 + u * KP_T + t;
      dv[u] = i < n ? D[i] : 0.f;  // (a zero distance weighs 0)
    }
  };
  load(i0);
  uint64_t st = *rng;  // (only the last block writes it, after its count)
  if (chosen[r] < 0) {
    if (blockIdx.x == 0 && t == 0) chosen[r + 1] = -1;
    return;
  }
  const float maxw = kpp_maxw(maxbits, r, &s_mx);
  uint64_t f = 0;
  for (int32_t j = 0; j < m; ++j) {
    float cur[KP_B / KP_T];
#pragma unroll
    for (int u = 0; u < KP_B / KP_T; ++u) cur[u] = dv[u];
    if (j + 1 < m) load(i0 + (j + 1) * KP_B);
#pragma unroll
    for (int u = 0; u < KP_B / KP_T; ++u) f += kpp_fixed(cur[u], maxw);
  }
  uint64_t sum;
  (void)block_excl_u64(f, wsum, &sum);
  if (t == 0) {
    uint64_t old = __hip_atomic_exchange(&bsum[blockIdx.x], sum, __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("" : "+v"(old) : : "memory");  // the exchange has returned
    s_last = atomicAdd(done, 1u) == (uint32_t)nb - 1u;
  }
  __syncthreads();
  if (!s_last) return;
  // thread t takes the sums of a run of consecutive blocks, so one scan over
  // the threads gives the total and every run's prefix
  const int64_t per = (nb + KP_T - 1) / KP_T;
  const int64_t b0 = t * per, b1 = b0 + per < nb ? b0 + per : nb;
  auto sum_of = [&](int64_t b) -> uint64_t {
    return __hip_atomic_load(&bsum[b], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  uint64_t part = 0;
  for (int64_t b = b0; b < b1; ++b) part += sum_of(b);
  if (t == 0) {
    *done = 0;  // for the next pick's launch
    s_blk = -1;
    s_row = -1;
  }
  uint64_t total;
  uint64_t before = block_excl_u64(part, wsum, &total);
  if (total == 0) {
    if (t == 0) chosen[r + 1] = -1;
    return;
  }
  const uint64_t u = swift_bounded(st, total);  // (every thread draws the same)
  if (t == 0) *rng = st;
  // the block holding u
  if (before <= u && u < before + part) {
    for (int64_t b = b0; b < b1; ++b) {
      const uint64_t v = per == 1 ? part : sum_of(b);
      if (u < before + v) {
        s_blk = b;
        s_base = before;
        break;
      }
      before += v;
    }
  }
  __syncthreads();
  // the row inside it (a block is always found: the blocks' sums partition
  // [0, total); the test keeps a broken invariant from reading out of range)
  const int64_t blk = s_blk;
  if (blk < 0) {
    if (t == 0) chosen[r + 1] = -1;
    return;
  }
  // consecutive rows per thread, so that thread order is row order
  uint64_t chunk = s_base;
  for (int32_t j = 0; j < m; ++j) {
    const int64_t i1 = (blk * m + j) * KP_B + (int64_t)t * (KP_B / KP_T);
    uint64_t fx[KP_B / KP_T], mine = 0;
#pragma unroll
    for (int v = 0; v < KP_B / KP_T; ++v) {
      fx[v] = i1 + v < n ? kpp_fixed(D[i1 + v], maxw) : 0;
      mine += fx[v];
    }
    uint64_t tot2;
    uint64_t ex = chunk + block_excl_u64(mine, wsum, &tot2);
#pragma unroll
    for (int v = 0; v < KP_B / KP_T; ++v) {
      if (fx[v] > 0 && ex <= u && u < ex + fx[v]) s_row = i1 + v;
      ex += fx[v];
    }
    chunk += tot2;
    if (u < chunk) break;  // (every thread's)
  }
  __syncthreads();
  if (t == 0) chosen[r + 1] = s_row;
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
static unsigned grid1d(int64_t n, int threads) {
  int64_t g = ceil_div(n, threads);
  return (unsigned)(g < 1 ? 1 : (g > 65535 * 32 ? 65535 * 32 : g));
}

// nearest centroid and its distance for each of the n rows of dx: the bf16
// screen with exact recomputation (qp.qh set) or the exact VALU scan
static void kmeans_assign(vsk_ctx *ctx, const float *cent, int32_t k, int32_t d,
                          int32_t ld, const float *dx, int64_t n, const ArgminQueries &qp,
                          int32_t *assign, float *dist) {
  if (qp.qh) {
    float *csq = static_cast<float *>(ctx->scratch_ptr("km.csq", sizeof(float) * (size_t)k));
    row_norms(ctx, cent, k, d, ld, csq, nullptr);
    screen_argmin(ctx, cent, csq, k, d, ld, dx, n, qp, assign, dist);
    return;
  }
  const int64_t chunk = 1 << 24;  // rows per launch (grid.x bound)
  for (int64_t r = 0; r < n; r += chunk) {
    const int64_t m = n - r < chunk ? n - r : chunk;
    FlatArgs a{};
    a.X = cent;
    a.ldx = ld;
    a.Q = dx + r * ld;
    a.ldq = ld;
    a.kdim = ld;
    a.nq = (int32_t)m;
    a.r0 = 0;
    a.r1 = k;
    a.metric = METRIC_L2_EXACT;
    a.amin = dist + r;
    launch_flat(ctx, a, MODE_ARGMIN, assign + r);
  }
}

// order[...] = the rows grouped by cluster, each cluster's rows ascending;
// off[c] = first position of cluster c, counts[c] = its rows
static void group_rows(vsk_ctx *ctx, const int32_t *assign, int64_t n, int32_t k,
                       int32_t *counts, int32_t *off, const int32_t **order) {
  KernelTimer tm(ctx, "kmeans_group", (double)n);
  fill_i32(ctx, counts, k, 0);
  k_count_clusters<<<grid1d(n, 256), 256, 0, ctx->stream>>>(assign, n, counts);
  check_launch("kmeans_count");
  VSK_HIP(hipMemcpyAsync(off, counts, sizeof(int32_t) * k, hipMemcpyDeviceToDevice,
                         ctx->stream));
  k_scan_excl<<<1, 1024, 0, ctx->stream>>>(off, k);
  check_launch("kmeans_scan");
  const int64_t nb = ceil_div(n, GR_B);
  int32_t *hist = static_cast<int32_t *>(
      ctx->scratch_ptr("km.hist", sizeof(int32_t) * 16 * (size_t)nb));
  int32_t *buf = static_cast<int32_t *>(
      ctx->scratch_ptr("km.radix", sizeof(int32_t) * 4 * (size_t)n));
  int32_t *ka = buf, *va = buf + n, *kb = buf + 2 * n, *vb = buf + 3 * n;
  const int32_t *kin = assign, *vin = nullptr;
  int shift = 0;
  do {
    k_grp_hist<<<(unsigned)nb, GR_T, 0, ctx->stream>>>(kin, n, shift, hist);
    check_launch("kmeans_radix_hist");
    k_scan_excl<<<1, 1024, 0, ctx->stream>>>(hist, 16 * nb);
    check_launch("kmeans_radix_scan");
    k_grp_scatter<<<(unsigned)nb, GR_T, 0, ctx->stream>>>(kin, vin, n, shift, hist,
                                                          ka, va);
    check_launch("kmeans_radix_scatter");
    kin = ka;
    vin = va;
    std::swap(ka, kb);
    std::swap(va, vb);
    shift += 4;
  } while (shift < 31 && ((k - 1) >> shift) > 0);
  *order = vin;
}

// the k starting rows of initializeRandom (:197-207): Fisher-Yates from the
// front on SeedableRNG(seed); positions touched are kept in a map
static std::vector<int64_t> init_random_rows(int64_t n, int32_t k, uint64_t seed) {
  std::unordered_map<int64_t, int64_t> perm;
  auto at = [&](int64_t i) {
    auto it = perm.find(i);
    return it == perm.end() ? i : it->second;
  };
  std::vector<int64_t> rows((size_t)k);
  uint64_t st = seed;
  for (int64_t i = 0; i < k; ++i) {
    if (i < n - 1) {
      const int64_t j = i + (int64_t)swift_bounded(st, (uint64_t)(n - i));
      const int64_t vi = at(i), vj = at(j);
      perm[i] = vj;
      perm[j] = vi;
    }
    rows[(size_t)i] = at(i);
  }
  return rows;
}

// k-means++ starting rows (see the file comment); false on degenerate data
static bool init_plusplus(vsk_ctx *ctx, const float *dx, int64_t n, int32_t d,
                          int32_t ld, int32_t k, uint64_t seed, int64_t *chosen) {
  KernelTimer tm(ctx, "kmeans_plusplus", (double)n * k);
  float *D = static_cast<float *>(ctx->scratch_ptr("km.kppD", sizeof(float) * (size_t)n));
  fill_i32(ctx, reinterpret_cast<int32_t *>(D), n, 0x7F800000);  // +inf
  const float skipm = 1.0f + (float)(d + 4) * 0x1p-22f;
  uint32_t *maxbits = static_cast<uint32_t *>(
      ctx->scratch_ptr("km.kppmax", sizeof(uint32_t) * (size_t)(k + 1) * KP_SLOTS));
  fill_i32(ctx, reinterpret_cast<int32_t *>(maxbits), (int64_t)(k + 1) * KP_SLOTS, 0);
  const int32_t m = (int32_t)ceil_div(n, (int64_t)KP_BLOCKS * KP_B);
  const int64_t nb = ceil_div(n, (int64_t)m * KP_B);
  uint64_t *bsum = static_cast<uint64_t *>(
      ctx->scratch_ptr("km.kppbsum", sizeof(uint64_t) * (size_t)nb));
  uint32_t *done =
      static_cast<uint32_t *>(ctx->scratch_ptr("km.kppdone", sizeof(uint32_t)));
  fill_i32(ctx, reinterpret_cast<int32_t *>(done), 1, 0);
  // [first row, stream state after drawing it]
  uint64_t st = seed;
  const int64_t first = (int64_t)swift_bounded(st, (uint64_t)n);
  const uint64_t init[2] = {(uint64_t)first, st};
  uint64_t *rng = static_cast<uint64_t *>(ctx->scratch_ptr("km.kpprng", sizeof(uint64_t)));
  VSK_HIP(hipMemcpyAsync(chosen, &init[0], sizeof(int64_t), hipMemcpyHostToDevice,
                         ctx->stream));
  VSK_HIP(hipMemcpyAsync(rng, &init[1], sizeof(uint64_t), hipMemcpyHostToDevice,
                         ctx->stream));
  // (an int8 dot product of 2^17 dims still fits 32 bits)
  const int32_t nch = (int32_t)ceil_div(d, 16);
  uint4 *codes = nullptr;
  float4 *par = nullptr;
  const size_t code_bytes = sizeof(uint4) * (size_t)ceil_div(n, 64) * 64 * nch;
  if (d <= 1 << 17) {
    // (in the memory that the Lloyd iterations' plane of the rows takes next:
    // twice as large, and written after the last pick)
    codes = static_cast<uint4 *>(ctx->scratch_ptr("km.q.qh", code_bytes));
    par = static_cast<float4 *>(ctx->scratch_ptr("km.kpppar", sizeof(float4) * (size_t)n));
    k_kpp_codes<<<(unsigned)std::min<int64_t>(ceil_div(n, KP_T / 64), 16384), KP_T, 0,
                  ctx->stream>>>(
        dx, ld, d, n, nch, reinterpret_cast<uint32_t *>(codes), par);
  }
  float *cc = nullptr;
  int32_t *near = nullptr;
  if (!codes || code_bytes > KP_NEAR || n > KP_NEAR_ROWS) {
    cc = static_cast<float *>(ctx->scratch_ptr("km.kppcc", sizeof(float) * (size_t)k));
    near = static_cast<int32_t *>(ctx->scratch_ptr("km.kppnear", sizeof(int32_t) * (size_t)n));
    fill_i32(ctx, near, n, -1);
  }
  for (int r = 0; r + 1 < k; ++r) {
    if (near && r > 0)
      k_kpp_cc<<<(unsigned)ceil_div(r, 4), 256, 0, ctx->stream>>>(dx, ld, d, chosen, r, cc);
    if (near)
      k_kpp_update_queued<<<(unsigned)std::min<int64_t>(ceil_div(n, 64), 16 * ctx->cu_count), 64,
                            0, ctx->stream>>>(dx, ld, d, n, chosen, r, codes, par, nch, skipm,
                                              cc, near, D, maxbits);
    else
      k_kpp_update<<<(unsigned)ceil_div(n, KP_T), KP_T, 0, ctx->stream>>>(
          dx, ld, d, n, chosen, r, codes, par, nch, skipm, D, maxbits);
    k_kpp_pick<<<(unsigned)nb, KP_T, 0, ctx->stream>>>(bsum, nb, m, D, n, maxbits, rng,
                                                       r, chosen, done);
  }
  check_launch("kmeans_plusplus");
  std::vector<int64_t> h((size_t)k);
  VSK_HIP(hipMemcpyAsync(h.data(), chosen, sizeof(int64_t) * k, hipMemcpyDeviceToHost,
                         ctx->stream));
  stream_sync(ctx);
  for (int64_t v : h)
    if (v < 0 || v >= n) return false;
  return true;
}

}  // namespace vsk

using namespace vsk;

vsk_status vsk_kmeans(vsk_ctx *ctx, const float *x, int64_t n, int32_t d,
                      int32_t k, const float *weights, int32_t init_method,
                      const float *init_centroids, uint64_t seed,
                      int32_t max_iter, float tolerance, float *out_centroids,
                      int32_t *out_assign, vsk_kmeans_result *result) {
  VSK_API_BEGIN(ctx);
  VSK_REQUIRE(n > 0, VSK_ERR_EMPTY_INPUT, "cannot cluster an empty dataset");
  VSK_REQUIRE(x && out_centroids && result, VSK_ERR_INVALID_ARGUMENT, "null buffer");
  VSK_REQUIRE(d > 0, VSK_ERR_INVALID_ARGUMENT, "dimension must be positive");
  VSK_REQUIRE(k > 0 && (int64_t)k <= n, VSK_ERR_INVALID_ARGUMENT,
              "invalid number of clusters: must be between 1 and the row count");
  VSK_REQUIRE(n <= 0x7FFFFFFFll, VSK_ERR_INVALID_BUFFER_SIZE,
              "k-means takes at most 2^31-1 rows");
  VSK_REQUIRE(init_method == VSK_KMEANS_INIT_RANDOM ||
                  init_method == VSK_KMEANS_INIT_CUSTOM ||
                  init_method == VSK_KMEANS_INIT_PLUSPLUS,
              VSK_ERR_INVALID_ARGUMENT, "unknown initialisation method");
  VSK_REQUIRE(init_method != VSK_KMEANS_INIT_CUSTOM || init_centroids,
              VSK_ERR_INVALID_ARGUMENT, "custom initialisation needs k x d centroids");
  VSK_REQUIRE(max_iter >= 0, VSK_ERR_INVALID_ARGUMENT, "negative iteration limit");
  CallScope cs(ctx);
  const int32_t ld = padded_ld(d);
  const float *dx = rows_to_device_padded(ctx, x, n, d, ld, "km.x");
  const float *dw = weights ? static_cast<const float *>(input_to_device(
                                  ctx, weights, sizeof(float) * n, "km.w"))
                            : nullptr;
  float *cbuf = static_cast<float *>(
      ctx->scratch_ptr("km.cent", sizeof(float) * 2 * (size_t)k * ld));
  float *cur0 = cbuf;
  // starting centroids
  if (init_method == VSK_KMEANS_INIT_CUSTOM) {
    if (ld != d) fill_i32(ctx, reinterpret_cast<int32_t *>(cur0), (int64_t)k * ld, 0);
    copy_rows(ctx, cur0, sizeof(float) * ld, init_centroids, sizeof(float) * d,
              sizeof(float) * d, k);
  } else {
    int64_t *rows = static_cast<int64_t *>(
        ctx->scratch_ptr("km.rows", sizeof(int64_t) * (size_t)k));
    if (init_method == VSK_KMEANS_INIT_RANDOM) {
      std::vector<int64_t> h = init_random_rows(n, k, seed);
      VSK_HIP(hipMemcpyAsync(rows, h.data(), sizeof(int64_t) * k, hipMemcpyHostToDevice,
                             ctx->stream));
      stream_sync(ctx);  // h goes out of scope
    } else {
      VSK_REQUIRE(init_plusplus(ctx, dx, n, d, ld, k, seed, rows),
                  VSK_ERR_INVALID_ARGUMENT,
                  "data is degenerate (all points are identical)");
    }
    k_gather_rows_i64<<<grid1d((int64_t)k * ld, 256), 256, 0, ctx->stream>>>(
        dx, ld, rows, k, cur0);
    check_launch("kmeans_gather");
  }
  // assignments and distances double-buffered: iteration i + 1 runs while
  // iteration i's inertia is summed on the auxiliary stream
  int32_t *assign2 = static_cast<int32_t *>(
      ctx->scratch_ptr("km.assign", sizeof(int32_t) * 2 * (size_t)n));
  float *dist2 = static_cast<float *>(
      ctx->scratch_ptr("km.dist", sizeof(float) * 2 * (size_t)n));
  int32_t *counts = static_cast<int32_t *>(
      ctx->scratch_ptr("km.counts", sizeof(int32_t) * 2 * (size_t)k));
  int32_t *off = counts + k;
  float *cntf = static_cast<float *>(ctx->scratch_ptr("km.cntf", sizeof(float) * (size_t)k));
  float *dinert = static_cast<float *>(ctx->scratch_ptr("km.inertia", 2 * sizeof(float)));
  uint64_t *rng = static_cast<uint64_t *>(ctx->scratch_ptr("km.rng", sizeof(uint64_t)));
  fill_u64(ctx, rng, 1, seed + 0x9E3779B97F4A7C15ull);
  float *h_inert = static_cast<float *>(ctx->pinned_ptr(2 * sizeof(float)));
  hipStream_t aux = ctx->aux_stream();
  hipEvent_t ev_assigned[2] = {ctx->take_event(), ctx->take_event()};
  hipEvent_t ev_summed[2] = {ctx->take_event(), ctx->take_event()};
  // the rows' fp16 plane for the screened assignment, made once
  ArgminQueries qp;
  if (max_iter > 0 && screen_argmin_applies(ctx, n, k, d))
    qp = half_argmin_queries(ctx, dx, n, d, ld, "km.q");
  // one Lloyd iteration i: centroids cbuf[i & 1] -> cbuf[(i + 1) & 1]
  auto enqueue = [&](int32_t i) {
    const float *cur = cbuf + (size_t)(i & 1) * k * ld;
    float *nxt = cbuf + (size_t)((i + 1) & 1) * k * ld;
    int32_t *assign = assign2 + (size_t)(i & 1) * n;
    float *dist = dist2 + (size_t)(i & 1) * n;
    kmeans_assign(ctx, cur, k, d, ld, dx, n, qp, assign, dist);
    VSK_HIP(hipEventRecord(ev_assigned[i & 1], ctx->stream));
    VSK_HIP(hipStreamWaitEvent(aux, ev_assigned[i & 1], 0));
    {
      KernelTimer tm(ctx, "kmeans_inertia", (double)n, aux);
      k_seq_sum<<<1, 64, 0, aux>>>(dist, n, dinert + (i & 1));
      check_launch("kmeans_inertia");
    }
    VSK_HIP(hipMemcpyAsync(h_inert + (i & 1), dinert + (i & 1), sizeof(float),
                           hipMemcpyDeviceToHost, aux));
    VSK_HIP(hipEventRecord(ev_summed[i & 1], aux));
    const int32_t *order = nullptr;
    group_rows(ctx, assign, n, k, counts, off, &order);
    {
      KernelTimer tm(ctx, "kmeans_means", (double)n * d);
      dim3 grid((unsigned)k, (unsigned)ceil_div(ld, 64));
      k_cluster_means<<<grid, 64, 0, ctx->stream>>>(dx, ld, d, order, off, counts, dw, nxt,
                                                    cntf);
      check_launch("kmeans_means");
    }
    k_refill_empty<<<1, 64, 0, ctx->stream>>>(cntf, k, dx, ld, d, n, rng, nxt);
    check_launch("kmeans_refill");
  };
  float prev = INFINITY;
  int32_t it = 0;
  bool conv = false;
  if (max_iter > 0) enqueue(0);
  while (it < max_iter && !conv) {
    // the next iteration goes in before this one's inertia is known; if
    // this one converged, its results (other buffers) are discarded
    if (it + 1 < max_iter) enqueue(it + 1);
    VSK_HIP(hipEventSynchronize(ev_summed[it & 1]));
    const float inertia = h_inert[it & 1];
    conv = fabsf(inertia - prev) < tolerance;
    prev = inertia;
    ++it;
  }
  for (hipEvent_t e : {ev_assigned[0], ev_assigned[1], ev_summed[0], ev_summed[1]})
    ctx->event_pool.push_back(e);
  const float *cur = cbuf + (size_t)(it & 1) * k * ld;
  const int32_t *assign = assign2 + (size_t)((it + 1) & 1) * n;  // iteration it - 1
  if (it == 0) fill_i32(ctx, assign2 + n, n, 0);
  copy_rows(ctx, out_centroids, sizeof(float) * d, cur, sizeof(float) * ld,
            sizeof(float) * d, k);
  if (out_assign)
    VSK_HIP(hipMemcpyAsync(out_assign, assign, sizeof(int32_t) * n,
                           is_device_ptr(out_assign) ? hipMemcpyDeviceToDevice
                                                     : hipMemcpyDeviceToHost,
                           ctx->stream));
  cs.finish();
  result->iterations = it;
  result->converged = conv ? 1 : 0;
  result->inertia = it > 0 ? prev : INFINITY;
  VSK_API_END(ctx);
}
