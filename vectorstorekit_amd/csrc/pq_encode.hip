// pq_encode.hip -- product-quantizer encoding on the matrix cores: codes of
// Codebook.encode (Quantization/ProductQuantizerCodebook.swift:12-30), the
// first codeword of smallest sequential fp32 |x_m - c|^2, for codebooks of
// 129 to 256 codewords of 4, 8 or 16 dimensions.
//
// The nearest codeword has the largest s(c) = x.c - |c|^2/2.  A bf16 MFMA
// gives s to about 16 bits: with x = xh + xl and c = ch + cl (bf16 each, the
// remainders below 2^-16 of them), xh.ch + xh.cl + xl.ch and the bias, split
// over three bf16 terms, are one sum of 3 DS + 3 products -- 27 of an MFMA's
// 32 at DS = 8.  The error of every s(c) is at most
//   E = 2^-13.9 T + (DS + 2) 2^-25 (|x| + |c|max)^2,  T = |x||c|max + |c|max^2/2:
// 3.1 2^-16 T from the three dropped products and remainders, 2 (3 DS + 3)
// 2^-24 T from the fp32 sum in any order and rounding mode, 2^-17 T from the
// codeword index packed into the score's 6 low bits; the last term is what
// the reference's own fp32 sum may be off by (half of it, in units of s).  A
// codeword whose score is below the best by more than 2 E therefore is not
// the reference's.  Rows with a second candidate group (the kernel's comment;
// some 0.3% of Gaussian data) are decided by the reference's sums over all
// codewords, as are rows whose magnitudes could under- or overflow and any
// NaN.
#include "flat.hpp"

namespace vsk {

typedef __bf16 pe_bf8 __attribute__((ext_vector_type(8)));
typedef float pe_f4 __attribute__((ext_vector_type(4)));
// (a segment starts at any multiple of 4 bytes)
typedef float pe_f4u __attribute__((ext_vector_type(4), aligned(4)));

// bf16 pairs by the hardware conversion (nearest even)
typedef __bf16 pe_bf2 __attribute__((ext_vector_type(2)));
__device__ inline uint32_t pe_cvt2(float a, float b) {
  const pe_bf2 v = {(__bf16)a, (__bf16)b};
  return __builtin_bit_cast(uint32_t, v);
}
__device__ inline float pe_f_lo(uint32_t p) { return __uint_as_float(p << 16); }
__device__ inline float pe_f_hi(uint32_t p) { return __uint_as_float(p & 0xFFFF0000u); }

constexpr int pe_steps(int ds) { return (3 * ds + 3 + 31) / 32; }  // MFMA k-steps
__device__ inline uint32_t pe_pack(uint16_t lo, uint16_t hi) {
  return (uint32_t)lo | ((uint32_t)hi << 16);
}

// The codebooks as MFMA operands, one wave per (segment, tile of 16
// codewords): lane (g, c) of k-step ks holds elements 32 ks + 8 g .. + 7 of
// codeword 16 i + c's vector (ch, cl, ch, three bias terms, zeros), at
// ops[((m * 16 + i) * NK + ks) * 64 + lane]; cmax[m * 16 + i] the tile's
// largest |c|^2 (+inf where it is too large or not a number)
template <int DS>
__global__ __launch_bounds__(64) void k_pq_encode_operands(const float *cb, int32_t ksub,
                                                           uint4 *ops, float *cmax) {
  constexpr int NK = pe_steps(DS);
  const int lane = threadIdx.x, grp = lane >> 4, col = lane & 15;
  const int m = blockIdx.y, i = blockIdx.x, c = 16 * i + col;
  const float *cw = cb + ((int64_t)m * ksub + c) * DS;
  const bool have = c < ksub;
  uint16_t hi[DS], lo[DS], bias[3];
  float sq = 0.f;
#pragma unroll
  for (int j = 0; j < DS; ++j) {
    const float v = have ? cw[j] : 0.f;
    hi[j] = bf16_rn(v);
    lo[j] = bf16_rn(v - __uint_as_float((uint32_t)hi[j] << 16));
    sq += v * v;
  }
  float b = have ? -0.5f * sq : -0x1p126f;  // (no codeword: never the best)
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    bias[j] = bf16_rn(b);
    b -= __uint_as_float((uint32_t)bias[j] << 16);
  }
#pragma unroll
  for (int ks = 0; ks < NK; ++ks) {
    uint16_t el[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      uint16_t v = 0;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int p = ks * 32 + g * 8 + e, sec = p / DS, j = p % DS, t = p - 3 * DS;
        const uint16_t vg = sec == 1          ? lo[j]
                            : sec < 3         ? hi[j]
                            : t >= 0 && t < 3 ? bias[t >= 0 && t < 3 ? t : 0]
                                              : (uint16_t)0;
        v = grp == g ? vg : v;
      }
      el[e] = v;
    }
    ops[((int64_t)(m * 16 + i) * NK + ks) * 64 + lane] =
        make_uint4(pe_pack(el[0], el[1]), pe_pack(el[2], el[3]), pe_pack(el[4], el[5]),
                   pe_pack(el[6], el[7]));
  }
  float mx = sq <= 0x1p120f ? sq : __int_as_float(0x7f800000);
#pragma unroll
  for (int o = 8; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
  if (lane == 0) cmax[m * 16 + i] = mx;
}

// A wave keeps one segment's whole codebook as MFMA operands in registers
// (16 tiles of 16 codewords) and walks the rows 64 at a time; the waves of a
// workgroup take the segments of the same rows, so that a row's cache lines
// are used whole.  A lane loads and splits one row's segment; the split goes
// through the wave's own LDS into the operand layout (a row's NK 64-byte
// vectors), 16 rows a tile.  The codeword side is the MFMA's row side, so a
// lane gets 64 scores of one row, in 16 groups of four codewords; it keeps
// the two largest group maxima and the first one's group (1.5 operations a
// score, which is what bounds the kernel), and the reference's own sums
// choose among the best group's four codewords.  Tracking the two largest
// scores themselves took 3 operations a score.  1M x 128, M = 16, 256
// codewords: 0.46 ms (0.10 ms of HBM reads, 0.31 ms of matrix and vector
// instructions issued one after the other), against 1.98 ms for the fp32 sums
// over all codewords, which stay for other codebook shapes.
//
// The codebooks sit in LDS as fp32: the gathers of the best groups (a random
// group a lane) and of the undecided rows would each wait on the L2.  The DS
// 16-byte pieces of a group of four codewords are stored rotated by the
// group, so that lanes on different groups meet different banks.
template <int DS>
__device__ inline int pe_slot(int c, int q) {
  const int g = c >> 2, piece = (c & 3) * (DS / 4) + q;
  return g * DS + (piece ^ (g & (DS - 1)));
}

template <int DS, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void k_pq_encode_mfma(
    const float *__restrict__ x, int64_t n, const float *__restrict__ cb,
    const uint4 *__restrict__ ops, const float *__restrict__ cm, int32_t M, int32_t ksub,
    int32_t segs, uint8_t *__restrict__ codes) {
#pragma clang fp contract(off)
  constexpr int NK = pe_steps(DS);
  extern __shared__ __attribute__((aligned(16))) uint4 lds[];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int grp = lane >> 4, col = lane & 15;
  const int32_t m0 = blockIdx.y * segs, m = m0 + w % segs;
  const int subs = WAVES / segs, sub = w / segs;
  // the workgroup's codebooks (padding codewords zero; never the best)
  for (int e = threadIdx.x; e < segs * 256 * (DS / 4); e += 64 * WAVES) {
    const int sg = e / (256 * (DS / 4)), c = e / (DS / 4) % 256, q = e % (DS / 4);
    pe_f4 v = {0.f, 0.f, 0.f, 0.f};
    if (m0 + sg < M && c < ksub)
      v = *reinterpret_cast<const pe_f4 *>(cb + ((int64_t)(m0 + sg) * ksub + c) * DS + 4 * q);
    lds[sg * 64 * DS + pe_slot<DS>(c, q)] = __builtin_bit_cast(uint4, v);
  }
  __syncthreads();
  if (m >= M || sub >= subs) return;  // (no barrier below)
  const int64_t ldx = (int64_t)M * DS;
  const uint4 *cbm = lds + (m - m0) * 64 * DS;
  auto codeword = [&](int c, int q) { return __builtin_bit_cast(pe_f4, cbm[pe_slot<DS>(c, q)]); };
  uint4 *sb = lds + segs * 64 * DS + w * 32 * NK * 4;
  float inf = __int_as_float(0x7f800000);
  asm volatile("" : "+v"(inf));
  // the codebook operands and |c|max
  pe_bf8 A[16][NK];
#pragma unroll
  for (int i = 0; i < 16; ++i)
#pragma unroll
    for (int ks = 0; ks < NK; ++ks)
      A[i][ks] =
          __builtin_bit_cast(pe_bf8, ops[((int64_t)(m * 16 + i) * NK + ks) * 64 + lane]);
  float cmax = cm[m * 16 + col];
#pragma unroll
  for (int o = 8; o > 0; o >>= 1) cmax = fmaxf(cmax, __shfl_xor(cmax, o));
  cmax = sqrtf(cmax);

  const int64_t step = (int64_t)gridDim.x * subs * 64;
  int64_t r0 = ((int64_t)blockIdx.x * subs + sub) * 64;
  float xn[DS];  // the next 64 rows' segments, a row a lane
  auto load = [&](int64_t rb) {
    const int64_t r = rb + lane < n ? rb + lane : n - 1;
    const float *p = x + r * ldx + (int64_t)m * DS;
#pragma unroll
    for (int j = 0; j < DS; j += 4) {
      const pe_f4u v = *reinterpret_cast<const pe_f4u *>(p + j);
#pragma unroll
      for (int u = 0; u < 4; ++u) xn[j + u] = v[u];
    }
  };
  if (r0 < n) load(r0);
  for (; r0 < n; r0 += step) {
    float xv[DS], sq = 0.f;
    uint32_t hi[DS / 2], lo[DS / 2];  // bf16 pairs
#pragma unroll
    for (int j = 0; j < DS; ++j) {
      xv[j] = xn[j];
      sq += xv[j] * xv[j];
    }
#pragma unroll
    for (int j = 0; j < DS / 2; ++j) {
      hi[j] = pe_cvt2(xv[2 * j], xv[2 * j + 1]);
      lo[j] = pe_cvt2(xv[2 * j] - pe_f_lo(hi[j]), xv[2 * j + 1] - pe_f_hi(hi[j]));
    }
    if (r0 + step < n) load(r0 + step);
    float top = 0.f, gap = 0.f;
#pragma unroll 1
    for (int t = 0; t < 4; ++t) {
      if (!(t & 1)) {  // the next 32 rows' operands
        if (lane >> 5 == t >> 1) {
#pragma unroll
          for (int ks = 0; ks < NK; ++ks)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
              uint32_t el[4];  // (a pair never straddles two sections: DS is even)
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                const int p = ks * 32 + g * 8 + 2 * e, sec = p / DS, j = p % DS / 2,
                          o = p - 3 * DS;
                el[e] = sec < 2 ? hi[j] : sec == 2 ? lo[j]
                        : o == 0 ? 0x3F803F80u : o == 2 ? 0x3F80u : 0u;
              }
              sb[((lane & 31) * NK + ks) * 4 + g] = make_uint4(el[0], el[1], el[2], el[3]);
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      }
      pe_bf8 b[NK];
#pragma unroll
      for (int ks = 0; ks < NK; ++ks)
        b[ks] = __builtin_bit_cast(pe_bf8, sb[((16 * (t & 1) + col) * NK + ks) * 4 + grp]);
      float m1 = -inf, m2 = -inf;
      // (the next tile's product is under way while one's scores are reduced;
      // a maximum is a median with an infinity the compiler cannot see: it
      // would canonicalise both operands of an fmaxf first)
      auto product = [&](int i) {
        pe_f4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < NK; ++ks)
          acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[i][ks], b[ks], acc, 0, 0, 0);
        return acc;
      };
      auto fmx = [&](float u, float v) { return __builtin_amdgcn_fmed3f(u, v, inf); };
      pe_f4 cur = product(0);
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const pe_f4 acc = cur;
        if (i + 1 < 16) cur = product(i + 1);
        const float four = fmx(fmx(acc[0], acc[1]), fmx(acc[2], acc[3]));
        const float s = __uint_as_float((__float_as_uint(four) & ~63u) | (uint32_t)(4 * i));
        m2 = __builtin_amdgcn_fmed3f(m1, m2, s);
        m1 = fmx(m1, s);
      }
      // the four lane groups hold other codewords of the same row: their two
      // largest, the group in the index's low bits
      m1 = __uint_as_float(__float_as_uint(m1) | (uint32_t)grp);
      {
        const auto u = __builtin_amdgcn_permlane16_swap(__float_as_uint(m1), __float_as_uint(m1),
                                                        false, false);
        const auto v = __builtin_amdgcn_permlane16_swap(__float_as_uint(m2), __float_as_uint(m2),
                                                        false, false);
        const float a0 = __uint_as_float(u[0]), a1 = __uint_as_float(u[1]);
        m2 = fmx(__builtin_amdgcn_fmed3f(a0, a1, -inf),
                 fmx(__uint_as_float(v[0]), __uint_as_float(v[1])));
        m1 = fmx(a0, a1);
      }
      {
        const auto u = __builtin_amdgcn_permlane32_swap(__float_as_uint(m1), __float_as_uint(m1),
                                                        false, false);
        const auto v = __builtin_amdgcn_permlane32_swap(__float_as_uint(m2), __float_as_uint(m2),
                                                        false, false);
        const float a0 = __uint_as_float(u[0]), a1 = __uint_as_float(u[1]);
        m2 = fmx(__builtin_amdgcn_fmed3f(a0, a1, -inf),
                 fmx(__uint_as_float(v[0]), __uint_as_float(v[1])));
        m1 = fmx(a0, a1);
      }
      if (grp == t) {  // (lane 16 t + col holds row 16 t + col)
        top = m1;
        gap = m1 - m2;
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    // the best group of four codewords: the reference's sums decide among
    // them (ascending, strict '<')
    int32_t code;
    {
      const uint32_t pos = __float_as_uint(top) & 63u;
      const int32_t c0 = (int32_t)(4 * pos);
      float best = inf;
      code = c0;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int32_t c = c0 + r < ksub ? c0 + r : ksub - 1;  // (padding: the last one again)
        float acc = 0.f;
#pragma unroll
        for (int j = 0; j < DS; j += 4) {
          const pe_f4 v = codeword(c, j / 4);
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const float d = xv[j + u] - v[u];
            acc = acc + d * d;
          }
        }
        if (acc < best) {
          best = acc;
          code = c;
        }
      }
    }
    // the margin 2 E, with room for its own roundings
    const float nx = sqrtf(sq), both = nx + cmax;
    const float margin = 0x1.27p-13f * (nx * cmax + 0.5f * cmax * cmax) +
                         (float)(DS + 2) * 0x1.04p-24f * (both * both) + 0x1p-100f;
    const bool sure = gap > margin && nx >= 0x1p-60f && nx <= 0x1p60f && cmax >= 0x1p-60f &&
                      cmax <= 0x1p60f;
    uint64_t todo = __ballot(!sure && r0 + lane < n);
    while (todo) {  // near ties between groups: all codewords
      const int rr = __builtin_ctzll(todo);
      todo &= todo - 1;
      float q[DS];
#pragma unroll
      for (int j = 0; j < DS; ++j)
        q[j] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(xv[j]), rr));
      float best = __int_as_float(0x7f800000);
      uint32_t bc = 0xFFFFFFFFu;
      for (int32_t c = lane; c < ksub; c += 64) {
        float acc = 0.f;
#pragma unroll
        for (int j = 0; j < DS; j += 4) {
          const pe_f4 v = codeword(c, j / 4);
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const float d = q[j + u] - v[u];
            acc = acc + d * d;
          }
        }
        if (acc < best) {
          best = acc;
          bc = (uint32_t)c;
        }
      }
      // (sums are not negative: their bits order as they do)
      uint64_t key = (uint64_t)__float_as_uint(best) << 32 | bc;
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) {
        const uint64_t k2 = (uint64_t)__shfl_xor((uint32_t)(key >> 32), o) << 32 |
                            __shfl_xor((uint32_t)key, o);
        key = k2 < key ? k2 : key;
      }
      // no sum below infinity: the reference keeps its start, codeword 0
      const int32_t c = (uint32_t)key == 0xFFFFFFFFu ? 0 : (int32_t)(uint32_t)key;
      if (lane == rr) code = c;
    }
    if (r0 + lane < n) codes[(r0 + lane) * M + m] = (uint8_t)code;
  }
}

template <int DS, int WAVES>
static void launch(vsk_ctx *ctx, const float *x, int64_t n, const float *cb, const uint4 *ops,
                   const float *cmax, int32_t M, int32_t ksub, uint8_t *codes) {
  const int32_t segs = M < WAVES ? M : WAVES;
  const int64_t gy = ceil_div(M, segs), per = (int64_t)(WAVES / segs) * 64;
  // one workgroup a CU (its registers fill it), all of them resident
  int64_t gx = ceil_div((int64_t)ctx->cu_count, gy);
  if (gx > ceil_div(n, per)) gx = ceil_div(n, per);
  constexpr int kMax = (WAVES * 64 * DS + WAVES * 32 * pe_steps(DS) * 4) * 16;  // 160 KB at most
  static_assert(kMax <= 160 * 1024, "codebooks and staging share one CU's LDS");
  VSK_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(k_pq_encode_mfma<DS, WAVES>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, kMax));
  const int lds = (segs * 64 * DS + WAVES * 32 * pe_steps(DS) * 4) * 16;
  k_pq_encode_mfma<DS, WAVES>
      <<<dim3((unsigned)gx, (unsigned)gy), 64 * WAVES, lds, ctx->stream>>>(x, n, cb, ops, cmax, M,
                                                                           ksub, segs, codes);
}

// (with at most 128 codewords half of the tiles would be padding)
bool pq_encode_mfma_applies(int32_t ksub, int32_t dsub) {
  return ksub > 128 && ksub <= 256 && (dsub == 4 || dsub == 8 || dsub == 16);
}

size_t pq_encode_operand_bytes(int32_t M, int32_t dsub) {
  return (size_t)M * 16 * (pe_steps(dsub) * 64 * sizeof(uint4) + sizeof(float));
}

static float *operand_cmax(void *ops, int32_t M, int32_t dsub) {
  return reinterpret_cast<float *>(static_cast<uint4 *>(ops) +
                                   (size_t)M * 16 * pe_steps(dsub) * 64);
}

void pq_encode_operands(vsk_ctx *ctx, const float *cb, int32_t M, int32_t ksub, int32_t dsub,
                        void *ops) {
  const dim3 grid(16, (unsigned)M);
  uint4 *o = static_cast<uint4 *>(ops);
  float *cm = operand_cmax(ops, M, dsub);
  if (dsub == 4) k_pq_encode_operands<4><<<grid, 64, 0, ctx->stream>>>(cb, ksub, o, cm);
  else if (dsub == 8) k_pq_encode_operands<8><<<grid, 64, 0, ctx->stream>>>(cb, ksub, o, cm);
  else k_pq_encode_operands<16><<<grid, 64, 0, ctx->stream>>>(cb, ksub, o, cm);
  check_launch("pq_encode_operands");
}

void pq_encode_mfma(vsk_ctx *ctx, const float *x, int64_t n, const float *cb, void *ops,
                    int32_t M, int32_t ksub, int32_t dsub, uint8_t *codes) {
  const uint4 *o = static_cast<const uint4 *>(ops);
  const float *cm = operand_cmax(ops, M, dsub);
  if (dsub == 4) launch<4, 16>(ctx, x, n, cb, o, cm, M, ksub, codes);
  else if (dsub == 8) launch<8, 16>(ctx, x, n, cb, o, cm, M, ksub, codes);
  else launch<16, 8>(ctx, x, n, cb, o, cm, M, ksub, codes);
}

}  // namespace vsk
