// gq_gemm_q8.hip -- the int8 mode of the batched GEMM (GQ_GEMM_INT8):
// Q4_K or Q6_K weights against activations packed per 32 elements exactly as
// KvDtype::Q8_0::pack (src/model/mod.rs:574-583: amax / 127, f16 scale xs,
// codes from the f32 scale), fp32 results.
//
// The format needs one scaling per (row, token, 32 elements).  On int8 MFMA
// that is a conversion, a product of the two scales and an FMA per result,
// 12 VALU instructions beside each 16-cycle MFMA, and the VALU was the bound.
// Here the integers are f16 operands instead, at the same MFMA rate for a
// depth of 32: a weight code times its sub-block scale is an integer of at
// most 11 bits (Q4_K: sc q <= 945), exact in f16 (Q6_K's sc (q - 32), up to 13
// bits, is its f16 rounding plus an exact rest, 0 up to 2048 and else 0 or +-1:
// two MFMAs into one result), and so is an activation code.  The fp32 dot D of
// 32 of them is exact, needs no conversion and already carries the weight's
// scale, so what is left per result is one FMA, acc += xs D (xs is the lane's
// own token's), and once per 256-element unit y += d acc.
// The Q4_K min term, y -= dmin sum_sb m_sb (xs sum q)_sb, is one bf16 MFMA per
// unit: m (6 bits, exact) against xs sum q in three bf16 (24 bits, exact, any
// exponent), the three at depths 0-7, 8-15 and 16-23.
// (Activations as f16 pairs hi + lo of xs q, whose dots chain through a whole
// unit on the MFMAs alone, took 151 us of kernel against 130 on 18944 x 3584 x
// 512, and their longer fp32 chains doubled the error of a short k.)
//
// 18944 x 3584 x 512 Q4_K: 204 us a call on int8 MFMA, 125 so (kernel 130 to 134
// under the profiler, which runs one launch at a time); 3584 x 18944 x 512 Q6_K
// 446 and 183 (kernel 181).  Q4_K / Q6_K, the MFMAs are busy for 25 / 34% of the
// kernel's cycles (of 93 / 90% of the CUs), VALU issue for 45 / 40%, and on a
// CU the LDS for 23 / 29%, with waves waiting for it in 2 / 5% of theirs: the
// bound is what a SIMD's two waves leave unhidden beside the MFMAs, that is the
// FMAs, staging W, the units' ends and the X loads, and not the A fragments'
// LDS reads.
#include <algorithm>
#include <type_traits>

#include "gq_gemm_dev.h"
#include "gq_internal.h"

namespace gq {

typedef _Float16 h16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 h16x2_t __attribute__((ext_vector_type(2)));
// (staged loads are held in these, not in uint4: the struct's copies across
// branches keep it in scratch memory)
typedef uint32_t u4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u2_t __attribute__((ext_vector_type(2)));

namespace {

// ----------------------------------------------------------- activations
// Codes as f16 MFMA B fragments [npad/16][kpad/32][64 lanes][8]: lane l holds
// token l % 16 and 8 of the block's elements, 8 (l / 16) + {0,2,1,3,4,6,5,7}
// (the order in which two-byte masks take the weights' codes apart); xs
// [npad/16][kpad/32][16]; and (Q4_K) xs sum(q) in bf16 thirds
// [npad/16][kpad/256][64][8] (lane l: token l % 16, third l / 16, the unit's 8
// blocks; zeros for l >= 48).  Tokens past n are all zero.  A wave packs one
// fragment.  I8 (the small kernel): the codes as int8 in the elements' order,
// [npad/16][kpad/32][64][8 bytes].
template <bool I8>
__global__ __launch_bounds__(256) void k_x_to_q8(const float *X, int n, int npad, int k, int units, uint16_t *xq,
                                                 float *xs, uint16_t *xm) {
  const int lane = threadIdx.x & 63, kbs = 8 * units;
  const long f = (long)blockIdx.x * 4 + (threadIdx.x >> 6);  // (token tile, block)
  const int nt = (int)(f / kbs), kb = (int)(f % kbs);
  if (16 * nt >= npad) return;  // (uniform per wave)
  const int t = 16 * nt + (lane & 15), sub = lane >> 4, c0 = 32 * kb + 8 * sub;
  float v[8];
  if ((k & 7) == 0) {
    float4 a = make_float4(0.f, 0.f, 0.f, 0.f), b = a;
    if (t < n && c0 < k) {
      a = *(const float4 *)(X + (long)t * k + c0);
      b = *(const float4 *)(X + (long)t * k + c0 + 4);
    }
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
    v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
  } else {
#pragma unroll
    for (int e = 0; e < 8; e++) v[e] = t < n && c0 + e < k ? X[(long)t * k + c0 + e] : 0.f;
  }
  float amax = 0.f;
#pragma unroll
  for (int e = 0; e < 8; e++) amax = fmaxf(amax, fabsf(v[e]));
  amax = fmaxf(amax, __shfl_xor(amax, 16, 64));
  amax = fmaxf(amax, __shfl_xor(amax, 32, 64));
  const float s = amax > 0.f ? amax / 127.0f : 1.0f;
  int q[8], sum = 0;
#pragma unroll
  for (int e = 0; e < 8; e++) {
    q[e] = (int)fminf(fmaxf(roundf(v[e] / s), -127.f), 127.f);
    sum += q[e];
  }
  const float sc = t < n ? __half2float(__float2half_rn(s)) : 0.f;
  if (sub == 0) xs[f * 16 + lane] = sc;
  if constexpr (I8) {
    uint32_t w[2] = {0, 0};
#pragma unroll
    for (int e = 0; e < 8; e++) w[e >> 2] |= ((uint32_t)q[e] & 0xFFu) << (8 * (e & 3));
    *(uint2 *)((uint8_t *)xq + (f * 64 + lane) * 8) = make_uint2(w[0], w[1]);
    return;
  }
  sum += __shfl_xor(sum, 16, 64);
  sum += __shfl_xor(sum, 32, 64);
  h16x8_t o = {(_Float16)(float)q[0], (_Float16)(float)q[2], (_Float16)(float)q[1], (_Float16)(float)q[3],
               (_Float16)(float)q[4], (_Float16)(float)q[6], (_Float16)(float)q[5], (_Float16)(float)q[7]};
  *(h16x8_t *)(xq + (f * 64 + lane) * 8) = o;
  if (xm) {
    const float x = sc * (float)sum, x1 = __uint_as_float(f2bf(x) << 16);
    // (past the f16 scale's range x is infinite, or 0 inf, and all of it is in x1)
    const float rest = fabsf(x) < INFINITY ? x - x1 : 0.f, x2 = __uint_as_float(f2bf(rest) << 16);
    xm[(((long)nt * units + (kb >> 3)) * 64 + lane) * 8 + (kb & 7)] =
        (uint16_t)f2bf(sub == 0 ? x1 : sub == 1 ? x2 : sub == 2 ? rest - x2 : 0.f);
  }
}

// ----------------------------------------------------------- kernel
struct Q8Args {
  const uint8_t *rec;     // stage records (Q4_K: ggml blocks)
  const uint16_t *xq, *xm;
  const float *xs;
  float *y, *part;        // part: partial products [ksplit][n][rows] instead
  int rows, n, kpad, ntiles, ksplit;
};

__device__ __forceinline__ uint32_t pkfma(uint32_t a, h16x2_t s, h16x2_t c) {
  const h16x2_t v = __builtin_bit_cast(h16x2_t, a);
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(v, s, c));
}

// Block tile 160 rows x 128 NJ tokens, 512 threads: wave w multiplies all 160
// rows by tokens 16 NJ w .., so no X fragment is needed by two waves: each is
// loaded from L2 straight into the registers of its wave, half a stage ahead
// (X through LDS measured slower, 172 against 130 us).  K-steps ("stages") of 64 = two sub-blocks.
// A stage ahead, five of the waves (a thread per row and half of the group's
// codes) turn W into f16 fragments in LDS and, on a unit's first stage, write
// the row's d (and dmin and mins).  One barrier per stage.
// PROD (k <= 256): y += (d xs) D instead, an instruction more per result and
// one rounding less, which shows where there is only one unit: relative error
// 5.4e-8 against 5.9e-8 (Q6_K) and 1.2e-7 against 1.3e-7 (Q4_K), at a price of 8 to
// 15% (18944 x 256 x 512: 24 against 21.5 us a call, Q6_K 26 against 23.6).  From
// two units on the other form's error is the smaller one.
template <int FMT, int NJ, bool PROD>
__global__ __launch_bounds__(512) void k_gemm_q8(Q8Args a) {
  constexpr bool Q4 = FMT == T_Q4_K;
  constexpr int NA = Q4 ? 1 : 2;  // f16 terms of a weight
  constexpr int RT = Q8_ROWS / 16;
  __shared__ __align__(16) uint16_t As[2][NA * 2 * RT * FR16];  // [buf][term][half][row tile] fragments
  __shared__ __align__(16) float Ds[2][Q8_ROWS], Dm[Q4 ? 2 : 1][Q4 ? Q8_ROWS : 4];
  __shared__ __align__(16) uint16_t Ms[Q4 ? 2 : 1][(Q4 ? Q8_ROWS : 1) * 8];  // bf16 mins of the row's unit
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int b = xcd_block(blockIdx.x, gridDim.x), split = b % a.ksplit, rest = b / a.ksplit;
  const int ntile = rest % a.ntiles, tile = rest / a.ntiles;
  const int rows = a.rows, m0 = tile * Q8_ROWS, n0 = ntile * 128 * NJ;
  const int units = a.kpad / 256;
  const int s0 = 4 * (int)((long)units * split / a.ksplit), s1 = 4 * (int)((long)units * (split + 1) / a.ksplit);

  // ---- W staging
  // Tasks (row, half): 0-255 on waves 0-3, 256-319 on wave 4 + s % 4, so that
  // the fifth wave's work goes around the SIMDs.
  const int wh = tid & 1;
  const auto row_of = [&](int s) { return wave < 4 ? tid >> 1 : wave == 4 + (s & 3) ? 128 + (lane >> 1) : -1; };
  u4_t c0 = {0, 0, 0, 0}, c1 = c0;  // Q4_K: quants; Q6_K: low bits of both quarters
  u4_t hd = c0;                       // Q4_K: the unit's header; Q6_K: high bits (x, y), scales (z), d (w)
  auto load_w = [&](int s) {
    const int wr = row_of(s);
    if (wr < 0) return;
    const uint8_t *wsrc = a.rec + (long)min(m0 + wr, rows - 1) * units * (Q4 ? 144 : 256);
    if constexpr (Q4) {
      const uint8_t *p = wsrc + (long)(s >> 2) * 144;
      c0 = *(const u4_t *)(p + 16 + 32 * (s & 3) + 16 * wh);
      hd = *(const u4_t *)p;
    } else {
      const uint8_t *p = wsrc + (long)s * 64;
      c0 = *(const u4_t *)(p + 16);
      c1 = *(const u4_t *)(p + 32);
      const u2_t hb = *(const u2_t *)(p + 48 + 8 * wh), sd = *(const u2_t *)p;
      hd = u4_t{hb.x, hb.y, sd.x, sd.y};
    }
  };
  auto store_w = [&](int s) {
    const int wr = row_of(s);
    if (wr < 0) return;
    const bool wok = m0 + wr < rows;
    const int buf = s & 1, ub = (s >> 2) & 1, rt = wr >> 4, r16 = wr & 15;
    if constexpr (Q4) {
      const int j = s & 3;
      uint32_t sc[2], mn;
      scale_min_k4(2 * j, hd.y, hd.z, hd.w, sc[0], mn);
      scale_min_k4(2 * j + 1, hd.y, hd.z, hd.w, sc[1], mn);
#pragma unroll
      for (int h = 0; h < 2; h++) {  // nibble h: sub-block h, elements 16 wh + byte
        // sc (1024 + q) - 1024 sc, exact
        const _Float16 sv = (_Float16)(wok ? (float)sc[h] : 0.f), cv = sv * (_Float16)-1024.f;
        const h16x2_t s2 = {sv, sv}, k2 = {cv, cv};
        uint32_t o[8];
#pragma unroll
        for (int i = 0; i < 4; i++) {
          o[2 * i] = pkfma(((c0[i] >> (4 * h)) & 0x000F000Fu) | 0x64006400u, s2, k2);
          o[2 * i + 1] = pkfma(((c0[i] >> (4 * h + 8)) & 0x000F000Fu) | 0x64006400u, s2, k2);
        }
        uint16_t *dst = &As[buf][((h * RT + rt) * 64 + r16 + 32 * wh) * 8];
        *(uint4 *)dst = make_uint4(o[0], o[1], o[2], o[3]);
        *(uint4 *)(dst + 128) = make_uint4(o[4], o[5], o[6], o[7]);
      }
      if (j == 0 && wh == 0) {
        Ds[ub][wr] = wok ? h2f(hd.x) : 0.f;
        Dm[ub][wr] = wok ? -h2f(hd.x >> 16) : 0.f;
        uint32_t o[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
          uint32_t sx, ma, mb;
          scale_min_k4(2 * e, hd.y, hd.z, hd.w, sx, ma);
          scale_min_k4(2 * e + 1, hd.y, hd.z, hd.w, sx, mb);
          o[e] = pack_bf16((float)ma, (float)mb);
        }
        *(uint4 *)&Ms[ub][wr * 8] = make_uint4(o[0], o[1], o[2], o[3]);
      }
    } else {
      // half wh: element 16 qq + i has its low 4 bits in nibble wh of byte i of
      // c0 / c1 and its high 2 bits at bits 2 i of dword qq of the high bits
#pragma unroll
      for (int qq = 0; qq < 2; qq++) {
        const u4_t c = qq ? c1 : c0;
        const uint32_t hw = qq ? hd.y : hd.x;
        const int sc = wok ? (int)(int8_t)(hd.z >> (8 * (2 * wh + qq))) : 0;
        const _Float16 sv = (_Float16)(float)sc;
        const h16x2_t s2 = {sv, sv}, off = {(_Float16)-1056.f, (_Float16)-1056.f};
        uint32_t oh[8], ol[8];
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const uint32_t l = c[i] >> (4 * wh), x = hw >> (8 * i);
          const uint32_t p[2] = {
              (l & 0x000F000Fu) | ((x << 4) & 0x30u) | ((x << 16) & 0x300000u) | 0x64006400u,
              ((l >> 8) & 0x000F000Fu) | ((x << 2) & 0x30u) | ((x << 14) & 0x300000u) | 0x64006400u};
#pragma unroll
          for (int e = 0; e < 2; e++) {
            const h16x2_t v = __builtin_bit_cast(h16x2_t, p[e]) + off;  // q - 32
            const h16x2_t hi = v * s2;
            oh[2 * i + e] = __builtin_bit_cast(uint32_t, hi);
            ol[2 * i + e] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(v, s2, -hi));
          }
        }
        uint16_t *dst = &As[buf][((wh * RT + rt) * 64 + r16 + 32 * qq) * 8];
        *(uint4 *)dst = make_uint4(oh[0], oh[1], oh[2], oh[3]);
        *(uint4 *)(dst + 128) = make_uint4(oh[4], oh[5], oh[6], oh[7]);
        uint16_t *rest = dst + 2 * RT * FR16;
        *(uint4 *)rest = make_uint4(ol[0], ol[1], ol[2], ol[3]);
        *(uint4 *)(rest + 128) = make_uint4(ol[4], ol[5], ol[6], ol[7]);
      }
      if ((s & 3) == 0 && wh == 0) Ds[ub][wr] = wok ? h2f(hd.w) : 0.f;
    }
  };

  // ---- X: fragments and scales of token tiles n0 / 16 + NJ wave + jn
  const long nt0 = (n0 >> 4) + NJ * wave;
  const uint16_t *xp = a.xq + nt0 * units * 4096 + lane * 8;
  const float *xsp = a.xs + nt0 * units * 128 + (lane & 15);
  h16x8_t bv[2][NJ];
  float xv[2][NJ];
  auto load_x = [&](int s, int ks) {
#pragma unroll
    for (int jn = 0; jn < NJ; jn++) {
      const int f = jn * units * 8 + 2 * s + ks;
      bv[ks][jn] = *(const h16x8_t *)(xp + (long)f * 512);
      xv[ks][jn] = xsp[(long)f * 16];
    }
  };
  u4_t xm[NJ];
  auto load_unit = [&](int u) {
    if constexpr (Q4) {
#pragma unroll
      for (int jn = 0; jn < NJ; jn++) xm[jn] = *(const u4_t *)(a.xm + (((nt0 + jn) * units + u) * 64 + lane) * 8);
    }
  };
  f32x4_t y[RT][NJ], acc[RT][NJ];
#pragma unroll
  for (int i = 0; i < RT; i++)
#pragma unroll
    for (int jn = 0; jn < NJ; jn++) y[i][jn] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  auto compute = [&](int s, int ks, auto first) {  // first: the unit's first half-stage
    const uint16_t *A = As[s & 1] + lane * 8;
    h16x8_t av[2][NA];  // one row tile ahead
    auto read_a = [&](int i) {
#pragma unroll
      for (int t = 0; t < NA; t++) av[i & 1][t] = *(const h16x8_t *)(A + ((t * 2 + ks) * RT + i) * FR16);
    };
    read_a(0);
    f32x4_t dq[2][NJ];
    auto fold = [&](int i) {  // acc += xs D
      if constexpr (PROD) {
        const f32x4_t dr = *(const f32x4_t *)&Ds[(s >> 2) & 1][16 * i + 4 * (lane >> 4)];
#pragma unroll
        for (int jn = 0; jn < NJ; jn++) {
#pragma unroll
          for (int r = 0; r < 4; r++) y[i][jn][r] = fmaf(dr[r] * xv[ks][jn], dq[i & 1][jn][r], y[i][jn][r]);
          asm volatile("" : "+v"(y[i][jn]));
        }
        return;
      }
#pragma unroll
      for (int jn = 0; jn < NJ; jn++) {
#pragma unroll
        for (int r = 0; r < 4; r++)
          acc[i][jn][r] = first ? xv[ks][jn] * dq[i & 1][jn][r] : fmaf(xv[ks][jn], dq[i & 1][jn][r], acc[i][jn][r]);
        asm volatile("" : "+v"(acc[i][jn]));
      }
    };
    // a row tile's FMAs run behind the next one's MFMAs
#pragma unroll
    for (int i = 0; i < RT; i++) {
      if (i + 1 < RT) read_a(i + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int jn = 0; jn < NJ; jn++) {
        const f32x4_t z = {0.f, 0.f, 0.f, 0.f};
        dq[i & 1][jn] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av[i & 1][NA - 1], bv[ks][jn], z, 0, 0, 0);
      }
      if constexpr (NA == 2) {
#pragma unroll
        for (int jn = 0; jn < NJ; jn++)
          dq[i & 1][jn] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av[i & 1][0], bv[ks][jn], dq[i & 1][jn], 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (i > 0) fold(i - 1);
      __builtin_amdgcn_sched_barrier(0);
    }
    fold(RT - 1);
  };
  // unit u done: y += d acc - dmin sum_sb m (xs sum q)
  auto finish = [&](int u) {
    const int ub = u & 1;
#pragma unroll
    for (int i = 0; i < RT; i++) {
      const f32x4_t dr = *(const f32x4_t *)&Ds[ub][16 * i + 4 * (lane >> 4)];
      f32x4_t mt[NJ], mr;
      if constexpr (Q4) {
        mr = *(const f32x4_t *)&Dm[ub][16 * i + 4 * (lane >> 4)];
        const bf16x8_t am = *(const bf16x8_t *)&Ms[ub][(16 * i + (lane & 15)) * 8];
#pragma unroll
        for (int jn = 0; jn < NJ; jn++) {
          const f32x4_t z = {0.f, 0.f, 0.f, 0.f};
          mt[jn] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(am, __builtin_bit_cast(bf16x8_t, xm[jn]), z, 0, 0, 0);
        }
      }
#pragma unroll
      for (int jn = 0; jn < NJ; jn++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
          if constexpr (!PROD) y[i][jn][r] = fmaf(dr[r], acc[i][jn][r], y[i][jn][r]);
          if constexpr (Q4) y[i][jn][r] = fmaf(mr[r], mt[jn][r], y[i][jn][r]);
        }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // A stage stages the next one's W first: the staging waves then run late, and
  // a SIMD's other wave has the MFMAs meanwhile (and is done with the unit's
  // FMAs while they multiply).
  load_w(s0);
  load_x(s0, 0);
  store_w(s0);
  if (s0 + 1 < s1) load_w(s0 + 1);
  __syncthreads();
  auto stage = [&](int s, auto first) {
    const bool more = s + 1 < s1, last = (s & 3) == 3;
    load_x(s, 1);
    if (more) store_w(s + 1);
    if (s + 2 < s1) load_w(s + 2);
    __builtin_amdgcn_sched_barrier(0);
    compute(s, 0, first);
    if (more) load_x(s + 1, 0);
    if (last) load_unit(s >> 2);
    __builtin_amdgcn_sched_barrier(0);
    compute(s, 1, std::false_type{});
    if (last) finish(s >> 2);
    __syncthreads();
  };
  for (int s = s0; s < s1; s += 4) {  // a unit
    stage(s, std::true_type{});
    if constexpr (Q4 || PROD) {  // (unrolled, they spill registers)
#pragma unroll 1
      for (int j = 1; j < 4; j++) stage(s + j, std::false_type{});
    } else {
      stage(s + 1, std::false_type{});
      stage(s + 2, std::false_type{});
      stage(s + 3, std::false_type{});
    }
  }
  // D layout: lane holds rows 4 (lane / 16) + r of token column lane % 16.
  float *Y = a.part ? a.part + (long)split * a.n * rows : a.y;
#pragma unroll
  for (int i = 0; i < RT; i++) {
    const int m = m0 + 16 * i + 4 * (lane >> 4);
#pragma unroll
    for (int jn = 0; jn < NJ; jn++) {
      const int t = n0 + 16 * (NJ * wave + jn) + (lane & 15);
      if (t >= a.n) continue;
      float *yp = Y + (long)t * rows + m;
      if (m + 3 < rows) {
        store4(yp, y[i][jn]);
      } else {
#pragma unroll
        for (int r = 0; r < 4; r++)
          if (m + r < rows) yp[r] = y[i][jn][r];
      }
    }
  }
}

// ----------------------------------------------------------- small kernel
// Q6_K launches that leave the kernel above mostly idle: a short depth, or few
// rows and tokens.  There the latency of a stage counts and not the rate, and
// a 160-row stage is a long one; a block here is 64 rows x 64 tokens on int8
// MFMA, 4 waves, each 16 rows by all the tokens.  A code minus 32 is an int8; the scales
// change every 16 elements, half an MFMA's depth, so each 32 elements are two
// MFMAs with the other group's half of A zero (lanes 0-31 hold elements 0-15,
// 32-63 the others), D = sc_a D_a + sc_b D_b in 32-bit integers (below 2^24,
// exact as f32), and from there on as above: acc += xs D, and y += d acc per
// unit (PROD: y += (d xs) D).  A stage ahead of its use, threads 0-127 turn
// the quants of (row tid / 2, half tid % 2) into A fragments, 128-191 write the
// row's scales and d, and all of them the stage's X fragments and scales.
// 600 x 256 x 200: 11 us a call, 16 on the kernel above; 4800 x 512 x 200: 17 and 23.
template <bool PROD>
__global__ __launch_bounds__(256) void k_gemm_q6_small(Q8Args a) {
  constexpr int NJ = Q6S / 16;
  __shared__ __align__(16) uint8_t Aq[2][2][4][512];  // [buf][half][row tile][lane slot x 8 codes]
  __shared__ __align__(16) int Sc[2][4][Q6S];         // [buf][group][row]
  __shared__ __align__(16) float Dd[2][Q6S];
  __shared__ __align__(16) float Xs[2][2][NJ][16];    // [buf][half][token tile][token]
  __shared__ __align__(16) uint8_t Xb[2][2][NJ][512];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rows = a.rows, m0 = blockIdx.x * Q6S, n0 = blockIdx.y * Q6S;
  const int stages = a.kpad / 64, kbs = a.kpad / 32;
  const uint8_t *xq = (const uint8_t *)a.xq;
  const int sr = tid < 128 ? tid >> 1 : tid - 128, sh = tid & 1;
  const bool sq = tid < 128, ss = tid >= 128 && tid < 192;
  const bool sok = m0 + sr < rows;
  const uint8_t *srow = a.rec + (long)min(m0 + min(sr, Q6S - 1), rows - 1) * stages * 64;
  u4_t c1 = {0, 0, 0, 0}, c2 = c1, xf;
  u2_t hb = {0, 0};  // high bits, or the scales (x) and d (y)
  float xsv = 0.f;
  // this thread's 16 bytes of the stage's X fragments: fragment (half, token tile) tid / 32
  const int xh = tid / (32 * NJ), xj = (tid >> 5) % NJ;
  const uint8_t *xfp = xq + (long)((n0 >> 4) + xj) * kbs * 512 + xh * 512 + 16 * (tid & 31);
  const float *xsp = a.xs + (long)((n0 >> 4) + ((tid >> 4) % NJ)) * kbs * 16 + (tid / (16 * NJ)) * 16 + (tid & 15);
  auto load = [&](int s) {
    const uint8_t *rp = srow + (long)s * 64;
    if (sq) {
      c1 = *(const u4_t *)(rp + 16);
      c2 = *(const u4_t *)(rp + 32);
      hb = *(const u2_t *)(rp + 48 + 8 * sh);
    } else if (ss) {
      hb = *(const u2_t *)rp;
    }
    if (tid < 32 * NJ) xsv = xsp[(long)s * 32];
    xf = *(const u4_t *)(xfp + (long)s * 1024);
  };
  auto store = [&](int buf) {
    if (sq) {
      // element 16 qq + i of half sh: its low 4 bits are nibble sh of byte i of
      // c1 / c2, its high 2 bits at bits 2 i of dword qq of hb
      uint8_t *fr = &Aq[buf][sh][sr >> 4][0];
#pragma unroll
      for (int j = 0; j < 4; j++) {  // codes 8 j .. 8 j + 7: lane slot (row % 16) + 16 j
        uint32_t out[2];
#pragma unroll
        for (int e = 0; e < 2; e++) {
          const int i0 = 8 * (j & 1) + 4 * e;
          const uint32_t lo = ((j >> 1 ? c2 : c1)[i0 >> 2] >> (4 * sh)) & 0x0F0F0F0Fu;
          const uint32_t b2 = (hb[j >> 1] >> (2 * i0)) & 0xFFu;
          const uint32_t hi = (b2 | (b2 << 6) | (b2 << 12) | (b2 << 18)) & 0x03030303u;
          out[e] = sok ? ((((lo | (hi << 4)) | 0x80808080u) - 0x20202020u) ^ 0x80808080u) : 0u;  // q - 32
        }
        *(uint2 *)(fr + ((sr & 15) + 16 * j) * 8) = make_uint2(out[0], out[1]);
      }
    } else if (ss) {
#pragma unroll
      for (int g = 0; g < 4; g++) Sc[buf][g][sr] = (int)(int8_t)(hb[0] >> (8 * g));
      Dd[buf][sr] = sok ? h2f(hb[1]) : 0.f;
    }
    if (tid < 32 * NJ) Xs[buf][tid / (16 * NJ)][(tid >> 4) % NJ][tid & 15] = xsv;
    *(u4_t *)&Xb[buf][xh][xj][16 * (tid & 31)] = xf;
  };
  f32x4_t y[NJ], acc[NJ];
#pragma unroll
  for (int jn = 0; jn < NJ; jn++) y[jn] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const int rr0 = 16 * wave + 4 * (lane >> 4);  // this lane's rows rr0 .. rr0 + 3 of the block
  auto compute = [&](int s) {
    const int buf = s & 1;
    const f32x4_t dd = *(const f32x4_t *)&Dd[buf][rr0];
    if (!PROD && (s & 3) == 0) {
#pragma unroll
      for (int jn = 0; jn < NJ; jn++) acc[jn] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const long c = *(const long *)&Aq[buf][h][wave][lane * 8];
      const long ca = lane < 32 ? c : 0, cb = lane < 32 ? 0 : c;  // groups 2 h and 2 h + 1
      const i32x4_t sa = *(const i32x4_t *)&Sc[buf][2 * h][rr0], sb = *(const i32x4_t *)&Sc[buf][2 * h + 1][rr0];
#pragma unroll
      for (int jn = 0; jn < NJ; jn++) {
        const long bx = *(const long *)&Xb[buf][h][jn][lane * 8];
        const i32x4_t z = {0, 0, 0, 0};
        const i32x4_t da = __builtin_amdgcn_mfma_i32_16x16x32_i8(ca, bx, z, 0, 0, 0);
        const i32x4_t db = __builtin_amdgcn_mfma_i32_16x16x32_i8(cb, bx, z, 0, 0, 0);
        const float xs = Xs[buf][h][jn][lane & 15];
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const float D = (float)(sa[r] * da[r] + sb[r] * db[r]);
          if constexpr (PROD) y[jn][r] = fmaf(dd[r] * xs, D, y[jn][r]);
          else acc[jn][r] = fmaf(xs, D, acc[jn][r]);
        }
      }
    }
    if (!PROD && (s & 3) == 3) {
#pragma unroll
      for (int jn = 0; jn < NJ; jn++)
#pragma unroll
        for (int r = 0; r < 4; r++) y[jn][r] = fmaf(dd[r], acc[jn][r], y[jn][r]);
    }
  };
  load(0);
  store(0);
  __syncthreads();
  for (int s = 0; s < stages; s++) {
    const bool more = s + 1 < stages;
    if (more) load(s + 1);
    compute(s);
    if (more) store((s + 1) & 1);
    __syncthreads();
  }
#pragma unroll
  for (int jn = 0; jn < NJ; jn++) {
    const int t = n0 + 16 * jn + (lane & 15);
    if (t >= a.n) continue;
#pragma unroll
    for (int r = 0; r < 4; r++)
      if (m0 + rr0 + r < rows) a.y[(long)t * rows + m0 + rr0 + r] = y[jn][r];
  }
}

template <int FMT>
void (*q8_kernel(int nj, int units))(Q8Args) {
  if (units == 1) return nj == 1 ? k_gemm_q8<FMT, 1, true> : k_gemm_q8<FMT, 2, true>;
  return nj == 1 ? k_gemm_q8<FMT, 1, false> : k_gemm_q8<FMT, 2, false>;
}
}  // namespace

size_t gemm_q8_workspace_bytes(const Layout &L, int n, int num_cus) {
  return q8_bytes(q8_plan(L.dtype, L.rows, L.units, n, num_cus), L.rows, L.units, n).total();
}

hipError_t launch_gemm_q8(const gq_weight *w, const float *X, int n, float *Y, void *workspace, int num_cus,
                          hipStream_t st) {
  const Layout &L = w->L;
  if (!w->gemm_raw) return hipErrorInvalidValue;
  const Q8Plan p = q8_plan(L.dtype, L.rows, L.units, n, num_cus);
  const Q8Bytes bytes = q8_bytes(p, L.rows, L.units, n);
  char *ws = (char *)workspace;
  uint16_t *xq = (uint16_t *)ws;
  float *xs = (float *)(ws += bytes.xq);
  uint16_t *xm = (uint16_t *)(ws += bytes.xs);
  float *part = (float *)(ws += bytes.xm);
  const long blocks = (long)(p.npad / 16) * L.units * 2, tiles = (long)p.tiles * p.ntiles * p.ksplit;
  if (blocks > 0x7fffffffL || tiles > 0x7fffffffL) return hipErrorInvalidValue;
  hipLaunchKernelGGL(p.small ? k_x_to_q8<true> : k_x_to_q8<false>, dim3((unsigned)blocks), dim3(256), 0, st, X, n,
                     p.npad, L.k, L.units, xq, xs, L.dtype == T_Q4_K ? xm : nullptr);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  Q8Args a{};
  a.rec = w->gemm_raw;
  a.xq = xq;
  a.xm = xm;
  a.xs = xs;
  a.y = Y;
  a.part = p.ksplit > 1 ? part : nullptr;
  a.rows = L.rows;
  a.n = n;
  a.kpad = L.units * 256;
  a.ntiles = p.ntiles;
  a.ksplit = p.ksplit;
  if (p.small) {
    hipLaunchKernelGGL(L.units == 1 ? k_gemm_q6_small<true> : k_gemm_q6_small<false>,
                       dim3((unsigned)p.tiles, (unsigned)p.ntiles), dim3(256), 0, st, a);
    return hipGetLastError();
  }
  void (*kern)(Q8Args) = L.dtype == T_Q4_K ? q8_kernel<T_Q4_K>(p.nj, L.units) : q8_kernel<T_Q6_K>(p.nj, L.units);
  hipLaunchKernelGGL(kern, dim3((unsigned)tiles), dim3(512), 0, st, a);
  if ((e = hipGetLastError()) != hipSuccess || p.ksplit == 1) return e;
  return launch_gemm_reduce(part, Y, (long)n * L.rows, p.ksplit, st);
}

}  // namespace gq
