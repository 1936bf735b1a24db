// gq_gemm.hip -- batched prefill GEMM Y[n][m] = sum_k W[m][k] X[n][k] for
// Q4_K, Q5_K, Q6_K and Q8_0 weights (gfx950 MFMA): the bf16 kernel for long
// batches, the K split's reduction, the GEMM copy of a weight, and the choice
// between the kernels.
//
// Replaces the prefill contraction of WeightMap::matmul_batch_into
// (src/model/mod.rs:414-464: dequant each row once, dot it with every
// token) and the reference's launch_only_batch / coop batch kernels
// (src/ops/wgpu_backend/resident.rs:76-183), which it does not follow.
//
// Two modes:
//  GQ_GEMM_BF16  Each 64-element group of a W row is dequantized exactly
//                (d*sc*q - dmin*m in fp32, as dequant_q4_k) and rounded to
//                bf16 into LDS; X is converted to bf16 once (round to
//                nearest even) by a prepass.  v_mfma_f32_16x16x32_bf16,
//                fp32 accumulation.
//  GQ_GEMM_INT8  gq_gemm_q8.hip.
//
// Tiling (bf16): a block computes 160 weight rows x 256 tokens (18944 rows
// x 512 tokens -> 238 blocks, one round on 256 CUs).  K advances 64
// elements (one Q4_K group) per stage, X fragments come straight from L2 into
// the multiply waves' registers.  Most batches of up to 128 tokens take
// gq_gemm_quad.hip's kernel instead (gemm_quad_faster).
#include <algorithm>
#include <type_traits>

#include "gq_gemm_dev.h"
#include "gq_internal.h"
#include "../../include/gq.h"

namespace gq {

constexpr int BM = 160, BN = 256, BK = 64;

// ----------------------------------------------------------- prepasses
// X fp32 [n][k] -> bf16 in MFMA B-operand fragments: fragment (token tile
// nt, k-step ks) of 16 tokens x 32 k is 64 lane slots of 8 bf16 (lane l:
// token 16nt + l%16, k 32ks + 8(l/16)), fragments ordered [nt][ks], so the
// GEMM loads each one as 1 KiB of contiguous memory.  Tokens are padded
// with zeros to npad, k to kpad.  One thread per slot.
__global__ void k_x_to_bf16_frag(const float *X, int n, int npad, int k, int kpad, uint16_t *out) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;  // slot
  const int ksteps = kpad / 32;
  if (i >= (long)(npad / 16) * ksteps * 64) return;
  const int l = (int)(i & 63);
  const long f = i >> 6;
  const int nt = (int)(f / ksteps), ks = (int)(f % ksteps);
  const int t = 16 * nt + (l & 15), c0 = 32 * ks + 8 * (l >> 4);
  uint32_t o[4];
  if ((k & 7) == 0) {  // the 8 values are one aligned 32-byte run (or all padding)
    float4 a = make_float4(0.f, 0.f, 0.f, 0.f), b = a;
    if (t < n && c0 < k) {
      a = *(const float4 *)(X + (long)t * k + c0);
      b = *(const float4 *)(X + (long)t * k + c0 + 4);
    }
    o[0] = f2bf(a.x) | (f2bf(a.y) << 16);
    o[1] = f2bf(a.z) | (f2bf(a.w) << 16);
    o[2] = f2bf(b.x) | (f2bf(b.y) << 16);
    o[3] = f2bf(b.z) | (f2bf(b.w) << 16);
  } else {
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const int c = c0 + 2 * e;
      const float a = t < n && c < k ? X[(long)t * k + c] : 0.f;
      const float b = t < n && c + 1 < k ? X[(long)t * k + c + 1] : 0.f;
      o[e] = f2bf(a) | (f2bf(b) << 16);
    }
  }
  *(uint4 *)(out + 8 * i) = make_uint4(o[0], o[1], o[2], o[3]);
}

// LDS reads written as asm and waited for inside: the compiler, seeing
// loads straight to LDS still outstanding, would otherwise wait for all of
// them (vmcnt(0)) before any LDS read; the callers wait for exactly the
// loads they read.
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
// Two 16-byte LDS reads, one wait.
__device__ __forceinline__ void lds_read2_a(const uint32_t (&ad)[2], uint4 (&v)[2]) {
  u32x4_t x0, x1;
  asm volatile(
      "ds_read_b128 %0, %2\n\t"
      "ds_read_b128 %1, %3\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(x0), "=&v"(x1)
      : "v"(ad[0]), "v"(ad[1])
      : "memory");
  v[0] = make_uint4(x0[0], x0[1], x0[2], x0[3]);
  v[1] = make_uint4(x1[0], x1[1], x1[2], x1[3]);
}
// Six 16-byte LDS reads, one wait.
__device__ __forceinline__ void lds_read6(const uint32_t (&ad)[6], uint4 (&v)[6]) {
  u32x4_t x0, x1, x2, x3, x4, x5;
  asm volatile(
      "ds_read_b128 %0, %6\n\t"
      "ds_read_b128 %1, %7\n\t"
      "ds_read_b128 %2, %8\n\t"
      "ds_read_b128 %3, %9\n\t"
      "ds_read_b128 %4, %10\n\t"
      "ds_read_b128 %5, %11\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(x0), "=&v"(x1), "=&v"(x2), "=&v"(x3), "=&v"(x4), "=&v"(x5)
      : "v"(ad[0]), "v"(ad[1]), "v"(ad[2]), "v"(ad[3]), "v"(ad[4]), "v"(ad[5])
      : "memory");
  v[0] = make_uint4(x0[0], x0[1], x0[2], x0[3]);
  v[1] = make_uint4(x1[0], x1[1], x1[2], x1[3]);
  v[2] = make_uint4(x2[0], x2[1], x2[2], x2[3]);
  v[3] = make_uint4(x3[0], x3[1], x3[2], x3[3]);
  v[4] = make_uint4(x4[0], x4[1], x4[2], x4[3]);
  v[5] = make_uint4(x5[0], x5[1], x5[2], x5[3]);
}

// get_scale_min_k4 (src/quant/q4_k.rs:26-35) without branches: both forms,
// then a select on j < 4.
__device__ __forceinline__ void scale_min_k4_sel(int j, uint32_t s0, uint32_t s1, uint32_t s2,
                                                 uint32_t &sc, uint32_t &m) {
  const uint32_t a = sbyte(s0, s1, s2, j & 7), b = sbyte(s0, s1, s2, j + 4);
  const uint32_t c = sbyte(s0, s1, s2, (j - 4) & 7);
  const uint32_t lo_sc = a & 63u, lo_m = b & 63u;
  const uint32_t hi_sc = (b & 0xFu) | ((c >> 6) << 4), hi_m = (b >> 4) | ((a >> 6) << 4);
  sc = j < 4 ? lo_sc : hi_sc;
  m = j < 4 ? lo_m : hi_m;
}

// ----------------------------------------------------------- bf16 GEMM weights
// The bf16 GEMM streams its own copy of a weight, made once: per row, one
// record per 64-element stage (K-step), holding exactly the bytes the
// stage's dequant needs, so that a producer fetches each stage's rows as
// whole 16-byte chunks:
//   Q4_K: the ggml block order itself (144-byte units); a stage reads the
//                unit's 16-byte header (d, dmin, 12 scale bytes; the same
//                bytes for the unit's 4 stages, so 3 of 4 reads hit L2) and
//                the group's 32 quant bytes (byte i holds element i in its
//                low and element 32 + i in its high nibble);
//   Q6_K (64 B): chunk 0 = the 4 int8 scales of the stage's 16-element
//                groups, then d (f16); chunks 1-2 = the low 4 bits of the
//                6-bit codes in the same nibble order as Q4_K; chunk 3 = the
//                high 2 bits, dword g (16-element group g) holding element
//                16 g + i at bits 2i, 2i + 1;
//   Q5_K (64 B): chunk 0 = the unit's 16-byte header (as Q4_K); chunks
//                1-2 = the group's 32 quant bytes (as Q4_K); chunk 3 = the
//                fifth bits, dword 2 h + qq holding element 32 h + 16 qq + i
//                at bit i;
//   Q8_0 (80 B): chunk 0 = the f16 d of the stage's two 32-element blocks;
//                chunks 1-4 = the 64 int8 codes.
template <int FMT> struct GemmFmt;
template <> struct GemmFmt<T_Q4_K> { static constexpr int C = 3; };
template <> struct GemmFmt<T_Q6_K> { static constexpr int C = 4; };
template <> struct GemmFmt<T_Q5_K> { static constexpr int C = 4; };
template <> struct GemmFmt<T_Q8_0> { static constexpr int C = 5; };
// Bytes of the copy per unit (4 stages) of a row.
__host__ __device__ constexpr int gemm_unit_bytes(int fmt) {
  return fmt == T_Q4_K ? 144 : fmt == T_Q8_0 ? 320 : 256;
}
// Offset of chunk c of stage s within a row of the copy.
template <int FMT>
__device__ __forceinline__ long gemm_chunk_off(int s, int c) {
  if constexpr (FMT == T_Q4_K) return (long)(s >> 2) * 144 + (c == 0 ? 0 : 16 + 32 * (s & 3) + 16 * (c - 1));
  else return (long)s * (16 * GemmFmt<FMT>::C) + 16 * c;
}
// The chunk of a stage record holding the quant bytes of dequant task
// (half h, quarter qq).
template <int FMT>
__host__ __device__ constexpr int gemm_qs_chunk(int h, int qq) {
  return FMT == T_Q8_0 ? 1 + 2 * h + qq : 1 + qq;
}

// Record of stage j (0..3) of one unit from the unit's ggml bytes u[] (Q6_K:
// ql 0..127, qh 128..191, scales 192..207, d at 208).
__device__ void q6k_stage_record(const uint8_t *u, int j, uint8_t *rec) {
  for (int i = 0; i < 64; i++) rec[i] = 0;
  for (int g = 0; g < 4; g++) {
    for (int i = 0; i < 16; i++) {
      const int x = 16 * g + i, e = 64 * j + x;  // element of the unit (dequant_q6_k order)
      const int nh = e >> 7, r = e & 127, p = r >> 5, l = r & 31;
      const uint8_t qlb = u[64 * nh + l + 32 * (p & 1)];
      const int lo = (p >> 1) ? qlb >> 4 : qlb & 15;
      const int hi = (u[128 + 32 * nh + l] >> (2 * p)) & 3;
      // low nibble: byte 16 (g & 1) + i of chunks 1-2, nibble g >> 1
      rec[16 + 16 * (g & 1) + i] |= (uint8_t)(lo << (4 * (g >> 1)));
      rec[48 + 4 * g + (i >> 2)] |= (uint8_t)(hi << (2 * (i & 3)));
      if (i == 0) rec[g] = u[192 + 8 * nh + (l >> 4) + 2 * p];
    }
  }
  rec[4] = u[208];
  rec[5] = u[209];
}

// One thread per (row, unit): the unit's part of the GEMM copy, from the
// tiled body.
__global__ void k_gemm_records(Layout L, const uint8_t *body, const uint16_t *dd, uint8_t *out) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (long)L.rows * L.units) return;
  const int r = (int)(i / L.units), u = (int)(i % L.units);
  const int t = r / L.rt, j = (r % L.rt) * L.units + u;
  uint8_t *dst = out + ((long)r * L.units + u) * gemm_unit_bytes(L.dtype);
  if (L.dtype == T_Q4_K) {
    for (int c = 0; c < 9; c++)
      *(uint4 *)(dst + 16 * c) = *(const uint4 *)(body + chunk_offset(L, t, j, c));
  } else if (L.dtype == T_Q6_K) {
    uint8_t ub[210];
    for (int c = 0; c < 13; c++) {
      const uint4 v = *(const uint4 *)(body + chunk_offset(L, t, j, c));
      __builtin_memcpy(ub + 16 * c, &v, 16);
    }
    const uint16_t dv = dd[unit_index(L, t, j)];
    ub[208] = (uint8_t)dv;
    ub[209] = (uint8_t)(dv >> 8);
    for (int s = 0; s < 4; s++) {
      uint8_t rb[64];
      q6k_stage_record(ub, s, rb);
      for (int q = 0; q < 4; q++) {
        uint4 v;
        __builtin_memcpy(&v, rb + 16 * q, 16);
        *(uint4 *)(dst + 64 * s + 16 * q) = v;
      }
    }
  } else {
    // Q5_K (the 176 B block) or Q8_0 (8 x 32 codes, then the 8 f16 d)
    const int nc = L.dtype == T_Q5_K ? 11 : 17;
    uint8_t ub[272];
    for (int c = 0; c < nc; c++) {
      const uint4 v = *(const uint4 *)(body + chunk_offset(L, t, j, c));
      __builtin_memcpy(ub + 16 * c, &v, 16);
    }
    for (int s = 0; s < 4; s++) {
      uint8_t rb[80];
      for (int i = 0; i < 80; i++) rb[i] = 0;
      if (L.dtype == T_Q5_K) {
        for (int i = 0; i < 16; i++) rb[i] = ub[i];
        for (int i = 0; i < 32; i++) rb[16 + i] = ub[48 + 32 * s + i];
        for (int h = 0; h < 2; h++)
          for (int l = 0; l < 32; l++)  // element 32 h + l of the stage: qh[l] bit 2 s + h
            rb[48 + 4 * (2 * h + (l >> 4)) + ((l & 15) >> 3)] |=
                (uint8_t)(((ub[16 + l] >> (2 * s + h)) & 1) << (l & 7));
        for (int q = 0; q < 4; q++) {
          uint4 v;
          __builtin_memcpy(&v, rb + 16 * q, 16);
          *(uint4 *)(dst + 64 * s + 16 * q) = v;
        }
      } else {
        for (int i = 0; i < 4; i++) rb[i] = ub[256 + 4 * s + i];  // d of blocks 2 s, 2 s + 1
        for (int i = 0; i < 64; i++) rb[16 + i] = ub[64 * s + i];
        for (int q = 0; q < 5; q++) {
          uint4 v;
          __builtin_memcpy(&v, rb + 16 * q, 16);
          *(uint4 *)(dst + 80 * s + 16 * q) = v;
        }
      }
    }
  }
}

// ----------------------------------------------------------- bf16 kernel, direct X
// Block tile 160 rows x 256 tokens, 512 threads, K-steps ("stages") of 64.
// Waves 0-3 multiply: wave w owns all 160 rows x tokens 64w .. 64w + 63 of
// the tile, so no X fragment is needed by two waves and X never passes
// through LDS: each multiply wave loads its B fragments (bf16, written in
// fragment order by a pre-pass) from global memory (L2) straight into
// registers, one stage ahead.  The only LDS operand is the dequantized W
// tile (fragment-major, two slots), read once per 4 MFMAs.  Waves 4-7
// produce it: each fetches, two stages ahead, the stage records of its own 40
// rows into a ring private to the wave (straight to LDS: a producer waits only
// for its own loads) and dequantizes them (Q4_K: d*sc*q - dmin*m; Q6_K:
// d*sc*(q - 32); rounded to bf16, RNE).  One barrier per stage.
// LDS traffic per stage: 20 KiB of A written, 4 x 20 KiB read; load path per
// stage: 32 KiB of X plus the W records.
// Blocks: (row tile, token tile, K split).  A launch covers up to
// GEMM_MAX_SEG matrices sharing the input (row tiles numbered across them);
// with ksplit > 1 a block covers stages [S*s/ksplit, S*(s+1)/ksplit) and
// writes a partial product, which k_gemm_reduce sums in a fixed order.
template <int FMT>
struct Direct {
  static constexpr int TBM = 160, TBN = 256;
  static constexpr int AT_ = TBM / 16;         // row tiles (10)
  static constexpr int A_FR_ = 2 * AT_;        // A fragments per stage
  static constexpr int C = GemmFmt<FMT>::C;
  static constexpr int PROWS = TBM / 4;        // rows per producer wave (40)
  static constexpr int WSLOTS = C * PROWS;
  static constexpr int WINS = (WSLOTS + 63) / 64;
  static constexpr int TASKS = 4 * PROWS;      // 16-element dequant tasks per producer wave
  static constexpr int ROUNDS = (TASKS + 63) / 64;
  static_assert(ROUNDS == 3, "3 dequant rounds");
  static constexpr int WR = 3;
};

template <int FMT>
__global__ __launch_bounds__(512) void k_gemm_bf16_direct(GemmArgs a) {
  using R = Direct<FMT>;
  constexpr int AT_ = R::AT_, PROWS = R::PROWS, WSLOTS = R::WSLOTS, C = R::C;
  constexpr int WINS = R::WINS, WR = R::WR, TBM = R::TBM, TBN = R::TBN;
  __shared__ __align__(16) uint16_t As[2][R::A_FR_ * FR16];
  __shared__ __align__(16) uint8_t Wg[4][WR][WSLOTS * 16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int b = xcd_block(blockIdx.x, gridDim.x), split = b % a.ksplit, rest = b / a.ksplit;
  const int ntile = rest % a.ntiles, tile = rest / a.ntiles;
  GemmSeg sg = a.seg[0];
#pragma unroll
  for (int i = 1; i < GEMM_MAX_SEG; i++)
    if (i < a.nseg && tile >= a.seg[i].tile_begin) sg = a.seg[i];
  // pair: tile rows 0-79 are gate rows m0 .. m0 + 79, 80-159 the same up rows
  const bool pair = a.pair != 0;
  const int m0 = (tile - sg.tile_begin) * (pair ? TBM / 2 : TBM), n0 = ntile * TBN, rows = sg.rows;
  const int stages_all = a.kpad / BK;
  const int s0 = (int)((long)stages_all * split / a.ksplit);
  const int stages = (int)((long)stages_all * (split + 1) / a.ksplit) - s0, last = stages - 1;
  const long row_stride = (long)(stages_all / 4) * gemm_unit_bytes(FMT);

  if (wave >= 4) {
    const int pw = wave - 4;
    // matrix row of this wave's tile row PROWS * pw + rr (pair: waves 6-7
    // hold the up rows)
    const int mrow0 = m0 + PROWS * (pair ? (pw & 1) : pw);
    const uint8_t *rec = pair && pw >= 2 ? a.seg[1].rec : sg.rec;
    // W chunk slots of this wave: q = 64 i + lane (q < WSLOTS): row
    // PROWS * pw + q / C, chunk q % C of the stage record.
    const uint8_t *wsrc[WINS];
    int wc[WINS];
#pragma unroll
    for (int i = 0; i < WINS; i++) {
      const int q = min(64 * i + lane, WSLOTS - 1);
      const int row = min(mrow0 + q / C, rows - 1);
      wsrc[i] = rec + (long)row * row_stride;
      wc[i] = q % C;
    }
    auto issue_w = [&](int s) {  // this wave's rows of local stage s (clamped) into slot s % WR
      const int sg_ = s0 + min(s, last);
#pragma unroll
      for (int i = 0; i < WINS; i++)
        if (64 * i + lane < WSLOTS)
          dma16(wsrc[i] + gemm_chunk_off<FMT>(sg_, wc[i]), &Wg[pw][s % WR][1024 * i]);
    };
    // Dequantize local stage s of this wave's rows: task t = 4 rr + 2 h + qq
    // (row rr, half h of the 64 elements, 16-element quarter qq of the half),
    // t = lane + 64 round.
    auto dequant = [&](int s) {
      const int j = (s0 + s) & 3;  // group of the unit (Q4_K scale pick)
      const uint8_t *wg = Wg[pw][s % WR];
      uint4 hd[3], qs[3], qh[3];
      {
        uint32_t ad[3 * 3];
#pragma unroll
        for (int round = 0; round < 3; round++) {
          const int t = min(lane + 64 * round, R::TASKS - 1);
          const int rr = t >> 2, h = (t >> 1) & 1, qq = t & 1;
          ad[3 * round] = (uint32_t)(uintptr_t)(lds_void_t *)(wg + 16 * C * rr);
          ad[3 * round + 1] =
              (uint32_t)(uintptr_t)(lds_void_t *)(wg + 16 * C * rr + 16 * gemm_qs_chunk<FMT>(h, qq));
          ad[3 * round + 2] = (uint32_t)(uintptr_t)(lds_void_t *)(wg + 16 * C * rr + 48);
        }
        if constexpr (FMT == T_Q4_K || FMT == T_Q8_0) {
          const uint32_t a6[6] = {ad[0], ad[1], ad[3], ad[4], ad[6], ad[7]};
          uint4 v[6];
          lds_read6(a6, v);
          hd[0] = v[0]; qs[0] = v[1]; hd[1] = v[2]; qs[1] = v[3]; hd[2] = v[4]; qs[2] = v[5];
        } else {
          const uint32_t a6[6] = {ad[0], ad[1], ad[2], ad[3], ad[4], ad[5]};
          uint4 v[6];
          lds_read6(a6, v);
          hd[0] = v[0]; qs[0] = v[1]; qh[0] = v[2]; hd[1] = v[3]; qs[1] = v[4]; qh[1] = v[5];
          const uint32_t a2[2] = {ad[6], ad[7]};
          uint4 w[2];
          lds_read2_a(a2, w);
          hd[2] = w[0]; qs[2] = w[1];
          const uint32_t a1[2] = {ad[8], ad[8]};
          lds_read2_a(a1, w);
          qh[2] = w[0];
        }
      }
#pragma unroll
      for (int round = 0; round < R::ROUNDS; round++) {
        const int t = lane + 64 * round;
        if (round < R::ROUNDS - 1 || t < R::TASKS) {
          const int rr = t >> 2, h = (t >> 1) & 1, qq = t & 1;
          const int r = PROWS * pw + rr;
          const bool ok = mrow0 + rr < rows;
          const uint32_t qw[4] = {qs[round].x, qs[round].y, qs[round].z, qs[round].w};
          const uint32_t sh = 4u * (uint32_t)h;
          uint32_t o[8];
          if constexpr (FMT == T_Q4_K) {
            uint32_t sc, mn;
            scale_min_k4_sel(2 * j + h, hd[round].y, hd[round].z, hd[round].w, sc, mn);
            const float ds = ok ? h2f(hd[round].x) * (float)sc : 0.f;
            const float nm = ok ? -(h2f(hd[round].x >> 16) * (float)mn) : 0.f;
#pragma unroll
            for (int i = 0; i < 4; i++) {
              const uint32_t qv = (qw[i] >> sh) & 0x0F0F0F0Fu;
              o[2 * i] = pack_bf16(fmaf(ds, cvt_ubyte<0>(qv), nm), fmaf(ds, cvt_ubyte<1>(qv), nm));
              o[2 * i + 1] = pack_bf16(fmaf(ds, cvt_ubyte<2>(qv), nm), fmaf(ds, cvt_ubyte<3>(qv), nm));
            }
          } else if constexpr (FMT == T_Q5_K) {
            // dequant_q5_k: d * sc * q - dmin * m, q = low nibble | fifth bit << 4
            uint32_t sc, mn;
            scale_min_k4_sel(2 * j + h, hd[round].y, hd[round].z, hd[round].w, sc, mn);
            const float ds = ok ? h2f(hd[round].x) * (float)sc : 0.f;
            const float nm = ok ? -(h2f(hd[round].x >> 16) * (float)mn) : 0.f;
            const int g = 2 * h + qq;
            const uint32_t hw = g == 0 ? qh[round].x : g == 1 ? qh[round].y : g == 2 ? qh[round].z : qh[round].w;
#pragma unroll
            for (int i = 0; i < 4; i++) {
              const uint32_t x4 = (hw >> (4 * i)) & 0xFu;
              const uint32_t hi = (x4 & 1u) | ((x4 & 2u) << 7) | ((x4 & 4u) << 14) | ((x4 & 8u) << 21);
              const uint32_t qv = ((qw[i] >> sh) & 0x0F0F0F0Fu) | (hi << 4);
              o[2 * i] = pack_bf16(fmaf(ds, cvt_ubyte<0>(qv), nm), fmaf(ds, cvt_ubyte<1>(qv), nm));
              o[2 * i + 1] = pack_bf16(fmaf(ds, cvt_ubyte<2>(qv), nm), fmaf(ds, cvt_ubyte<3>(qv), nm));
            }
          } else if constexpr (FMT == T_Q8_0) {
            // dequant_q8_0: d * q, exact in fp32, then bf16
            const float d = ok ? h2f(h ? hd[round].x >> 16 : hd[round].x) : 0.f;
#pragma unroll
            for (int i = 0; i < 4; i++) {
              const uint32_t w = qw[i];
              o[2 * i] = pack_bf16(d * (float)(int8_t)(w & 0xFFu), d * (float)(int8_t)((w >> 8) & 0xFFu));
              o[2 * i + 1] = pack_bf16(d * (float)(int8_t)((w >> 16) & 0xFFu), d * (float)(int8_t)(w >> 24));
            }
          } else {
            // dequant_q6_k: (d * sc) * (q - 32), one rounding: fma(ds, q, -32 ds)
            const int g = 2 * h + qq;
            const int sc8 = (int)(int8_t)(hd[round].x >> (8 * g));
            const float ds = ok ? h2f(hd[round].y) * (float)sc8 : 0.f;
            const float nm = -32.0f * ds;
            const uint32_t hw = g == 0 ? qh[round].x : g == 1 ? qh[round].y : g == 2 ? qh[round].z : qh[round].w;
#pragma unroll
            for (int i = 0; i < 4; i++) {
              const uint32_t b2 = (hw >> (8 * i)) & 0xFFu;
              const uint32_t hi = (b2 | (b2 << 6) | (b2 << 12) | (b2 << 18)) & 0x03030303u;
              const uint32_t qv = ((qw[i] >> sh) & 0x0F0F0F0Fu) | (hi << 4);
              o[2 * i] = pack_bf16(fmaf(ds, cvt_ubyte<0>(qv), nm), fmaf(ds, cvt_ubyte<1>(qv), nm));
              o[2 * i + 1] = pack_bf16(fmaf(ds, cvt_ubyte<2>(qv), nm), fmaf(ds, cvt_ubyte<3>(qv), nm));
            }
          }
          uint16_t *dst = &As[s & 1][((h * AT_ + (r >> 4)) * 64 + (r & 15) + 32 * qq) * 8];
          *(uint4 *)dst = make_uint4(o[0], o[1], o[2], o[3]);
          *(uint4 *)(dst + 128) = make_uint4(o[4], o[5], o[6], o[7]);
        }
      }
    };
    issue_w(0);
    issue_w(1);
    wait_vm<WINS>();  // W of stage 0
    dequant(0);
    wait_lgkm0();
    __builtin_amdgcn_s_barrier();
    for (int kt = 0; kt < stages; kt++) {
      issue_w(kt + 2);
      wait_vm<WINS>();  // W of stage kt + 1
      if (kt + 1 < stages) dequant(kt + 1);
      wait_lgkm0();
      __builtin_amdgcn_s_barrier();
    }
    wait_vm<0>();  // drain the clamped loads before the block ends
    return;
  }

  // ---- multiply waves: 160 rows x 64 tokens each
  const int ksteps = a.kpad / 32;
  // fragment (token tile 4 * wave + jn of the block, k-step ks):
  // xp + (jn * ksteps + ks) * 512
  const uint16_t *xp = a.xb + ((long)((n0 >> 4) + 4 * wave) * ksteps * 64 + lane) * 8;
  // B fragments of the current stage, per 32-k half; a half is reloaded
  // with the next stage's as soon as its MFMAs are issued (half a stage of
  // lead for the L2 latency, 32 registers).
  bf16x8_t bv[2][4];
  auto load_b = [&](int s, int ks) {
    const int kk = 2 * (s0 + s) + ks;
#pragma unroll
    for (int jn = 0; jn < 4; jn++) bv[ks][jn] = *(const bf16x8_t *)(xp + ((long)jn * ksteps + kk) * 512);
  };
  f32x4_t acc[AT_][4];
#pragma unroll
  for (int i = 0; i < AT_; i++)
#pragma unroll
    for (int jn = 0; jn < 4; jn++) acc[i][jn] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  load_b(0, 0);
  load_b(0, 1);
  __builtin_amdgcn_s_barrier();  // stage 0 in LDS
  for (int kt = 0; kt < stages; kt++) {
    const uint16_t *A = As[kt & 1];
#pragma unroll
    for (int ks = 0; ks < 2; ks++) {
      // A fragments one ahead: the read of i + 1 is in flight during the
      // 4 MFMAs of i (the scheduler may not hoist more: registers).
      bf16x8_t av[2];
      av[0] = *(const bf16x8_t *)(A + ((ks * AT_) * 64 + lane) * 8);
#pragma unroll
      for (int i = 0; i < AT_; i++) {
        if (i + 1 < AT_) av[(i + 1) & 1] = *(const bf16x8_t *)(A + ((ks * AT_ + i + 1) * 64 + lane) * 8);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int jn = 0; jn < 4; jn++)
          acc[i][jn] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[i & 1], bv[ks][jn], acc[i][jn], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (kt + 1 < stages) load_b(kt + 1, ks);
    }
    __builtin_amdgcn_s_barrier();
  }
  // D layout: lane holds rows 4*(lane/16)+r (weight rows) of column lane%16 (token).
  if (pair) {  // h = silu(g) * u (ffn_gate_up, cpu_path.rs:225-227) as bf16 fragments
    const int hks = a.hkpad / 32;
#pragma unroll
    for (int i = 0; i < AT_ / 2; i++) {
      const int m = m0 + 16 * i + 4 * (lane >> 4);
      if (m >= a.hkpad) continue;
#pragma unroll
      for (int jn = 0; jn < 4; jn++) {
        const int t = n0 + 64 * wave + 16 * jn + (lane & 15);
        float h[4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const float g = acc[i][jn][r], u = acc[i + AT_ / 2][jn][r];
          h[r] = t < a.n && m + r < rows ? g / (1.0f + expf(-g)) * u : 0.f;
        }
        // columns m .. m + 3 of token t: half of a fragment slot of 8
        uint16_t *dst = a.hb + (((long)(t >> 4) * hks + (m >> 5)) * 64 + (t & 15) + 16 * ((m & 31) >> 3)) * 8 + (m & 7);
        *(uint2 *)dst = make_uint2(f2bf(h[0]) | (f2bf(h[1]) << 16), f2bf(h[2]) | (f2bf(h[3]) << 16));
      }
    }
    return;
  }
  float *Y = sg.part ? sg.part + (long)split * a.n * rows : sg.y;
#pragma unroll
  for (int i = 0; i < AT_; i++) {
    const int m = m0 + 16 * i + 4 * (lane >> 4);
#pragma unroll
    for (int jn = 0; jn < 4; jn++) {
      const int t = n0 + 64 * wave + 16 * jn + (lane & 15);
      if (t >= a.n) continue;
      float *yp = Y + (long)t * rows + m;
      if (m + 3 < rows) {
        store4(yp, acc[i][jn]);
      } else {
#pragma unroll
        for (int r = 0; r < 4; r++)
          if (m + r < rows) yp[r] = acc[i][jn][r];
      }
    }
  }
}

// y[t][r] = (add ? y[t][r] : 0) + sum_s part[s][t][r], s in order, for the
// segments of one launch at once (segment i owns blocks blk0[i] ..
// blk0[i + 1] - 1: one launch instead of one per matrix).
struct ReduceSegs {
  const float *part[GEMM_MAX_SEG];
  float *y[GEMM_MAX_SEG];
  long count[GEMM_MAX_SEG];
  int blk0[GEMM_MAX_SEG + 1];
  int nseg;
};
__global__ void k_gemm_reduce(ReduceSegs r, int ksplit, int add) {
  int si = 0;
#pragma unroll
  for (int j = 1; j < GEMM_MAX_SEG; j++)
    if (j < r.nseg && (int)blockIdx.x >= r.blk0[j]) si = j;
  const float *part = r.part[si];
  float *y = r.y[si];
  const long count = r.count[si];
  const long i = ((long)(blockIdx.x - r.blk0[si]) * blockDim.x + threadIdx.x) * 4;
  if (i >= count) return;
  if (i + 3 < count) {
    float4 s = add ? *(const float4 *)(y + i) : make_float4(0.f, 0.f, 0.f, 0.f);
    for (int k = 0; k < ksplit; k++) {
      const float4 p = *(const float4 *)(part + (long)k * count + i);
      s.x += p.x; s.y += p.y; s.z += p.z; s.w += p.w;
    }
    *(float4 *)(y + i) = s;
  } else {
    for (long e = i; e < count; e++) {
      float s = add ? y[e] : 0.f;
      for (int k = 0; k < ksplit; k++) s += part[(long)k * count + e];
      y[e] = s;
    }
  }
}

// ----------------------------------------------------------- host side
size_t gemm_records_bytes(const Layout &L) {
  return (size_t)L.rows * L.units * gemm_unit_bytes(L.dtype);
}

hipError_t launch_gemm_records(const gq_weight *w, uint8_t *out, hipStream_t st) {
  const Layout &L = w->L;
  const long n = (long)L.rows * L.units;
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_gemm_records, dim3((unsigned)((n + 127) / 128)), dim3(128), 0, st, L,
                     w->body, w->d, out);
  return hipGetLastError();
}

namespace {
struct GemmPlan {
  bool quad;                        // gq_gemm_quad.hip's kernel
  int tbm, tbn, ntiles, tiles, ksplit;
};
GemmPlan gemm_plan(const gq_weight *const *ws, int count, int n, bool quad, int num_cus) {
  GemmPlan p;
  p.quad = quad;
  p.tbm = p.quad ? GEMM_QUAD_ROWS : BM;
  p.tbn = p.quad ? 16 * gemm_quad_nt(n) : BN;
  p.ntiles = (n + p.tbn - 1) / p.tbn;
  int mt = 0;
  long rows = 0;
  for (int i = 0; i < count; i++) {
    mt += (ws[i]->L.rows + p.tbm - 1) / p.tbm;
    rows += ws[i]->L.rows;
  }
  p.tiles = mt * p.ntiles;
  const int U = ws[0]->L.units;
  p.ksplit = p.quad ? gemm_quad_ksplit(ws[0]->L.dtype, p.tiles, rows, U, n, num_cus)
                    : gemm_ksplit(p.tiles, U * 4, num_cus);
  return p;
}
}  // namespace

// The short-batch kernel takes up to 128 tokens (the largest batch whose
// accumulators and X fragments fit a wave's registers), on weights in the quad
// layout (all dense ones; not stacked experts of other than 16 m rows), where
// it is the faster one.
bool gemm_uses_quad(const gq_weight *w, int n, int num_cus) {
  return w->L.quad && n <= GEMM_QUAD_MAX && gemm_quad_faster(w->L.dtype, w->L.rows, w->L.units, n, num_cus);
}

// bf16 of X in fragment form for a batch of n (quad: gemm_uses_quad).
size_t gemm_x_elems(int units, int n, bool quad) {
  if (quad) return (size_t)16 * gemm_quad_nt(n) * ((units + 3) / 4) * 1024;
  return (size_t)((n + GEMM_NPAD - 1) / GEMM_NPAD * GEMM_NPAD) * units * 256;
}

namespace {
hipError_t launch_reduce(ReduceSegs &r, int ksplit, bool add, hipStream_t st) {
  int blocks = 0;
  for (int i = 0; i < r.nseg; i++) {
    r.blk0[i] = blocks;
    blocks += (int)((r.count[i] / 4 + 255) / 256 + 1);
  }
  r.blk0[r.nseg] = blocks;
  hipLaunchKernelGGL(k_gemm_reduce, dim3((unsigned)blocks), dim3(256), 0, st, r, ksplit, add ? 1 : 0);
  return hipGetLastError();
}
}  // namespace

size_t gemm_part_floats(const gq_weight *const *ws, int count, int n, bool quad, int num_cus, bool add) {
  const GemmPlan p = gemm_plan(ws, count, n, quad, num_cus);
  if (p.ksplit == 1 && !add) return 0;
  size_t rows = 0;
  for (int i = 0; i < count; i++) rows += (size_t)ws[i]->L.rows;
  return (size_t)p.ksplit * n * rows;
}

static size_t gemm_bf16_bytes(const gq_weight *w, int n, bool quad, int num_cus) {
  const size_t xb = gemm_x_elems(w->L.units, n, quad) * 2;
  return ((xb + 255) & ~(size_t)255) + gemm_part_floats(&w, 1, n, quad, num_cus, false) * 4 + 256;
}

size_t gemm_workspace_bytes(const gq_weight *w, int n, int mode, int num_cus) {
  if (mode == GQ_GEMM_BF16) {
    if (w->L.dtype != T_Q4_K && w->L.dtype != T_Q6_K && w->L.dtype != T_Q5_K && w->L.dtype != T_Q8_0)
      return (size_t)-1;
    return gemm_bf16_bytes(w, n, gemm_uses_quad(w, n, num_cus), num_cus);
  }
  if (w->L.dtype != T_Q4_K && w->L.dtype != T_Q6_K) return (size_t)-1;
  return gemm_q8_workspace_bytes(w->L, n, num_cus);
}

// Bytes that serve any call on w of up to gemm_room_tokens(n) tokens, in either
// mode, and the X of any bf16 call of up to n rounded up to 512.  (A shorter
// batch has fewer blocks and so may split K further, into more partial
// products than a longer one.)  The weight keeps the last answer: the search
// costs some tens of microseconds, and most calls ask the same again.
size_t gemm_workspace_bound(const gq_weight *w, int n, int num_cus) {
  const long nr = gemm_room_tokens(n);
  uint64_t *memo = const_cast<uint64_t *>(&w->gemm_room);  // nr / 256 << 41 | bytes / 256
  const uint64_t m = __atomic_load_n(memo, __ATOMIC_RELAXED);
  if (m >> 41 == (uint64_t)nr / 256) return (size_t)(m & ((1ull << 41) - 1)) * 256;
  if (nr > 0x7fffff00) return 0;
  const int nmax = (int)nr;
  size_t b = 0;
  for (int t = 1; w->L.quad && t <= GEMM_QUAD_MAX; t++)  // (a split per batch)
    b = std::max(b, gemm_bf16_bytes(w, t, true, num_cus));
  for (int t = GEMM_NPAD; t <= nmax; t += GEMM_NPAD)  // (a split per token tile)
    b = std::max(b, gemm_bf16_bytes(w, t, false, num_cus));
  if (nmax < 512) b = std::max(b, gemm_x_elems(w->L.units, 512, false) * 2 + 256);
  if (w->L.dtype == T_Q4_K || w->L.dtype == T_Q6_K)
    b = std::max(b, q8_bytes_bound(w->L.rows, w->L.units, nmax, num_cus));
  b = (b + 255) & ~(size_t)255;
  if (b >> 8 < 1ull << 41) __atomic_store_n(memo, (uint64_t)nr / 256 << 41 | b / 256, __ATOMIC_RELAXED);
  return b;
}

hipError_t launch_x_to_frag(const float *X, int n, int k, uint16_t *xb, hipStream_t st) {
  const int kpad = (k + 255) / 256 * 256;
  const int npad = (n + GEMM_NPAD - 1) / GEMM_NPAD * GEMM_NPAD;
  const long slots = (long)(npad / 16) * (kpad / 32) * 64;
  hipLaunchKernelGGL(k_x_to_bf16_frag, dim3((unsigned)((slots + 255) / 256)), dim3(256), 0, st, X,
                     n, npad, k, kpad, xb);
  return hipGetLastError();
}

hipError_t launch_gemm_bf16(const gq_weight *const *ws, float *const *ys, int count,
                            const uint16_t *xb, int n, bool quad, float *part, bool add, int num_cus,
                            hipStream_t st, int *defer) {
  if (count < 1 || count > GEMM_MAX_SEG || n <= 0 || (quad && n > GEMM_QUAD_MAX)) return hipErrorInvalidValue;
  const int fmt = ws[0]->L.dtype;
  const GemmPlan p = gemm_plan(ws, count, n, quad, num_cus);
  const bool parts = add || p.ksplit > 1;  // partial products, summed by k_gemm_reduce
  GemmArgs a{};
  a.nseg = count;
  a.ksplit = p.ksplit;
  a.n = n;
  a.kpad = ws[0]->L.units * 256;
  a.xb = xb;
  int tb = 0;
  size_t po = 0;
  for (int i = 0; i < count; i++) {
    if (ws[i]->L.dtype != fmt || ws[i]->L.units != ws[0]->L.units || !(quad ? ws[i]->L.quad != 0 : ws[i]->gemm_raw != nullptr))
      return hipErrorInvalidValue;
    a.seg[i].rec = ws[i]->gemm_raw;
    a.seg[i].body = ws[i]->body;
    a.seg[i].d = ws[i]->d;
    a.seg[i].y = ys[i];
    a.seg[i].rows = ws[i]->L.rows;
    a.seg[i].tile_begin = tb;
    a.seg[i].part = parts ? part + po : nullptr;
    tb += (ws[i]->L.rows + p.tbm - 1) / p.tbm;
    po += (size_t)p.ksplit * n * ws[i]->L.rows;
  }
  if (parts && !part) return hipErrorInvalidValue;
  a.ntiles = p.quad ? tb : p.ntiles;
  const long nb = (long)tb * p.ntiles * p.ksplit;
  if (nb > 0x7fffffffL) return hipErrorInvalidValue;
  hipError_t e;
  if (p.quad) {
    e = launch_gemm_quad(a, fmt, (int)nb, st);
  } else {
    void (*kern)(GemmArgs);
    if (fmt == T_Q5_K) kern = k_gemm_bf16_direct<T_Q5_K>;
    else if (fmt == T_Q8_0) kern = k_gemm_bf16_direct<T_Q8_0>;
    else if (fmt == T_Q4_K) kern = k_gemm_bf16_direct<T_Q4_K>;
    else if (fmt == T_Q6_K) kern = k_gemm_bf16_direct<T_Q6_K>;
    else return hipErrorInvalidValue;
    hipLaunchKernelGGL(kern, dim3((unsigned)nb), dim3(512), 0, st, a);
    e = hipGetLastError();
  }
  if (e != hipSuccess || !parts) return e;
  if (defer && add) {
    *defer = p.ksplit;
    return hipSuccess;
  }
  ReduceSegs r{};
  r.nseg = count;
  for (int i = 0; i < count; i++) {
    r.part[i] = a.seg[i].part;
    r.y[i] = a.seg[i].y;
    r.count[i] = (long)n * a.seg[i].rows;
  }
  return launch_reduce(r, p.ksplit, add, st);
}

hipError_t launch_gemm_reduce(const float *part, float *y, long count, int ksplit, hipStream_t st) {
  ReduceSegs r{};
  r.nseg = 1;
  r.part[0] = part;
  r.y[0] = y;
  r.count[0] = count;
  return launch_reduce(r, ksplit, false, st);
}

hipError_t launch_gemm_bf16_swiglu(const gq_weight *gate, const gq_weight *up, const uint16_t *xb, int n,
                                   uint16_t *hb, int num_cus, hipStream_t st) {
  (void)num_cus;
  if (n <= GEMM_QUAD_MAX) return hipErrorNotSupported;  // the short-batch kernel's
  const Layout &L = gate->L;
  if (up->L.dtype != L.dtype || up->L.units != L.units || up->L.rows != L.rows || !gate->gemm_raw ||
      !up->gemm_raw)
    return hipErrorNotSupported;
  if (L.dtype != T_Q4_K && L.dtype != T_Q6_K && L.dtype != T_Q5_K && L.dtype != T_Q8_0)
    return hipErrorNotSupported;
  GemmArgs a{};
  a.nseg = 1;
  a.ntiles = (n + BN - 1) / BN;
  a.ksplit = 1;
  a.n = n;
  a.kpad = L.units * 256;
  a.xb = xb;
  a.pair = 1;
  a.hkpad = (L.rows + 255) / 256 * 256;
  a.hb = hb;
  a.seg[0].rec = gate->gemm_raw;
  a.seg[0].rows = L.rows;
  a.seg[0].tile_begin = 0;
  a.seg[1].rec = up->gemm_raw;
  a.seg[1].rows = L.rows;
  // 80 output rows per tile, over every padded column of hb (rows past F
  // give zeros)
  const long nb = (long)((a.hkpad + BM / 2 - 1) / (BM / 2)) * a.ntiles;
  if (nb > 0x7fffffffL) return hipErrorInvalidValue;
  void (*kern)(GemmArgs) = L.dtype == T_Q4_K   ? k_gemm_bf16_direct<T_Q4_K>
                           : L.dtype == T_Q6_K ? k_gemm_bf16_direct<T_Q6_K>
                           : L.dtype == T_Q5_K ? k_gemm_bf16_direct<T_Q5_K>
                                               : k_gemm_bf16_direct<T_Q8_0>;
  hipLaunchKernelGGL(kern, dim3((unsigned)nb), dim3(512), 0, st, a);
  return hipGetLastError();
}

hipError_t launch_gemm(const gq_weight *w, const float *X, int n, float *Y, int mode,
                       void *workspace, size_t ws_bytes, int num_cus, hipStream_t st) {
  (void)ws_bytes;
  const Layout &L = w->L;
  if (mode == GQ_GEMM_BF16) {
    uint16_t *xb = (uint16_t *)workspace;
    const bool quad = gemm_uses_quad(w, n, num_cus);
    const size_t xbb = gemm_x_elems(L.units, n, quad) * 2;
    float *part = (float *)((char *)workspace + ((xbb + 255) & ~(size_t)255));
    hipError_t e = quad ? launch_x_to_quad(X, n, L.k, xb, st) : launch_x_to_frag(X, n, L.k, xb, st);
    if (e != hipSuccess) return e;
    return launch_gemm_bf16(&w, &Y, 1, xb, n, quad, part, false, num_cus, st);
  }
  return launch_gemm_q8(w, X, n, Y, workspace, num_cus, st);
}

}  // namespace gq
