// gq_gemm_quad.hip -- bf16 GEMM for batches of up to 128 tokens, straight
// from the quad-layout weights (gfx950 MFMA).
//
// Same contraction and operands as gq_gemm.hip's bf16 mode (weights: bf16 of
// the exact dequant, activations: bf16, fp32 accumulation; WeightMap::
// matmul_batch_into, src/model/mod.rs:414-464); the 160 x 256 tiles there
// spend 256 columns of work on any shorter batch.
//
// A short batch is bound by the weight stream (and, from about 48 tokens, by
// the dequant VALU and MFMA issue beside it), so each weight byte is read
// once, by one lane, with 1 KiB contiguous loads, and dequantized once, in
// registers, for all tokens.  In the quad layout lane 16 q + r of an item
// load holds whole units: (row r, unit q) of 16 rows x 4 units.  The order of
// a contraction's depth is free as long as both operands use it, so an MFMA
// step's k-group q is taken from unit q: step s multiplies elements 8 s ..
// 8 s + 7 of the four units, and a lane's dequantized codes are its A operand
// as they stand (no LDS round trip, no shuffle).  X is written in that order
// by the pre-pass: fragment (token tile, quad, step) holds, in lane 16 q + c,
// elements 1024 quad + 256 q + 8 s .. + 7 of token c.
//
// Block: 112 rows (waves 0-6, 16 each) x all tokens, one block of 8 waves per
// CU; wave 7 streams the X fragments straight to an LDS ring that the seven
// multiply waves share (X from L2 once per block).  A wave of its own issues
// them because a wave's loads complete in order: X behind the weight stream
// would wait for HBM.  (Blocks of 4 + 1 waves ran one to a CU, not two, so
// that each SIMD's VALU sat idle behind its only wave's latencies.)  K is
// split over quads where the rows alone do not fill the CUs.  One barrier per
// piece of PS steps.
//
// What bounds it now: latency between the dequant's VALU (about 30 instructions
// per 8 elements and lane, 4 cycles each; issuing for 36% of the kernel's time on
// the SIMDs that hold a block) and the MFMAs (13%), with two waves a SIMD; the K
// split leaves the blocks 2 or 3 quads each.  3584 x 18944 Q6_K at 37 tokens: 70 us
// a call on 160 x 256 tiles, 31.5 so (kernel 63.5 and 25.8 under the profiler).
#include <algorithm>

#include "gq_gemm_dev.h"
#include "gq_internal.h"

namespace gq {

namespace {

template <int FMT> struct QW;
template <> struct QW<T_Q4_K> { static constexpr int HDR = 0; };
template <> struct QW<T_Q5_K> { static constexpr int HDR = 0; };
template <> struct QW<T_Q6_K> { static constexpr int HDR = 12; };
template <> struct QW<T_Q8_0> { static constexpr int HDR = 16; };

template <int FMT>
struct QItem {
  uint4 ch[unit_chunks(FMT)];
  uint32_t d;  // Q6_K
};

// Scale and offset of the run that elements 8 s .. 8 s + 7 of a unit belong
// to: an element is fma(ds, code, nm) (Q8_0: ds * code), each as the
// row dequant computes it.
template <int FMT>
__device__ __forceinline__ void run_scale(const QItem<FMT> &R, int s, float &ds, float &nm) {
  if constexpr (FMT == T_Q4_K || FMT == T_Q5_K) {
    const uint4 hd = R.ch[0];
    uint32_t sc, m;
    scale_min_k4(s >> 2, hd.y, hd.z, hd.w, sc, m);
    ds = h2f(hd.x) * (float)sc;
    nm = -(h2f(hd.x >> 16) * (float)m);
  } else if constexpr (FMT == T_Q6_K) {
    const int h = s >> 4, t = (s >> 2) & 3, so = 8 * h + ((s & 3) >> 1) + 2 * t;
    ds = h2f(R.d) * (float)(int8_t)(dw(R.ch + 12, so >> 2) >> (8 * (so & 3)));
    nm = -32.0f * ds;
  } else {
    const int b = s >> 2;
    ds = h2f(dw(R.ch + 16, b >> 1) >> (16 * (b & 1)));
    nm = 0.f;
  }
}

// Elements 8 s .. 8 s + 7 of the lane's unit as bf16 (round to nearest even).
template <int FMT>
__device__ __forceinline__ bf16x8_t dequant8(const QItem<FMT> &R, int s, float ds, float nm) {
  uint32_t o[4];
#pragma unroll
  for (int i = 0; i < 2; i++) {  // 4 codes each
    uint32_t q;
    if constexpr (FMT == T_Q4_K || FMT == T_Q5_K) {
      const int j = s >> 3, h = (s >> 2) & 1, w = 2 * (s & 3) + i;  // dword w of the group's 8
      const uint32_t v = dw(R.ch + (FMT == T_Q5_K ? 3 : 1) + 2 * j, w);
      q = (h ? v >> 4 : v) & 0x0F0F0F0Fu;
      if constexpr (FMT == T_Q5_K) {
        const uint32_t qh = dw(R.ch + 1, w);
        const int is = 2 * j + h;  // the fifth bit's place
        q |= (is < 4 ? qh << (4 - is) : qh >> (is - 4)) & 0x10101010u;
      }
    } else if constexpr (FMT == T_Q6_K) {
      const int h = s >> 4, t = (s >> 2) & 3, w = 2 * (s & 3) + i;
      const uint32_t v = dw(R.ch + 4 * h + 2 * (t & 1), w), hv = dw(R.ch + 8 + 2 * h, w);
      q = ((t & 2) ? v >> 4 : v) & 0x0F0F0F0Fu;
      q |= (t == 0 ? hv << 4 : t == 1 ? hv << 2 : t == 2 ? hv : hv >> 2) & 0x30303030u;
    } else {
      q = dw(R.ch, 2 * s + i);
    }
    if constexpr (FMT == T_Q8_0) {
      o[2 * i] = pack_bf16(ds * (float)(int8_t)q, ds * (float)(int8_t)(q >> 8));
      o[2 * i + 1] = pack_bf16(ds * (float)(int8_t)(q >> 16), ds * (float)(int8_t)(q >> 24));
    } else {
      asm("" : "+v"(q));  // (keeps the masks above out of the byte conversions)
      o[2 * i] = pack_bf16(fmaf(ds, ub<0>(q), nm), fmaf(ds, ub<1>(q), nm));
      o[2 * i + 1] = pack_bf16(fmaf(ds, ub<2>(q), nm), fmaf(ds, ub<3>(q), nm));
    }
  }
  return __builtin_bit_cast(bf16x8_t, make_uint4(o[0], o[1], o[2], o[3]));
}

// The block's barrier between pieces (LDS reads of the piece done).
__device__ __forceinline__ void piece_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

constexpr int NCW = GEMM_QUAD_ROWS / QROWS;  // multiply waves

// NT token tiles of 16; a piece is PS steps (PS * NT KiB of X), the ring
// holds NXR pieces (the producer counts at most 63 loads in flight).
template <int NT>
struct QRing {
  static constexpr int PS = NT <= 4 ? 8 : 4;
  static constexpr int FR = PS * NT;   // fragments per piece
  static constexpr int NXR = FR <= 8 ? 6 : FR <= 16 ? 5 : FR <= 24 ? 4 : 3;
  static constexpr int PPQ = 32 / PS;  // pieces per quad
  static_assert((NXR - 2) * FR <= 63, "vmcnt");
};

template <int FMT, int NT>
__global__ __launch_bounds__(64 * (NCW + 1)) void k_gemm_quad(GemmArgs a) {
  using R = QRing<NT>;
  constexpr int PS = R::PS, NXR = R::NXR, PPQ = R::PPQ, FR = R::FR, C = unit_chunks(FMT);
  __shared__ __align__(16) uint16_t Xs[NXR][FR * FR16];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // splits outermost: an XCD's blocks (a contiguous range) share one or two
  // slices of X in its L2
  const int b = xcd_block(blockIdx.x, gridDim.x), tiles = a.ntiles;
  const int split = b / tiles, tile = b % tiles;
  const int U = a.kpad / 256, Tq = (U + 3) >> 2;
  const int q0 = (int)((long)Tq * split / a.ksplit), q1 = (int)((long)Tq * (split + 1) / a.ksplit);
  const int pieces = (q1 - q0) * PPQ;

  if (wave == NCW) {  // X pieces q0 PPQ .. into the ring, NXR - 1 ahead
    const uint16_t *src = a.xb + ((long)q0 * 32 * 64 + lane) * 8;
    auto issue = [&](int p) {
      const int pc = min(p, pieces - 1);  // (past the end: the last piece again, into a free slot)
#pragma unroll
      for (int f = 0; f < FR; f++) {
        const int s = f / NT, nt = f % NT;
        dma16(src + ((long)nt * Tq * 32 + (long)pc * PS + s) * FR16, &Xs[p % NXR][f * FR16]);
      }
    };
    for (int p = 0; p < NXR - 1; p++) issue(p);
    wait_vm<(NXR - 2) * FR>();
    __builtin_amdgcn_s_barrier();
    for (int p = 0; p < pieces; p++) {
      issue(p + NXR - 1);
      wait_vm<(NXR - 2) * FR>();  // piece p + 1 in LDS
      __builtin_amdgcn_s_barrier();
    }
    wait_vm<0>();  // drain the clamped loads before the block ends
    return;
  }

  GemmSeg sg = a.seg[0];
#pragma unroll
  for (int i = 1; i < GEMM_MAX_SEG; i++)
    if (i < a.nseg && tile >= a.seg[i].tile_begin) sg = a.seg[i];
  const int rows = sg.rows, G = (rows + QROWS - 1) / QROWS;
  const int gw = NCW * (tile - sg.tile_begin) + wave;  // this wave's row group
  const int g = min(gw, G - 1);                      // (past the end: the last one's loads, no stores)
  const int nr = min(QROWS, rows - QROWS * g);
  const int q = lane >> 4, r = lane & 15;
  auto load = [&](QItem<FMT> &it, int t) {
    const int nq = min(4, U - 4 * t);
    const long base = (long)g * QROWS * U + (long)t * 4 * nr;  // quad_item_unit
    const int l = r < nr && q < nq ? nr * q + r : 0;            // lanes without a unit re-read lane 0's
    const uint8_t *bp = sg.body + base * (C * 16);
    const int cs = 16 * nr * nq;
#pragma unroll
    for (int c = 0; c < C; c++) it.ch[c] = ldw4(bp + (uint32_t)(c * cs + 16 * l));
    if constexpr (FMT == T_Q6_K) it.d = ldh(sg.d + base + l);
  };
  f32x4_t acc[NT];
#pragma unroll
  for (int i = 0; i < NT; i++) acc[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  QItem<FMT> cur, nxt;
  load(cur, q0);
  piece_barrier();  // piece 0 in LDS
  int p = 0;
  for (int t = q0; t < q1; t++) {
    if (t + 1 < q1) load(nxt, t + 1);
    if (4 * t + q >= U) {  // no such unit: a zero A operand (X is zero there, the unit must be finite)
      cur.ch[QW<FMT>::HDR] = make_uint4(0, 0, 0, 0);
      cur.d = 0;
    }
    // Software pipeline over the quad's 32 steps: while step s multiplies,
    // step s + 1 is dequantized and its X fragments are read (a piece's first
    // fragments after the barrier that publishes them).
    float ds, nm;
    bf16x8_t av[2], bv[2][NT];
    auto deq = [&](int s) {
      if (s % (FMT == T_Q6_K ? 2 : 4) == 0) run_scale<FMT>(cur, s, ds, nm);
      av[s & 1] = dequant8<FMT>(cur, s, ds, nm);
    };
    deq(0);
#pragma unroll
    for (int pc = 0; pc < PPQ; pc++, p++) {
      const uint16_t *B = Xs[p % NXR] + lane * 8;
      auto read = [&](int i) {
#pragma unroll
        for (int nt = 0; nt < NT; nt++) bv[i & 1][nt] = *(const bf16x8_t *)(B + (i * NT + nt) * FR16);
      };
      read(0);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < PS; i++) {
        const int s = PS * pc + i;
        if (i + 1 < PS) read(i + 1);
#pragma unroll
        for (int nt = 0; nt < NT; nt++)
          acc[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[s & 1], bv[i & 1][nt], acc[nt], 0, 0, 0);
        if (s + 1 < 32) deq(s + 1);
        __builtin_amdgcn_sched_group_barrier(0x100, NT, 0);  // the reads first,
#pragma unroll
        for (int nt = 0; nt < NT; nt++) {                    // then VALU between the MFMAs
          __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x2, 32 / NT, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      piece_barrier();
    }
    cur = nxt;
  }
  // D layout: lane holds rows 4 (lane / 16) + i of token lane % 16.
  if (gw >= G) return;
  float *Y = sg.part ? sg.part + (long)split * a.n * rows : sg.y;
  const int m = QROWS * g + 4 * q;
#pragma unroll
  for (int nt = 0; nt < NT; nt++) {
    const int t = 16 * nt + r;
    if (t >= a.n) continue;
    float *yp = Y + (long)t * rows + m;
    if (m + 3 < rows) {
      store4(yp, acc[nt]);
    } else {
#pragma unroll
      for (int i = 0; i < 4; i++)
        if (m + i < rows) yp[i] = acc[nt][i];
    }
  }
}

// X fp32 [n][k] -> bf16 quad fragments [npad/16][Tq][32 steps][64 lanes][8],
// zero past n and k.  A wave converts 4 consecutive steps of 16 tokens at
// one unit: 128-byte reads per token, 256-byte runs written.
__global__ __launch_bounds__(256) void k_x_to_quad_frag(const float *X, int n, int npad, int k, int Tq,
                                                        uint16_t *out) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  const int l = (int)(i & 63);
  const long w = i >> 6;  // (token tile, quad, unit, step / 4)
  const int nt = (int)(w / (32 * Tq)), rem = (int)(w % (32 * Tq)), t = rem >> 5, q = (rem >> 3) & 3;
  if (16 * nt >= npad) return;
  const int s = 4 * (rem & 7) + (l >> 4), c = l & 15;
  const int tok = 16 * nt + c, col = 1024 * t + 256 * q + 8 * s;
  float v[8];
  if ((k & 7) == 0) {  // one aligned 32-byte run, or all padding
    float4 a = make_float4(0.f, 0.f, 0.f, 0.f), b = a;
    if (tok < n && col < k) {
      a = *(const float4 *)(X + (long)tok * k + col);
      b = *(const float4 *)(X + (long)tok * k + col + 4);
    }
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
    v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
  } else {
#pragma unroll
    for (int e = 0; e < 8; e++) v[e] = tok < n && col + e < k ? X[(long)tok * k + col + e] : 0.f;
  }
  uint32_t o[4];
#pragma unroll
  for (int e = 0; e < 4; e++) o[e] = f2bf(v[2 * e]) | (f2bf(v[2 * e + 1]) << 16);
  *(uint4 *)(out + ((((long)nt * Tq + t) * 32 + s) * 64 + c + 16 * q) * 8) = make_uint4(o[0], o[1], o[2], o[3]);
}

template <int FMT>
void (*quad_kernel(int nt))(GemmArgs) {
  switch (nt) {
  case 1: return k_gemm_quad<FMT, 1>;
  case 2: return k_gemm_quad<FMT, 2>;
  case 3: return k_gemm_quad<FMT, 3>;
  case 4: return k_gemm_quad<FMT, 4>;
  case 6: return k_gemm_quad<FMT, 6>;
  default: return k_gemm_quad<FMT, 8>;
  }
}

}  // namespace

hipError_t launch_x_to_quad(const float *X, int n, int k, uint16_t *xb, hipStream_t st) {
  const int Tq = (k + 1023) / 1024, npad = 16 * gemm_quad_nt(n);
  const long threads = (long)(npad / 16) * Tq * 32 * 64;
  hipLaunchKernelGGL(k_x_to_quad_frag, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, st, X, n, npad, k,
                     Tq, xb);
  return hipGetLastError();
}

hipError_t launch_gemm_quad(const GemmArgs &a, int fmt, int blocks, hipStream_t st) {
  const int nt = gemm_quad_nt(a.n);
  void (*kern)(GemmArgs) = nullptr;
  switch (fmt) {
  case T_Q4_K: kern = quad_kernel<T_Q4_K>(nt); break;
  case T_Q5_K: kern = quad_kernel<T_Q5_K>(nt); break;
  case T_Q6_K: kern = quad_kernel<T_Q6_K>(nt); break;
  case T_Q8_0: kern = quad_kernel<T_Q8_0>(nt); break;
  default: return hipErrorInvalidValue;
  }
  hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(64 * (NCW + 1)), 0, st, a);
  return hipGetLastError();
}

}  // namespace gq
