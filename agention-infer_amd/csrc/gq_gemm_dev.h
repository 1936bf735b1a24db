// gq_gemm_dev.h -- device pieces shared by the GEMM kernels: bf16 packing,
// byte conversions, loads straight to LDS with their waits, and the block
// numbering over the XCDs.
#pragma once
#include "gq_device.h"

namespace gq {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef int i32x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void_t;

// Four floats to p, aligned to 4 bytes: one store (global memory takes 16 bytes at
// any dword).  A result row of any other than 4 m rows starts anywhere, and a dword
// store per element there is four times the requests.
typedef float f32x4u_t __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ void store4(float *p, f32x4_t v) { *(f32x4u_t *)p = v; }

constexpr int FR16 = 512;  // bf16 per 1 KiB MFMA operand fragment

// fp32 -> bf16 bits, round to nearest even (NaN kept quiet).
__device__ __forceinline__ uint32_t f2bf(float f) {
  const uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (u >> 16) | 0x40u;
  return (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
}

// s_waitcnt vmcnt(N), leaving the other counters alone (gfx9 encoding).
template <int N>
__device__ __forceinline__ void wait_vm() {
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (0x7 << 4) | (0xF << 8));
}
__device__ __forceinline__ void wait_lgkm0() { __builtin_amdgcn_s_waitcnt(0xC07F); }

__device__ __forceinline__ void dma16(const void *g, void *lds) {
  __builtin_amdgcn_global_load_lds(g, (lds_void_t *)lds, 16, 0, 0);
}

// Byte K of w (0..255) as float: one v_cvt_f32_ubyteK.  Written as asm
// because the compiler otherwise folds a preceding nibble mask into a
// v_bfe per element.
template <int K>
__device__ __forceinline__ float cvt_ubyte(uint32_t w) {
  float f;
  if constexpr (K == 0) asm("v_cvt_f32_ubyte0 %0, %1" : "=v"(f) : "v"(w));
  else if constexpr (K == 1) asm("v_cvt_f32_ubyte1 %0, %1" : "=v"(f) : "v"(w));
  else if constexpr (K == 2) asm("v_cvt_f32_ubyte2 %0, %1" : "=v"(f) : "v"(w));
  else asm("v_cvt_f32_ubyte3 %0, %1" : "=v"(f) : "v"(w));
  return f;
}

__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
  const bf16x2_t v = {(__bf16)a, (__bf16)b};  // v_cvt_pk_bf16_f32: round to nearest even
  return __builtin_bit_cast(uint32_t, v);
}

// Workgroups are dealt to the 8 XCDs round-robin by id (id % 8).  The
// GEMM's block index is renumbered so that each XCD takes a contiguous range
// of it: the token tiles (and K splits) of one row tile then run on one XCD
// and read its W tile through the same L2.
__device__ __forceinline__ int xcd_block(int id, int n) {
  const int x = id & 7, j = id >> 3, q = n >> 3, r = n & 7;
  return x * q + min(x, r) + j;
}

}  // namespace gq
