// int4 operands on the int8 matrix cores (gfx950): nibble unpacking and the
// epilogue's output narrowing, shared by the GEMM kernels and the fused
// decode kernel.
//
// A packed dword w holds 8 nibbles; the two dwords
//   lo = (w << 4) & 0xF0F0F0F0   (even k, each byte = 16 * nibble value)
//   hi =  w       & 0xF0F0F0F0   (odd k)
// are 8 int8 values scaled by 16 with the sign in the byte's top bit.  A and
// B go through the same k permutation, so a dot product of unpacked operands
// is 256 times the nibble dot product, removed exactly by an arithmetic >> 8.
#pragma once

#include <type_traits>

#include "common.h"
#include "rowquant.h"

namespace dscq {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

__device__ __forceinline__ v4i unpack8(uint32_t w0, uint32_t w1) {
  v4i r;
  r[0] = (int)((w0 << 4) & 0xF0F0F0F0u);
  r[1] = (int)(w0 & 0xF0F0F0F0u);
  r[2] = (int)((w1 << 4) & 0xF0F0F0F0u);
  r[3] = (int)(w1 & 0xF0F0F0F0u);
  return r;
}

template <typename OutT>
__device__ __forceinline__ OutT to_out(float v);
// The reference rounds the fp32 result, then narrows it to fp16 (two
// roundings).  Left alone, the compiler folds a preceding fp32 multiply / add
// into the narrowing (v_fma_mixlo_f16: one rounding), which differs on exact
// fp16 ties; the empty asm pins the fp32 value first.
template <>
__device__ __forceinline__ __half to_out<__half>(float v) {
  asm("" : "+v"(v));
  return __float2half_rn(v);
}
template <>
__device__ __forceinline__ float to_out<float>(float v) {
  return v;
}

// Two fp32 results narrowed to fp16 (round to nearest even) and packed, low
// half first: one v_cvt_pk_f16_f32.  The values are pinned first, so no
// preceding multiply or add is folded into the narrowing (one rounding of the
// fp32 result, as to_out<__half>).
__device__ __forceinline__ uint32_t pack_h2(float lo, float hi) {
  typedef float f2 __attribute__((ext_vector_type(2)));
  typedef _Float16 h2 __attribute__((ext_vector_type(2)));
  asm("" : "+v"(lo), "+v"(hi));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f2){lo, hi}, h2));
}

// bfloat16 results: round to nearest even of the fp32 value, pinned likewise.
template <>
__device__ __forceinline__ bf16 to_out<bf16>(float v) {
  asm("" : "+v"(v));
  return __builtin_bit_cast(bf16, (__bf16)v);
}
__device__ __forceinline__ uint32_t pack_b2(float lo, float hi) {
  typedef float f2 __attribute__((ext_vector_type(2)));
  typedef __bf16 b2 __attribute__((ext_vector_type(2)));
  asm("" : "+v"(lo), "+v"(hi));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f2){lo, hi}, b2));
}
// SiLU-gated MLP activation of two bf16 pairs: h = bf16(bf16(silu(g)) * u), a bf16
// model's roundings.  silu(g) = g / (1 + e^-g) by the hardware exp2 and reciprocal
// is within 60 ulps of the fp32 value (|g| 2^-24 log2(e) ln(2) of the exponent's
// argument, |g| < 128 where it matters, plus a few), so its bf16 rounding is that
// value's unless the low half lies within 128 ulps of a tie; there, and where the
// reciprocal would be subnormal, it is recomputed with expf and IEEE division, as
// torch's silu does.
__device__ __forceinline__ uint32_t silu_mul_bf16x2(uint32_t g2, uint32_t u2) {
  float h[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const float g = __uint_as_float(i ? g2 & 0xFFFF0000u : g2 << 16);
    const float u = __uint_as_float(i ? u2 & 0xFFFF0000u : u2 << 16);
    const float e = __builtin_amdgcn_exp2f(g * -1.4426950408889634f);
    float s = g * __builtin_amdgcn_rcpf(1.0f + e);
    const uint32_t low = __float_as_uint(s) & 0xFFFFu;
    if (low - (0x8000u - 128u) <= 256u || !(e < 0x1p125f)) {
      asm volatile("" ::: "memory");  // keeps the exact form behind the branch
      s = g / (1.0f + expf(-g));
    }
    h[i] = (float)(__bf16)s * u;
  }
  return pack_b2(h[0], h[1]);
}

template <typename OutT>
__device__ __forceinline__ uint32_t pack_pair(float lo, float hi) {
  if constexpr (std::is_same<OutT, bf16>::value) return pack_b2(lo, hi);
  else return pack_h2(lo, hi);
}

// The same for either 16-bit type (fp16: silu_mul_f16x2 of rowquant.h).
template <typename OutT>
__device__ __forceinline__ uint32_t silu_mul_x2(uint32_t g2, uint32_t u2) {
  if constexpr (std::is_same<OutT, bf16>::value) return silu_mul_bf16x2(g2, u2);
  else return silu_mul_f16x2(g2, u2);
}

}  // namespace dscq
