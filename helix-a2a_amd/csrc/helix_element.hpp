// helix_element.hpp -- element conversions and log-sum-exp arithmetic shared by the combine kernels.
#pragma once

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace helix {

using u32x2 = uint32_t __attribute__((ext_vector_type(2)));
using u32x4 = uint32_t __attribute__((ext_vector_type(4)));

// Element conversions of partial_o (4 elements per 8-byte piece).
template <int kDtype>
__device__ __forceinline__ void widen4(u32x2 piece, float (&f)[4]);
template <>
__device__ __forceinline__ void widen4<0>(u32x2 piece, float (&f)[4]) {  // bf16: the upper half of an fp32
  f[0] = __uint_as_float(piece.x << 16);
  f[1] = __uint_as_float(piece.x & 0xFFFF0000u);
  f[2] = __uint_as_float(piece.y << 16);
  f[3] = __uint_as_float(piece.y & 0xFFFF0000u);
}
template <>
__device__ __forceinline__ void widen4<1>(u32x2 piece, float (&f)[4]) {  // fp16
  f[0] = __half2float(__ushort_as_half(static_cast<unsigned short>(piece.x & 0xFFFFu)));
  f[1] = __half2float(__ushort_as_half(static_cast<unsigned short>(piece.x >> 16)));
  f[2] = __half2float(__ushort_as_half(static_cast<unsigned short>(piece.y & 0xFFFFu)));
  f[3] = __half2float(__ushort_as_half(static_cast<unsigned short>(piece.y >> 16)));
}

__device__ __forceinline__ float shuffle_xor(float v, int mask) { return __shfl_xor(v, mask, 64); }

// exp and ln on the hardware's base-2 units (v_exp_f32 / v_log_f32, about 1 ulp):
// the result is rounded to 8 or 11 mantissa bits anyway. exp(-inf) = 0,
// ln(0) = -inf, ln(x < 0) = NaN hold.
__device__ __forceinline__ float fast_exp(float x) { return __builtin_amdgcn_exp2f(x * 1.4426950408889634f); }
__device__ __forceinline__ float fast_log(float x) { return __builtin_amdgcn_logf(x) * 0.6931471805599453f; }

// log-sum-exp of head h from the 8-byte statistics piece {s0, s1} that holds it;
// NaN and +-inf count as "no contribution".
//   mode 0: piece h = {lse, unused}     mode 1: piece h = {running max, running sum}
//   mode 2: piece h/2 = {lse of head 2*(h/2), lse of head 2*(h/2)+1}
// With base2 the log-sum-exp values are base-2 logarithms (the is_lse_base_on_e=False of
// patches/dcp_alltoall_helix.py:183-186); they are brought to natural logarithms here.
__device__ __forceinline__ float lse_of_stats(uint32_t s0, uint32_t s1, int statsMode, uint32_t h, bool base2) {
  float x = __uint_as_float((statsMode == 2 && (h & 1u)) ? s1 : s0);
  if (statsMode == 1) x = x + fast_log(__uint_as_float(s1));  // running max + ln(running sum)
  else if (base2) x *= 0.6931471805599453f;
  return (isnan(x) || isinf(x)) ? -INFINITY : x;
}

// four fp32 -> one 8-byte piece of bf16 (v_cvt_pk_bf16_f32: round to nearest even, NaN stays NaN) or fp16
template <int kDtype>
__device__ __forceinline__ u32x2 narrow_piece(const float (&acc)[4]);
template <>
__device__ __forceinline__ u32x2 narrow_piece<0>(const float (&acc)[4]) {
  using f32x2 = float __attribute__((ext_vector_type(2)));
  using bf16x2 = __bf16 __attribute__((ext_vector_type(2)));
  const bf16x2 lo = __builtin_convertvector(f32x2{acc[0], acc[1]}, bf16x2);
  const bf16x2 hi = __builtin_convertvector(f32x2{acc[2], acc[3]}, bf16x2);
  u32x2 r = {__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, hi)};
  return r;
}
template <>
__device__ __forceinline__ u32x2 narrow_piece<1>(const float (&acc)[4]) {
  using f32x2 = float __attribute__((ext_vector_type(2)));
  using f16x2 = _Float16 __attribute__((ext_vector_type(2)));
  const f16x2 lo = __builtin_convertvector(f32x2{acc[0], acc[1]}, f16x2);  // round to nearest even
  const f16x2 hi = __builtin_convertvector(f32x2{acc[2], acc[3]}, f16x2);
  u32x2 r = {__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, hi)};
  return r;
}

}  // namespace helix
