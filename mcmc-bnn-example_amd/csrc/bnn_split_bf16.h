// FP32 values as sums of three bf16 parts, and the matrix instruction that takes them.
#pragma once

#include <hip/hip_runtime.h>

#include "bnn_kernel_common.h"

namespace bnn {

// A number that is infinite, or rounds to an infinite bf16 (beyond 3.3895e38), has no such parts: m and l come out NaN,
// and so does every product with them.  A wave whose sums come out NaN takes its tiles again, those with a NaN among
// their row sums on FP32 matrix instructions, which carry infinity as FP32 arithmetic does (again_in_fp32).
constexpr float LARGEST_BF16 = 0x1.FEp127f;
typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));

// D = A B + C on v_mfma_f32_16x16x32_bf16: lane 16 q + n holds A[n][8 q + i], B[8 q + i][n] (i < 8) and
// C[4 q + j][n] (j < 4).  Products are exact in FP32; what the sums round to is measured against 64 bits in the
// tests.
__device__ __forceinline__ f4 mfma_bf16(bf8 a, bf8 b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// x = h + m + l: h is x rounded to bf16 (to nearest), m the rest rounded to bf16, l what is left.  A 24-bit
// significand leaves at most 16 bits after h and 8 after m, so the split is exact (down to the subnormal
// range of the parts).  Two values per v_cvt_pk_bf16_f32; the rounded values are taken apart with a shift and a mask.
// DOT: v_dot2_f32_bf16 with (-1, 0) or (0, -1) subtracts a rounded value without taking it apart (the difference is an
// FP32 number, so nothing is rounded): 7 instructions for two values instead of 11.  It runs on the pipe of the matrix
// instructions, though, and none of them overlaps with it: better where the card is limited by power (64 -> 128 -> 1:
// 29.8 against 30.4 ms for the same tiles), worse where it is limited by that pipe and the vector instructions
// (22 -> 40 -> 1: 1375 against 1329 cycles per tile).
template <bool DOT = false>
__device__ __forceinline__ void split2(f2 x, bf2& h, bf2& m, bf2& l) {
  if constexpr (DOT) {
    // (in scalar registers: as an inline constant the pair (-1, 0) would hang on how the instruction widens it)
    unsigned c0 = 0x0000BF80u, c1 = 0xBF800000u;
    asm("" : "+s"(c0), "+s"(c1));
    const bf2 first = __builtin_bit_cast(bf2, c0), second = __builtin_bit_cast(bf2, c1);
    h = __builtin_convertvector(x, bf2);
    const f2 r = {__builtin_amdgcn_fdot2_f32_bf16(h, first, x[0], false),
                  __builtin_amdgcn_fdot2_f32_bf16(h, second, x[1], false)};
    m = __builtin_convertvector(r, bf2);
    const f2 r2 = {__builtin_amdgcn_fdot2_f32_bf16(m, first, r[0], false),
                   __builtin_amdgcn_fdot2_f32_bf16(m, second, r[1], false)};
    l = __builtin_convertvector(r2, bf2);
  } else {
    h = __builtin_convertvector(x, bf2);
    const f2 r = {x[0] - (float)h[0], x[1] - (float)h[1]};
    m = __builtin_convertvector(r, bf2);
    const f2 r2 = {r[0] - (float)m[0], r[1] - (float)m[1]};
    l = __builtin_convertvector(r2, bf2);
  }
}
// The parts of w * scale for a weight that stays the same for many rows: the rounding of the product goes into the
// last part.
__device__ __forceinline__ void split_scaled(float w, float scale, __bf16& h, __bf16& m, __bf16& l) {
  const float hi = w * scale;
  const float lo = __builtin_fmaf(w, scale, -hi);
  h = (__bf16)hi;
  const float r = hi - (float)h;
  m = (__bf16)r;
  l = (__bf16)((r - (float)m) + lo);
}
// ... of numbers up to the largest FP32 one: h stays finite
__device__ __forceinline__ void split2_any(f2 x, bf2& h, bf2& m, bf2& l) {
  const f2 t = {__builtin_fabsf(x[0]) > LARGEST_BF16 ? __builtin_copysignf(LARGEST_BF16, x[0]) : x[0],
                __builtin_fabsf(x[1]) > LARGEST_BF16 ? __builtin_copysignf(LARGEST_BF16, x[1]) : x[1]};
  h = __builtin_convertvector(t, bf2);
  const f2 r = {x[0] - (float)h[0], x[1] - (float)h[1]};
  m = __builtin_convertvector(r, bf2);
  const f2 r2 = {r[0] - (float)m[0], r[1] - (float)m[1]};
  l = __builtin_convertvector(r2, bf2);
}
template <bool DOT = false>
__device__ __forceinline__ void split4(f4 x, bf4& h, bf4& m, bf4& l) {
  bf2 h0, m0, l0, h1, m1, l1;
  split2<DOT>(f2{x[0], x[1]}, h0, m0, l0);
  split2<DOT>(f2{x[2], x[3]}, h1, m1, l1);
  h = __builtin_shufflevector(h0, h1, 0, 1, 2, 3);
  m = __builtin_shufflevector(m0, m1, 0, 1, 2, 3);
  l = __builtin_shufflevector(l0, l1, 0, 1, 2, 3);
}
__device__ __forceinline__ bf8 join(bf4 a, bf4 b) { return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7); }
template <bool DOT = false>
__device__ __forceinline__ void split8(f4 x0, f4 x1, bf8& h, bf8& m, bf8& l) {
  bf4 h0, m0, l0, h1, m1, l1;
  split4<DOT>(x0, h0, m0, l0);
  split4<DOT>(x1, h1, m1, l1);
  h = join(h0, h1);
  m = join(m0, m1);
  l = join(l0, l1);
}

}  // namespace bnn
