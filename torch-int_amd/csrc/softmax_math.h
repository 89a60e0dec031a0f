// Arithmetic shared by the kernels that turn attention scores into int8 probabilities: one fixed
// sequence of IEEE fp32 operations, so every kernel (and a CPU restatement of the same sequence)
// produces the same bits.
#pragma once
#include "ti_common.h"

namespace ti {

// e^x for x <= 0: Cody-Waite reduction x = n ln2 + r, |r| <= ln2/2, degree-6
// polynomial in Horner form with fma, scaling by 2^n.  x below -87 gives 0, NaN too.  About 1 ulp.
// Straight-line on purpose: the out-of-range case is a select at the end, not a branch around the polynomial.  A branch per
// value costs three scalar instructions and a fetch bubble, and keeps the four values of a lane from overlapping.
// Adding 1.5 * 2^23 rounds to the nearest integer (ties to even) and leaves n in the low bits of the sum, from where one
// shift-and-add puts it into the exponent of the polynomial: p is in [0.7, 1.42] and, where n is -126, above 1, so the
// result is an ordinary number.  Same bits as rint, a conversion and a multiplication by 2^n, for every x, in four
// instructions fewer.
__device__ __forceinline__ float exp_nonpos(float x) {
  const float t = x * 1.44269504088896341f;
  const float shifted = t + 12582912.0f;
  const float n = shifted - 12582912.0f;
  float r = __builtin_fmaf(n, -0.693145751953125f, x);        // ln2 high part (exact product for |n| < 2^11)
  r = __builtin_fmaf(n, -1.42860682030941723e-6f, r);         // ln2 low part
  float p = 1.0f / 720.0f;
  p = __builtin_fmaf(p, r, 1.0f / 120.0f);
  p = __builtin_fmaf(p, r, 1.0f / 24.0f);
  p = __builtin_fmaf(p, r, 1.0f / 6.0f);
  p = __builtin_fmaf(p, r, 0.5f);
  p = __builtin_fmaf(p, r, 1.0f);
  p = __builtin_fmaf(p, r, 1.0f);
  const float v = __int_as_float((int)((unsigned)__float_as_int(p) + ((unsigned)__float_as_int(shifted) << 23)));
  return x > -87.0f ? v : 0.0f;
}

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    const float o = __shfl_xor(v, off, 64);
    v = v > o ? v : o;
  }
  return v;
}
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v = v + __shfl_xor(v, off, 64);
  return v;
}

}  // namespace ti
