/* Quotients by a corrected product: the bits of the IEEE division in fewer
 * steps of the dependent chain.  tests/test_quotients.py compares them with the
 * division for every binary32 argument. */
#ifndef HEXDYN_DIV_H
#define HEXDYN_DIV_H

#include <hip/hip_runtime.h>

namespace hexdyn {

// 1 / x with IEEE round-to-nearest for |x| in [2^-100, 2^100]: the hardware
// reciprocal with one FMA correction is the correctly rounded quotient there.
// Callers take the division outside it.
__device__ __forceinline__ bool recip_in_range(float x) {
  const float a = fabsf(x);
  return a >= 0x1p-100f && a <= 0x1p100f;
}
__device__ __forceinline__ float recip(float x) {
  const float y0 = __builtin_amdgcn_rcpf(x);
  return __builtin_fmaf(__builtin_fmaf(-x, y0, 1.0f), y0, y0);
}

// s / n for a neighbour count n in 3..7, rn = RN(1/n): the product with one
// FMA residual correction is the correctly rounded quotient for quotients in
// [2^-120, FLT_MAX] and for +0, which a relu leaves often; other inputs take
// the division.
__device__ __forceinline__ float div_count(float s, float n, float rn) {
  const float q0 = s * rn;
  const float a = fabsf(q0);
  if ((a >= 0x1p-120f && a <= 0x1.fffffep127f) || __float_as_uint(s) == 0u)
    return __builtin_fmaf(__builtin_fmaf(-q0, n, s), rn, q0);
  return s / n;
}

}  // namespace hexdyn

#endif /* HEXDYN_DIV_H */
