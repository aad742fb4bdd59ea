// GELU in its erf form, for the epilogues of products.
#pragma once
#include "common.h"

namespace nga {

// x Phi(x). Phi(-|x|) = 2^(-x^2 / (2 ln 2) + R(|x|)): R, the logarithm of a scaled erfc, is smooth, here its minimax polynomial on
// [0, 7.5], weighted by what an error of it does to the result (beyond, its value at 7.5). No branches: with erff's, which diverge, the
// kernel of gemm_nt.hip takes 274 us for 190 at 19,264 x 4,096 of K 1,024, that of gemm_skinny.hip 17.0 for 14.7 at 1,024 x 4,096 (its
// stores included). By itself in fp32, largest error against 64 bits, with erff / so: x in [-6, -5] 8.3e-8 / 1.8e-10, [-4, -3] 6.0e-8 /
// 5.9e-9, [-2, -1] 4.7e-8 / 5.5e-8, [-1, 0] 3.5e-8 / 4.9e-8, [0, 1] 8.4e-8 / 9.3e-8, [1, 3] 2.5e-7 / 2.1e-7; relative 1.3e-4 at most
// down to -7.5, where 1 + erf has no digit left from -5.5 on. The rounding to bf16 behind it is up to 2^-8:
// of its results 7e-6 to 1.1e-5 above -1 round another way than in 64 bits (erff 6e-6 to 1.0e-5), below 1.6e-5 to 1.5 % (3e-5 to 99 %). Root mean square in
// fp32, erff / so: [-0.5, 0] 4.4e-9 / 6.7e-9, [0, 0.5] 7.4e-9 / 9.9e-9, elsewhere smaller than erff's: [-2, -1] 1.9e-8 / 1.1e-8, [1, 2] 4.8e-8 / 4.3e-8.
__device__ __forceinline__ float gelu_f(float x) {
  const float a = fabsf(x), c = __builtin_amdgcn_fmed3f(a, 0.f, 7.5f);
  float p = __builtin_fmaf(-1.84474267e-8f, c, 6.14227645e-7f);
  p = __builtin_fmaf(p, c, -8.58164822e-6f);
  p = __builtin_fmaf(p, c, 6.38452766e-5f);
  p = __builtin_fmaf(p, c, -2.39952234e-4f);
  p = __builtin_fmaf(p, c, -7.65839359e-5f);
  p = __builtin_fmaf(p, c, 7.03580119e-3f);
  p = __builtin_fmaf(p, c, -5.24996445e-2f);
  p = __builtin_fmaf(p, c, 2.62145728e-1f);
  p = __builtin_fmaf(p, c, -1.15110648f);
  p = __builtin_fmaf(p, c, -0.99999994f);
  const float q = __builtin_amdgcn_exp2f(__builtin_fmaf(-0.721347511f * a, a, p));
  return x * (x < 0.f ? q : 1.f - q);
}

}  // namespace nga
