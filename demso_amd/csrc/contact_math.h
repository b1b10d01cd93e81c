// contact_math.h -- the contact-list walk's root and quotients: the floats of
// sqrtf and of a division in fewer operations.
#pragma once

#include <hip/hip_runtime.h>
#include <math.h>

namespace dem {

// RN(sqrt(x)) and y = 1 / sqrt(x) to within 2^-20 (NaN where x is not in
// [2^-96, 2^96]: NaN, 0 and the far ends take sqrtf).  s = x y is corrected
// once by Newton's step for the root, s + (x - s s) y / 2, with the residual
// exact in a fused operation, as Markstein corrects a root: that rounds
// correctly for every mantissa if y is the rounded 1 / sqrt(x), and misses a
// few if y is a unit off, so what v_rsq gives decides
// (tests/contact_math_check.hip compares all 1.6 billion of these floats with
// sqrtf).  Five operations instead of sqrtf's seventeen, which scale and test
// two neighbours.
__device__ __forceinline__ float root(float x, float& y) {
  y = __builtin_nanf("");
  if (__builtin_expect(!(x >= 0x1p-96f && x <= 0x1p96f), 0)) return sqrtf(x);
  y = __builtin_amdgcn_rsqf(x);
  const float s = x * y;
  return __builtin_fmaf(__builtin_fmaf(-s, s, x), 0.5f * y, s);
}

// a / b and c / b rounded to float, given y within 2^-20 of 1 / b (or NaN).
// 1 / b in double (e = 1 - b y, y (1 + e + e^2): within 2^-52 of it for every
// b and y that root() returns), times a: within 2^-51 of a / b, which lies at
// least 2^-49 from every midpoint of two normal floats (a midpoint of 25 bits
// times b's 24 has 49), so the product rounds to the same float.  Where a
// quotient is subnormal or NaN (so for y NaN) both are divided.  Thirteen
// operations for the two instead of 22.
__device__ __forceinline__ void quotients(float a, float c, float b, float y, float& qa, float& qc) {
  const double bd = (double)b, yd = (double)y;
  const double e = __builtin_fma(-bd, yd, 1.0);
  const double inv = __builtin_fma(yd, __builtin_fma(e, e, e), yd);
  qa = (float)((double)a * inv);
  qc = (float)((double)c * inv);
  constexpr int kOdd = 0x3 | 0x10 | 0x80;  // NaN, subnormal
  if (__builtin_expect(__builtin_amdgcn_classf(qa, kOdd) || __builtin_amdgcn_classf(qc, kOdd), 0)) {
    qa = a / b;
    qc = c / b;
  }
}

}  // namespace dem
