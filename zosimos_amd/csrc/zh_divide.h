// zh_divide.h -- divisions by constants of the SrLab2 non-linearity, for device
// code and for the host test that compares them with the division.
#pragma once
#ifndef __HIPCC_RTC__  // hiprtc has the functions built in
#include <math.h>
#endif

namespace zh {

// x / c for a constant c in 3 instructions for the general division's 11: the
// product with rc = 1/c, corrected by its exact remainder (Markstein).  This is
// the rounded quotient, the sign of zero included, over every finite x for c =
// 24389, for 2700 but where x / 2700 lies half way between two subnormals
// (div_2700), and for 1.16 where |x| > 6.2e-32.  Infinite x gives NaN.
__host__ __device__ __forceinline__ float div_const(float x, float c, float rc) {
  const float q = x * rc;
  return fmaf(-fmaf(q, c, -x), rc, q);
}

// x / 2700.  A quotient half way between two subnormals is no float's exact
// remainder times the rounded 1/2700, so ties went the wrong way; they need an x
// of 1350 (2k + 1) units of 2^-149, which has more than 24 bits from 2^-124 on.
__host__ __device__ __forceinline__ float div_2700(float x) {
  if (x != 0.0f && fabsf(x) < 0x1p-124f) return x / 2700.0f;
  return div_const(x, 2700.0f, 1.0f / 2700.0f);
}

}  // namespace zh
