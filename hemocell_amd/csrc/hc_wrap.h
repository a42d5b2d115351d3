// hc_wrap.h -- node coordinates on periodic axes, as plain arithmetic shared by the
// kernels and a CPU test.
#pragma once
#include <cmath>
#include <cstdint>

#ifdef __HIPCC__
#include <hip/hip_runtime.h>
#define HC_ANY __host__ __device__ __forceinline__
#else
#define HC_ANY inline
#endif

namespace hcg {

constexpr double kNearNodes = 4503599627370496.0;  // 2^52

// Coordinate of node fl (an integer, |fl| < kNearNodes) on a periodic axis of size n.
HC_ANY int wrap_node(double fl, int n) {
  double m = fl - (double)n * floor(fl / (double)n);
  if (m < 0.0) m += (double)n;
  if (m >= (double)n) m -= (double)n;
  return (int)m;
}

// The same for any finite integer (the rounded product above leaves any difference from
// 2^52 on).  A pass is exact: the quotient is off by its rounding only, and the fused
// multiply-add leaves a remainder within 2 n of an |fl| below 2^52 n, within a 2^52th of
// a larger one, where another pass follows.  Passes end for any input: no comparison
// holds for a NaN.
HC_ANY int wrap_far(double fl, int n) {
  double m = fl;
  do {
    m = fma(-floor(m / (double)n), (double)n, m);
  } while (fabs(m) > (double)n);
  if (m < 0.0) m += (double)n;
  if (m >= (double)n) m -= (double)n;
  return (int)m;
}

}  // namespace hcg
