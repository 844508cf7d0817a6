// dgx_dd.hpp -- double-double helpers of the basis conversion kernels
// (dgx_kernels.hip, dgx_general.hip).
#pragma once

#include <hip/hip_runtime.h>

namespace dgx
{

// Double-double arithmetic (hi + lo) for the state basis conversions: the
// state itself is known to 1 ulp, and the residual's sensitivity to the state
// (the stiff acoustic part of the operator) would amplify a conversion error
// of a few ulps, so V = B3 U is formed with error-free transformations
// (Knuth two-sum, FMA two-product) and rounded once.
struct DD
{
  double hi, lo;
};

// (not contracted: s = a + b fused with the product that b is would not be the
// sum whose error e is)
__device__ __forceinline__ DD dd_two_sum(double a, double b)
{
#pragma clang fp contract(off)
  double s  = a + b;
  double bb = s - a;
  double e  = (a - (s - bb)) + (b - bb);
  return {s, e};
}

__device__ __forceinline__ DD dd_fast(double a, double b)
{
#pragma clang fp contract(off)
  double s = a + b;
  return {s, b - (s - a)};
}

// (x.hi + x.lo) * (c + clo) + acc, renormalised per term; the compiler may fuse
// the product with the first sum, which costs the result an ulp now and then.
// Kept for the mixed forms: another last bit of a state can flip the rounding of
// an FP32 trace record.
__device__ __forceinline__ DD dd_fma(DD x, double c, double clo, DD acc)
{
  const double p = x.hi * c;
  double e = fma(x.hi, c, -p);
  e = fma(x.hi, clo, e);
  e = fma(x.lo, c, e);
  const double s = acc.hi + p, bb = s - acc.hi;
  const double lo = (acc.hi - (s - bb)) + (p - bb) + (acc.lo + e), h = s + lo;
  return {h, lo - (h - s)};
}

// Sum over a line of (x[m].hi + x[m].lo) (c[m] + clo[m]) in double-double: the
// leading products are added error-free, the errors and the small products
// plainly, and the sum is renormalised once.  The lower part is about n ulps of
// the sum, so its own rounding is below n ulp^2, as with a renormalisation per
// term (12 operations a term, 4 for the first, against 15).  LO = false:
// x.lo = 0.
template <int N, bool LO, typename X, typename C>
__device__ __forceinline__ DD dd_dot(X x, C c)
{
  double hi = 0.0, lo = 0.0;
#pragma unroll
  for (int m = 0; m < N; ++m)
  {
    const DD xm = x(m), cm = c(m);
    const double p = xm.hi * cm.hi;
    double e = fma(xm.hi, cm.hi, -p);
    e = fma(xm.hi, cm.lo, e);
    if (LO)
      e = fma(xm.lo, cm.hi, e);
    if (m == 0)
    {
      hi = p;
      lo = e;
      continue;
    }
    const DD s = dd_two_sum(hi, p);
    hi = s.hi;
    lo += s.lo + e;
  }
  return dd_fast(hi, lo);
}

}  // namespace dgx
