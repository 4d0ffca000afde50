// IEEE double division and square root without the range handling of the
// compiler's general sequences, for operands known to be far from the ends of
// the exponent range, and division of several numerators by one denominator.
//
// Method: the hardware's reciprocal (square root) estimate is refined by
// Newton steps in fused arithmetic, and the quotient (root) corrected by its
// exactly computed remainder (Markstein, "Computation of elementary functions on
// the IBM RISC System/6000 processor", IBM J. Res. Dev. 34, 1990).  The remainder
// is exact, and no intermediate leaves the normal range, for
//   |b| in [2^-900, 2^900], |a| zero or in [2^-900, 2^1000], |a/b| in [2^-1000, 2^1000]
// for the quotient a/b, and x in [2^-700, 2^900] for the root: callers check
// their operands and fall back to `/` and sqrt().  Markstein's theorem gives the
// correctly rounded quotient from a correctly rounded reciprocal.  The refined
// one is that but for denominators whose reciprocal lies within ~2^-100 of the
// middle of two doubles; that the quotients are the IEEE ones there as well, and
// the roots, rests on a test: random operands, such denominators, and quotients
// and roots nearest to the middle of two doubles, all bit for bit.  Of a zero
// numerator the quotient is a zero, whose sign may differ from a/b's; callers'
// results are then equal as numbers.
#pragma once
#include <hip/hip_runtime.h>

namespace m2c {

// a denominator and its refined reciprocal
struct Recip {
  double b, y;
  __device__ __forceinline__ explicit Recip(double b_) : b(b_) {
    y = __builtin_amdgcn_rcp(b);
    y = __builtin_fma(__builtin_fma(-b, y, 1.0), y, y);
    y = __builtin_fma(__builtin_fma(-b, y, 1.0), y, y);
  }
  __device__ __forceinline__ double quot(double a) const {
    const double q = a * y;
    return __builtin_fma(__builtin_fma(-b, q, a), y, q);
  }
};

// the same interface with the general division
struct PlainRecip {
  double b;
  __device__ __forceinline__ explicit PlainRecip(double b_) : b(b_) {}
  __device__ __forceinline__ double quot(double a) const { return a / b; }
};

__device__ __forceinline__ double root_in_range(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y, h = 0.5 * y;
  const double r = __builtin_fma(-h, g, 0.5);
  g = __builtin_fma(g, r, g);
  h = __builtin_fma(h, r, h);
  g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
  return __builtin_fma(__builtin_fma(-g, g, x), h, g);
}

// The arithmetic of a formula: Fast for operands in range, General for any.
struct FastMath {
  using R = Recip;
  static __device__ __forceinline__ double root(double x) { return root_in_range(x); }
};
struct GeneralMath {
  using R = PlainRecip;
  static __device__ __forceinline__ double root(double x) { return sqrt(x); }
};

// lo <= |x| <= hi (false for NaN)
__device__ __forceinline__ bool in_range(double x, double lo, double hi) { return (fabs(x) >= lo) & (fabs(x) <= hi); }

}  // namespace m2c
