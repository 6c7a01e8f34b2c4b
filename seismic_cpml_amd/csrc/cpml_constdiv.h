// Correctly rounded division by a number that stays the same for a whole
// launch (24 DELTAX, DELTAX, 24): x / d bit for bit, in 4 instructions and
// a range test of 2 instead of the 11 (one of them a quarter-rate reciprocal)
// of an IEEE division.
//
// With 1/d = c + cl, c the largest number not above it (so cl >= 0 and the sign
// of a zero survives), and ch = RN(1/d):
//   q0 = RN(x c + RN(x cl))   is less than one unit in the last place off x/d,
//   e  = q0 d - x             is exact (one fused multiply-add),
//   q  = RN(q0 - e ch)        is RN(x / d): q0 - e ch differs from x/d by
//     |x/d - q0| |ch d - 1|.  Near a midpoint of two neighbouring numbers
//     (the only place where that could matter) |x/d - q0| is half a unit, so
//     with d in [1, 2) and p bits the difference is under d 2^(-2p-1), while
//     x/d is at least 2^(1-2p)/d away from the midpoint (Markstein 1990).
// It holds for x = 0 and lo <= |x| < hi, where nothing is subnormal or
// overflows; callers take the IEEE division elsewhere (NaN goes either way).
#pragma once

#include <cmath>
#include <cstdint>
#include <cstring>
#include <limits>

#ifdef __HIPCC__
#define CPML_HD __host__ __device__ __forceinline__
#else
#define CPML_HD inline
#endif

namespace cpml {

// A number that orders |x| below a power of two bound and puts 0 on top:
// twice the magnitude bits, less one.
CPML_HD uint32_t magnitude_key(float x) {
  uint32_t u;
  std::memcpy(&u, &x, sizeof u);
  return (u << 1) - 1u;
}
CPML_HD uint32_t magnitude_key(double x) {
  uint64_t u;
  std::memcpy(&u, &x, sizeof u);
  const uint32_t low = (uint32_t)u;  // a double whose high word is 0 is not 0
  return (((uint32_t)(u >> 32) << 1) | (low != 0u ? 1u : 0u)) - 1u;
}

template <typename T>
struct ConstDiv {
  T d;             // the divisor
  T c, cl, ch;     // 1/d = c + cl rounded down; 1/d to nearest
  T hi;            // quot() holds for |x| < hi ...
  uint32_t lo;     // ... and magnitude_key(x) >= lo

  CPML_HD T quot(T x) const {
    const T q0 = std::fma(x, c, x * cl);
    const T e = std::fma(q0, d, -x);
    return std::fma(-e, ch, q0);
  }
  CPML_HD bool in_range(T x) const { return std::fabs(x) < hi && magnitude_key(x) >= lo; }
};

// Host: the constants of a positive divisor.  A divisor outside 2^-20 .. 2^40
// is always divided by plainly (hi = 0).
template <typename T>
inline ConstDiv<T> const_div(T d) {
  ConstDiv<T> k;
  k.d = d;
  k.ch = T(1) / d;
  k.c = k.ch;
  if (std::fma(d, k.c, T(-1)) > T(0)) k.c = std::nextafter(k.c, T(0));
  k.cl = std::fabs(std::fma(d, k.c, T(-1)) / d);  // 1 - d c >= 0 is exact
  constexpr int small = sizeof(T) == 4 ? -96 : -960;
  const bool fits = d >= T(0x1p-20) && d <= T(0x1p40);
  k.hi = fits ? std::ldexp(d < T(1) ? d : T(1), std::numeric_limits<T>::max_exponent - 3) : T(0);
  k.lo = magnitude_key(std::ldexp(d > T(1) ? d : T(1), small));
  return k;
}

#ifdef __HIPCC__
// a / A, b / B, c / C, d / D with one range test for the four.
template <typename T>
__device__ __forceinline__ void const_divide(T &a, const ConstDiv<T> &A, T &b,
                                             const ConstDiv<T> &B, T &c, const ConstDiv<T> &C,
                                             T &d, const ConstDiv<T> &D) {
  // the bounds of the divisors are uniform: scalar code
  const T hi = min(min(A.hi, B.hi), min(C.hi, D.hi));
  const uint32_t lo = max(max(A.lo, B.lo), max(C.lo, D.lo));
  const T m = fmax(fmax(fabs(a), fabs(b)), fmax(fabs(c), fabs(d)));
  const uint32_t k = min(min(magnitude_key(a), magnitude_key(b)),
                         min(magnitude_key(c), magnitude_key(d)));
  const T qa = A.quot(a), qb = B.quot(b), qc = C.quot(c), qd = D.quot(d);
  if (__builtin_expect(m >= hi || k < lo, 0)) {
    a = a / A.d;
    b = b / B.d;
    c = c / C.d;
    d = d / D.d;
  } else {
    a = qa, b = qb, c = qc, d = qd;
  }
}
// The same of three numbers and one divisor.
template <typename T>
__device__ __forceinline__ void const_divide(const ConstDiv<T> &D, T &a, T &b, T &c) {
  const T m = fmax(fmax(fabs(a), fabs(b)), fabs(c));
  const uint32_t k = min(min(magnitude_key(a), magnitude_key(b)), magnitude_key(c));
  const T qa = D.quot(a), qb = D.quot(b), qc = D.quot(c);
  if (__builtin_expect(m >= D.hi || k < D.lo, 0)) {
    a = a / D.d;
    b = b / D.d;
    c = c / D.d;
  } else {
    a = qa, b = qb, c = qc;
  }
}
#endif

}  // namespace cpml
