// Correctly rounded division by a divisor known in advance.
//
// The Thomas recurrences divide by data-independent pivots d_k.  With
// yb = RN(1/b) prepared once (an IEEE division), the quotient RN(a/b) is
//   q0 = RN(a*yb);  r0 = a - b*q0 (fma);  q1 = RN(q0 + r0*yb)  -> faithful
//   r1 = a - b*q1 (exact, fma);  q2 = RN(q1 + r1*yb)            -> RN(a/b)
// (Markstein's theorem: if yb = RN(1/b) and q1 is within one ulp of a/b, the
// remainder r1 is exact and RN(q1 + r1*yb) is the correctly rounded quotient),
// valid when no intermediate underflows or overflows, which the callers'
// magnitudes guarantee.  It replaces the hardware division sequence, whose
// numerator-dependent part is twice as long, on the serial critical path of
// each line solve; results are bit-identical to a/b (tested on the CPU
// against division and end to end on the GPU against the oracle), up to the
// sign of a zero quotient.
#pragma once

#ifdef __HIPCC__
#define VLS_HD __host__ __device__
#else
#define VLS_HD
#endif

#include <cmath>
#include <cstdint>

namespace vls {

VLS_HD inline double div_known(double a, double b, double yb) {
  double q0 = a * yb;
  double r0 = std::fma(-b, q0, a);
  double q1 = std::fma(r0, yb, q0);
  double r1 = std::fma(-b, q1, a);
  return std::fma(r1, yb, q1);
}

// Division by a pivot in two operations: with rh = RN(1/d) and
// rl = RN(1/d - rh), fma(a, rh, RN(a rl)) (N. Brisebarre, J.-M. Muller and
// S. K. Raina, "Accelerating correctly rounded floating-point division when
// the divisor is known in advance", IEEE Trans. Computers 53 (2004)).  The
// value that the fma rounds is within 2 |rl d| 2^-53 of a/d, relatively.  With
// D = 2^t D' (D' odd) the 53-bit integer significand of d, a quotient differs
// from a midpoint of two neighbouring doubles by an odd multiple of
// 2^t / (2 D) ulp, so the result can only be wrong for the numerators at the
// first of these distances, at most two significands A with
// 2^53 A or 2^54 A = +-2^t (mod D); pivot_division_exact solves for them and
// compares the result with a / d there, which makes the rounding proven for a
// given d (no intermediate may underflow, as above: a rl is subnormal for a
// below about 2^-968).  An elimination row is a
// chain of dependent operations: c16 y, the subtraction, and 2 here against 5
// of div_known (one FP64 operation: 7 to 9 cycles).  At 129x129x64 k_line_rows
// went from 15.0 to 13.8 us, k_line from 9.4 to 8.8, the column splines with
// the moment from 18.5 to 17.7.
VLS_HD inline double div_pivot(double a, double rh, double rl) { return std::fma(a, rh, a * rl); }

inline double pivot_remainder(double d, double rh) { return std::fma(-d, rh, 1.0) / d; }

// Calls fn(a) for the 53-bit significands a whose quotient a / d lies at the
// first distance from a midpoint; false if fn returned false, or for too many
// of them (d with few significant bits).  D = 2^t odd is d's significand.
template <class F>
inline bool nearest_to_ties(uint64_t odd, int t, F fn) {
  typedef unsigned __int128 u128;
  // inverse of 2^k modulo the odd part of D
  auto inv_pow2 = [&](int k) {
    uint64_t x = 1 % odd;
    for (; k > 0; k--) x = (x & 1) ? (uint64_t)(((u128)x + odd) >> 1) : x >> 1;
    return x;
  };
  for (int k = 53; k <= 54; k++) {
    const uint64_t r = k > t ? inv_pow2(k - t) : 1 % odd;
    for (uint64_t a0 : {r, odd - r}) {
      // the 53-bit significands congruent to a0
      const uint64_t lo = 1ull << 52, hi = 1ull << 53;
      uint64_t A = a0 >= lo ? a0 : a0 + (lo - a0 + odd - 1) / odd * odd;
      int tried = 0;
      for (; A < hi; A += odd) {
        if (++tried > 4096) return false;
        if (!fn((double)A)) return false;
      }
    }
  }
  return true;
}
// d's 53-bit significand, its odd part and the power of two in it
inline uint64_t significand(double d, uint64_t &odd, int &t) {
  int e = 0;
  const uint64_t D = (uint64_t)std::ldexp(std::frexp(std::fabs(d), &e), 53);
  odd = D;
  t = 0;
  while (!(odd & 1)) odd >>= 1, t++;
  return D;
}

// Whether div_pivot(a, rh, rl) is RN(a / d) for every a (host).  The bounds
// below are those of rh, rl as the set-up makes them: others are refused.
inline bool pivot_division_exact(double d, double rh, double rl) {
  if (!std::isnormal(d) || rh != 1.0 / d || rl != pivot_remainder(d, rh)) return false;
  uint64_t odd;
  int t;
  const uint64_t D = significand(d, odd, t);
  if (odd == 1) return rl == 0.0;  // a power of two: a * rh is exact
  // 4 |rl d| D bounds the error in units of 1 / (2 D) ulp: below 2^t no
  // numerator is near enough to a midpoint, below 3 2^t only the first ones
  if (4.0 * std::fabs(rl * d) * (double)D < std::ldexp(1.0, t)) return true;
  if (!(4.0 * std::fabs(rl * d) * (double)D < 3.0 * std::ldexp(1.0, t))) return false;
  return nearest_to_ties(odd, t, [&](double a) { return div_pivot(a, rh, rl) == a / d; });
}

}  // namespace vls
