// Operand ranges in which every division of a stencil by a geometry value, a physical constant or
// the density is exact with qdiv_in (qdiv.hpp), so that a kernel tests its inputs once per cell
// instead of the operands of each of its divisions.
//
// A kernel may take the untested form for a cell when, over the cells its stencil reads,
//   every transported value is 0 or has magnitude in 2^-RANGE_L .. 2^RANGE_U,
//   the density lies in 2^-RANGE_R .. 2^RANGE_RU,
// and the geometry (cell sizes, their halves and squares, face denominators, extrapolation weights)
// and the static fields are in range (checked once at set-up: geometry_in_range, field_in_range).
// The bounds follow from the operations: a sum of multiples of 2^g is a multiple of 2^g, a product
// of multiples of 2^g1 and 2^g2 that is not 0 is at least 2^(g1+g2), and a double of magnitude at
// least 2^k is a multiple of 2^(k-52).  Followed through the deepest chain (interpolation,
// extrapolation, limited flux times face velocity, difference over the cell), every dividend is 0
// or at least 2^-960 and every quotient too; tests/test_division_ranges.py walks the chains.
// Nothing overflows either: the largest product stays below 2^900.  Infinities, NaN and denormals
// are out of range, so the untested form also may order values with the hardware's min and max and
// need not tell +0 from -0 inside a sum that ends in + 0.0.
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>

#include "qdiv.hpp"

namespace spruce {

constexpr int RANGE_G = 48;     // lengths (cell sizes, halves, face sums): 2^-48 .. 2^48
constexpr int RANGE_L = 170;    // transported values: 0 or at least 2^-170 (7e-52)
constexpr int RANGE_U = 150;    // and at most 2^150
constexpr int RANGE_R = 150;    // density: at least 2^-150 (7e-46)
constexpr int RANGE_RU = 40;    // and at most 2^40
constexpr int RANGE_RCP = 700;  // divisors of recip_in, arguments of sqrt_in: 2^-700 .. 2^700
constexpr int RANGE_Q = 760;    // quotients by recip_in: 0 or 2^-760 .. 2^760
constexpr double RANGE_U_V = 0x1p+150, RANGE_R_V = 0x1p-150, RANGE_RU_V = 0x1p+40;

// a cell size whose half and whose sums of up to three halves of neighbours are in range
inline bool geometry_in_range(double d) { return d >= 0x1p-46 && d <= 0x1p+46; }
inline bool field_in_range(double v) { return v == 0.0 || (fabs(v) >= 0x1p-170 && fabs(v) <= RANGE_U_V); }

#ifdef __HIPCC__
// Accumulates one lane's test over the values of a cell.
struct RangeTest {
  int emin = 0;          // least binary exponent seen; 0 and (caught by the other test) inf, NaN count as 0
  bool high = false;     // a value above 2^RANGE_U, infinite or NaN
  __device__ __forceinline__ void add(double v) {
    emin = min(emin, __builtin_amdgcn_frexp_exp(v));
    high = high || !(__builtin_fabs(v) <= RANGE_U_V);
  }
  __device__ __forceinline__ void density(double rho) { high = high || !(rho >= RANGE_R_V && rho <= RANGE_RU_V); }
  // frexp_exp(2^-L) is 1 - L
  __device__ __forceinline__ bool out() const { return high || emin < 1 - RANGE_L; }
};

// The reciprocal that the hardware's IEEE division of doubles works with, without the scaling its
// extreme exponents need: qdiv_in(a, b, recip_in(b)) is then that division's own sequence, a/b
// correctly rounded: 8 instructions instead of 11, and 3 for each further dividend.  For b within
// 2^-RANGE_RCP .. 2^RANGE_RCP and a = 0, or a within 2^-960 .. 2^900 and a/b within 2^-RANGE_Q .. 2^RANGE_Q: there
// 1/b, the quotient and the last place of the residual a - b q are normal numbers and the exponents differ
// by less than the 768 from which on the division scales its operands.  2.1e9 random operands over these
// ranges gave no difference from the division, nor sqrt_in from the square root.
__device__ __forceinline__ double recip_in(double b) {
  double y = __builtin_amdgcn_rcp(b);
  y = fma(y, fma(-b, y, 1.0), y);
  return fma(y, fma(-b, y, 1.0), y);
}

// sqrt(x) correctly rounded for x in 2^-RANGE_RCP .. 2^RANGE_RCP: Newton steps from v_rsq_f64 and two corrections
// by the exact residual, the sequence of the compiler's own square root without its scaling and
// its tests for 0 and infinity.
__device__ __forceinline__ double sqrt_in(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  double s = x * y, h = 0.5 * y;
  const double r = fma(-h, s, 0.5);
  h = fma(h, r, h);
  s = fma(s, r, s);
  s = fma(fma(-s, s, x), h, s);
  return fma(fma(-s, s, x), h, s);
}

// The hardware's minimum and maximum: std::min and std::max where neither operand is NaN, up to the
// sign of a zero.  Written as instructions because the compiler's own form first canonicalises both
// operands.
__device__ __forceinline__ double hw_min(double a, double b) {
  double r;
  asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ double hw_max(double a, double b) {
  double r;
  asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
#endif

}  // namespace spruce
