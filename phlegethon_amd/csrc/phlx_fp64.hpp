// phlx_fp64.hpp -- FP64 quotients and square roots of the kernels: the bits of
// a / b and sqrt(x) in fewer instructions than the compiler's expansions.
// Host code that provides the three hardware functions can include it too (the
// arithmetic is checked that way, with seeds of any error up to the bound).
#pragma once

#ifdef __HIPCC__
#include <hip/hip_runtime.h>
#define PHLX_FP64_FN __device__ __forceinline__
namespace phlx {
// v_rcp_f64, v_rsq_f64: relative error < 2^-24
PHLX_FP64_FN double hw_rcp(double x) { return __builtin_amdgcn_rcp(x); }
PHLX_FP64_FN double hw_rsq(double x) { return __builtin_amdgcn_rsq(x); }
// v_div_fixup_f64: q, or the result of a / b where a or b is a zero, an
// infinity or NaN
PHLX_FP64_FN double hw_div_fixup(double q, double b, double a) {
  return __builtin_amdgcn_div_fixup(q, b, a);
}
}  // namespace phlx
#else
#include <cmath>
#define PHLX_FP64_FN inline
namespace phlx {
double hw_rcp(double x);
double hw_rsq(double x);
double hw_div_fixup(double q, double b, double a);
using std::fma;
}  // namespace phlx
#endif

namespace phlx {

// Quotients of one denominator.  The compiler's a / b is v_div_scale twice,
// reciprocal, four FMAs, product, remainder, v_div_fmas, v_div_fixup: 11
// instructions per quotient, nothing shared.  Here the hardware reciprocal is
// refined in one third-order step, r (1 + e + e^2), to half an ulp; a quotient is
// the product with it corrected by its exact FMA remainder (Markstein's
// theorem), and v_div_fixup puts zeros, infinities and NaN right: 4 instructions
// and 4 per quotient (3 for 1 / b).  (Without v_div_fixup an infinite
// EoS target and a face with a zero sound speed came out NaN; it costs 256^3 MHD
// 0.8 % of a step, 133 x 120 x 97 flattened hydro 1.0 %, 512^3 Helmholtz MHD 1.3 %.)
// What the missing scaling and the single step cost:
//   - 2^-1020 <= |b| <= 2^1020, or b a zero, an infinity or NaN.  A subnormal b
//     gives NaN, or 0 for a = 0.  The callers' denominators are densities, speeds
//     and their differences, cell widths, temperatures, energies, conductivities,
//     and the limiter's sum of two slopes whose product is positive (> 2^-538).
//   - for 2^-960 <= |a|, |a / b| <= 2^1000 the bits of a / b, unless that lies
//     within 2^-45 ulp of the midpoint of two numbers: there either of the two
//     (none of 1.6e10 pairs differed on gfx950, exponents to +-480, mantissas next
//     to all ones and all zeros among them; nor did their roots).
//   - below, where the remainder underflows, within 1.5 ulp of a / b: a product of
//     slopes under 1e-289 (the limiter in a decaying tail), a field as small.
struct Recip {
  double b, r;
  PHLX_FP64_FN explicit Recip(double v) : b(v) {
    const double r0 = hw_rcp(v);
    const double e = fma(-v, r0, 1.0);
    r = fma(r0, fma(e, e, e), r0);
  }
  PHLX_FP64_FN double div(double a) const { return hw_div_fixup(div_finite(a), b, a); }
  // for a normal b and a finite a
  PHLX_FP64_FN double div_finite(double a) const {
    const double q = a * r;
    return fma(fma(-b, q, a), r, q);
  }
  PHLX_FP64_FN double inv() const { return hw_div_fixup(inv_finite(), b, 1.0); }
  PHLX_FP64_FN double inv_finite() const { return fma(fma(-b, r, 1.0), r, r); }
};

// The square root: two steps of Goldschmidt's iteration from the hardware's
// reciprocal root, to an ulp, and one correction by the exact remainder, without
// the compiler's rescaling and its tests of the ends of the range (13
// instructions instead of 19).  The bits of sqrt(x) for x >= 2^-960 (with the
// midpoints' exception above), a zero, an infinity, NaN or x < 0; below 2^-960,
// where the remainder underflows, within 1.5 ulp: the squared velocity of a gas
// slower than 1e-144 in LHLLC, its square in LHLLD.
PHLX_FP64_FN double dsqrt(double x) {
  const double y = hw_rsq(x);
  double s = x * y, h = 0.5 * y;
  // y is an infinity or 0: x is -0, +0 or infinite, its own root (v_cmp_class on x
  // would hold its mask in a register: 2D hydro at 4 waves per SIMD instead of 5,
  // 3000^2 992 -> 1060 us per step)
  const bool own = h == y;
  double r = fma(-h, s, 0.5);
  s = fma(s, r, s);
  h = fma(h, r, h);
  r = fma(-h, s, 0.5);
  s = fma(s, r, s);
  s = fma(fma(-s, s, x), h, s);
  return own ? x : s;
}

}  // namespace phlx
