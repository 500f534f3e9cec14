// gemhip_math.h -- constants and scalar arithmetic shared by every transport kernel.
//
// Everything here must round exactly like the reference build (gfortran for the
// x86-64 baseline: no FMA, IEEE divide and sqrt, glibc pow).  The library is
// compiled with -ffp-contract=off, so a*b+c stays two rounded operations; a divide
// stays one, or is div_rcp, which gives its result from the divisor's correctly
// rounded reciprocal.  (The energy and momentum sources are held to a tolerance and contract.)
// The header also compiles as plain C++ on the host (GEMHIP_HD expands to nothing) so
// the CPU tests can check the scalar routines against libm.
#pragma once

#include <stdint.h>
#include <math.h>

#if defined(__HIPCC__)
#define GEMHIP_HD __host__ __device__ __forceinline__
#else
#define GEMHIP_HD inline
#endif

namespace gemhip {

constexpr int LSP = 7;  // phys_consts.in.f90:41

// phys_consts.in.f90:24-26, 82-84
constexpr double kB = 1.38064852e-23;
constexpr double elchrg = 1.60217662e-19;
constexpr double amu = 1.660539040e-27;
constexpr double mindensdiv = 1.0e-5;
constexpr double mindens = 1.0e-100, mindensnull = 1.0e-20;

// ms = [16,30,28,32,14,1,5.485799090e-4]*amu (phys_consts.in.f90:43); the product is
// a single IEEE multiply, identical whether folded at compile time or not.
GEMHIP_HD double ms(int isp) {
  return (isp == 1 ? 16.0 : isp == 2 ? 30.0 : isp == 3 ? 28.0 : isp == 4 ? 32.0
          : isp == 5 ? 14.0 : isp == 6 ? 1.0 : 5.485799090e-4) * amu;
}
// qs = [1,1,1,1,1,1,-1]*elchrg (phys_consts.in.f90:45)
GEMHIP_HD double qs(int isp) { return (isp < LSP ? 1.0 : -1.0) * elchrg; }
// gammas (phys_consts.in.f90:47-53)
GEMHIP_HD double gammas(int isp) {
  return (isp == 2 || isp == 3 || isp == 4) ? 7.0 / 5.0 : 5.0 / 3.0;
}
// collisions.f90:51-53: default-real literals converted to real64, so each value is
// the single-precision number nearest the decimal, widened.
GEMHIP_HD double thermal_coeff(int isp) {
  return isp == 1 ? (double)0.1019e-12f : isp == 2 ? (double)0.0747e-12f
       : isp == 3 ? (double)0.0754e-12f : isp == 4 ? (double)0.0701e-12f
       : isp == 5 ? (double)0.1068e-12f : (double)0.3986e-12f;
}

// Fortran MIN/MAX as gfortran evaluates them on ordered operands.
GEMHIP_HD double fmin_f(double a, double b) { return (b < a) ? b : a; }
GEMHIP_HD double fmax_f(double a, double b) { return (b > a) ? b : a; }

// x / b from y = RN(1/b), correctly rounded: q0 = RN(x y) is within a few ulps of x/b,
// the FMA residual x - b q0 is exact, and one correction step q0 + r y, rounded once,
// gives RN(x/b) (Markstein's theorem for a correctly rounded reciprocal).  v_div_fixup_f64
// gives the quotients of zeros (with their sign), infinities and NaN.  The residual is exact
// while x and the quotient are above 2^-960 or so; below, the result may be off by an ulp.
__device__ __forceinline__ double div_rcp(double x, double b, double y) {
  const double q0 = x * y;
  const double r = __builtin_fma(-b, q0, x);
  return __builtin_amdgcn_div_fixup(__builtin_fma(r, y, q0), b, x);
}

// advec.f90:438-447
GEMHIP_HD double minmod(double a, double b) {
  if (a * b <= 0.0) return 0.0;
  return (fabs(a) < fabs(b)) ? a : b;
}

GEMHIP_HD double fma_exact(double a, double b, double c) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_fma(a, b, c);
#else
  return fma(a, b, c);
#endif
}

// x**2.5 rounded to nearest, which is what glibc's pow returns for these arguments
// (its error bound is below 0.52 ulp and exact-or-correct for x^n.5 in practice; the
// CPU test checks agreement on millions of samples).  x^2.5 = x^2 * sqrt(x) is formed
// in double-double: x^2 exactly by an FMA product split, sqrt(x) to ~2^-104 by one
// Newton correction (e/(2s), with `ih` a reciprocal of 2s to about an ulp), then one final
// rounding.  For arguments between 2^-400 and 2^400, where nothing in between over- or
// underflows.
GEMHIP_HD double pow25_core(double x, double s, double ih) {
  const double e = fma_exact(-s, s, x);     // x - s*s exactly
  const double sl = e * ih;                 // sqrt(x) ~= s + sl
  const double qh = x * x;
  const double ql = fma_exact(x, x, -qh);   // x*x = qh + ql exactly
  const double ph = qh * s;
  const double pl = fma_exact(qh, s, -ph) + (qh * sl + ql * s);
  return ph + pl;
}

#if defined(__HIP_DEVICE_COMPILE__)
// sqrt(x), correctly rounded, and a reciprocal of 2 sqrt(x), for x between 2^-400 and 2^400:
// v_rsq_f64, one Goldschmidt step, two residual corrections of the root (the sequence the
// compiler's sqrt uses inside its scaling for the arguments excluded here) and a Newton step
// of the reciprocal.
__device__ __forceinline__ double sqrt_rcp(double x, double& ih) {
  const double r = __builtin_amdgcn_rsq(x);
  double g = x * r, h = 0.5 * r;
  const double d = __builtin_fma(-h, g, 0.5);
  g = __builtin_fma(g, d, g);
  h = __builtin_fma(h, d, h);
  g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
  g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
  ih = __builtin_fma(h, __builtin_fma(-h, g + g, 1.0), h);
  return g;
}

// x**2.5 and sqrt(x).  Arguments outside the core's range are scaled by an even power of two
// first (zero, negative, infinite and NaN arguments give pow's results), in a branch taken
// only by waves that hold one: written as a plain conditional around the library pow, it was
// turned into selects and every cell of the diffusion evaluated the library pow too (1600 of
// the solve's 4200 cycles per row on a 128x64x1 grid).
__device__ __forceinline__ double pow25(double x, double& root) {
  const bool out = !(x > 0x1p-400 && x < 0x1p+400);
  double ih;
  if (__builtin_expect(__any(out), 0)) {
    const int k = out ? __builtin_amdgcn_frexp_exp(x) >> 1 : 0;
    const double m = __builtin_amdgcn_ldexp(x, -2 * k);
    const double s = sqrt_rcp(m, ih);
    const double y = __builtin_amdgcn_ldexp(pow25_core(m, s, ih), 5 * k);
    root = sqrt(x);
    return x > 0.0 && x < __builtin_inf() ? y : x == 0.0 ? 0.0
           : __builtin_fabs(x) == __builtin_inf() ? __builtin_inf() : __builtin_nan("");
  }
  root = sqrt_rcp(x, ih);
  return pow25_core(x, root, ih);
}
__device__ __forceinline__ double pow25(double x) {
  double root;
  return pow25(x, root);
}
#else
GEMHIP_HD double pow25(double x, double& root) {
  root = sqrt(x);
  if (!(x > 0x1p-400 && x < 0x1p+400)) return pow(x, 2.5);
  return pow25_core(x, root, 1.0 / (2.0 * root));
}
GEMHIP_HD double pow25(double x) {
  double root;
  return pow25(x, root);
}
#endif

}  // namespace gemhip
