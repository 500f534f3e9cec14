// kernels_sources.hip -- the source/loss substep of a time step (src/libgemini.cpp:223-232):
// source_loss_energy, source_loss_momentum and source_loss_mass (multifluid.f90:130-175,
// 472-549) with their collisional and chemical rates (sources.f90, collisions.f90:58-159)
// and the exponential time differencing of calculus.in.f90:174-196.
//
// Each substep is one pass over the padded grid, one thread per cell.  The interior cells
// form their production and loss rates in registers and advance the conserved quantity;
// every cell (ghosts included, as the reference's whole-array statements do) then converts
// back to temperature / velocity / electron density.  The rates never touch HBM.
//
// Arithmetic follows the reference's expressions, with liberties that cost a few ulp per
// operation at most: products and sums of the energy and momentum passes contract into FMAs
// (which takes them from 3.59 and 3.71 ms to 3.33 and 3.65 at 512x256x192; the mass pass gains
// nothing by it and rounds each on its own), a divide by a compile-time constant (a mass sum,
// 3) is a multiply by its correctly rounded reciprocal, a Coulomb pair's powers of 1/Teff come
// from one reciprocal root (to an ulp or so, where the reference divides and takes a power)
// and its drift functions from polynomials.  The transcendental functions of the other rates
// (exp, log, log10, tanh, sin, and x**p for the fitted exponents) are the device library's,
// which agree with glibc to about an ulp; x**0.5 is the correctly rounded sqrt.  These passes
// therefore match the reference to rounding (the tests hold them to 1e-12 of each field's
// magnitude) rather than bit for bit.
//
// Ion-ion (Coulomb) terms: Teff, Wsj, Phisj and Psisj of coulomb_colln are symmetric in
// the species pair, so each unordered pair is evaluated once and feeds both species.  The
// pairs run in lexicographic order, which adds each species' terms in the reference's
// isp2 order; self-collision terms are exact zeros and are skipped.
//
// On 512x256x192 the energy pass moves 13.6 GB in 3.3 ms, the momentum pass 17.5 GB in 3.7, the
// mass pass 10.9 GB in 1.97: 4.1, 4.7 and 5.5 TB/s, with vector instructions at some 70, 57 and
// 60 % of the FP64 issue rate.  At two waves a SIMD the energy pass is still held by issue and
// latency, the other two by both.  The first two had some 8000 instructions a cell, at 5.5 and
// 6.5 ms: erf and exp in every pair; register arrays indexed by a rolled loop's pair, or 130
// KB of unrolled code that misses the instruction cache; the edge logarithms of a gradient
// inlined once per use.  Blocks of 128 threads are 2 to 4 % faster than 256.  Momentum
// takes 135 registers (3 waves per SIMD), reading its momenta where they are used; energy 225
// (two; at 168 it spills and took 5.1 ms against 3.33).
#include "gemhip_internal.h"

#pragma clang fp contract(fast)

namespace gemhip {
namespace {

constexpr int TPB = 128;
constexpr double PI = 3.141592653589793;   // 4*atan(1.0_wp), phys_consts.in.f90:20

// collisions.f90:11-47: default-real literals widened to real64
__device__ __forceinline__ double tab_csn(int isp, int isp2) {
  constexpr float t[7][4] = {
      {-1, 6.82e-10f, 6.64e-10f, -1},        {2.44e-10f, 4.34e-10f, 4.27e-10f, 0.69e-10f},
      {2.58e-10f, -1, 4.49e-10f, 0.74e-10f}, {2.31e-10f, 4.13e-10f, -1, 0.65e-10f},
      {4.42e-10f, 7.47e-10f, 7.25e-10f, 1.45e-10f}, {-1, 33.6e-10f, 32.0e-10f, -1},
      {-1, -1, -1, -1}};
  return (double)t[isp - 1][isp2 - 1];
}
__device__ __forceinline__ double tab_c2sn1(int isp, int isp2) {
  constexpr float t[7][4] = {
      {3.67e-11f, 0, 0, 4.63e-12f}, {0, 0, 0, 0}, {0, 5.14e-11f, 0, 0}, {0, 0, 2.59e-11f, 0},
      {0, 0, 0, 0}, {6.61e-11f, 0, 0, 2.65e-10f}, {-1, -1, -1, -1}};
  return (double)t[isp - 1][isp2 - 1];
}
__device__ __forceinline__ double tab_c2sn2(int isp, int isp2) {
  constexpr float t[7][4] = {
      {0.064f, 0, 0, -1}, {0, 0, 0, 0}, {0, 0.069f, 0, 0}, {0, 0, 0.073f, 0},
      {0, 0, 0, 0}, {0.047f, 0, 0, 0.083f}, {-1, -1, -1, -1}};
  return (double)t[isp - 1][isp2 - 1];
}
// phys_consts.in.f90:60: mn = [16,28,32,1]*amu
__device__ __forceinline__ double mn(int isp2) {
  return (isp2 == 1 ? 16.0 : isp2 == 2 ? 28.0 : isp2 == 3 ? 32.0 : 1.0) * amu;
}

// calculus.in.f90:174-196
__device__ __forceinline__ double etd(double f, double P, double L, double dt) {
#pragma clang fp contract(off)
  const double Ldt = L * dt;
  const double expL = exp(-1.0 * Ldt);
  if (Ldt > 1e-10) return f * expL + (P / L) * (1.0 - expL);
  return f + P * dt;
}

// collisions.f90:58-114 at one cell (nn2 = nn(isp2), Tsp = Ts(isp))
__device__ __forceinline__ double maxwell(int isp, int isp2, double nn2, double Tn, double Tsp) {
  if (isp < LSP) {
    const double csn = tab_csn(isp, isp2);
    if (csn < 0) {
      const double c1 = tab_c2sn1(isp, isp2);
      if (isp == 1 && isp2 == 4) {
        const double Teff = Tn + Tsp / 16.0;
        return ((c1 * sqrt(Teff)) * nn2) * 1e-6;
      }
      const double Teff = 0.5 * (Tn + Tsp);
      const double b = 1.0 - tab_c2sn2(isp, isp2) * log10(Teff);
      return (((c1 * (b * b)) * sqrt(Teff)) * nn2) * 1e-6;
    }
    return (csn * nn2) * 1e-6;
  }
  const double T = Tsp;
  switch (isp2) {
    case 1: return (((8.9e-11 * (1.0 + 5.7e-4 * T)) * sqrt(T)) * nn2) * 1e-6;
    case 2: return (((2.33e-11 * (1.0 - 1.21e-4 * T)) * T) * nn2) * 1e-6;
    case 3: return (((1.82e-10 * (1.0 + 3.6e-2 * sqrt(T))) * sqrt(T)) * nn2) * 1e-6;
    default: return (((4.5e-9 * (1.0 - 1.35e-4 * T)) * sqrt(T)) * nn2) * 1e-6;
  }
}

// collisions.f90:22-31 (Csj), times the 1e-6 of :146
__device__ __forceinline__ double csj_1e6(int x, int y) {
  constexpr float t[7][7] = {
      {0.22f, 0.26f, 0.25f, 0.26f, 0.22f, 0.077f, 1.87e-3f}, {0.14f, 0.16f, 0.16f, 0.17f, 0.13f, 0.042f, 9.97e-4f},
      {0.15f, 0.17f, 0.17f, 0.18f, 0.14f, 0.045f, 1.07e-3f}, {0.13f, 0.16f, 0.15f, 0.16f, 0.12f, 0.039f, 9.347e-4f},
      {0.25f, 0.28f, 0.28f, 0.28f, 0.24f, 0.088f, 2.136e-3f}, {1.23f, 1.25f, 1.25f, 1.25f, 1.23f, 0.90f, 29.7e-3f},
      {54.5f, 54.5f, 54.5f, 54.5f, 54.5f, 54.5f, 38.537f}};
  return (double)t[x - 1][y - 1] * 1e-6;
}

// Psi = exp(-x) and Phi = 3 int_0^1 t^2 exp(-x t^2) dt for x = W**2 in [0, 1]: their power
// series, sum (-x)^k/k! and sum 3 (-x)^k/(k! (2k+3)), interpolated at Chebyshev points (with the
// rounded coefficients off by 3.7e-17 and 6.1e-17 at most, near x = 1).  Then, for x above 1,
// h(u) = 3/2 + 3/4 sqrt(pi) u exp(x) erfc(1/u) with u = 1/sqrt(x), in powers of 2 u - 1: fitted
// where exp(-x) matters (u above 0.156), its share of Phi off by 2.6e-17 of Phi at most; and 1/k!.
// Tables in memory, so that they are read into scalar registers.
__constant__ double c_drift[57] = {
    1.0, -0.5999999999999948, 0.21428571428546575, -0.05555555555090525, 0.011363636318628153,
    -0.0019230766656642064, 0.0002777768425337601, -3.5011761846027854e-05, 3.912431467016512e-06,
    -3.898097348795919e-07, 3.327267488170533e-08, -1.9011473537307833e-09,
    1.0, -0.999999999999999, 0.4999999999999427, -0.16666666666540417, 0.041666666652193346,
    -0.008333333234481316, 0.0013888884549085943, -0.00019841141919339013, 2.4798998659720724e-05,
    -2.7521178006932173e-06, 2.721363367981267e-07, -2.2905624278899246e-08, 1.2719039650810423e-09,
    1.66975389374294, 0.3117227437994364, 0.11114017474596585, -0.0289303739213432,
    0.004581320932399893, 0.0008654691675095566, -0.0011654640359131995, 0.0005916453698633884,
    -0.00017255696227433563, -7.169342455466241e-06, 4.8919590990281544e-05, -3.839188796818616e-05,
    1.895223840237792e-05, -5.702602069219486e-06, 2.1974621485947115e-07, 7.00313799736029e-07,
    -3.1185083070019743e-07, 4.806131617009341e-08,
    1.0, 1.0, 1.0 / 2.0, 1.0 / 6.0, 1.0 / 24.0, 1.0 / 120.0, 1.0 / 720.0, 1.0 / 5040.0, 1.0 / 40320.0,
    1.0 / 362880.0, 1.0 / 3628800.0, 1.0 / 39916800.0, 1.0 / 479001600.0, 1.0 / 6227020800.0};
template <int DEG>
__device__ __forceinline__ double horner(const double* c, double x) {
  double b = c[DEG];
#pragma unroll
  for (int k = DEG - 1; k >= 0; --k) b = __builtin_fma(b, x, c[k]);
  return b;
}

// 1/sqrt(x) to about an ulp: v_rsq_f64 and two Newton steps; and 1/x by one residual correction
__device__ __forceinline__ double rsqrt2(double x, double& rcp) {
  double y = __builtin_amdgcn_rsq(x);
  y = __builtin_fma(0.5 * y, __builtin_fma(-(x * y), y, 1.0), y);
  y = __builtin_fma(0.5 * y, __builtin_fma(-(x * y), y, 1.0), y);
  const double q = y * y;
  rcp = __builtin_fma(q, __builtin_fma(-x, q, 1.0), q);
  return y;
}

// The pair-symmetric part of coulomb_colln (collisions.f90:138-157) for species a < b:
// 1/Teff**1.5 and W**2, from one reciprocal root.
struct Pair { double iT15, W2; };
__device__ __forceinline__ Pair coulomb_pair(double ma, double mb, double Ta, double Tb, double va, double vb) {
  double iTeff;
  const double y = rsqrt2(__builtin_fma(mb, Ta, ma * Tb) * (1.0 / (mb + ma)), iTeff);
  const double dv = va - vb;
  return {iTeff * y, ((dv * dv) * (((ma * mb) / (ma + mb)) / (2.0 * kB))) * iTeff};
}

// Phisj and Psisj above x = W**2 = 1: Phi = (3/4 sqrt(pi) erf(W)/W - 3/2 exp(-x))/x with erf as
// 1 - exp(-x) (exp(x) erfc(W)).  Off by 5e-16 at most where that form with the library's erf is
// off by 9e-16.
__device__ __forceinline__ void drift_far(double x, double& Phi, double& Psi) {
  x = x > 1e300 ? 1e300 : x;                     // (of an infinite drift: both are zero)
  double rcp;
  const double u = rsqrt2(x, rcp);
  // exp(-x) = 2**n exp(r), |r| <= log(2)/2: the Taylor series to r**13 (off by 4e-18).  (Zero
  // where x is no number, which Phi shows.)
  const double xe = x < 800.0 ? x : 800.0;
  const double n = __builtin_rint(xe * -1.4426950408889634);
  double r = __builtin_fma(n, -0.6931471805599453, -xe);
  r = __builtin_fma(n, -2.3190468138462996e-17, r);
  Psi = __builtin_amdgcn_ldexp(horner<13>(c_drift + 43, r), (int)n);
  const double e = Psi * horner<17>(c_drift + 25, __builtin_fma(2.0, u, -1.0));
  Phi = rcp * __builtin_fma((3.0 / 4.0) * sqrt(PI), u, -e);
}
constexpr double W2_NEAR = 1.0;
// the species of pair k of (1,2), (1,3), .., (6,7)
__device__ __forceinline__ constexpr int pair_a(int k) { return k < 6 ? 1 : k < 11 ? 2 : k < 15 ? 3 : k < 18 ? 4 : k < 20 ? 5 : 6; }
__device__ __forceinline__ constexpr int pair_b(int k) { return k < 6 ? k + 2 : k < 11 ? k - 3 : k < 15 ? k - 7 : k < 18 ? k - 10 : k < 20 ? k - 12 : 7; }

// The Coulomb terms of all species pairs.  add(x, y, iT15 Phi, iT15 Psi) takes species x's share
// of its collisions with y.  Up to W**2 = 1 (a drift of 1.5 km/s between heavy ions, 6 between
// H+ and O+, hundreds between ions and electrons) Phi and Psi are the series; a wave with a
// lane that is beyond in any pair of a group of seven (or has no number) branches for the group.
// Each branch ends a run of instructions, and a pair's chain is long: by single pairs ordinary
// cells took 4 % longer than by sevens (255x113x67 energy 284 us and 273).  Left to a loop of
// their own over the partner, whose values it read again, with erf and exp evaluated for both
// species of a pair, the pairs beyond cost more than they had before there was a series: H+
// flowing out at 20 km/s 491 and 617 us (energy and momentum, 255x113x67, erf and exp in every
// pair), 552 and 348 (that loop), 371 and 312 now; two pairs in three beyond 560 and 689, 883 and
// 630, 375 and 347.
template <bool PSI, int NX, typename ADD>
__device__ __forceinline__ void coulomb_terms(const double* T, const double* v1, ADD add) {
  constexpr int G = 7;                           // pairs of a group
#pragma unroll
  for (int k = 0; k < 21; k += G) {
    double iT15[G], W2[G], phi[G], psi[G];
    bool far = false;
#pragma unroll
    for (int j = 0; j < G; ++j) {
      const int a = pair_a(k + j), b = pair_b(k + j);
      const Pair p = coulomb_pair(ms(a), ms(b), T[a - 1], T[b - 1], v1[a - 1], v1[b - 1]);
      iT15[j] = p.iT15;
      W2[j] = p.W2;
      far = far || !(W2[j] <= W2_NEAR);
      const double s = horner<11>(c_drift, W2[j]);
      phi[j] = W2[j] < 0.01 ? 1.0 : s;
      psi[j] = PSI ? horner<12>(c_drift + 12, W2[j]) : 0.0;
    }
    if (__builtin_expect(__any(far), 0)) {
#pragma unroll
      for (int j = 0; j < G; ++j) {
        const int a = pair_a(k + j), b = pair_b(k + j);
        double phi_f, psi_f;
        drift_far(W2[j], phi_f, psi_f);
        if (!(W2[j] <= W2_NEAR)) {
          phi[j] = phi_f;
          psi[j] = psi_f;
        }
        // an infinite Teff (which has no reciprocal root above): no collisions, no drift
        if (T[a - 1] == __builtin_inf() || T[b - 1] == __builtin_inf()) {
          iT15[j] = 0.0;
          phi[j] = psi[j] = 1.0;
        }
      }
    }
#pragma unroll
    for (int j = 0; j < G; ++j) {
      const int a = pair_a(k + j), b = pair_b(k + j);
      const double f = iT15[j] * phi[j], q = iT15[j] * psi[j];
      add(a, b, f, q);
      if (b <= NX) add(b, a, f, q);
    }
    __builtin_amdgcn_sched_barrier(0);           // (keeps one group's values in registers)
  }
}

// the values are formed here: the compiler would move their operations down, past the branches,
// to the next use, and keep what they are formed from in registers instead
__device__ __forceinline__ void pin(double& a, double& b) { __asm__ volatile("" : "+v"(a), "+v"(b)); }

struct Cell {
  int i1, i2, i3;
  bool interior;
  long k;          // interior index (i1-1) + lx1*((i2-1) + lx2*(i3-1))
};
__device__ __forceinline__ Cell decode(const DevGrid& g, long c) {
  Cell q;
  q.i1 = (int)(c % g.L1) - 1;
  const long r = c / g.L1;
  q.i2 = (int)(r % g.L2) - 1;
  q.i3 = (int)(r / g.L2) - 1;
  q.interior = q.i1 >= 1 && q.i1 <= g.lx1 && q.i2 >= 1 && q.i2 <= g.lx2 && q.i3 >= 1 && q.i3 <= g.lx3;
  q.k = (long)(q.i1 - 1) + (long)g.lx1 * ((long)(q.i2 - 1) + (long)g.lx2 * (long)(q.i3 - 1));
  return q;
}

// ---- source_loss_energy: srcsEnergy (sources.f90:292-374), Qeionize, ETD, rhoe2T ----
__global__ __launch_bounds__(TPB) void k_src_energy(DevGrid g, DevState s, DevSources a, double dt) {
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= g.N) return;
  const Cell q = decode(g, c);
  double n[LSP], e[LSP];
#pragma unroll
  for (int i = 0; i < LSP; ++i) {
    n[i] = s.ns[i * g.N + c];
    e[i] = s.rhoes[i * g.N + c];
  }
  if (q.interior) {
    const long ni = (long)g.lx1 * g.lx2 * g.lx3, k = q.k;
    double T[LSP], v1[LSP], v2[LSP], v3[LSP], P[LSP], L[LSP];
#pragma unroll
    for (int i = 0; i < LSP; ++i) {
      T[i] = s.Ts[i * g.N + c];
      v1[i] = s.vs1[i * g.N + c];
      v2[i] = s.vs2[i * g.N + c];
      v3[i] = s.vs3[i * g.N + c];
    }
    const double Tn = s.Tn[k], vn1 = a.vn1[k], vn2 = a.vn2[k], vn3 = a.vn3[k];
    double nnk[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) nnk[j] = a.nn[j * ni + k];
    // ion-neutral and electron-neutral: heat transfer and friction.  Every production term
    // of species isp carries the factor ns ms/(gamma-1), which is applied at the end.
#pragma unroll
    for (int isp = 1; isp <= LSP; ++isp) {
      const double m = ms(isp);
      const double d1 = v1[isp - 1] - vn1, d2 = v2[isp - 1] - vn2, d3 = v3[isp - 1] - vn3;
      const double dv2 = ((d1 * d1) + (d2 * d2)) + (d3 * d3);
      double Pp = 0.0, Ll = 0.0;
#pragma unroll
      for (int isp2 = 1; isp2 <= 4; ++isp2) {
        const double nu = maxwell(isp, isp2, nnk[isp2 - 1], Tn, T[isp - 1]);
        const double fact = nu * (2.0 / (m + mn(isp2)));
        Pp = Pp + fact * (kB * Tn + (mn(isp2) / 3.0) * dv2);
        Ll = Ll + fact;
      }
      P[isp - 1] = Pp;
      L[isp - 1] = m * Ll;
      pin(P[isp - 1], L[isp - 1]);
      __builtin_amdgcn_sched_barrier(0);
    }
    // ion-ion and ion-electron (Coulomb)
    coulomb_terms<true, LSP>(T, v1, [&](int x, int y, double phi, double psi) {
      const double d1 = v1[x - 1] - v1[y - 1], d2 = v2[x - 1] - v2[y - 1], d3 = v3[x - 1] - v3[y - 1];
      const double dv2 = ((d1 * d1) + (d2 * d2)) + (d3 * d3);
      const double c2 = csj_1e6(x, y) * (2.0 / (ms(x) + ms(y)));
      const double ny = n[y - 1], npsi = ny * psi;
      P[x - 1] = P[x - 1] + (c2 * kB) * (npsi * T[y - 1]) + (c2 * (ms(y) / 3.0)) * (ny * (phi * dv2));
      L[x - 1] = L[x - 1] + (c2 * ms(x)) * npsi;
      pin(P[x - 1], L[x - 1]);
    });
#pragma unroll
    for (int i = 1; i <= LSP; ++i) P[i - 1] = (n[i - 1] * (ms(i) * (1.0 / (gammas(i) - 1.0)))) * P[i - 1];
    // inelastic electron-neutral collisions (sources.f90:350-373)
    const double sfact = (elchrg / kB) * (gammas(LSP) - 1.0);
    const double Te = T[LSP - 1], nn2 = nnk[1], nn3 = nnk[2];
    double nu = (((sfact * 6.9e-14) * nn3) * 1e-6) / sqrt(Te);
    double iePT = nu * Tn, ieLT = nu;
    nu = (((sfact * 2.9e-14) * nn2) * 1e-6) / sqrt(Te);
    iePT = iePT + nu * Tn;
    ieLT = ieLT + nu;
    double f = 1.06e4 + 7.51e3 * tanh(1.10e-3 * (Te - 1800.0));
    const double gg = (3300.0 + 1.233 * (Te - 1000.0)) - (2.056e-4 * (Te - 1000.0)) * (Te - 4000.0);
    double fact = ((((sfact * 2.99e-12) * nn2) * 1e-6) * exp(((f * (Te - 2000.0)) / Te) / 2000.0)) *
                  (exp((-(gg * (Te - Tn)) / Te) / Tn) - 1.0);
    iePT = iePT - fmax_f(fact, 0.0);
    f = 3300.0 - 839.0 * sin(1.91e-4 * (Te - 2700.0));
    fact = ((((sfact * 5.196e-13) * nn3) * 1e-6) * exp(((f * (Te - 700.0)) / Te) / 700.0)) *
           (exp((-(2770.0 * (Te - Tn)) / Te) / Tn) - 1.0);
    iePT = iePT - fmax_f(fact, 0.0);
    P[LSP - 1] = P[LSP - 1] + (((iePT * n[LSP - 1]) * kB) / (gammas(LSP) - 1.0));
    L[LSP - 1] = L[LSP - 1] + ieLT;
    // energy_source_loss_solve (multifluid.f90:474-495)
    P[LSP - 1] = P[LSP - 1] + a.Qeionize[k];
#pragma unroll
    for (int i = 0; i < LSP; ++i) {
      e[i] = etd(e[i], P[i], L[i], dt);
      s.rhoes[i * g.N + c] = e[i];
    }
  }
#pragma unroll
  for (int isp = 1; isp <= LSP; ++isp) {
    const double t = (((gammas(isp) - 1.0) / kB) * e[isp - 1]) / fmax_f(n[isp - 1], mindensdiv);
    s.Ts[(isp - 1) * g.N + c] = fmax_f(t, 100.0);
  }
}

// The divisors of an x1 gradient at cell i1 (centred, or one-sided at the ends: gradient.f90:
// 136-146) and their correctly rounded reciprocals, for the gradients of a cell's seven log
// pressures, six viscosities and two metric factors.
struct Grad {
  double d, yd, h, yh;
  __device__ __forceinline__ double operator()(double diff) const { return div_rcp(div_rcp(diff, d, yd), h, yh); }
};

// ---- source_loss_momentum: srcsMomentum_curv (sources.f90:228-289), ETD, velocities ----
__global__ __launch_bounds__(TPB, 3) void k_src_momentum(DevGrid g, DevState s, DevSources a, double dt) {
  // log p of the block's cells and of the one before and after them: x1 neighbours are
  // neighbouring threads (a cell outside the grid is no interior cell's neighbour)
  __shared__ double lp[LSP][TPB + 2];
  const int t = threadIdx.x;
  const long c0 = (long)blockIdx.x * TPB, c = c0 + t;
  auto logp = [&](int i, long cc) { return log((s.ns[i * g.N + cc] * kB) * s.Ts[i * g.N + cc]); };
  if (c < g.N) {
#pragma unroll
    for (int i = 0; i < LSP; ++i) lp[i][t + 1] = logp(i, c);
  }
  if (t < 2 * LSP) {
    const int i = t % LSP, u = t < LSP ? 0 : TPB + 1;
    const long cc = c0 + u - 1;
    if (cc >= 0 && cc < g.N) lp[i][u] = logp(i, cc);
  }
  __syncthreads();
  if (c >= g.N) return;
  const Cell q = decode(g, c);
  double n[LSP], r[LSP - 1];
#pragma unroll
  for (int i = 0; i < LSP; ++i) n[i] = s.ns[i * g.N + c];
  if (q.interior) {
    const long ni = (long)g.lx1 * g.lx2 * g.lx3, k = q.k;
    const int i1 = q.i1;
    const bool ghosted = !(g.isglobal[0] || g.isglobal[1]);
    double T[LSP], v1[LSP], P[LSP - 1], L[LSP - 1];
#pragma unroll
    for (int i = 0; i < LSP; ++i) {
      T[i] = s.Ts[i * g.N + c];
      v1[i] = s.vs1[i * g.N + c];
    }
    const double Tn = s.Tn[k], vn1 = a.vn1[k];
    double nnk[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) nnk[j] = a.nn[j * ni + k];
#pragma unroll
    for (int isp = 1; isp <= LSP - 1; ++isp) {
      double Ll = 0.0;
#pragma unroll
      for (int isp2 = 1; isp2 <= 4; ++isp2) Ll = Ll + maxwell(isp, isp2, nnk[isp2 - 1], Tn, T[isp - 1]);
      P[isp - 1] = Ll * vn1;                     // (times ns ms, applied at the end)
      L[isp - 1] = Ll;
      pin(P[isp - 1], L[isp - 1]);
      __builtin_amdgcn_sched_barrier(0);
    }
    coulomb_terms<false, LSP - 1>(T, v1, [&](int x, int y, double phi, double) {
      const double nphi = csj_1e6(x, y) * (n[y - 1] * phi);
      L[x - 1] = L[x - 1] + nphi;
      P[x - 1] = P[x - 1] + nphi * v1[y - 1];
      pin(P[x - 1], L[x - 1]);
    });
#pragma unroll
    for (int i = 1; i < LSP; ++i) P[i - 1] = (n[i - 1] * ms(i)) * P[i - 1];
    // geometric factors, ambipolar field, gravity (sources.f90:248-288)
    const double h1 = g.h1[c], h2 = g.h2[c], h3 = g.h3[c];
    const double h1h2h3 = (h1 * h2) * h3;
    // (sources.f90:259-270: centred over the ghost cells when the subdomain touches neither x1
    // end, otherwise over the interior with one-sided differences at i1 = 1 and lx1)
    const double dsum = g.dx1[i1 + 1] + g.dx1[i1], ysum = g.rdx1s[i1], yh1 = 1.0 / h1;
    const Grad mid{dsum, ysum, h1, yh1};
    const int lo = i1 == 1 ? 0 : -1, hi = i1 == g.lx1 ? 0 : 1;
    const Grad one = i1 == 1 ? Grad{g.dx1[1], g.rdx1[1], h1, yh1}
                   : i1 == g.lx1 ? Grad{g.dx1[g.lx1], g.rdx1[g.lx1], h1, yh1} : mid;
    auto dlogp = [&](int isp) {
      if (ghosted)
        return mid(lp[isp - 1][t + 2] - lp[isp - 1][t]);
      return one(lp[isp - 1][t + 1 + hi] - lp[isp - 1][t + 1 + lo]);
    };
    const double dh2dx1 = mid(g.h2[c + 1] - g.h2[c - 1]);
    const double dh3dx1 = mid(g.h3[c + 1] - g.h3[c - 1]);
    const double Te = T[LSP - 1];
    const double Epol1 = ((kB * Te) / qs(LSP)) * dlogp(LSP);
    const double E1f = a.alt[c] < 100e3 ? 0.0 : a.E1[c];
    const double g1 = a.g1[k];
#pragma unroll
    for (int isp = 1; isp <= LSP - 1; ++isp) {
      const double nsp = n[isp - 1], m = ms(isp);
      const double pr = (nsp * kB) * T[isp - 1];
      const double ionpress = pr * dlogp(isp);
      const double* Qs = a.Q + (long)(isp - 1) * ni;
      const double gQ = one(Qs[k + hi] - Qs[k + lo]);
      const double w2 = s.vs2[(isp - 1) * g.N + c], w3 = s.vs3[(isp - 1) * g.N + c];
      const double geom = (((((w2 * w2) * h3) * dh2dx1 + ((w3 * w3) * h2) * dh3dx1) * nsp) * m) / h1h2h3;
      const double Pp = ((((P[isp - 1] + (nsp * qs(isp)) * (E1f + Epol1)) - ionpress) - gQ) + geom) +
                        (nsp * m) * g1;
      r[isp - 1] = etd(s.rhovs1[(isp - 1) * g.N + c], Pp, L[isp - 1], dt);   // (so late: registers)
      s.rhovs1[(isp - 1) * g.N + c] = r[isp - 1];
    }
  } else {
#pragma unroll
    for (int i = 0; i < LSP - 1; ++i) r[i] = s.rhovs1[i * g.N + c];
  }
  // momentum_source_loss_solve (multifluid.f90:510-527), whole padded grid
  double chrgflux = 0.0;
#pragma unroll
  for (int isp = 1; isp <= LSP - 1; ++isp) {
    const double v = r[isp - 1] / (ms(isp) * fmax_f(n[isp - 1], mindensdiv));
    s.vs1[(isp - 1) * g.N + c] = v;
    chrgflux = chrgflux + (n[isp - 1] * qs(isp)) * v;
  }
  const double ve = -(((1.0 / fmax_f(n[LSP - 1], mindensdiv)) / qs(LSP)) * chrgflux);
  s.vs1[(LSP - 1) * g.N + c] = ve;
  s.rhovs1[(LSP - 1) * g.N + c] = (n[LSP - 1] * ms(LSP)) * ve;
}

// kreac fits of srcsContinuity: ((((c0 s1 c1 t) s2 c2 t^2) s3 c3 t^3) s4 c4 t^4)
__device__ __forceinline__ double poly4(double t, double c0, double c1, double c2, double c3,
                                        double c4, bool p1, bool p2, bool p3, bool p4) {
#pragma clang fp contract(off)
  const double t2 = t * t, t3 = t2 * t, t4 = t2 * t2;
  double r = c0;
  r = p1 ? r + c1 * t : r - c1 * t;
  r = p2 ? r + c2 * t2 : r - c2 * t2;
  r = p3 ? r + c3 * t3 : r - c3 * t3;
  r = p4 ? r + c4 * t4 : r - c4 * t4;
  return r;
}

// ---- source_loss_mass: srcsContinuity (sources.f90:18-225), Prionize, ETD, ne ----
// CLEAN (the sources block, libgemini.cpp:225-231): clean_param 3 and 1 follow the three
// source passes, with clean_param 2 (velocities only) between them, so this last pass
// also applies them to its cell: temperatures floored at 100 K (ghost and null cells at
// 100 K), ion densities floored at mindens with the electrons their sum (ghost cells at
// mindensdiv, null cells at mindensnull).  Its own reads of Ts come first.
template <bool CLEAN>
__global__ __launch_bounds__(TPB) void k_src_mass(DevGrid g, DevState s, DevSources a, double dt,
                                                  const int* nul) {
#pragma clang fp contract(off)
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= g.N) return;
  const Cell q = decode(g, c);
  if (CLEAN) {
    const bool null = q.interior && nul && nul[q.k] != 0;
    if (!q.interior || null) {
#pragma unroll
      for (int i = 0; i < LSP; ++i) {
        s.Ts[i * g.N + c] = 100.0;
        s.ns[i * g.N + c] = !q.interior ? mindensdiv : (i == 0 ? mindensnull * 1e-2 : mindensnull);
      }
      return;
    }
  }
  double n[LSP];
#pragma unroll
  for (int i = 0; i < LSP; ++i) n[i] = s.ns[i * g.N + c];
  if (q.interior) {
    const long ni = (long)g.lx1 * g.lx2 * g.lx3, k = q.k;
    double P[LSP] = {0, 0, 0, 0, 0, 0, 0}, L[LSP] = {0, 0, 0, 0, 0, 0, 0};
    const double Tn = s.Tn[k];
    const double T1 = s.Ts[c], T3 = s.Ts[2 * g.N + c], T6 = s.Ts[5 * g.N + c];
    const double Te = s.Ts[6 * g.N + c], ne = n[LSP - 1];
    const double d1 = s.vs1[c] - a.vn1[k], d2 = s.vs2[c] - a.vn2[k], d3 = s.vs3[c] - a.vn3[k];
    const double dv2 = ((d1 * d1) + (d2 * d2)) + (d3 * d3);
    auto NN = [&](int j) { return a.nn[(long)(j - 1) * ni + k]; };
    const double e07 = (double)0.7f, e085 = (double)0.85f, e039 = (double)0.39f;
    const double e023 = (double)0.23f, em041 = -(double)0.41f, e044 = (double)0.44f;
    const double em02 = -(double)0.2f, e070 = (double)0.70f, e056 = (double)0.56f;
    const double X16 = (((16.0 * amu) / 3.0) / kB) * dv2, X28 = (((28.0 * amu) / 3.0) / kB) * dv2;
    double Teff, kreac = 0.0, b;
    // O+ + N2 -> NO+ + N
    Teff = (28.0 / (16.0 + 28.0)) * ((X16 + T1) - Tn) + Tn;
    if (Teff <= 3725.0)
      kreac = poly4(Teff / 300.0, 1.71676e-12, 7.19934e-13, 1.33276e-13, 9.28213e-15, 6.39557e-16, false, true, false, true);
    if (Teff > 3725.0 && Teff <= 30000.0)
      kreac = poly4(Teff / 300.0, -1.52489e-11, 7.67112e-13, 1.19064e-13, 1.30858e-15, 4.67756e-18, true, true, false, true);
    if (Teff > 30000.0)
      kreac = poly4(100.0, -1.52489e-11, 7.67112e-13, 1.19064e-13, 1.30858e-15, 4.67756e-18, true, true, false, true);
    b = (kreac * NN(2)) * 1e-6;
    P[1] = P[1] + b * n[0]; L[0] = L[0] + b;
    // O+ + O2 -> O2+ + O
    Teff = (32.0 / (16.0 + 32.0)) * ((X16 + T1) - Tn) + Tn;
    if (Teff <= 4800.0)
      kreac = poly4(Teff / 300.0, 2.78932e-11, 6.92612e-12, 8.67684e-13, 3.47251e-14, 5.07097e-16, false, true, false, true);
    if (Teff > 4800.0 && Teff <= 30000.0) {
      const double t = Teff / 300.0;
      kreac = ((-1.74046e-11 + (3.02328e-12 * Teff) / 300.0) - 2.39214e-15 * (t * t)) - 4.02394e-17 * ((t * t) * t);
    }
    if (Teff > 30000.0)
      kreac = ((-1.74046e-11 + 3.02328e-12 * 100.0) - 2.39214e-15 * 10000.0) - 4.02394e-17 * 1000000.0;
    b = (kreac * NN(3)) * 1e-6;
    P[3] = P[3] + b * n[0]; L[0] = L[0] + b;
    // O+ + NO -> NO+ + O
    Teff = (30.0 / (16.0 + 30.0)) * ((X16 + T1) - Tn) + Tn;
    if (Teff <= 3800.0)
      kreac = poly4(Teff / 300.0, 6.40408e-13, 1.33888e-13, 7.65103e-14, 3.11509e-15, 6.62374e-17, false, true, false, true);
    if (Teff > 3800.0 && Teff <= 30000.0)
      kreac = poly4(Teff / 300.0, -7.48312e-13, 2.31502e-13, 3.07160e-14, 2.65436e-16, 7.76665e-19, true, true, false, true);
    if (Teff > 30000.0)
      kreac = poly4(100.0, -7.48312e-13, 2.31502e-13, 3.07160e-14, 2.65436e-16, 7.76665e-19, true, true, false, true);
    b = (kreac * NN(6)) * 1e-6;
    P[1] = P[1] + b * n[0]; L[0] = L[0] + b;
    // O+ + e -> O + hv
    b = ((3.7e-12 * pow(250.0 / Te, e07)) * ne) * 1e-6;
    L[0] = L[0] + b;
    // N2+ + O -> O+ + N2
    Teff = (16.0 / (28.0 + 16.0)) * ((X28 + T3) - Tn) + Tn;
    kreac = Teff <= 1500.0 ? 1e-11 * pow(300.0 / Teff, e023) : 3.6e-12 * pow(300.0 / Teff, em041);
    b = (kreac * NN(1)) * 1e-6;
    P[0] = P[0] + b * n[2]; L[2] = L[2] + b;
    // N+ + O -> O+ + N
    b = (5e-13 * NN(1)) * 1e-6;
    P[0] = P[0] + b * n[4]; L[4] = L[4] + b;
    // H+ + O -> O+ + H
    b = (((6.e-10 * (8.0 / 9.0)) * sqrt((T6 + Tn / 4.0) / (Tn + T6 / 16.0))) * NN(1)) * 1e-6;
    P[0] = P[0] + b * n[5]; L[5] = L[5] + b;
    // O+ + H -> H+ + O
    b = (6.0e-10 * NN(4)) * 1e-6;
    P[5] = P[5] + b * n[0]; L[0] = L[0] + b;
    // O2+ + N2 -> NO+ + NO (the reference takes nn(:,:,:,3))
    b = (5e-16 * NN(3)) * 1e-6;
    P[1] = P[1] + b * n[3]; L[3] = L[3] + b;
    // O2+ + N -> NO+ + O
    b = (1.2e-10 * NN(5)) * 1e-6;
    P[1] = P[1] + b * n[3]; L[3] = L[3] + b;
    // O2+ + NO -> NO+ + O2
    b = (4.6e-10 * NN(6)) * 1e-6;
    P[1] = P[1] + b * n[3]; L[3] = L[3] + b;
    // N2+ + O -> NO+ + N
    kreac = Teff <= 1500.0 ? 1.4e-10 * pow(300.0 / Teff, e044) : 5.2e-11 * pow(300.0 / Teff, em02);
    b = (kreac * NN(1)) * 1e-6;
    P[1] = P[1] + b * n[2]; L[2] = L[2] + b;
    // N2+ + NO -> NO+ + N2
    b = (4.1e-10 * NN(6)) * 1e-6;
    P[1] = P[1] + b * n[2]; L[2] = L[2] + b;
    // N+ + O2 -> NO+ + O
    b = (2.6e-10 * NN(3)) * 1e-6;
    P[1] = P[1] + b * n[4]; L[4] = L[4] + b;
    // NO+ + e -> N + O
    b = ((4.2e-7 * pow(300.0 / Te, e085)) * ne) * 1e-6;
    L[1] = L[1] + b;
    // N2+ + O2 -> O2+ + N2
    Teff = (32.0 / (28.0 + 32.0)) * ((X28 + T3) - Tn) + Tn;
    b = ((5e-11 * (300.0 / Teff)) * NN(3)) * 1e-6;
    P[3] = P[3] + b * n[2]; L[2] = L[2] + b;
    // N2+ + e -> N + N
    b = ((1.8e-7 * pow(300.0 / Te, e039)) * ne) * 1e-6;
    L[2] = L[2] + b;
    // N+ + O2 -> O2+ + N
    b = (3.1e-10 * NN(3)) * 1e-6;
    P[3] = P[3] + b * n[4]; L[4] = L[4] + b;
    // O2+ + e -> O + O
    kreac = Te <= 1200.0 ? 1.95e-7 * pow(300.0 / Te, e070) : 7.38e-8 * pow(1200.0 / Te, e056);
    b = (kreac * ne) * 1e-6;
    L[3] = L[3] + b;
    // N+ + H -> H+ + N
    b = (3.6e-12 * NN(4)) * 1e-6;
    P[5] = P[5] + b * n[4]; L[4] = L[4] + b;
    // H+ + e -> H + hv
    b = ((3.7e-12 * pow(250.0 / Te, e07)) * ne) * 1e-6;
    L[5] = L[5] + b;
    // mass_source_loss_solve (multifluid.f90:532-549)
#pragma unroll
    for (int i = 0; i < LSP - 1; ++i) {
      n[i] = etd(n[i], P[i] + a.Prionize[i * ni + k], L[i], dt);
      if (CLEAN) n[i] = fmax_f(n[i], mindens);
      s.ns[i * g.N + c] = n[i];
    }
    if (CLEAN) {
#pragma unroll
      for (int i = 0; i < LSP; ++i) s.Ts[i * g.N + c] = fmax_f(s.Ts[i * g.N + c], 100.0);
    }
  }
  double sum = 0.0;
#pragma unroll
  for (int i = 0; i < LSP - 1; ++i) sum = sum + n[i];
  s.ns[(LSP - 1) * g.N + c] = sum;
}

int blocks_of(long n) { return (int)((n + TPB - 1) / TPB); }

__global__ void k_zero(double* p, long n) {
  for (long k = (long)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (long)gridDim.x * blockDim.x)
    p[k] = 0.0;
}

}  // namespace

// zero n doubles with a kernel (a memset node would be unsafe if a caller captures the call)
void launch_zero(double* p, long n, hipStream_t st) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_zero, dim3((int)min(blocks_of(n), 16384L)), dim3(TPB), 0, st, p, n);
}

void launch_source_loss_energy(const DevGrid& g, const DevState& s, const DevSources& a,
                               double dt, hipStream_t st) {
  timing_begin("source_energy", st);
  hipLaunchKernelGGL(k_src_energy, dim3(blocks_of(g.N)), dim3(TPB), 0, st, g, s, a, dt);
  timing_end("source_energy", st);
}

void launch_source_loss_momentum(const DevGrid& g, const DevState& s, const DevSources& a,
                                 double dt, hipStream_t st) {
  timing_begin("source_momentum", st);
  hipLaunchKernelGGL(k_src_momentum, dim3(blocks_of(g.N)), dim3(TPB), 0, st, g, s, a, dt);
  timing_end("source_momentum", st);
}

void launch_source_loss_mass(const DevGrid& g, const DevState& s, const DevSources& a,
                             double dt, hipStream_t st, const int* clean_nul, bool clean) {
  timing_begin("source_mass", st);
  if (clean)
    hipLaunchKernelGGL(k_src_mass<true>, dim3(blocks_of(g.N)), dim3(TPB), 0, st, g, s, a, dt,
                       clean_nul);
  else
    hipLaunchKernelGGL(k_src_mass<false>, dim3(blocks_of(g.N)), dim3(TPB), 0, st, g, s, a, dt,
                       nullptr);
  timing_end("source_mass", st);
}

}  // namespace gemhip
