// kernels_adjoint.hip -- discrete adjoint of the electron energy path of one transport step.
//
// Only the electron temperature depends on the fitting parameters (a per-column scale
// kappa on the electron thermal conductivity and a downward top heat flux q), so the
// adjoint state is one field, lambda = dL/dTe.  The forward step is, for electrons
// (reference order src/libgemini.cpp:155-208):
//   e = ne kB Te / (gamma-1)                           T2rhoe        multifluid.f90:193-202
//   ghost fill of e, periodic x3 wrap                  advec.f90:21-149, mpihalo.f90:147-152
//   e <- S3 e, e <- S1 e, x3 wrap, e <- S2 e           MC-limited sweeps, advec.f90:233-447
//   Te' = max((gamma-1) e / (kB max(ne', nmin)), 100)  rhoe2T        multifluid.f90:179-189
//   Te'' = max(TRBDF2(Te'; kappa, q), 100)             PDEparabolic.f90:19-218
// Each map is differentiated exactly with the branches the forward took (upwind side,
// minmod selection, floors) frozen, and the adjoint runs the maps in reverse:
//   * TRBDF2: the two pivoted band solves are recomputed per column as the forward does,
//     then the transposed systems M2^T w2 = mu and M1^T w1 = (4/dt) w2 are solved with
//     the stored factors (U^T forward substitution, then the row eliminations and
//     interchanges transposed in reverse order), and w1, w2 are chained through the
//     matrix and right-hand-side entries to the conductivity (d lambda_e / dT in closed
//     form), kappa and q;
//   * sweeps: lambda_in(j) = lambda_out(j) + sum over the interface fluxes and limited
//     slopes that read cell j, gathered per cell (no atomics);
//   * ghost fill and wrap: each overwritten ghost hands its adjoint to the cell it was
//     copied or scaled from and is cleared;
//   * conversions: pointwise.
// The inputs each map needs (electron densities, the energy density entering each sweep,
// interface velocities, the temperature entering the diffusion) are taken from a tape
// recorded by the forward step.
#include "diffusion_cell.h"

namespace gemhip {

namespace {

constexpr int TPB = 256;

inline unsigned grid_for(long n) {
  long b = (n + TPB - 1) / TPB;
  return (unsigned)(b > 8192 ? 8192 : b);          // grid-stride loops cover the rest
}
inline unsigned grid_exact(long n) { return (unsigned)((n + TPB - 1) / TPB); }

__device__ __forceinline__ int clampi(int v, int lo, int hi) { return v < lo ? lo : (v > hi ? hi : v); }

// ------------------------------------------------------------------ tape helpers
// electron interface velocities (advec.f90:155-229), the values the forward sweeps use
__global__ void k_tape_vels(DevGrid g, const double* vs1, const double* vs2, const double* vs3,
                            double* v1, double* v2, double* v3) {
  const long n1 = (long)(g.lx1 + 1) * g.lx2 * g.lx3;
  const long n2 = (long)g.lx1 * (g.lx2 + 1) * g.lx3;
  const long n3 = (long)g.lx1 * g.lx2 * (g.lx3 + 1);
  for (long t = (long)blockIdx.x * blockDim.x + threadIdx.x; t < n1 + n2 + n3;
       t += (long)gridDim.x * blockDim.x) {
    if (t < n1) {
      const int k = (int)(t % (g.lx1 + 1)) + 1;
      const long line = t / (g.lx1 + 1);
      const int i2 = (int)(line % g.lx2) + 1, i3 = (int)(line / g.lx2) + 1;
      v1[t] = v1i_at(g, vs1 + gix(g, 0, i2, i3), k);
    } else if (t < n1 + n2) {
      const long u = t - n1;
      const int i1 = (int)(u % g.lx1) + 1;
      const long r = u / g.lx1;
      const int k = (int)(r % (g.lx2 + 1)) + 1, i3 = (int)(r / (g.lx2 + 1)) + 1;
      v2[u] = 0.5 * (vs2[gix(g, i1, k - 1, i3)] + vs2[gix(g, i1, k, i3)]);
    } else {
      const long u = t - n1 - n2;
      const int i1 = (int)(u % g.lx1) + 1;
      const long r = u / g.lx1;
      const int i2 = (int)(r % g.lx2) + 1, k = (int)(r / g.lx2) + 1;
      v3[u] = 0.5 * (vs3[gix(g, i1, i2, k - 1)] + vs3[gix(g, i1, i2, k)]);
    }
  }
}

// ------------------------------------------------------------------ pointwise maps
// rhoe2T (with its floor) and the diffusion's floor on ghost cells, transposed:
// lambda <- lambda [Te' > 100] (gamma-1)/kB / max(ne', nmin)
__global__ void k_adj_rhoe2T(DevGrid g, double* lam, const double* TD, const double* NE1) {
  const double c = (gammas(LSP) - 1.0) / kB;
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < g.N;
       i += (long)gridDim.x * blockDim.x)
    lam[i] = TD[i] > 100.0 ? lam[i] * (c / fmax_f(NE1[i], mindensdiv)) : 0.0;
}

// T2rhoe transposed: out = in ne kB / (gamma-1)
__global__ void k_adj_T2rhoe(DevGrid g, const double* in, double* out, const double* NE0) {
  const double gm1 = gammas(LSP) - 1.0;
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < g.N;
       i += (long)gridDim.x * blockDim.x)
    out[i] = in[i] * ((NE0[i] * kB) / gm1);
}

// ------------------------------------------------------------------ ghost fill, wrap
// advec.f90:107-132 transposed (x3 ends, every x1 and x2 position)
__global__ void k_adj_bc_x3(DevGrid g, double* lam) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long)g.L1 * g.L2) return;
  const int i1 = (int)(t % g.L1) - 1, i2 = (int)(t / g.L1) - 1;
  if (g.isglobal[5]) {
    const long a = gix(g, i1, i2, g.lx3 + 1), b = gix(g, i1, i2, g.lx3 + 2);
    lam[gix(g, i1, i2, g.lx3)] += lam[a] + lam[b];
    lam[a] = 0.0;
    lam[b] = 0.0;
  }
  if (g.isglobal[4]) {
    const long a = gix(g, i1, i2, 0), b = gix(g, i1, i2, -1);
    lam[gix(g, i1, i2, 1)] += lam[a] + lam[b];
    lam[a] = 0.0;
    lam[b] = 0.0;
  }
}

// advec.f90:83-104 transposed (x2 ends, every x1 and x3 position)
__global__ void k_adj_bc_x2(DevGrid g, double* lam) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long)g.L1 * g.L3) return;
  const int i1 = (int)(t % g.L1) - 1, i3 = (int)(t / g.L1) - 1;
  if (g.isglobal[3]) {
    const long a = gix(g, i1, g.lx2 + 1, i3), b = gix(g, i1, g.lx2 + 2, i3);
    lam[gix(g, i1, g.lx2, i3)] += lam[a] + lam[b];
    lam[a] = 0.0;
    lam[b] = 0.0;
  }
  if (g.isglobal[2]) {
    const long a = gix(g, i1, 0, i3), b = gix(g, i1, -1, i3);
    lam[gix(g, i1, 1, i3)] += lam[a] + lam[b];
    lam[a] = 0.0;
    lam[b] = 0.0;
  }
}

// advec.f90:42-79 transposed for the energy density: e(0) = (e(1)/n(1)) n(0) etc., with
// the densities as the fill leaves them when e is filled (interior columns get their
// density ghosts extrapolated first, advec.f90:45-50)
__global__ void k_adj_bc_x1(DevGrid g, double* lam, const double* NE0) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long)g.L2 * g.L3) return;
  const int i2 = (int)(t % g.L2) - 1, i3 = (int)(t / g.L2) - 1;
  const bool inner = i2 >= 1 && i2 <= g.lx2 && i3 >= 1 && i3 <= g.lx3;
  const long o = gix(g, 0, i2, i3);
  const double* n = NE0 + o;         // n[i1]
  double* l = lam + o;
  const int lx1 = g.lx1;
  if (g.isglobal[1]) {
    double nP1 = n[lx1 + 1], nP2 = n[lx1 + 2];
    if (inner) {
      const double coeff = n[lx1 - 1] / n[lx1 - 2];
      nP1 = fmin_f(coeff * n[lx1], n[lx1]);
      nP2 = fmin_f(coeff * nP1, nP1);
    }
    l[lx1] += (nP1 / n[lx1]) * l[lx1 + 1] + (nP2 / n[lx1]) * l[lx1 + 2];
    l[lx1 + 1] = 0.0;
    l[lx1 + 2] = 0.0;
  }
  if (g.isglobal[0]) {
    double n0 = n[0], nm1 = n[-1];
    if (inner) {
      const double coeff = n[2] / n[3];
      n0 = fmin_f(coeff * n[1], n[1]);
      nm1 = fmin_f(coeff * n0, n0);
    }
    l[1] += (n0 / n[1]) * l[0] + (nm1 / n[1]) * l[-1];
    l[0] = 0.0;
    l[-1] = 0.0;
  }
}

// mpihalo.f90:147-152 (one process along x3, depth 2) transposed; needs lx3 >= 2
__global__ void k_adj_halo(DevGrid g, double* lam) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long)g.L1 * g.lx2) return;
  const int i1 = (int)(t % g.L1) - 1, i2 = (int)(t / g.L1) + 1;
  for (int h = 0; h < 2; ++h) {
    const long gh = gix(g, i1, i2, -1 + h);
    lam[gix(g, i1, i2, g.lx3 - 1 + h)] += lam[gh];
    lam[gh] = 0.0;
  }
  for (int h = 0; h < 2; ++h) {
    const long gh = gix(g, i1, i2, g.lx3 + 1 + h);
    lam[gix(g, i1, i2, 1 + h)] += lam[gh];
    lam[gh] = 0.0;
  }
}

// ------------------------------------------------------------------ sweeps
// advec.f90:384-435 along direction DIR, transposed with the limiter and upwind choices
// the forward made on f.  One thread per ghosted cell; cells that are not on an interior
// line of the direction are left unchanged by the sweep, so their adjoint is copied.
//   out(i) = f(i) - dt (ha2i(i+1) phi(i+1) - ha2i(i) phi(i)) / dxi(i) / ha1(i), 1 <= i <= lx
//   phi(i) = v<0: f(i) v - (v/2)(dx(i) + v dt/h1i(i)) slope(i)
//            v>=0: f(i-1) v + (v/2)(dx(i) - v dt/h1i(i)) slope(i-1)
//   slope(k) = minmod(central, minmod(2 left, 2 right)), 0 <= k <= lx+1
template <int DIR>
__global__ void k_adj_sweep(DevGrid g, const double* lam_out, double* lam_in, const double* f,
                            const double* vi, double dt) {
  const int lx = DIR == 1 ? g.lx1 : DIR == 2 ? g.lx2 : g.lx3;
  const double* dx = DIR == 1 ? g.dx1 : DIR == 2 ? g.dx2 : g.dx3;           // dx[k], k=0..lx+2
  const double* dxi = (DIR == 1 ? g.dx1i : DIR == 2 ? g.dx2i : g.dx3i) - 1;  // dxi[k], k=1..lx
  const long st = DIR == 1 ? 1L : DIR == 2 ? (long)g.L1 : (long)g.L1 * g.L2;
  for (long c = (long)blockIdx.x * blockDim.x + threadIdx.x; c < g.N;
       c += (long)gridDim.x * blockDim.x) {
    const int i1 = (int)(c % g.L1) - 1;
    const int i2 = (int)((c / g.L1) % g.L2) - 1;
    const int i3 = (int)(c / ((long)g.L1 * g.L2)) - 1;
    int j, a, b;
    bool line;
    if (DIR == 1) { j = i1; a = i2; b = i3; line = a >= 1 && a <= g.lx2 && b >= 1 && b <= g.lx3; }
    else if (DIR == 2) { j = i2; a = i1; b = i3; line = a >= 1 && a <= g.lx1 && b >= 1 && b <= g.lx3; }
    else { j = i3; a = i1; b = i2; line = a >= 1 && a <= g.lx1 && b >= 1 && b <= g.lx2; }
    if (!line || lx <= 1) { lam_in[c] = lam_out[c]; continue; }
    auto cell = [&](int k) { return c + (long)(k - j) * st; };
    auto fidx = [&](int i) -> long {                 // interface i of this line
      if (DIR == 1) return (i - 1) + (long)(g.lx1 + 1) * ((a - 1) + (long)g.lx2 * (b - 1));
      if (DIR == 2) return (a - 1) + (long)g.lx1 * ((i - 1) + (long)(g.lx2 + 1) * (b - 1));
      return (a - 1) + (long)g.lx1 * ((b - 1) + (long)g.lx2 * (i - 1));
    };
    // p(k) = dt lam_out(k) / dxi(k) / ha1(k) on the updated cells, k = j-2..j+2
    double P[5];
#pragma unroll
    for (int o = 0; o < 5; ++o) {
      const int k = j - 2 + o;
      P[o] = 0.0;
      if (k >= 1 && k <= lx) {
        const long ck = cell(k);
        P[o] = ((dt * lam_out[ck]) / dxi[k]) / ((g.h1[ck] * g.h2[ck]) * g.h3[ck]);
      }
    }
    // interfaces i = j-1..j+2: flux adjoint and its two upwind coefficients
    double LPHI[4], V[4], CM[4], CP[4];
    bool IV[4];
#pragma unroll
    for (int o = 0; o < 4; ++o) {
      const int i = j - 1 + o;
      IV[o] = i >= 1 && i <= lx + 1;
      LPHI[o] = V[o] = CM[o] = CP[o] = 0.0;
      if (IV[o]) {
        const long fi = fidx(i);
        double ha2i, h1i;
        if (DIR == 1) { ha2i = g.h2x1i[fi] * g.h3x1i[fi]; h1i = g.h1x1i[fi]; }
        else if (DIR == 2) { ha2i = g.h1x2i[fi] * g.h3x2i[fi]; h1i = g.h2x2i[fi]; }
        else { ha2i = g.h1x3i[fi] * g.h2x3i[fi]; h1i = g.h3x3i[fi]; }
        const double v = vi[fi];
        V[o] = v;
        LPHI[o] = ha2i * (P[o + 1] - P[o]);
        CM[o] = -((0.5 * v) * (dx[i] + (v / h1i) * dt));
        CP[o] = (0.5 * v) * (dx[i] - (v / h1i) * dt);
      }
    }
    // f(j-2..j+2) for the limiter choices
    double F[5];
#pragma unroll
    for (int o = 0; o < 5; ++o) {
      const int k = j - 2 + o;
      F[o] = (k >= -1 && k <= lx + 2) ? f[cell(k)] : 0.0;
    }
    double acc = lam_out[c];
    if (IV[1] && V[1] < 0.0) acc += V[1] * LPHI[1];          // phi(j) reads f(j) when v<0
    if (IV[2] && V[2] >= 0.0) acc += V[2] * LPHI[2];         // phi(j+1) reads f(j) when v>=0
#pragma unroll
    for (int o = 0; o < 3; ++o) {                            // slopes k = j-1, j, j+1
      const int k = j - 1 + o;
      if (k < 0 || k > lx + 1) continue;
      double ls = 0.0;                                       // d L / d slope(k)
      if (IV[o] && V[o] < 0.0) ls += LPHI[o] * CM[o];
      if (IV[o + 1] && V[o + 1] >= 0.0) ls += LPHI[o + 1] * CP[o + 1];
      if (ls == 0.0) continue;
      const double fm = F[o], f0 = F[o + 1], fp = F[o + 2];  // f(k-1), f(k), f(k+1)
      const double lsl = (f0 - fm) / dx[k], rsl = (fp - f0) / dx[k + 1];
      const double csl = (fp - fm) / (dx[k] + dx[k + 1]);
      const double l2 = 2.0 * lsl, r2 = 2.0 * rsl;
      int msel;
      double m;
      if (l2 * r2 <= 0.0) { m = 0.0; msel = 0; }
      else if (fabs(l2) < fabs(r2)) { m = l2; msel = 2; }
      else { m = r2; msel = 3; }
      int sel;
      if (csl * m <= 0.0) sel = 0;
      else if (fabs(csl) < fabs(m)) sel = 1;
      else sel = msel;
      // d slope(k) / d f(j) for the chosen form
      if (o == 1) {
        if (sel == 2) acc += (2.0 * ls) / dx[k];
        else if (sel == 3) acc -= (2.0 * ls) / dx[k + 1];
      } else if (o == 0) {                                   // f(j) = f(k+1)
        if (sel == 1) acc += ls / (dx[k] + dx[k + 1]);
        else if (sel == 3) acc += (2.0 * ls) / dx[k + 1];
      } else {                                               // f(j) = f(k-1)
        if (sel == 1) acc -= ls / (dx[k] + dx[k + 1]);
        else if (sel == 2) acc -= (2.0 * ls) / dx[k];
      }
    }
    lam_in[c] = acc;
  }
}

// ------------------------------------------------------------------ TRBDF2
// d lambda_e / dT of the electron conductivity (collisions.f90:185-195)
__device__ __forceinline__ double lambda_e_dT(const CellIn<true>& c, double lam_e) {
  const double T = c.T, sq = sqrt(T);
  const double br = ((c.n1 * 1.1e-16) * (1.0 + 5.7e-4 * T) + ((c.n2 * 2.82e-17) * sq) * (1.0 - 1.21e-4 * T))
                    + (c.n3 * 2.2e-16) * (1.0 + 3.6e-2 * sq);
  const double dbr = (c.n1 * 1.1e-16) * 5.7e-4
                     + (c.n2 * 2.82e-17) * ((0.5 / sq) * (1.0 - 1.21e-4 * T) - sq * 1.21e-4)
                     + (c.n3 * 2.2e-16) * (3.6e-2 * (0.5 / sq));
  const double den = 1.0 + ((3.22e4 * (T * T)) / c.n) * br;
  const double dden = (3.22e4 / c.n) * ((2.0 * T) * br + (T * T) * dbr);
  return lam_e * (2.5 / T - dden / den);
}

// scratch slots per (row, column): groups of 64 columns, in a group row by row, in a row slot
// by slot, 64 columns each, so that a lane reaches its row's slots from one address
enum : int {
  A0 = 0, A1, A2, AY, AL, AI,      // TR: s1 s2 s3 and rhs -> pivot row, rhs (then BDF2's) -> U^T
                                   // solve -> w1; multiplier; 1/pivot
  B0, B1, B2, BY, BL, BI,          // BDF2: the same, BY: dL/dTe after the step -> mu -> U^T solve
                                   // -> w2 (BL of row 1 is SINGULAR for a column without an adjoint)
  X1, X2,                          // TR and BDF2 solutions (X2 before: the rhs term in T)
  NSA
};
constexpr double SINGULAR = 2.0;   // (a multiplier is at most 1)

// one column of the scratch
struct Col {
  double* p;                       // row 1, slot NSA/2 (immediate offsets reach 4 KB either way)
  __device__ Col(const double* scratch, int N, long col)
      : p(const_cast<double*>(scratch) + (((col >> 6) * N * NSA + NSA / 2) * 64 + (col & 63))) {}
  __device__ double& operator()(int i, int k) const { return p[(long)(i - 1) * (NSA * 64) + (k - NSA / 2) * 64]; }
};

struct AdjArgs {
  const double* TD;      // electron temperature entering the diffusion (ghosted field)
  const double* NE1;     // electron density at the diffusion (ghosted field)
  double* lam;           // in: dL/dTe after the step; out: dL/dTe' (interior rows)
  double* gk;            // += dL/dkappa per column
  double* gq;            // += dL/dq per column (null without a heat flux)
  double dt, Teinf;
};

// pivoted elimination step bringing in row (a, b, cc | d) against the pending row
// (r0, r1 | rb), as dgbtf2 + dgbtrs do it (kernels_diffusion.hip): stores the pivot row, its
// reciprocal and rhs and the multiplier.  An interchange shows in the third entry, which is
// +0 without one (and -0 where an interchange brings a zero).  The zero tests of the band
// routines only skip work that changes nothing (of finite entries), and are left out.
template <bool RHS>
__device__ __forceinline__ bool adj_elim(const Col& q, int j, int s0, double& r0, double& r1,
                                         double& rb, double a, double b, double cc, double d) {
  const bool swap = fabs(a) > fabs(r0);
  const double p0 = swap ? a : r0, p1 = swap ? b : r1, p2 = swap ? (cc == 0.0 ? -0.0 : cc) : 0.0;
  const double o0 = swap ? r0 : a, o1 = swap ? r1 : b, o2 = swap ? 0.0 : cc;
  const double rp = 1.0 / p0, l = rp * o0;
  q(j, s0) = p0; q(j, s0 + 1) = p1; q(j, s0 + 2) = p2;
  q(j, s0 + 4) = l; q(j, s0 + 5) = rp;
  r0 = o1 + l * (-p1);
  r1 = o2 + l * (-p2);
  if (RHS) {
    const double pd = swap ? d : rb, od = swap ? rb : d;
    q(j, s0 + 3) = pd;
    rb = od + l * (-pd);
  }
  return p0 == 0.0;
}
__device__ __forceinline__ bool interchanged(double p2) { return __double_as_longlong(p2) != 0; }

// Every pass below walks the rows of a column in order with a loop-carried recurrence.
// Row data are fetched P rows ahead into a register ring, so the loads of later rows are
// in flight while the recurrence runs (the loop over a full ring is unrolled, its ring
// slots are registers); the last count % P rows are fetched as they come.
template <int P, int DIR, class Raw, class Fetch, class Body>
__device__ __forceinline__ void stream_rows(int first, int count, Fetch fetch, Body body) {
  Raw ring[P];
#pragma unroll
  for (int u = 0; u < P; ++u) fetch(first + DIR * u, ring[u]);
  const int nfull = count / P;
  for (int c = 0; c < nfull; ++c) {
#pragma unroll
    for (int u = 0; u < P; ++u) {
      const int i = first + DIR * (c * P + u);
      const Raw v = ring[u];
      fetch(i + DIR * P, ring[u]);
      body(i, v);
    }
  }
  for (int k = nfull * P; k < count; ++k) {
    const int i = first + DIR * k;
    Raw v;
    fetch(i, v);
    body(i, v);
  }
}

constexpr int PF = 12;           // ring depth of the passes (8: 8 % slower, 16: spills)

struct R4 { double a, b, c, d; };

// dtbsv (upper, no transpose) over stored rows s0..s0+2 with the rhs in AY, into slot sx;
// with MU, also mu(i) = dL/dx(i) through the output floor into BY
template <bool MU>
__device__ __forceinline__ void adj_backsub(const Col& q, int N, int s0, int sx) {
  double x1 = 0.0, x2 = 0.0;                         // x(i+1), x(i+2)
  struct R { double a, b, c, y, d, e; };
  stream_rows<PF, -1, R>(N, N, [&](int i, R& r) {
    const int c = clampi(i, 1, N);
    r.a = q(c, s0); r.b = q(c, s0 + 1); r.c = q(c, s0 + 2); r.y = q(c, s0 + 5); r.d = q(c, AY);
    if (MU) r.e = q(c, BY);
  }, [&](int i, const R& r) {
    const double x = div_rcp((r.d - x2 * r.c) - x1 * r.b, r.a, r.y);
    q(i, sx) = x;
    if (MU) q(i, BY) = x >= 100.0 ? r.e : 0.0;
    x2 = x1;
    x1 = x;
  });
}

// M^T w = rhs for a matrix factored by adj_elim into slots s0...  The rhs is slot s0+3, or
// with CW the interior rows of cw * (slot BY); slot s0+3 ends holding w.
// U^T z = rhs top-down (z(i-1), the chain's last value, comes off last; the error is the same in
// either order), then the eliminations transposed bottom-up: z(j) -= l_j z(j+1), then the
// interchange.
template <bool CW>
__device__ __forceinline__ void adj_solveT(const Col& q, int N, int s0, double cw = 0.0) {
  double zm1 = 0.0, zm2 = 0.0;                       // z(i-1), z(i-2)
  double u1m1 = 0.0, u2m1 = 0.0, u2m2 = 0.0;         // U1(i-1), U2(i-1), U2(i-2)
  struct R { double a, b, c, y, d; };
  stream_rows<PF, 1, R>(1, N, [&](int i, R& r) {
    const int c = clampi(i, 1, N);
    r.a = q(c, s0); r.b = q(c, s0 + 1); r.c = q(c, s0 + 2); r.y = q(c, s0 + 5);
    r.d = q(c, CW ? BY : s0 + 3);
  }, [&](int i, const R& r) {
    const double rhs = !CW ? r.d : (i >= 2 && i <= N - 1 ? cw * r.d : 0.0);
    const double z = div_rcp((rhs - u2m2 * zm2) - u1m1 * zm1, r.a, r.y);
    q(i, s0 + 3) = z;
    zm2 = zm1; zm1 = z;
    u2m2 = u2m1;
    u1m1 = r.b; u2m1 = r.c;
  });
  double carry = q(N, s0 + 3);
  struct T { double z, l, c; };
  stream_rows<PF, -1, T>(N - 1, N - 1, [&](int j, T& r) {
    const int c = clampi(j, 1, N);
    r.z = q(c, s0 + 3); r.l = q(c, s0 + 4); r.c = q(c, s0 + 2);
  }, [&](int j, const T& r) {
    const double a = r.z - r.l * carry;
    const bool swap = interchanged(r.c);
    q(j + 1, s0 + 3) = swap ? a : carry;
    carry = swap ? carry : a;
  });
  q(1, s0 + 3) = carry;
}

// Electron inputs of row r of column (i2, i3)
__device__ __forceinline__ CellIn<true> adj_cell(const DevGrid& g, const DevState& s, const AdjArgs& A,
                                                 int r, int i2, int i3, long col) {
  const long c = gix(g, r, i2, i3), k = (long)g.lx1 * col + r - 1, ni = (long)g.lx1 * g.lx2 * g.lx3;
  CellIn<true> v;
  v.T = A.TD[c];
  v.n = A.NE1[c];
  v.h1 = g.h1[c]; v.h2 = g.h2[c]; v.h3 = g.h3[c];
  v.n1 = s.nn[k]; v.n2 = s.nn[ni + k]; v.n3 = s.nn[2 * ni + k];
  v.J = s.J1[c];
  v.kap = s.kappa ? s.kappa[col] : 1.0;
  return v;
}

// row i's entries from the coefficients C, B of the row and D of it and its neighbours
struct RowTerms { double s1, s2, s3; };
__device__ __forceinline__ RowTerms adj_row(const DevGrid& g, int i, double C, double B, double Dm,
                                            double Dc, double Dp) {
  const double* dx1i = g.dx1i - 1;
  const double Dh = 0.5 * (Dm + Dc), Dh1 = 0.5 * (Dc + Dp);
  RowTerms t;
  t.s1 = ((C * Dh) / dx1i[i]) / g.dx1[i];
  t.s3 = ((C * Dh1) / dx1i[i]) / g.dx1[i + 1];
  t.s2 = B / (g.dx1[i + 1] + g.dx1[i]);
  return t;
}

// The adjoint of TRBDF2 in three kernels.  Its recurrences run one lane per column, and a
// grid of a few thousand columns gives a wave to one CU in five: everything that is no
// recurrence is done by cell, in tiles that read the fields along x1 and the scratch along
// the columns (LDS turns one into the other).  192x64x48: 228 us, of which some 160 are the
// recurrences; one kernel with a lane per column took 728, most of it in two passes that read
// the fields with the stride of a column.
constexpr int TR_ROWS = 32, TC = 16, LDT = TR_ROWS + 1;      // a tile's rows and columns in LDS

// s1, s2, s3 of the rows 2..N-1 and the right-hand sides, into the slots A0..AY, B0..B2 and X2;
// dL/dTe of all rows into BY
__global__ __launch_bounds__(TPB) void k_adj_terms(DevGrid g, DevState s, AdjArgs A, double* scratch) {
  __shared__ double lT[TC * LDT], lC[TC * LDT], lB[TC * LDT], lD[TC * LDT],
      lL[TC * LDT];
  const long ncol = (long)g.lx2 * g.lx3;
  const int N = g.lx1;
  const unsigned row_tiles = (N - 2 + TR_ROWS - 3) / (TR_ROWS - 2);
  const int first = (int)(blockIdx.x % row_tiles) * (TR_ROWS - 2) + 1;  // the tile's rows first..
  const long col0 = (long)(blockIdx.x / row_tiles) * TC;
  const double gm1kB = (gammas(LSP) - 1.0) / kB;
  for (int u = threadIdx.x; u < TR_ROWS * TC; u += TPB) {
    const int rr = u % TR_ROWS, cc = u / TR_ROWS, r = first + rr;
    const long col = col0 + cc;
    if (r <= N && col < ncol) {
      const int i2 = (int)(col % g.lx2) + 1, i3 = (int)(col / g.lx2) + 1;
      const CellIn<true> c = adj_cell(g, s, A, r, i2, i3, col);
      double C, B, D;
      cell_coeffs<true, true>(c, LSP, gm1kB, C, B, D);
      const int o = cc * LDT + rr;
      lT[o] = c.T; lC[o] = C; lB[o] = B; lD[o] = D;
      lL[o] = A.lam[gix(g, r, i2, i3)];
    }
  }
  __syncthreads();
  const double dt2 = A.dt / 2.0, dt3 = A.dt / 3.0, c13 = 1.0 / 3.0;
  for (int u = threadIdx.x; u < TR_ROWS * TC; u += TPB) {
    const int cc = u % TC, rr = u / TC, i = first + rr;
    const long col = col0 + cc;
    if (i > N || col >= ncol) continue;
    const int o = cc * LDT + rr;
    const Col q(scratch, N, col);
    if (i == 1 || i == N) q(i, BY) = lL[o];
    if (rr < 1 || rr > TR_ROWS - 2 || i > N - 1) continue;
    const RowTerms t = adj_row(g, i, lC[o], lB[o], lD[o - 1], lD[o], lD[o + 1]);
    const double t1 = t.s1 / 2.0, t2 = t.s2 / 2.0, t3 = t.s3 / 2.0;
    const double a = -t1 + t2, c = -t3 - t2;
    q(i, A0) = t.s1; q(i, A1) = t.s2; q(i, A2) = t.s3;
    q(i, B0) = t.s1; q(i, B1) = t.s2; q(i, B2) = t.s3;
    q(i, AY) = ((lT[o] / dt2 - a * lT[o - 1]) - (t3 + t1) * lT[o]) - c * lT[o + 1];
    q(i, X2) = -((c13 * lT[o]) / dt3);
    q(i, BY) = lL[o];
  }
}

// The two solves and their transposes: a block of two waves to 64 columns, a lane per column
// in each.  The waves factor the TR and the BDF2 matrix side by side; the first goes on
// through the passes that depend on each other.  Bound by its chains: rows times eight passes
// times a row's dependent operations and their issue by a lone wave, some 250 cycles; so
// pivots keep their reciprocals (div_rcp is exact), an interchange is read off the pivot row,
// and a row's slots lie within the immediate offsets of one address (246 us without the three).
__global__ __launch_bounds__(128) void k_adj_trbdf2(DevGrid g, DevState s, AdjArgs A,
                                                     double* scratch) {
  __shared__ int bad[64];
  const long ncol = (long)g.lx2 * g.lx3;
  const int lane = threadIdx.x & 63;
  const bool second = threadIdx.x >= 64;
  const long col = (long)blockIdx.x * 64 + lane;
  const bool active = col < ncol;
  const int N = g.lx1;
  const int i2 = (int)(col % g.lx2) + 1, i3 = (int)(col / g.lx2) + 1;
  const long kb = (long)N * col;
  const Col q(scratch, N, active ? col : ncol - 1);
  const double* dx1 = g.dx1;
  const double dt2 = A.dt / 2.0, K1 = 1.0 / dt2;
  const double dt3 = A.dt / 3.0, K2 = 1.0 / dt3;
  const double c43 = 4.0 / 3.0;
  double Tmin = 0.0, Tmax = 0.0, aN = 0.0, bN = 1.0;
  bool sing = false;
  if (active) {
    const double Tn1 = s.Tn[kb], TnN = s.Tn[kb + N - 1];
    if (g.gridflag == 0) { Tmin = Tn1; Tmax = TnN; }
    else if (g.gridflag == 1) { Tmax = TnN; Tmin = A.Teinf; }
    else { Tmin = Tn1; Tmax = A.Teinf; }
    if (s.qtop) {
      const CellIn<true> c = adj_cell(g, s, A, N, i2, i3, col);
      aN = -1.0 / dx1[N];
      bN = 1.0 / dx1[N];
      Tmax = (s.qtop[col] * c.h1) / (cell_lambda<true, false>(c, LSP) * c.kap);
    }
    // pass A (top-down): the factorisation, the TR right-hand side eliminated alongside (rows
    // read ahead of the pivot rows that replace them)
    double e0 = 1.0, e1 = 0.0, eb = Tmin;            // pending row (row 1: identity)
    if (!second) {
      stream_rows<PF, 1, R4>(2, N - 2, [&](int i, R4& r) {
        const int c = clampi(i, 1, N);
        r.a = q(c, A0); r.b = q(c, A1); r.c = q(c, A2); r.d = q(c, AY);
      }, [&](int i, const R4& r) {
        const double t1 = r.a / 2.0, t2 = r.b / 2.0, t3 = r.c / 2.0;
        sing |= adj_elim<true>(q, i - 1, A0, e0, e1, eb, -t1 + t2, (K1 + t3) + t1, -t3 - t2, r.d);
      });
      sing |= adj_elim<true>(q, N - 1, A0, e0, e1, eb, aN, bN, 0.0, Tmax);   // boundary row N
      q(N, A0) = e0; q(N, A1) = 0.0; q(N, A2) = 0.0; q(N, AY) = eb; q(N, AI) = 1.0 / e0;
    } else {
      stream_rows<PF, 1, R4>(2, N - 2, [&](int i, R4& r) {
        const int c = clampi(i, 1, N);
        r.a = q(c, B0); r.b = q(c, B1); r.c = q(c, B2);
      }, [&](int i, const R4& r) {
        sing |= adj_elim<false>(q, i - 1, B0, e0, e1, eb, -r.a + r.b, (K2 + r.c) + r.a, -r.c - r.b, 0.0);
      });
      sing |= adj_elim<false>(q, N - 1, B0, e0, e1, eb, aN, bN, 0.0, 0.0);
      q(N, B0) = e0; q(N, B1) = 0.0; q(N, B2) = 0.0; q(N, BI) = 1.0 / e0;
    }
    sing |= e0 == 0.0;
  }
  if (second) bad[lane] = sing;
  __syncthreads();
  if (second || !active) return;
  if (sing || bad[lane]) {                           // no adjoint of a singular solve
    q(1, BL) = SINGULAR;
    return;
  }
  // pass B: TR solution
  adj_backsub<false>(q, N, A0, X1);
  // pass C: BDF2 right-hand side through the stored eliminations (row 1: Tmin, row N: Tmax)
  // into AY
  {
    double rb = Tmin;
    stream_rows<PF, 1, R4>(1, N - 1, [&](int j, R4& r) {
      const int c = clampi(j, 1, N - 1);
      r.a = q(c + 1, X2); r.b = q(c + 1, X1); r.c = q(c, B2); r.d = q(c, BL);
    }, [&](int j, const R4& r) {
      const double d = j + 1 >= N ? Tmax : r.a + div_rcp(c43 * r.b, dt3, K2);
      const bool swap = interchanged(r.c);
      const double pd = swap ? d : rb, od = swap ? rb : d;
      q(j, AY) = pd;
      rb = od + r.d * (-pd);
    });
    q(N, AY) = rb;
  }
  // pass D: BDF2 solution, and mu = dL/dx2 through the output floor into BY
  adj_backsub<true>(q, N, B0, X2);
  // passes E-F: w2
  adj_solveT<false>(q, N, B0);
  // passes G-H: w1 from dL/dx1 = (4/3)/(dt/3) w2 on the interior rows
  adj_solveT<true>(q, N, A0, c43 / dt3);
}

// Chain w1, w2 through the matrix and rhs entries of rows 2..N-1
//   dL/dM1(i,k) = -w1(i) (x1(k) + T(k))   (M1 x1 = (2/(dt/2) - M1) T on those rows)
//   dL/dM2(i,k) = -w2(i) x2(k)
// to s1 = C Dh(i)/dx1i/dx1(i), s3 = C Dh(i+1)/dx1i/dx1(i+1) (TR uses s/2), then Dh, D,
// lambda = kappa lambda_e(T), and the direct T terms of both right-hand sides.  A block walks
// the rows of TC columns in tiles with two rows more on each side, and sums a column's
// dL/dkappa in row order.
__global__ __launch_bounds__(TPB) void k_adj_chain(DevGrid g, DevState s, AdjArgs A, const double* scratch) {
  // T C B D x1 x2 w1 w2; then u v tm tc tn in place of x1 .. w2 and B, the kappa terms in x1
  __shared__ double l[8][TC * LDT];
  constexpr int CELLS = TR_ROWS * TC / TPB;
  const long ncol = (long)g.lx2 * g.lx3;
  const long col0 = (long)blockIdx.x * TC;
  const int N = g.lx1;
  const double gm1kB = (gammas(LSP) - 1.0) / kB;
  const double dt2 = A.dt / 2.0, K1 = 1.0 / dt2, dt3 = A.dt / 3.0, c13 = 1.0 / 3.0;
  const double* dx1i = g.dx1i - 1;
  double gk = 0.0;
  for (int first = -1; first + 2 <= N; first += TR_ROWS - 4) {          // tile rows first..first+31
    CellIn<true> in[CELLS];
    double lam_e[CELLS];
#pragma unroll
    for (int v = 0; v < CELLS; ++v) {
      const int u = threadIdx.x + v * TPB, rr = u % TR_ROWS, cc = u / TR_ROWS, r = first + rr;
      const long col = col0 + cc;
      lam_e[v] = 0.0;
      if (r < 1 || r > N || col >= ncol) continue;
      in[v] = adj_cell(g, s, A, r, (int)(col % g.lx2) + 1, (int)(col / g.lx2) + 1, col);
      const int o = cc * LDT + rr;
      lam_e[v] = cell_lambda<true, false>(in[v], LSP);
      l[0][o] = in[v].T;
      cell_coeffs<true, true>(in[v], LSP, gm1kB, l[1][o], l[2][o], l[3][o]);
    }
#pragma unroll
    for (int v = 0; v < CELLS; ++v) {
      const int u = threadIdx.x + v * TPB, cc = u % TC, rr = u / TC, r = first + rr;
      const long col = col0 + cc;
      if (r < 1 || r > N || col >= ncol) continue;
      const Col q(scratch, N, col);
      const int o = cc * LDT + rr;
      l[4][o] = q(r, X1); l[5][o] = q(r, X2); l[6][o] = q(r, AY); l[7][o] = q(r, BY);
    }
    __syncthreads();
    double uu[CELLS], vv[CELLS], tm[CELLS], tc[CELLS], tn[CELLS];
#pragma unroll
    for (int v = 0; v < CELLS; ++v) {
      const int t = threadIdx.x + v * TPB, rr = t % TR_ROWS, cc = t / TR_ROWS, i = first + rr;
      uu[v] = vv[v] = tm[v] = tc[v] = tn[v] = 0.0;
      if (rr < 1 || rr > TR_ROWS - 2 || i < 2 || i > N - 1 || col0 + cc >= ncol) continue;
      const int o = cc * LDT + rr;
      const double *T = l[0] + o, *x1 = l[4] + o, *x2 = l[5] + o, *D = l[3] + o;
      const double C = l[1][o], w1 = l[6][o], w2 = l[7][o];
      const RowTerms s_ = adj_row(g, i, C, l[2][o], D[-1], D[0], D[1]);
      const double t1 = s_.s1 / 2.0, t2 = s_.s2 / 2.0, t3 = s_.s3 / 2.0;
      const double a = -t1 + t2, c = -t3 - t2;
      const double G1a = -w1 * (x1[-1] + T[-1]), G1b = -w1 * (x1[0] + T[0]), G1c = -w1 * (x1[1] + T[1]);
      const double G2a = -w2 * x2[-1], G2b = -w2 * x2[0], G2c = -w2 * x2[1];
      const double gs1 = 0.5 * (G1b - G1a) + (G2b - G2a);
      const double gs3 = 0.5 * (G1b - G1c) + (G2b - G2c);
      uu[v] = gs1 * ((C / dx1i[i]) / g.dx1[i]);        // to Dh(i)
      vv[v] = gs3 * ((C / dx1i[i]) / g.dx1[i + 1]);    // to Dh(i+1)
      tm[v] = -w1 * a;                                 // row i: -a T(i-1)
      tc[v] = w1 * (K1 - (t3 + t1)) - (c13 / dt3) * w2;
      tn[v] = -w1 * c;                                 // row i: -c T(i+1)
    }
    __syncthreads();
#pragma unroll
    for (int v = 0; v < CELLS; ++v) {
      const int t = threadIdx.x + v * TPB, o = (t / TR_ROWS) * LDT + t % TR_ROWS;
      l[4][o] = uu[v]; l[5][o] = vv[v]; l[6][o] = tm[v]; l[7][o] = tn[v];
    }
    __syncthreads();
    double kterm[CELLS];
#pragma unroll
    for (int v = 0; v < CELLS; ++v) {
      const int t = threadIdx.x + v * TPB, rr = t % TR_ROWS, cc = t / TR_ROWS, j = first + rr;
      const long col = col0 + cc;
      kterm[v] = 0.0;
      if (rr < 2 || rr > TR_ROWS - 3 || j < 1 || j > N || col >= ncol) continue;
      const int o = cc * LDT + rr;
      double* lam = A.lam + gix(g, j, (int)(col % g.lx2) + 1, (int)(col / g.lx2) + 1);
      const Col q(scratch, N, col);
      if (q(1, BL) == SINGULAR) {
        *lam = __builtin_nan("");
        continue;
      }
      // dL/dDh(j) and (j+1); D(j) = lambda(j) h2 h3 / h1 enters both
      const double gDh = l[5][o - 1] + uu[v], gDh1 = vv[v] + l[4][o + 1];
      const double gT = (l[7][o - 1] + tc[v]) + l[6][o + 1];
      double glam = (0.5 * (gDh + gDh1)) * ((in[v].h2 * in[v].h3) / in[v].h1);
      if (s.qtop && j == N) {                          // row N rhs: q h1(N) / lambda(N)
        const double gg = q(N, AY) + q(N, BY);
        const double lamN = lam_e[v] * in[v].kap;
        glam += -gg * (((s.qtop[col] * in[v].h1) / lamN) / lamN);
        if (A.gq) A.gq[col] += gg * (in[v].h1 / lamN);
      }
      kterm[v] = glam * lam_e[v];
      *lam = gT + glam * (in[v].kap * lambda_e_dT(in[v], lam_e[v]));
    }
    // (B is not read any more; rows of other tiles and of singular columns hold 0)
#pragma unroll
    for (int v = 0; v < CELLS; ++v) {
      const int t = threadIdx.x + v * TPB;
      l[2][(t / TR_ROWS) * LDT + t % TR_ROWS] = kterm[v];
    }
    __syncthreads();
    if (threadIdx.x < TC) {
#pragma unroll
      for (int rr = 2; rr <= TR_ROWS - 3; ++rr) gk += l[2][threadIdx.x * LDT + rr];
    }
    __syncthreads();
  }
  const long col = col0 + threadIdx.x;
  if (threadIdx.x < TC && col < ncol && A.gk && Col(scratch, N, col)(1, BL) != SINGULAR) A.gk[col] += gk;
}

}  // namespace

size_t adjoint_scratch_bytes(const DevGrid& g) {
  return (size_t)NSA * g.lx1 * (((long)g.lx2 * g.lx3 + 63) / 64 * 64) * sizeof(double);
}

void launch_tape_vels(const DevGrid& g, const DevState& s, double* v1, double* v2, double* v3,
                      hipStream_t st) {
  const long so = (long)(LSP - 1) * g.N;
  const long n = (long)(g.lx1 + 1) * g.lx2 * g.lx3 + (long)g.lx1 * (g.lx2 + 1) * g.lx3 +
                 (long)g.lx1 * g.lx2 * (g.lx3 + 1);
  hipLaunchKernelGGL(k_tape_vels, dim3(grid_for(n)), dim3(TPB), 0, st, g, s.vs1 + so,
                     s.vs2 + so, s.vs3 + so, v1, v2, v3);
}

void launch_adjoint_step(const DevGrid& g, const DevState& s, const AdjTape& t, double dt,
                         double Teinf, double* lam, double* work, double* gk, double* gq,
                         double* scratch, hipStream_t st) {
  const long ncol = (long)g.lx2 * g.lx3;
  const dim3 cells(grid_for(g.N)), blk(TPB);
  AdjArgs A{t.TD, t.NE1, lam, gk, gq, dt, Teinf};
  timing_begin("adj_trbdf2", st);
  const unsigned tiles = (unsigned)((ncol + TC - 1) / TC);
  const unsigned row_tiles = (g.lx1 - 2 + TR_ROWS - 3) / (TR_ROWS - 2);     // (lx1 >= 4)
  hipLaunchKernelGGL(k_adj_terms, dim3(row_tiles * tiles), dim3(TPB), 0, st, g, s, A, scratch);
  hipLaunchKernelGGL(k_adj_trbdf2, dim3((unsigned)((ncol + 63) / 64)), dim3(128), 0, st, g, s, A,
                     scratch);
  hipLaunchKernelGGL(k_adj_chain, dim3(tiles), dim3(TPB), 0, st, g, s, A, scratch);
  timing_end("adj_trbdf2", st);
  timing_begin("adj_advection", st);
  hipLaunchKernelGGL(k_adj_rhoe2T, cells, blk, 0, st, g, lam, t.TD, t.NE1);
  hipLaunchKernelGGL(k_adj_sweep<2>, cells, blk, 0, st, g, lam, work, t.ES2, t.V2, dt);
  const dim3 hal(grid_exact((long)g.L1 * g.lx2));
  if (g.flagper) hipLaunchKernelGGL(k_adj_halo, hal, blk, 0, st, g, work);
  hipLaunchKernelGGL(k_adj_sweep<1>, cells, blk, 0, st, g, work, lam, t.ES1, t.V1, dt);
  hipLaunchKernelGGL(k_adj_sweep<3>, cells, blk, 0, st, g, lam, work, t.ES3, t.V3, dt);
  if (g.flagper) hipLaunchKernelGGL(k_adj_halo, hal, blk, 0, st, g, work);
  else hipLaunchKernelGGL(k_adj_bc_x3, dim3(grid_exact((long)g.L1 * g.L2)), blk, 0, st, g, work);
  hipLaunchKernelGGL(k_adj_bc_x2, dim3(grid_exact((long)g.L1 * g.L3)), blk, 0, st, g, work);
  hipLaunchKernelGGL(k_adj_bc_x1, dim3(grid_exact((long)g.L2 * g.L3)), blk, 0, st, g, work, t.NE0);
  hipLaunchKernelGGL(k_adj_T2rhoe, cells, blk, 0, st, g, work, lam, t.NE0);
  timing_end("adj_advection", st);
}

}  // namespace gemhip
