// kernels_diffusion.hip -- field-aligned energy diffusion (TRBDF2 / backward Euler).
//
// Reference: src/multifluid/multifluid.f90:309-342 (energy_diffusion),
// src/collisions/collisions.f90:162-199 (thermal_conduct),
// src/numerical/diffusion/diffusion.f90:24-152 (diffusion_prep, column loops),
// src/numerical/diffusion/PDEparabolic.f90:19-346 (TRBDF21D, backEuler1D) and the
// LAPACK dgbsv call of src/vendor/lapack95/gbsv.in.f90:58-97.
//
// Each column (fixed x2, x3, species) is solved by one lane, reproducing operation for
// operation what the reference computes for it: the conductivity and the band matrix
// entries in the reference's expression order, then LAPACK's banded LU with partial
// pivoting (dgbtf2: idamax pivot search, dscal by the reciprocal pivot, dger update;
// dgbtrs: row swaps and dger on the right-hand side; dtbsv: column-oriented back
// substitution).  The matrix is tridiagonal stored with kl=ku=2, so of the band only the
// three diagonals and the pivoting fill-in can be non-zero; every other term LAPACK forms
// is a multiply by an exact zero and leaves values unchanged, so those terms are not
// formed.  Divisions are IEEE divisions or give their results (div_rcp), and the file is
// built with -ffp-contract=off, which makes the result bit-identical to the reference
// arithmetic apart from x**2.5 (correctly rounded here, libm pow there).
#include <type_traits>

#include "diffusion_cell.h"

namespace gemhip {

namespace {

struct Coef {
  double K;        // 1/(dt/2) (TR), 1/(dt/3) (BDF2) or 1/dt (backward Euler)
  double dt2, dt3, dt;
  double c13, c43; // 1/3._wp and 4/3._wp
};

// ---------------------------------------------------------------- column-group kernel
// One wavefront (the whole workgroup) owns 64 systems, one lane each: the 64 columns of a
// column group for the electrons, or 32 columns (half a group) of two ion species.  The two
// ions of a wave read the columns' metric factors once.  It makes four passes over the rows:
//   1 (top-down): the input rows arrive in chunks of R rows, loaded by the wave
//     cooperatively (lane -> (row, column), so each load instruction reads whole 64-byte
//     segments), the next chunk's loads in flight while a chunk is used.  Conductivity and
//     the cell factors C, B, D of each (row, column) go through LDS; each lane then forms
//     its rows' three parabolic terms and runs the pivoted elimination of the first solve
//     (TR, or backward Euler).  It keeps the terms and the temperature of every row, and
//     the elimination's state at the first row of every block of R rows; the pivot rows
//     themselves are not kept;
//   2 (bottom-up, block by block): the block's pivot rows formed again in registers from
//     its kept state, and back substitution through them (into Ts for backward Euler; for
//     TRBDF2 the BDF2 right-hand side of each row, in the temperature's place);
//   3 (top-down, TRBDF2): the elimination of the BDF2 system, its state kept per block;
//   4 (bottom-up, TRBDF2): as pass 2, into Ts.
// Every value is formed with the operations, and in the order, LAPACK's dgbtf2, dgbtrs
// and dtbsv would use on the reference's band matrix; forming a pivot row a second time
// from the same state gives the same bits.
//
// Why the pivot rows are formed twice: the full-size launch is bound by HBM traffic, and
// the solve's arithmetic is a fifth of its time.  Keeping both factorisations took nine
// 8-byte slots per row and species, each written and read (a pivot row, its right-hand
// side and a multiplier for each solve); the terms, the temperature and the block states
// take 3.4 slots for an ion and 4.4 for the electrons.  With the ions' shared metric factors
// the cheaper x**2.5 and divisions, and no tests for zero entries: 512x256x192 7.91 -> 5.84 ms,
// 255x113x67 0.87 -> 0.57, 301x127x75 1.19 -> 0.79 (backward Euler 256x128x96 0.66 -> 0.485).
//
// Rows are kept lane-interleaved in HBM (one 512-byte segment per row and slot for the
// wave) and outputs are staged through LDS so global stores are coalesced.  Blocks are
// numbered so that the species of a column group run on one XCD, the electron groups (the
// longest waves) first.
//
// Divisions by values that depend on the row or the step alone (coordinate differences, dt/2,
// dt/3) are multiplications by correctly rounded reciprocals with one correction (div_rcp),
// which gives the IEEE quotient; every other division is one.
//
// The steady state of every pass issues its memory operations unconditionally (clamped
// indices; rows 1 and N have slots that no system uses, where rows past the ends land), so
// the compiler's wait counters stay exact and loads issued ahead stay in flight.  Lanes of a
// group past the last column solve the last column again and write the same values to the
// same places.
constexpr int LP = 65;         // padded LDS row (conflict-free transposed access)
#ifndef DIFF_CHUNK
#define DIFF_CHUNK 8           // rows per chunk: 4 x 8 x 65 doubles of LDS per wave
#endif
#ifndef DIFF_BATCH_E
#define DIFF_BATCH_E 2         // electron cells per lane whose inputs are loaded together
#endif
// slots of a row: the parabolic terms of its lower and upper neighbour and (electrons) of
// the drift; the input temperature, which pass 2 replaces by the BDF2 right-hand side
enum : int { ST1 = 0, ST3 = 1, STV = 2, ST2 = 3 };
constexpr int NCK = 3;         // kept elimination state: r0, r1, rb

// units of a column group: one wave of electrons, six of ions (half of its columns, a pair
// of species)
__host__ __device__ inline long diffusion_groups(const DevGrid& g) {
  return ((long)g.lx2 * g.lx3 + 63) / 64;
}
__host__ __device__ inline int kept_blocks(const DevGrid& g) { return (g.lx1 + 6) / 4 + 1; }
__host__ __device__ inline long unit_doubles(const DevGrid& g, bool elec) {
  return ((long)g.lx1 * (elec ? 4 : 3) + (long)kept_blocks(g) * NCK) * 64;
}

__device__ __forceinline__ int clampi(int v, int lo, int hi) { return v < lo ? lo : (v > hi ? hi : v); }

__device__ __forceinline__ void column_of(const DevGrid& g, int gcol, int& i2, int& i3) {
  i2 = gcol % g.lx2 + 1;
  i3 = gcol / g.lx2 + 1;
}
// a grid array at a wave-uniform index, by a scalar load (a vector load would be the newest
// vector memory operation, and waiting for it would wait for every kept row in flight)
__device__ __forceinline__ double ld_row(const double* p, int i) {
  return ((const __attribute__((address_space(4))) double*)p)[i];
}

// a pointer to HBM that is the same for the whole wave, in scalar registers
typedef __attribute__((address_space(1))) double gdouble;
__device__ __forceinline__ gdouble* uniform_ptr(double* p) {
  const unsigned long a = (unsigned long)p;
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)a);
  const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(a >> 32));
  return (gdouble*)(((unsigned long)hi << 32) | lo);
}

// State of the pivoted elimination between steps: the row at pivot position j holds
// (r0, r1) in columns j, j+1 (column j+2 is always zero there) and right-hand side rb.
struct Elim {
  double r0, r1, rb;
  bool singular;
};
struct Pivot {
  double u0, u1, u2, y;
};

// Pivoted elimination step (dgbtf2 with dgbtrs's forward solve) bringing in the row
// (a, b, cc | d): returns the pivot row, advances the state.  A zero pivot leaves the other
// row as it is.  Written without branches: a step under a branch could not overlap the next
// row's independent work.  (The band routines also skip zero entries; while the entries and the
// pivot's reciprocal are finite, the product of one changes at most the sign of a zero, which no
// temperature shows.  Columns with an infinite or NaN temperature or density, a step of zero or of
// infinity come out alike with and without the tests.  These took 6 % of the solve at 255x113x67
// and 10 % at 128x64x1.)  Rows interchange at most cells where
// the diffusion number is large, so steps that assume the pending row is the larger, with
// these as the way out, took twice as long.
__device__ __forceinline__ Pivot elim_step(Elim& e, double a, double b, double cc, double d,
                                           bool& swap, double* mult = nullptr) {
  swap = fabs(a) > fabs(e.r0);
  Pivot p;
  p.u0 = swap ? a : e.r0;
  p.u1 = swap ? b : e.r1;
  p.u2 = swap ? cc : 0.0;
  p.y = swap ? d : e.rb;
  const double o0 = swap ? e.r0 : a, o1 = swap ? e.r1 : b, o2 = swap ? 0.0 : cc,
               od = swap ? e.rb : d;
  const bool live = p.u0 != 0.0;
  const double rp = 1.0 / p.u0;
  const double l = live ? rp * o0 : 0.0;
  if (mult) *mult = l;
  e.r0 = o1 + l * (-p.u1);
  e.r1 = o2 + l * (-p.u2);
  e.rb = od + l * (-p.y);
  e.singular = e.singular | !live;
  return p;
}

// one row of dtbsv, column-oriented: x(i+2) U2 comes off first, then x(i+1) U1
__device__ __forceinline__ double back_step(const Pivot& p, double x1, double x2) {
  return ((p.y - x2 * p.u2) - x1 * p.u1) / p.u0;
}

template <int R, bool BE, bool ELEC, bool EXT>
__device__ __forceinline__ void diffusion_unit(const DevGrid& g, const DevState& s,
                                               double* scratch, const Coef& k1, const Coef& bdf,
                                               double Teinf, long cg, int half, int pair,
                                               double (*sT)[LP], double (*sC)[LP],
                                               double (*sB)[LP], double (*sD)[LP]) {
  constexpr int NC = ELEC ? 64 : 32;                 // columns of the wave
  constexpr int NSP = ELEC ? 1 : 2;                  // species of the wave
  constexpr int CPI = 64 / R;                        // columns per load instruction
  constexpr int NK = NC / CPI;                       // and cells per lane of a chunk
  constexpr int NS = ELEC ? 4 : 3;
  const int lane = threadIdx.x;
  const int N = g.lx1;
  const int isp0 = ELEC ? LSP : 2 * pair + 1;
  const int isp = ELEC ? LSP : isp0 + (lane >> 5);
  const int l0 = ELEC ? 0 : half * 32;               // the wave's first lane in the group
  const int col = group_column(g, cg, l0 + (lane & (NC - 1)));
  const long gps = diffusion_groups(g);
  gdouble* row0 = uniform_ptr(
      scratch + (ELEC ? cg * unit_doubles(g, true)
                      : gps * unit_doubles(g, true) +
                            ((cg * 2 + half) * 3 + pair) * unit_doubles(g, false)));
  gdouble* ck0 = row0 + (long)N * NS * 64;
  // Kept rows are non-temporal (the nt bit: streamed through L2 at low priority): each is
  // written once and read a pass later, and as ordinary accesses they evicted the input
  // lines that the cooperative loads of the next chunk still needed.
  // (addresses: a wave-uniform row pointer plus the lane)
  const unsigned ln = lane;
  auto put = [&](int i, int k, double v) { __builtin_nontemporal_store(v, row0 + ((long)(i - 1) * NS + k) * 64 + ln); };
  auto get = [&](int i, int k) { return __builtin_nontemporal_load(row0 + ((long)(i - 1) * NS + k) * 64 + ln); };
  auto keep_state = [&](int m, const Elim& e) {
    gdouble* c = ck0 + (long)m * NCK * 64;
    __builtin_nontemporal_store(e.r0, c + ln);
    __builtin_nontemporal_store(e.r1, c + 64 + ln);
    __builtin_nontemporal_store(e.rb, c + 128 + ln);
  };
  const long ni = (long)g.lx1 * g.lx2 * g.lx3;
  const long kb = (long)g.lx1 * col;
  const double* dx1 = g.dx1;
  const double* dx1i = g.dx1i - 1;
  double Tmin, Tmax;
  {
    const double Tn1 = s.Tn[kb], TnN = s.Tn[kb + N - 1];
    if (g.gridflag == 0) { Tmin = Tn1; Tmax = TnN; }
    else if (g.gridflag == 1) { Tmax = TnN; Tmin = Teinf; }
    else { Tmin = Tn1; Tmax = Teinf; }
  }
  // row N: the reference's Dirichlet row, or under the extension with a top heat flux the
  // Neumann row (T(N) - T(N-1))/dx1(N) = q h1(N)/lambda(N)
  double aN = 0.0, bN = 1.0;
  if (EXT && ELEC && s.qtop) {
    CellIn<ELEC> top;
    cell_load<ELEC, EXT>(g, s, (long)(LSP - 1) * g.N, gix(g, 0, col % g.lx2 + 1, col / g.lx2 + 1),
                         kb, ni, N, top, hcol_index(g, col, N), col);
    aN = -1.0 / dx1[N];
    bN = 1.0 / dx1[N];
    Tmax = (s.qtop[col] * top.h1) / cell_lambda<ELEC, EXT>(top, isp);
  }
  // cooperative mapping of a chunk: lane -> (row lr, column sub-index cs)
  const int lr = lane % R, cs = lane / R;
  // Row phase of the chunk windows: a column's row 1 sits 2 cells into its stride, so
  // windows of R rows from row 1 straddle 64-byte sectors, and a sector's other part is
  // fetched again a chunk later (long after the L2 dropped it).  The wave's windows start
  // ph rows early instead, which puts the windows of lane 0's column, and of every column
  // that shares its sector phase (all of an interleaved group's), on sector boundaries.
  // The steps before row 1 are not real.  Blocks of kept state use the same windows.
  int c2, c3;
  column_of(g, group_column(g, cg, l0), c2, c3);
  constexpr int RA = R < 8 ? R : 8;                  // (R a power of two)
  const double* Ts0 = s.Ts + (long)(isp0 - 1) * g.N;
  const int ph = __builtin_amdgcn_readfirstlane(
      (int)(((unsigned long)(Ts0 + gix(g, 0, c2, c3) + 1) >> 3) & 7) % RA);
  const int mb = (N - 1 + ph) / R;                   // block and chunk of row N
  int cbk[NK];                                       // gix(0, i2, i3) of the columns this lane loads
  int kbk[ELEC ? NK : 1];                            // and their interior offsets lx1*(column)
  int gck[EXT && ELEC ? NK : 1];                     // and column numbers (extension only)
#pragma unroll
  for (int k = 0; k < NK; ++k) {
    const int gcol = group_column(g, cg, l0 + k * CPI + cs);
    int a2, a3;
    column_of(g, gcol, a2, a3);
    cbk[k] = (int)gix(g, 0, a2, a3);
    if (ELEC) kbk[k % (ELEC ? NK : 1)] = g.lx1 * gcol;
    if (EXT && ELEC) gck[k % (EXT && ELEC ? NK : 1)] = gcol;
  }

  // inputs of a chunk: rows r0..r0+R-1 (clamped to 1..N) of the wave's columns.  The electrons
  // (nine values a cell) load theirs in batches, the first a chunk ahead.
  constexpr int NB = ELEC ? (NK < DIFF_BATCH_E ? NK : DIFF_BATCH_E) : NK;
  CellIn<ELEC> in[NB][NSP];
  auto issue = [&](int r0, int k0, CellIn<ELEC> (*c)[NSP]) {
    const int r = clampi(r0 + lr, 1, N);
    // hcol slot of this lane's first column at row r: the group's 64 columns are contiguous
    // (slots past the last column repeat it, as these lanes do)
    const long hrow = ((long)cg * N + (r - 1)) * 64 + l0 + cs;
#pragma unroll
    for (int k = 0; k < NB; ++k) {
      const int kk = k0 + k;
      if (ELEC) {
        cell_load<ELEC, EXT>(g, s, (long)(LSP - 1) * g.N, cbk[kk], kbk[kk % (ELEC ? NK : 1)], ni, r,
                             c[k][0], hrow + kk * CPI, gck[kk % (EXT && ELEC ? NK : 1)]);
      } else {
        const long hc = hrow + kk * CPI;
        const double h1 = g.hcol[hc], h2 = g.hcol[g.hstride + hc], h3 = g.hcol[2 * g.hstride + hc];
#pragma unroll
        for (int q = 0; q < NSP; ++q) {
          const long so = (long)(isp0 + q - 1) * g.N;
          c[k][q].T = s.Ts[so + cbk[kk] + r];
          c[k][q].n = s.ns[so + cbk[kk] + r];
          c[k][q].h1 = h1; c[k][q].h2 = h2; c[k][q].h3 = h3;
        }
      }
    }
  };
  auto convert = [&](int k0, CellIn<ELEC> (*c)[NSP]) {
#pragma unroll
    for (int k = 0; k < NB; ++k) {
#pragma unroll
      for (int q = 0; q < NSP; ++q) {
        double C_, B_, D_;
        cell_coeffs<ELEC, EXT>(c[k][q], isp0 + q, (gammas(isp0 + q) - 1.0) / kB, C_, B_, D_);
        const int cc = q * 32 + (k0 + k) * CPI + cs;
        sT[lr][cc] = c[k][q].T; sC[lr][cc] = C_; sD[lr][cc] = D_;
        if (ELEC) sB[lr][cc] = B_;
      }
    }
  };

  // a row of each matrix from its parabolic terms (PDEparabolic.f90:19-145 TR half step,
  // :146-216 BDF2, :221-346 backward Euler); the ions' drift term is an exact zero
  auto first_row = [&](double t1f, double t2f, double t3f, double Tm, double Tc, double Tp,
                       double& a, double& b, double& c, double& d) {
    if (BE) {
      a = -t1f + t2f; b = (k1.K + t3f) + t1f; c = -t3f - t2f;
      d = div_rcp(Tc, k1.dt, k1.K);
    } else {
      const double t1 = t1f / 2.0, t2 = t2f / 2.0, t3 = t3f / 2.0;
      a = -t1 + t2; b = (k1.K + t3) + t1; c = -t3 - t2;
      d = ((div_rcp(Tc, k1.dt2, k1.K) - a * Tm) - (t3 + t1) * Tc) - c * Tp;
    }
  };

  // the record of the electron columns' interchanges (fitting extension, adjoint tapes)
  const int nw = (N + 31) / 32;
  int* prec = (EXT && ELEC && s.pivrec) ? s.pivrec + (long)col * 2 * nw : nullptr;
  int sbits = 0;
  auto record = [&](int stage, int j, bool swap) {   // step j (1..N-1) of the TR or BDF2 solve
    if (!(EXT && ELEC) || !prec) return;
    sbits |= (swap ? 1 : 0) << (j & 31);
    if ((j & 31) == 31 || j == N - 1) {
      prec[stage * nw + (j >> 5)] = sbits;
      sbits = 0;
    }
  };

  // ---- pass 1
  Elim e{1.0, 0.0, Tmin, false};
  {
    double Tm = 0.0, Tc = 0.0, Cc = 0.0, Bc = 0.0, Dm = 0.0, Dc = 1.0;
    issue(1 - ph, 0, in);
    for (int m = 0; m <= mb; ++m) {
      const int r0 = m * R + 1 - ph;
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int k0 = 0; k0 < NK; k0 += NB) {
        CellIn<ELEC> nxt[NB][NSP];
        if (k0 + NB < NK) issue(r0, k0 + NB, nxt);
        convert(k0, in);
        if (k0 + NB < NK) {
#pragma unroll
          for (int k = 0; k < NB; ++k) in[k][0] = nxt[k][0];
        }
      }
      issue(r0 + R, 0, in);
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int k = 0; k < R; ++k) {
        // row r's arrival completes the terms of row ro = r-1 (2..N-1)
        const int r = r0 + k, ro = r - 1, rc = clampi(ro, 2, N - 1), rs = clampi(ro, 1, N);
        const double Tp = sT[k][lane], Cp = sC[k][lane], Dp = sD[k][lane];
        const double Bp = ELEC ? sB[k][lane] : 0.0;
        const double dxi = ld_row(dx1i, rc), dxl = ld_row(dx1, rc), dxr = ld_row(dx1, rc + 1);
        const double ydxi = ld_row(g.rdx1i, rc), ydxl = ld_row(g.rdx1, rc), ydxr = ld_row(g.rdx1, rc + 1);
        const double Dhr = 0.5 * (Dm + Dc), Dhr1 = 0.5 * (Dc + Dp);
        const double t1f = div_rcp(div_rcp(Cc * Dhr, dxi, ydxi), dxl, ydxl);
        const double t3f = div_rcp(div_rcp(Cc * Dhr1, dxi, ydxi), dxr, ydxr);
        const double t2f = ELEC ? div_rcp(Bc, dxr + dxl, ld_row(g.rdx1s, rc)) : 0.0;
        put(rs, ST1, t1f);
        put(rs, ST3, t3f);
        put(rs, STV, Tc);
        if (ELEC) put(rs, ST2, t2f);
        if (k == 2) keep_state(m, e);                // before the step of position r0 = r - 2
        if (r >= 3 && r <= N) {
          double a, b, c, d;
          bool sw;
          first_row(t1f, t2f, t3f, Tm, Tc, Tp, a, b, c, d);
          elim_step(e, a, b, c, d, sw);
          record(0, r - 2, sw);
        }
        Tm = Tc; Tc = Tp;
        Cc = Cp; Bc = Bp;
        Dm = Dc; Dc = Dp;
      }
    }
    put(N, STV, Tc);                                 // (the window may end on row N)
    bool sw;
    elim_step(e, aN, bN, 0.0, Tmax, sw);             // boundary row N
    record(0, N - 1, sw);
    if (mb * R + 1 - ph == N) keep_state(mb, e);     // position N starts its block
    if (e.r0 == 0.0) e.singular = true;
  }

  // The rows of a block's steps: terms of row r = position + 1, reloaded for the next block
  // as soon as a step has used them.
  double t1[R], t3[R], t2[ELEC ? R : 1], v[R], ckn[NCK];
  auto load_terms = [&](int r, int u) {
    const int rr = clampi(r, 1, N);
    t1[u] = get(rr, ST1);
    t3[u] = get(rr, ST3);
    if (ELEC) t2[u % (ELEC ? R : 1)] = get(rr, ST2);
  };
  auto load_state = [&](int m) {
#pragma unroll
    for (int q = 0; q < NCK; ++q) ckn[q] = __builtin_nontemporal_load(ck0 + ((long)(m < 0 ? 0 : m) * NCK + q) * 64 + ln);
  };
  // Final temperatures go out through LDS, one block of R rows at a time (rows past N and
  // before 1 are never stored: those lanes store row N or 1 again).
  auto flush_out = [&](int j0) {
    __builtin_amdgcn_wave_barrier();
    const int rr = clampi(j0 + lr, 1, N);
#pragma unroll
    for (int q = 0; q < NSP; ++q) {
      double* To = s.Ts + (long)(isp0 + q - 1) * g.N;
#pragma unroll
      for (int kk = 0; kk < NK; ++kk) To[cbk[kk] + rr] = sT[rr - j0][q * 32 + kk * CPI + cs];
    }
    __builtin_amdgcn_wave_barrier();
  };

  // A TR factorisation that is singular leaves dgbsv's right-hand side as the solution: the
  // lanes concerned put the BDF2 right-hand side of that solution in place now (a slow pass
  // that never runs on physical inputs) and pass 2 leaves it there.
  const bool tr_sing = __any(e.singular);
  auto bdf_rhs = [&](double T, double x) {
    return -div_rcp(bdf.c13 * T, bdf.dt3, bdf.K) + div_rcp(bdf.c43 * x, bdf.dt3, bdf.K);
  };
  if (!BE && tr_sing && e.singular) {
    double Tm = get(1, STV), Tc = get(2, STV);
    for (int r = 2; r <= N - 1; ++r) {
      const double Tp = get(r + 1, STV);
      double a, b, c, d;
      first_row(get(r, ST1), ELEC ? get(r, ST2) : 0.0, get(r, ST3), Tm, Tc, Tp, a, b, c, d);
      put(r, STV, bdf_rhs(Tc, d));
      Tm = Tc; Tc = Tp;
    }
  }

  // ---- pass 2
  {
    double x1 = 0.0, x2 = 0.0, va = 0.0, vb = 0.0;   // va, vb: temperatures of the two rows above
    auto block = [&](auto edge_, int m) {
      constexpr bool EDGE = decltype(edge_)::value;
      const int j0 = m * R + 1 - ph;
      Elim q{ckn[0], ckn[1], ckn[2], false};
      double w[R + 2];
      Pivot P[R];
#pragma unroll
      for (int u = 0; u < R; ++u) w[u] = v[u];
      w[R] = va; w[R + 1] = vb;
      va = w[0]; vb = w[1];
      load_state(m - 1);
#pragma unroll
      for (int u = 0; u < R; ++u) v[u] = get(clampi(j0 - R + u, 1, N), STV);
#pragma unroll
      for (int u = 0; u < R; ++u) {
        const int j = j0 + u;                        // row j+1 comes in
        double a, b, c, d;
        bool sw;
        first_row(t1[u], ELEC ? t2[u % (ELEC ? R : 1)] : 0.0, t3[u], w[u], w[u + 1], w[u + 2], a, b, c, d);
        load_terms(j + 1 - R, u);
        if (EDGE && j >= N - 1) { a = aN; b = bN; c = 0.0; d = Tmax; }
        if (EDGE && j >= N) P[u] = Pivot{q.r0, 0.0, 0.0, q.rb};
        else if (!EDGE || j >= 1) P[u] = elim_step(q, a, b, c, d, sw);
        else P[u] = Pivot{1.0, 0.0, 0.0, 0.0};
      }
#pragma unroll
      for (int u = R - 1; u >= 0; --u) {
        const int i = j0 + u;
        if (EDGE && (i > N || i < 1)) continue;
        double x = back_step(P[u], x1, x2);
        if (BE) {
          if (tr_sing && e.singular) x = i == 1 ? Tmin : i == N ? Tmax : div_rcp(w[u], k1.dt, k1.K);
          sT[u][lane] = fmax_f(x, 100.0);
        } else {
          double d = bdf_rhs(w[u], x);
          if (tr_sing && e.singular) d = w[u];       // (already the right-hand side)
          put(i, STV, d);
        }
        x2 = x1;
        x1 = x;
      }
      if (BE) flush_out(j0);
    };
    load_state(mb);
    {
      const int j0 = mb * R + 1 - ph;
#pragma unroll
      for (int u = 0; u < R; ++u) {
        v[u] = get(clampi(j0 + u, 1, N), STV);
        load_terms(j0 + u + 1, u);
      }
    }
    for (int m = mb; m >= 0; --m) {
      const int j0 = m * R + 1 - ph;
      if (j0 >= 1 && j0 + R <= N - 1) block(std::false_type{}, m);
      else block(std::true_type{}, m);
    }
  }
  if (BE) return;

  // ---- pass 3: the BDF2 elimination; v holds the right-hand sides of the steps' rows
  Elim f{1.0, 0.0, Tmin, false};
  auto load_row = [&](int r, int u) {
    load_terms(r, u);
    v[u] = get(clampi(r, 1, N), STV);
  };
  auto bdf_row = [&](int u, double& a, double& b, double& c, double& d) {
    const double t2f = ELEC ? t2[u % (ELEC ? R : 1)] : 0.0;
    a = -t1[u] + t2f; b = (bdf.K + t3[u]) + t1[u]; c = -t3[u] - t2f; d = v[u];
  };
  {
#pragma unroll
    for (int u = 0; u < R; ++u) load_row(2 - ph + u, u);
    auto block = [&](auto edge_, int m) {
      constexpr bool EDGE = decltype(edge_)::value;
      const int j0 = m * R + 1 - ph;
      keep_state(m, f);
#pragma unroll
      for (int u = 0; u < R; ++u) {
        const int j = j0 + u;
        double a, b, c, d;
        bool sw;
        bdf_row(u, a, b, c, d);
        load_row(j + 1 + R, u);
        if (EDGE && (j < 1 || j > N - 1)) continue;
        if (EDGE && j == N - 1) { a = aN; b = bN; c = 0.0; d = Tmax; }
        elim_step(f, a, b, c, d, sw);
        record(1, j, sw);
      }
    };
    for (int m = 0; m <= mb; ++m) {
      const int j0 = m * R + 1 - ph;
      if (j0 >= 1 && j0 + R <= N - 1) block(std::false_type{}, m);
      else block(std::true_type{}, m);
    }
    if (f.r0 == 0.0) f.singular = true;
  }

  // ---- pass 4
  {
    double x1 = 0.0, x2 = 0.0;
    auto block = [&](auto edge_, int m) {
      constexpr bool EDGE = decltype(edge_)::value;
      const int j0 = m * R + 1 - ph;
      Elim q{ckn[0], ckn[1], ckn[2], false};
      Pivot P[R];
      load_state(m - 1);
#pragma unroll
      for (int u = 0; u < R; ++u) {
        const int j = j0 + u;
        double a, b, c, d;
        bool sw;
        bdf_row(u, a, b, c, d);
        load_row(j + 1 - R, u);
        if (EDGE && j >= N - 1) { a = aN; b = bN; c = 0.0; d = Tmax; }
        if (EDGE && j >= N) P[u] = Pivot{q.r0, 0.0, 0.0, q.rb};
        else if (!EDGE || j >= 1) P[u] = elim_step(q, a, b, c, d, sw);
        else P[u] = Pivot{1.0, 0.0, 0.0, 0.0};
      }
#pragma unroll
      for (int u = R - 1; u >= 0; --u) {
        if (EDGE && (j0 + u > N || j0 + u < 1)) continue;
        const double x = back_step(P[u], x1, x2);
        sT[u][lane] = fmax_f(x, 100.0);
        x2 = x1;
        x1 = x;
      }
      flush_out(j0);
    };
    load_state(mb);
    {
      const int j0 = mb * R + 1 - ph;
#pragma unroll
      for (int u = 0; u < R; ++u) load_row(j0 + u + 1, u);
    }
    for (int m = mb; m >= 0; --m) {
      const int j0 = m * R + 1 - ph;
      if (j0 >= 1 && j0 + R <= N - 1) block(std::false_type{}, m);
      else block(std::true_type{}, m);
    }
  }
  // a singular BDF2 factorisation likewise (slow, never on physical inputs): the right-hand
  // sides, which pass 4 left in place, are the solution
  if (__any(f.singular) && f.singular) {
    int a2, a3;
    column_of(g, col, a2, a3);
    double* To = s.Ts + (long)(isp - 1) * g.N + gix(g, 0, a2, a3);
    for (int r = 1; r <= N; ++r) {
      const double d = r == 1 ? Tmin : r == N ? Tmax : get(r, STV);
      To[r] = fmax_f(d, 100.0);
    }
  }
}

// Unit v of a launch: the electron groups first (their waves are the longest, so the last
// wave round is shorter), then the six ion units of each run of 8 groups; unit v runs on XCD
// v % 8, and every unit of column group cg on XCD cg % 8.
template <int R, bool BE, bool EXT>
__device__ __forceinline__ void diffusion_block(const DevGrid& g, const DevState& s, long v,
                                                double* scratch, const Coef& k1, const Coef& bdf,
                                                double Teinf, double (*sT)[LP], double (*sC)[LP],
                                                double (*sB)[LP], double (*sD)[LP]) {
  const long gps = diffusion_groups(g), ne = (gps + 7) / 8 * 8;
  if (v < ne) {
    if (v < gps)
      diffusion_unit<R, BE, true, EXT>(g, s, scratch, k1, bdf, Teinf, v, 0, 0, sT, sC, sB, sD);
    return;
  }
  const long b = v - ne, slot = b / 8, cg = slot / 6 * 8 + b % 8;
  const int half = (int)(slot % 6) / 3, pair = (int)(slot % 6) % 3;
  // (a half past the last column has none of its own)
  if (cg >= gps || (!group_interleaved(g, cg) && cg * 64 + half * 32 >= (long)g.lx2 * g.lx3)) return;
  diffusion_unit<R, BE, false, EXT>(g, s, scratch, k1, bdf, Teinf, cg, half, pair, sT, sC, sB, sD);
}

template <int R, bool BE, bool EXT = false>
__global__ __launch_bounds__(64, 2) void k_diffusion(DevGrid g, DevState s, double* scratch,
                                                     Coef k1, Coef bdf, double Teinf) {
  __shared__ double sT[R][LP], sC[R][LP], sB[R][LP], sD[R][LP];
  diffusion_block<R, BE, EXT>(g, s, blockIdx.x, scratch, k1, bdf, Teinf, sT, sC, sB, sD);
}

// ---------------------------------------------------------------- small grids
// A grid with few columns leaves most of the GPU idle under the kernel above, whose waves then
// take 1.5 us a row: four passes of a serial chain, the cells' conductivity and factors formed
// by the same wave.  Here a workgroup of 4 to 16 waves owns W columns of one species and keeps
// everything in LDS (nine doubles a row and column): all form the matrices' rows, then one
// wave eliminates both systems at once (lanes 0-31 the first solve, 32-63 the BDF2
// matrix, one instruction stream) and keeps the pivot rows in the place of the rows it has
// used, so nothing is formed twice and each pass is one chain of a few dozen instructions.
// Same operations and order as above.  128x64x1 53.8 us, 96x24x20 46.5, 64x24x16 35 (the wave
// kernel 188, 148 and 103; with the rows formed by the solving wave, and zero tests in it, this
// one 65, 57 and 41).
//
// LDS rows of Q_SLOTS x W doubles and one more (which spreads the rows over the banks for the
// threads of the first phase, which run along x1): row r at r RS.  Rows 0, N+1 and N+2 exist
// and hold nothing: the walks read a row or two ahead.
enum : int { Q_T1 = 0, Q_T3 = 1, Q_T2 = 2, Q_Y = 3,      // terms, then the first matrix's row
                                                         // and rhs, then U0 U1 U2 and the rhs
             Q_T = 4,                                    // temperature, then the BDF2 rhs, x
             Q_V = 5, Q_SLOTS = 9 };                     // C B D, then the BDF2 row, then V0 V1
                                                         // V2 and multiplier
__host__ __device__ inline size_t small_lds_bytes(int N, int W) {
  return (size_t)(N + 3) * (Q_SLOTS * W + 1) * sizeof(double) +
         (size_t)((N + 31) / 32) * W * sizeof(int);
}

// threads of a block: two of the wide blocks seldom share a CU, and their four or two waves a
// SIMD hide the latency of the cells' inputs (256 threads: 96x24x20 51 us, 64x24x16 38; these
// 46.5 and 35)
__host__ __device__ constexpr int small_threads(int W) { return W >= 8 ? W * 64 : 256; }

template <int W, bool BE, bool EXT>
__global__ __launch_bounds__(small_threads(W)) void k_diffusion_small(DevGrid g, DevState s, Coef k1, Coef bdf,
                                                         double Teinf) {
  extern __shared__ double lds[];
  const int N = g.lx1, tid = threadIdx.x;
  const int ncol = g.lx2 * g.lx3;
  const int c0 = blockIdx.x * W;                       // first column
  const int isp = LSP - (int)blockIdx.y;               // (electrons first: the longer blocks)
  const bool elec = isp == LSP;
  const long so = (long)(isp - 1) * g.N, ni = (long)g.lx1 * ncol;
  constexpr int RS = Q_SLOTS * W + 1;                  // doubles of a row
  int* swb = (int*)(lds + (N + 3) * RS);               // BDF2 interchange words [word][W]
  auto at = [&](int q, int r, int c) -> double& { return lds[r * RS + q * W + c]; };
  const double gm1kB = (gammas(isp) - 1.0) / kB;
  // temperature and the factors C, B, D of one cell, from HBM
  auto cell = [&](int r, int col, double& T, double& C, double& B, double& D) {
    const int i2 = col % g.lx2 + 1, i3 = col / g.lx2 + 1;
    const long cb = gix(g, r, i2, i3), kb = (long)g.lx1 * col + r - 1;
    const double h1 = g.h1[cb], h2 = g.h2[cb], h3 = g.h3[cb];
    if (elec) {
      CellIn<true> in;
      in.T = s.Ts[so + cb]; in.n = s.ns[so + cb];
      in.h1 = h1; in.h2 = h2; in.h3 = h3;
      in.n1 = s.nn[kb]; in.n2 = s.nn[ni + kb]; in.n3 = s.nn[2 * ni + kb];
      in.J = s.J1[cb];
      in.kap = EXT && s.kappa ? s.kappa[col] : 1.0;
      cell_coeffs<true, EXT>(in, isp, gm1kB, C, B, D);
      T = in.T;
    } else {
      CellIn<false> in;
      in.T = s.Ts[so + cb]; in.n = s.ns[so + cb];
      in.h1 = h1; in.h2 = h2; in.h3 = h3;
      cell_coeffs<false, false>(in, isp, gm1kB, C, B, D);
      T = in.T;
    }
  };
  const double* dx1i = g.dx1i - 1;
  // the parabolic terms of row r from C(r), B(r), D(r-1..r+1)
  auto terms = [&](int r, double C, double B, double Dm, double D, double Dp, double& t1, double& t2,
                   double& t3) {
    const double dxi = dx1i[r], dxl = g.dx1[r], dxr = g.dx1[r + 1], yi = g.rdx1i[r];
    t1 = div_rcp(div_rcp(C * (0.5 * (Dm + D)), dxi, yi), dxl, g.rdx1[r]);
    t3 = div_rcp(div_rcp(C * (0.5 * (D + Dp)), dxi, yi), dxr, g.rdx1[r + 1]);
    t2 = elec ? div_rcp(B, dxr + dxl, g.rdx1s[r]) : 0.0;
  };
  // ---- terms: threads along x1 (columns past the last repeat it)
  for (int t = tid; t < N * W; t += small_threads(W)) {
    const int c = t / N, r = t - c * N + 1;
    double T, C, B, D;
    cell(r, min(c0 + c, ncol - 1), T, C, B, D);
    at(Q_T, r, c) = T;
    at(Q_V, r, c) = C; at(Q_V + 1, r, c) = B; at(Q_V + 2, r, c) = D;
  }
  __syncthreads();
  for (int t = tid; t < N * W; t += small_threads(W)) {
    const int c = t / N, r = t - c * N + 1;
    if (r == 1 || r == N) continue;
    double t1, t2, t3;
    terms(r, at(Q_V, r, c), at(Q_V + 1, r, c), at(Q_V + 2, r - 1, c), at(Q_V + 2, r, c),
          at(Q_V + 2, r + 1, c), t1, t2, t3);
    at(Q_T1, r, c) = t1; at(Q_T3, r, c) = t3; at(Q_T2, r, c) = t2;
  }
  __syncthreads();
  // first solve: TR takes half of each term; backward Euler the whole, as BDF2
  auto rhs1 = [&](double a, double tsum, double cc, double Tm, double Tc, double Tp) {
    if (BE) return div_rcp(Tc, k1.dt, k1.K);
    return ((div_rcp(Tc, k1.dt2, k1.K) - a * Tm) - tsum * Tc) - cc * Tp;
  };
  constexpr double half = BE ? 1.0 : 0.5;
  // ---- the matrices' rows, so that the solving wave has only their elimination to do
  for (int t = tid; t < N * W; t += small_threads(W)) {
    const int c = t / N, r = t - c * N + 1;
    if (r == 1 || r == N) continue;
    const double f1 = at(Q_T1, r, c), f2 = at(Q_T2, r, c), f3 = at(Q_T3, r, c);
    const double t1 = f1 * half, t2 = f2 * half, t3 = f3 * half;
    const double a = -t1 + t2, cc = -t3 - t2;
    at(Q_T1, r, c) = a; at(Q_T1 + 1, r, c) = (k1.K + t3) + t1; at(Q_T1 + 2, r, c) = cc;
    at(Q_Y, r, c) = rhs1(a, t3 + t1, cc, at(Q_T, r - 1, c), at(Q_T, r, c), at(Q_T, r + 1, c));
    if (!BE) {
      at(Q_V, r, c) = -f1 + f2; at(Q_V + 1, r, c) = (bdf.K + f3) + f1; at(Q_V + 2, r, c) = -f3 - f2;
      at(Q_V + 3, r, c) = 0.0;                         // (a right-hand side that nothing uses)
    }
  }
  __syncthreads();
  // ---- the solves: the first wave; lanes past W repeat the last column
  if (__builtin_amdgcn_readfirstlane(tid >> 6) == 0) {
    const int lane = tid & 63, c = min(lane & 31, W - 1);
    const bool second = !BE && lane >= 32;             // the BDF2 factorisation
    const int col = min(c0 + c, ncol - 1);
    double Tmin, Tmax, aN = 0.0, bN = 1.0;
    {
      const long kb = (long)g.lx1 * col;
      const double Tn1 = s.Tn[kb], TnN = s.Tn[kb + N - 1];
      if (g.gridflag == 0) { Tmin = Tn1; Tmax = TnN; }
      else if (g.gridflag == 1) { Tmax = TnN; Tmin = Teinf; }
      else { Tmin = Tn1; Tmax = Teinf; }
    }
    if (EXT && elec && s.qtop) {                       // (see diffusion_unit)
      const int i2 = col % g.lx2 + 1, i3 = col / g.lx2 + 1;
      CellIn<true> top;
      cell_load<true, true>(g, s, so, gix(g, 0, i2, i3), (long)g.lx1 * col, ni, N, top,
                            hcol_index(g, col, N), col);
      aN = -1.0 / g.dx1[N];
      bN = 1.0 / g.dx1[N];
      Tmax = (s.qtop[col] * top.h1) / cell_lambda<true, true>(top, isp);
    }
    const int nw = (N + 31) / 32;
    int* prec = (EXT && elec && s.pivrec) ? s.pivrec + ((long)col * 2 + (second ? 1 : 0)) * nw : nullptr;
    const int out = second ? Q_V : Q_T1;
    Elim e{1.0, 0.0, Tmin, false};
    const double* in = &at(out, 2, c);                 // the next row
    double na = in[0], nb = in[W], nc = in[2 * W], nd = in[3 * W];
    double* po = &at(out, 1, c);                       // pivot rows
    // step j brings row j+1 in; the bits of its interchanges, 32 steps a word
    auto step = [&](bool last) -> bool {
      double a = na, b = nb, cc = nc, d = nd, l;
      in += RS;
      na = in[0]; nb = in[W]; nc = in[2 * W]; nd = in[3 * W];
      if (last) { a = aN; b = bN; cc = 0.0; d = Tmax; }
      bool sw;
      const Pivot p = elim_step(e, a, b, cc, d, sw, &l);
      po[0] = p.u0; po[W] = p.u1; po[2 * W] = p.u2;
      po[3 * W] = second ? l : p.y;
      po += RS;
      return sw;
    };
    auto word = [&](int j, int bits) {
      if (second) swb[(j >> 5) * W + c] = bits;
      if (EXT && prec) prec[j >> 5] = bits;
    };
    for (int j0 = 0; j0 < N - 1; j0 += 32) {
      int bits = 0;
      const int je = min(j0 + 32, N - 1);              // row N's step comes after the loops
#pragma unroll 4
      for (int j = max(j0, 1); j < je; ++j) bits |= (step(false) ? 1 : 0) << (j & 31);
      if (je == N - 1 && (je & 31)) bits |= (step(true) ? 1 : 0) << (je & 31);
      word(j0, bits);
    }
    if (((N - 1) & 31) == 0) word(N - 1, step(true) ? 1 : 0);
    if (e.r0 == 0.0) e.singular = true;
    at(out, N, c) = e.r0; at(out + 1, N, c) = 0.0; at(out + 2, N, c) = 0.0;
    if (!second) at(out + 3, N, c) = e.rb;
    const int sing = e.singular ? 1 : 0;
    const bool s1 = __shfl(sing, lane & 31) != 0, s2 = __shfl(sing, (lane & 31) + 32) != 0;
    __builtin_amdgcn_wave_barrier();
    // dgbsv leaves the right-hand side where a factorisation is singular (never on physical
    // inputs): formed again from HBM, in the place of the eliminated one
    if (__any(s1) && s1) {
      at(Q_Y, 1, c) = Tmin;
      at(Q_Y, N, c) = Tmax;
      double T0, T1, T2, C0, C1, C2, B0, B1, B2, D0, D1, D2;
      cell(1, col, T0, C0, B0, D0);
      cell(2, col, T1, C1, B1, D1);
      for (int r = 2; r < N; ++r) {
        cell(r + 1, col, T2, C2, B2, D2);
        double t1, t2, t3;
        terms(r, C1, B1, D0, D1, D2, t1, t2, t3);
        t1 *= half; t2 *= half; t3 *= half;
        at(Q_Y, r, c) = rhs1(-t1 + t2, t3 + t1, -t3 - t2, T0, T1, T2);
        T0 = T1; D0 = D1; T1 = T2; C1 = C2; B1 = B2; D1 = D2;
      }
    }
    __builtin_amdgcn_wave_barrier();
    // back substitution through the pivot rows at slots q0.., rhs in Q_Y
    auto back = [&](int q0, bool singular, auto put) {
      double x1 = 0.0, x2 = 0.0;
      const double* pq = &at(0, N, c);
      Pivot n{pq[q0 * W], pq[(q0 + 1) * W], pq[(q0 + 2) * W], pq[Q_Y * W]};
      double* pT = &at(Q_T, N, c);
#pragma unroll 4
      for (int i = N; i >= 1; --i) {
        const Pivot p = n;
        pq -= RS;
        n = Pivot{pq[q0 * W], pq[(q0 + 1) * W], pq[(q0 + 2) * W], pq[Q_Y * W]};
        const double v = back_step(p, x1, x2), x = singular ? p.y : v;
        *pT = put(*pT, x);
        pT -= RS;
        x2 = x1;
        x1 = x;
      }
    };
    auto floor100 = [&](double, double x) { return fmax_f(x, 100.0); };
    if (BE) {
      back(Q_T1, s1, floor100);
    } else {
      back(Q_T1, s1, [&](double T, double x) {
        return -div_rcp(bdf.c13 * T, bdf.dt3, bdf.K) + div_rcp(bdf.c43 * x, bdf.dt3, bdf.K);
      });
      __builtin_amdgcn_wave_barrier();
      // BDF2 forward solve through the kept interchanges and multipliers
      const double* pi = &at(0, 1, c);                 // row j: multiplier; row j+1: rhs
      double* py = &at(Q_Y, s2 ? 2 : 1, c);
      double rb = Tmin, nd = pi[Q_T * W + RS], nl = pi[(Q_V + 3) * W];
      if (s2) at(Q_Y, 1, c) = Tmin;
      auto fwd = [&](int w, int j, bool last) {
        const double d = last ? Tmax : nd, l = nl;
        pi += RS;
        nd = pi[Q_T * W + RS];
        nl = pi[(Q_V + 3) * W];
        const bool sw = (w >> (j & 31)) & 1;
        const double pd = sw ? d : rb, od = sw ? rb : d;
        const double nod = od + l * (-pd);
        rb = pd != 0.0 ? nod : od;
        *py = s2 ? d : pd;
        py += RS;
      };
      for (int j0 = 0; j0 < N - 1; j0 += 32) {
        const int w = swb[(j0 >> 5) * W + c], je = min(j0 + 32, N - 1);
#pragma unroll 4
        for (int j = max(j0, 1); j < je; ++j) fwd(w, j, false);
        if (je == N - 1 && (je & 31)) fwd(w, je, true);
      }
      if (((N - 1) & 31) == 0) fwd(swb[((N - 1) >> 5) * W + c], N - 1, true);
      if (!s2) at(Q_Y, N, c) = rb;
      __builtin_amdgcn_wave_barrier();
      back(Q_V, s2, floor100);
    }
  }
  __syncthreads();
  for (int t = tid; t < N * W; t += small_threads(W)) {
    const int c = t / N, r = t - c * N + 1, col = c0 + c;
    if (col < ncol) s.Ts[so + gix(g, r, col % g.lx2 + 1, col / g.lx2 + 1)] = at(Q_T, r, c);
  }
}

}  // namespace

void launch_floor_ghosts(const DevGrid& g, double* Ts, hipStream_t st);

namespace {
__host__ __device__ inline Coef tr_coef(double dt) {
  Coef c{};
  c.dt2 = dt / 2.0; c.K = 1.0 / c.dt2; c.dt = dt;
  return c;
}
__host__ __device__ inline Coef bdf_coef(double dt) {
  Coef c{};
  c.dt3 = dt / 3.0; c.K = 1.0 / c.dt3; c.dt = dt;
  c.c13 = 1.0 / 3.0; c.c43 = 4.0 / 3.0;
  return c;
}

__device__ __forceinline__ double uniform_double(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readfirstlane((int)b), hi = __builtin_amdgcn_readfirstlane((int)(b >> 32));
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
__device__ __forceinline__ BatchMember load_uniform(const BatchMember* p) {
  BatchMember b;
  static_assert(sizeof(BatchMember) % 4 == 0, "copied by words");
  const auto* w = (const __attribute__((address_space(4))) int*)p;
#pragma unroll
  for (unsigned k = 0; k < sizeof(BatchMember) / 4; ++k) ((int*)&b)[k] = w[k];
  return b;
}

// The TRBDF2 solve of every member of a batched step: a persistent grid of one-wave blocks
// taking the members' units in turn, numbered as each member's own launch numbers them
// (every member's count is a multiple of 8, so a group keeps its XCD).  The coefficients are
// formed from each member's dt as launch_energy_diffusion forms them.
template <int R>
__global__ __launch_bounds__(64, 2) void kb_diffusion(const BatchMember* M, const long* pre, int n,
                                                      long total) {
  __shared__ double sT[R][LP], sC[R][LP], sB[R][LP], sD[R][LP];
  const long* p = pre + (long)BK_DIFF * (n + 1);
  for (long t = blockIdx.x; t < total; t += gridDim.x) {
    // (the member's table entry by scalar loads: as vector loads its 60 uniform values took
    // vector registers, and the kernel spilled)
    const int m = __builtin_amdgcn_readfirstlane(batch_member(p, n, t));
    const BatchMember b = load_uniform(M + m);
    Coef tr = tr_coef(b.dt), bdf = bdf_coef(b.dt);
    tr.dt2 = uniform_double(tr.dt2); tr.K = uniform_double(tr.K);
    bdf.dt3 = uniform_double(bdf.dt3); bdf.K = uniform_double(bdf.K);
    diffusion_block<R, false, false>(b.g, b.s, t - p[m], b.scratch, tr, bdf, b.Teinf, sT, sC, sB, sD);
  }
}
}  // namespace


// the metric factors in column-group order (DevGrid::hcol), one thread per entry; lanes
// past the last column repeat it
__global__ void k_fill_hcol(DevGrid g, double* hcol) {
  const long ncol = (long)g.lx2 * g.lx3;
  for (long t = (long)blockIdx.x * blockDim.x + threadIdx.x; t < g.hstride;
       t += (long)gridDim.x * blockDim.x) {
    const int lane = (int)(t & 63);
    const long q = t >> 6;
    const int r = (int)(q % g.lx1) + 1;
    const long gcol = group_column(g, q / g.lx1, lane);
    const long cb = gix(g, 0, (int)(gcol % g.lx2) + 1, (int)(gcol / g.lx2) + 1);
    hcol[t] = g.h1[cb + r];
    hcol[g.hstride + t] = g.h2[cb + r];
    hcol[2 * g.hstride + t] = g.h3[cb + r];
  }
}
// the correctly rounded reciprocals of one axis' divisors (DevGrid::rdx1, rdx1i, rdx1s)
__global__ void k_fill_rdx(const double* dx, const double* dxi, int lx, double* r) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x, L = lx + 3;
  if (i >= L) return;
  r[i] = 1.0 / dx[i];
  r[L + i] = 1.0 / dxi[clampi(i - 1, 0, lx - 1)];
  r[2 * L + i] = 1.0 / (dx[min(i + 1, lx + 2)] + dx[i]);
}

long pivot_record_ints(const DevGrid& g) { return (long)g.lx2 * g.lx3 * 2 * ((g.lx1 + 31) / 32); }

long diffusion_hcol_doubles(const DevGrid& g) {
  return 3 * (((long)g.lx2 * g.lx3 + 63) / 64) * g.lx1 * 64;
}
long rdx_doubles(const DevGrid& g) { return 3L * (g.lx1 + g.lx2 + g.lx3 + 9); }

void launch_fill_hcol(const DevGrid& g, double* hcol, hipStream_t st) {
  hipLaunchKernelGGL(k_fill_hcol, dim3(4096), dim3(256), 0, st, g, hcol);
}

void launch_fill_rdx(DevGrid& g, double* rdx, hipStream_t st) {
  const double* dx[] = {g.dx1, g.dx2, g.dx3};
  const double* dxi[] = {g.dx1i, g.dx2i, g.dx3i};
  const double** out[] = {&g.rdx1, &g.rdx1i, &g.rdx1s, &g.rdx2, &g.rdx2i, &g.rdx2s, &g.rdx3, &g.rdx3i,
                          &g.rdx3s};
  const int lx[] = {g.lx1, g.lx2, g.lx3};
  for (int a = 0; a < 3; ++a) {
    const int L = lx[a] + 3;
    hipLaunchKernelGGL(k_fill_rdx, dim3((L + 255) / 256), dim3(256), 0, st, dx[a], dxi[a], lx[a], rdx);
    for (int k = 0; k < 3; ++k) *out[3 * a + k] = rdx + k * L;
    rdx += 3 * L;
  }
}

// the kept rows and elimination states of every unit
size_t diffusion_scratch_bytes(const DevGrid& g) {
  const size_t gps = (size_t)diffusion_groups(g);
  return gps * (size_t)(unit_doubles(g, true) + 6 * unit_doubles(g, false)) * sizeof(double);
}

// the size a grid is held to by the allocation-free entry point, whose limit is part of its
// interface: nine doubles, an interchange bit and a flag per row and system of 64-column groups
size_t diffusion_noalloc_bytes(const DevGrid& g) {
  const size_t sys = (size_t)diffusion_groups(g) * LSP * 64;
  return sys * ((size_t)g.lx1 * 9 * sizeof(double) + (size_t)((g.lx1 + 31) / 32 + 1) * sizeof(int));
}

namespace {
// Columns per block of the small-grid kernel, 0 where the wave kernel is faster: the fewest
// that leave at most one block per CU (the solving waves of two would share a SIMD), else the
// most that fit the LDS, if that makes at most three blocks per CU.  A block costs its CU 0.45
// us a row or more, at once or in turn, the wave kernel 1.3-1.8 us a row for all at these sizes
// (us, wave kernel and this: 2.5 blocks 98x40x36 145 and 135; 2.73 16x40x40 43 and 31, 64x40x40
// 102 and 92, 128x40x40 182 and 172; 3.9 64x48x48 107 and 121; 6.2 9x60x60 34 and 48, 33x60x61
// 68 and 120; 22 9x115x113 47 and 147).
int small_columns(const DevGrid& g) {
  constexpr size_t LDS = 160 * 1024;
  constexpr long CUS = 256;
  const long ncol = (long)g.lx2 * g.lx3;
  int best = 0;
  for (int W = 2; W <= 16; W *= 2) {
    const size_t b = small_lds_bytes(g.lx1, W);
    if (b > LDS) break;
    const long blocks = (ncol + W - 1) / W * LSP;
    if (blocks <= CUS) return W;
    best = blocks <= 3 * CUS ? W : 0;
  }
  return best;
}

template <int W>
void small_launch(const DevGrid& g, const DevState& s, int diffsolvetype, double Teinf,
                  const Coef& tr, const Coef& bdf, const Coef& be, hipStream_t st) {
  const dim3 grd((unsigned)(((long)g.lx2 * g.lx3 + W - 1) / W), LSP), blk(small_threads(W));
  const size_t b = small_lds_bytes(g.lx1, W);
  if (diffsolvetype == 1)
    hipLaunchKernelGGL((k_diffusion_small<W, true, false>), grd, blk, b, st, g, s, be, bdf, Teinf);
  else if (s.kappa || s.qtop)
    hipLaunchKernelGGL((k_diffusion_small<W, false, true>), grd, blk, b, st, g, s, tr, bdf, Teinf);
  else
    hipLaunchKernelGGL((k_diffusion_small<W, false, false>), grd, blk, b, st, g, s, tr, bdf, Teinf);
}

template <int R>
void diffusion_launch(const DevGrid& g, const DevState& s, int diffsolvetype, double Teinf,
                      double* scratch, const Coef& tr, const Coef& bdf, const Coef& be,
                      hipStream_t st) {
  switch (R == 4 ? 0 : small_columns(g)) {             // (the 4-row variant: waves always)
    case 16: return small_launch<16>(g, s, diffsolvetype, Teinf, tr, bdf, be, st);
    case 8: return small_launch<8>(g, s, diffsolvetype, Teinf, tr, bdf, be, st);
    case 4: return small_launch<4>(g, s, diffsolvetype, Teinf, tr, bdf, be, st);
    case 2: return small_launch<2>(g, s, diffsolvetype, Teinf, tr, bdf, be, st);
  }
  const dim3 grd((unsigned)((diffusion_groups(g) + 7) / 8 * 8 * LSP)), blk(64);
  if (diffsolvetype == 1)
    hipLaunchKernelGGL((k_diffusion<R, true>), grd, blk, 0, st, g, s, scratch, be, bdf, Teinf);
  else if (s.kappa || s.qtop)                         // fitting extension (TRBDF2 only)
    hipLaunchKernelGGL((k_diffusion<R, false, true>), grd, blk, 0, st, g, s, scratch, tr, bdf, Teinf);
  else
    hipLaunchKernelGGL((k_diffusion<R, false>), grd, blk, 0, st, g, s, scratch, tr, bdf, Teinf);
}
}  // namespace

void launch_batch_diffusion(const BatchTable& t, int diff_chunk, hipStream_t st) {
  const long total = t.total[BK_DIFF];
  const unsigned b = (unsigned)(total < t.blocks_diff ? total : t.blocks_diff);
  if (diff_chunk == 4)
    hipLaunchKernelGGL(kb_diffusion<4>, dim3(b ? b : 1), dim3(64), 0, st, t.m, t.pre, t.n, total);
  else
    hipLaunchKernelGGL(kb_diffusion<DIFF_CHUNK>, dim3(b ? b : 1), dim3(64), 0, st, t.m, t.pre, t.n,
                       total);
  // (no ghost floor: the batched step's surface conversions floored the ghost temperatures
  // at 100 K, and the solve writes interior rows only)
}

void launch_energy_diffusion(const DevGrid& g, const DevState& s, double dt, int diffsolvetype,
                             double Teinf, double* scratch, hipStream_t st, const Tuning& tune,
                             bool floor_ghosts) {
  Coef be{};
  be.dt = dt; be.K = 1.0 / dt;
  timing_begin("trbdf2", st);
  if (tune.diff_chunk == 4)
    diffusion_launch<4>(g, s, diffsolvetype, Teinf, scratch, tr_coef(dt), bdf_coef(dt), be, st);
  else
    diffusion_launch<DIFF_CHUNK>(g, s, diffsolvetype, Teinf, scratch, tr_coef(dt), bdf_coef(dt), be, st);
  timing_end("trbdf2", st);
  if (!floor_ghosts) return;
  timing_begin("floor_ghosts", st);
  launch_floor_ghosts(g, s.Ts, st);
  timing_end("floor_ghosts", st);
}

}  // namespace gemhip
