// bdf_group.h -- the Gear-BDF integrator of one cell on a group of lanes.
//
// A cell is integrated by G = 8 or 16 neighbouring lanes of a wave (G >= the
// SA reacting species), so a wave holds 64/G cells.  Lane `sub` of a group
// holds species sub of every vector of DDRIV3's state (Nordsieck columns,
// weights, SAVE1, SAVE2, FAC) and row `sub` of the factored iteration matrix;
// the scalars (t, h, order, counters) are held alike in all lanes of the
// group, which therefore take every branch together.  Values pass between the
// lanes of a group by DPP and through the group's slice of LDS, which also
// holds the cell's rate constants.
//
// Why a group and not a lane per cell: one cell per lane needs ~250 doubles of
// state in a lane (512 registers, one wave per SIMD, and scratch for the
// larger mechanisms), so the FP64 dependency chains ran with nothing to hide
// them, and a wave's 64 cells each waited for the stages of the others.  In a
// group the vector work of a stage is one instruction instead of SA and a
// lane's state fits 168 registers (three waves per SIMD, no scratch).  What
// bounds a grid that fills the chip is the VALU (busy 79 % of the time on an
// igniting mixture: the scalar work of a step, its divisions, powers and
// ordered sums, is done in all G lanes alike); a small grid is bound by the
// way of one cell through its steps.  Against one cell per lane (bdf_lane.h),
// kernel time in stiffness order: 65,536 KEROMNES flame cells 2.03 -> 1.45 ms,
// 262,144 cells with hot kernels 2.71 -> 1.15, 65,536 igniting ones 3.57 ->
// 1.66, 65,536 KONNOV flame cells (13 species) 83 -> 10.9; one cell per lane
// stays ahead where cells that cost alike fill the chip (1M flame cells: 11.9
// ms, 14.8 here).
//
// Also measured: two species to a lane (4 lanes per cell, 233 registers, two
// waves per SIMD): 26 % fewer VALU instructions, but latency-bound; 8 % faster
// than this on 2.1M cells of hot kernels, equal or slower (up to 40 %) elsewhere.
//
// Every decision and every rounding follows the reference operation by
// operation (this TU is built with -ffp-contract=off): sums over species or
// reactions run in the reference's order, whichever lane forms the terms.
//
// Reference: computing_module/src/current_build/chemical_kinetics_solver.f90
// (RHS :495-540) and SLATEC SDRIVE in computing_module/src/third_party/slatec/
// (ddriv3.f90, ddstp.f90, ddntl.f90, ddpst.f90, ddcor.f90, ddpsc.f90,
// ddscl.f90, ddntp.f90, dgefa.f90, dgesl.f90, dnrm2.f90).
#pragma once
#include "chem_device.h"

namespace nrg {

constexpr int G = SA <= 8 ? 8 : 16;         // lanes per cell
constexpr int CPW = WAVE / G;               // cells per wave
static_assert(SA <= 16, "a cell's reacting species must fit a group of 16 lanes");

typedef __attribute__((address_space(3))) double lds_double;

constexpr int imax(int a, int b) { return a > b ? a : b; }

// ---------------------------------------------------------------------------
// A cell's slice of LDS, in doubles:
//   [0, 2 REC_PAIRS)   the cell record (chem_device.h)
//   CZERO, CZERO+1     0.0 (an absent term)
//   CONE               1.0 (the factor of an absent operand)
//   CZ .. CZ+SA        y of the right-hand side being formed, by active slot
//   CX ..              exchange space: rates of the reactions (fwd, rev, fwd),
//                      rows of the iteration matrix, norm terms
// ---------------------------------------------------------------------------
constexpr int CZERO = 2 * REC_PAIRS;
constexpr int CONE = CZERO + 2;
constexpr int CZ = CONE + 1;
constexpr int CX = (CZ + SA + 1) & ~1;
constexpr int LDP = (SA + 1) | 1;           // row pitch of a matrix in the exchange space (a spare column at least)

constexpr int RROUNDS = (R + G - 1) / G;    // reactions per lane in rhs_group

// Most terms of a species in fun's sums (chemical_kinetics_solver.f90:528-535).
constexpr int max_terms()
{
  int best = 0;
  for (int a = 0; a < SA; ++a) {
    int n = 0;
    for (int r = 0; r < R; ++r)
      for (int c = 0; c < 3; ++c) {
        if (c < topo::nl[r] && topo::left[r][c] == kSp.full[a]) ++n;
        if (c < topo::nr[r] && topo::right[r][c] == kSp.full[a]) ++n;
      }
    best = imax(best, n);
  }
  return best;
}
constexpr int NTERM = max_terms();
constexpr int CX_SIZE = imax(imax(3 * R, SA * LDP), imax(6 * G, S));
// even (pairs stay 16-byte aligned) with an odd number of pairs: the slices of
// a wave's cells start in different banks
constexpr int CELL_EVEN = (CX + CX_SIZE + 1) & ~1;
constexpr int CELL_DOUBLES = (CELL_EVEN / 2) % 2 ? CELL_EVEN : CELL_EVEN + 2;
static_assert(CELL_DOUBLES < 8192, "16-bit byte offsets");

// ---------------------------------------------------------------------------
// Tables of the right-hand side for each lane of a group, as byte offsets into
// the cell's slice, two 16-bit entries to a word (one copy per wave in LDS: as
// loop-invariant values in registers they would be kept unpacked, two registers
// to a word):
//   words [0, OPW): for reaction q G + sub of round q, the operands of the
//     forward and of the reverse product in the order of their terms (fun,
//     :520-527), three each, CONE where a term is absent;
//   words [OPW, ..): for species sub, its terms in the order fun adds them:
//     where (fwd, rev) stands if it is consumed, (rev, fwd) if it is produced,
//     CZERO past the last one.  A reaction's rates are stored (fwd, rev, fwd).
// ---------------------------------------------------------------------------
constexpr int OPW = 3 * RROUNDS;
constexpr int TABW = (OPW + (NTERM + 1) / 2 + 3) & ~3;
constexpr int operand_offset(int sp, int r) { return sp == S ? 2 * REC_M + kMSlot.v[r] : CZ + act_of(sp); }
struct GroupTable {
  unsigned w[G][TABW];
};
constexpr GroupTable make_group_table()
{
  GroupTable t{};
  for (int sub = 0; sub < G; ++sub) {
    for (int q = 0; q < RROUNDS; ++q) {
      unsigned o[6] = {};
      for (int i = 0; i < 6; ++i) o[i] = CONE;
      const int r = q * G + sub;
      if (r < R)
        for (int c = 0; c < 3; ++c) {
          if (c < topo::nl[r]) o[c] = operand_offset(topo::left[r][c], r);
          if (c < topo::nr[r]) o[3 + c] = operand_offset(topo::right[r][c], r);
        }
      for (int i = 0; i < 3; ++i) t.w[sub][3 * q + i] = 8u * (o[2 * i] | (o[2 * i + 1] << 16));
    }
    unsigned l[2 * ((NTERM + 1) / 2)] = {};
    for (int i = 0; i < 2 * ((NTERM + 1) / 2); ++i) l[i] = CZERO;
    int n = 0;
    if (sub < SA)
      for (int r = 0; r < R; ++r) {
        for (int c = 0; c < 3; ++c)
          if (c < topo::nl[r] && topo::left[r][c] == kSp.full[sub]) l[n++] = CX + 3 * r;
        for (int c = 0; c < 3; ++c)
          if (c < topo::nr[r] && topo::right[r][c] == kSp.full[sub]) l[n++] = CX + 3 * r + 1;
      }
    for (int i = 0; i < (NTERM + 1) / 2; ++i) t.w[sub][OPW + i] = 8u * (l[2 * i] | (l[2 * i + 1] << 16));
  }
  return t;
}
// most terms of a side among the reactions of round q
constexpr int round_terms(int q, int side)
{
  int best = 0;
  for (int r = q * G; r < R && r < (q + 1) * G; ++r) best = imax(best, side ? topo::nr[r] : topo::nl[r]);
  return best;
}
static __device__ const GroupTable group_table = make_group_table();

// the species of term a (0..2 left, 3..5 right) of reaction r, -1 if it has none
constexpr int term_species(int r, int a)
{
  return a < 3 ? (a < topo::nl[r] ? topo::left[r][a] : -1) : (a - 3 < topo::nr[r] ? topo::right[r][a - 3] : -1);
}
// How many terms of reaction r the species with the most terms in it has
constexpr int most_terms(int r)
{
  int best = 0;
  for (int s = 0; s < S; ++s) {
    int n = 0;
    for (int a = 0; a < 6; ++a) n += term_species(r, a) == s ? 1 : 0;
    best = imax(best, n);
  }
  return best;
}
constexpr int most_terms_of_all()
{
  int best = 1;
  for (int r = 0; r < R; ++r) best = imax(best, most_terms(r));
  return best;
}
// Table of the exact Jacobian for each lane, in the same form: for reaction
// q G + i of round q, where the derivative of its rate by species sub stands in
// the exchange space (6 to a reaction of the round, by term), CZERO where it has
// none: word n JW2 + r / 2 for the n-th term of the species.
constexpr int JW2 = (R + 1) / 2;
constexpr int JTERMS = most_terms_of_all();
constexpr int JTABW = (JTERMS * JW2 + 3) & ~3;
struct JacTable {
  unsigned w[G][JTABW];
};
constexpr JacTable make_jac_table()
{
  JacTable t{};
  for (int sub = 0; sub < G; ++sub)
    for (int r = 0; r < R; ++r) {
      unsigned o[JTERMS] = {};
      for (int i = 0; i < JTERMS; ++i) o[i] = CZERO;
      int n = 0;
      for (int a = 0; a < 6; ++a)
        if (sub < SA && term_species(r, a) == kSp.full[sub < SA ? sub : 0]) o[n++] = (unsigned)(CX + 6 * (r % G) + a);
      for (int i = 0; i < JTERMS; ++i) t.w[sub][i * JW2 + r / 2] |= (8u * o[i]) << (16 * (r % 2));
    }
  return t;
}
static __device__ const JacTable jac_table = make_jac_table();

// Is species s inert, and the active slot of one that is not (s per lane).
NRG_DI bool inert_species(int s)
{
  bool in = false;
#pragma unroll
  for (int i = 0; i < NI; ++i) in = in || s == kSp.inert[i];
  return in;
}
NRG_DI int active_slot(int s)
{
  int a = s;
#pragma unroll
  for (int i = 0; i < NI; ++i) a -= s > kSp.inert[i] ? 1 : 0;
  return a;
}
// The species of an active slot (per lane).
NRG_DI int slot_species(int a)
{
  int s = a;
#pragma unroll
  for (int i = 0; i < NI; ++i) s += s >= kSp.inert[i] ? 1 : 0;
  return s;
}

NRG_DI lds_double *at_addr(unsigned addr) { return (lds_double *)(uintptr_t)addr; }
// base + 16-bit half HALF of w, in one instruction
template <int HALF>
NRG_DI unsigned add_half(unsigned w, unsigned base)
{
  unsigned d;
  if (HALF)
    asm("v_mad_u32_u16 %0, %1, 1, %2 op_sel:[1,0,0,0]" : "=v"(d) : "v"(w), "v"(base));
  else
    asm("v_mad_u32_u16 %0, %1, 1, %2" : "=v"(d) : "v"(w), "v"(base));
  return d;
}

// What the lanes of a group wrote before is read after.  A wave's LDS
// instructions execute in order, so only the compiler has to be held.
NRG_DI void wave_sync()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

NRG_DI bool wave_any(bool p) { return __any(p ? 1 : 0) != 0; }

// ---------------------------------------------------------------------------
// Lane moves.  row_newbcast takes a lane of each row of 16 (64 bits at once),
// in the quads that `banks` names; quad_perm moves within a quad.
// ---------------------------------------------------------------------------
template <int CTRL>
NRG_DI double dpp32(double v)
{
  const long long x = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)x, CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(x >> 32), CTRL, 0xf, 0xf, true);
  return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}
// v, but lane K of the row in the quads of BANKS (and lane K2 in those of BANKS2)
template <int K, int BANKS, int K2 = 0, int BANKS2 = 0>
NRG_DI double row_pass(double v)
{
  const long long x = __double_as_longlong(v);
  long long r = __builtin_amdgcn_update_dpp(x, x, 0x150 + (K & 15), 0xf, BANKS, false);
  if (BANKS2) r = __builtin_amdgcn_update_dpp(r, x, 0x150 + (K2 & 15), 0xf, BANKS2, false);
  return __longlong_as_double(r);
}

// ---------------------------------------------------------------------------
// FP64 division and square root without the scaling steps of the compiler's
// expansions, the same instructions otherwise: the same bits where those would
// not scale, and only there.  A numerator below 2^-969 has a remainder that FP64
// does not hold (the last bit goes), and a quotient above 2^1023 gives NaN
// instead of infinity.  Concentrations, densities, time steps and tables come
// from the caller with any exponent, so these are used only where the operands
// are known: in norm_usual and norms (the ratio of two components from 2^-900 up,
// and sums of squares that are 0 or above 2^-67), in solve (which see) and for what
// a norm is divided by.  Everything else divides.
// ---------------------------------------------------------------------------
// v_rcp_f64 and two Newton steps: the reciprocal a division starts from.
NRG_DI double recip(double d)
{
  double r = __builtin_amdgcn_rcp(d);
  double e = __builtin_fma(-d, r, 1.0);
  r = __builtin_fma(r, e, r);
  e = __builtin_fma(-d, r, 1.0);
  return __builtin_fma(r, e, r);
}
// n / d from r = recip(d): quotient, remainder, correction, and the fix-up of
// zeros, infinities and NaN.  The bits of n / d where n is 0, infinite, NaN or above
// 2^-969, and |d| and |n / d| within 2^+-1000.
NRG_DI double div_by(double n, double d, double r)
{
  const double q = n * r;
  const double e = __builtin_fma(-d, q, n);
  return __builtin_amdgcn_div_fixup(__builtin_fma(e, r, q), d, n);
}
// without the fix-up: n and d finite, d != 0 (else the result is not used)
NRG_DI double quot_raw(double n, double d)
{
  const double r = recip(d), q = n * r;
  return __builtin_fma(__builtin_fma(-d, q, n), r, q);
}
NRG_DI double root(double x)
{
  const double y = __builtin_amdgcn_rsq(x);
  double s = x * y, h = y * 0.5;
  const double r = __builtin_fma(-h, s, 0.5);
  s = __builtin_fma(s, r, s);
  h = __builtin_fma(h, r, h);
  double d = __builtin_fma(-s, s, x);
  s = __builtin_fma(d, h, s);
  d = __builtin_fma(-s, s, x);
  s = __builtin_fma(d, h, s);
  return x == 0.0 ? x : s;
}

constexpr double NRM_CUTLO = 8.232e-11;
constexpr double NRM_HITEST = 1.304e19 / (double)S;

enum Pc : int {
  PC_260 = 0,      // DDRIV3 label 260: weights and guards, then DDSTP entry
  PC_NTL_F,        // DDNTL after its f(y)
  PC_ATTEMPT,      // DDSTP label 100: predict, then f(y_pred)
  PC_PRED_F,       // after f(y_pred) (label 110)
  PC_JAC_DONE,     // after the Jacobian + LU (DDPST)
  PC_CORR,         // label 130: corrector (DDCOR)
  PC_CORR_F,       // after f(y) of a corrector iteration
  PC_ERRTEST,      // label 170: error test, accept, step/order selection
  PC_RETRACT,      // retract the prediction after a failed attempt
  PC_POW,          // the step-size candidates' powers
  PC_SCALE,        // apply a pending DDSCL rescale, then continue
  // a cell that asked for something resumes at the low four bits
  PC_WAIT_F = 16,      // ... once f(y) is in save2
  PC_WAIT_JAC = 32,    // ... once its iteration matrix is factored
  PC_DONE = 64,        // finished: the outcome in the low bits
  PC_IDLE = 128        // no cell
};
enum CellOutcome { OUT_OK = 0, OUT_MXSTEP = 2, OUT_STEP_ZERO = 3, OUT_REPEATED_FAIL = 4,
                   OUT_SINGULAR = 5, OUT_EPS = 6 };
// which step-size choice waits for its powers
enum PowUse : int { POW_FIRST = 0, POW_SELECT, POW_CONV, POW_ERR };
// work counters, counter i in lane i of the group
enum WorkLane : int { WORK_NFE = 0, WORK_NJE, WORK_NCORR, WORK_NATT };

NRG_DI double el_of(const BdfCoef &mc, int j, int nq) { return mc.el[nq - 1][j - 1]; }
// What the error test compares, nrm / (TQ(2, nq) sqrt(N)), and the same over sqrt(N):
// div_by gives a quotient's bits from 2^-969 up, and below that no decision hangs on
// them (EPS is at least UROUND here, and the powers end at UROUND).
NRG_DI double over_tq2(const BdfCoef &mc, double nrm, int nq) { return div_by(nrm, mc.den[1][nq - 1], mc.rden2[nq - 1]); }
// v / (TQ(k, nq) sqrt(N))
NRG_DI double over_tq(const BdfCoef &mc, double v, int k, int nq)
{
  return v / mc.den[k - 1][nq - 1];
}

// Net stoichiometric coefficient of species s in reaction r (right - left terms).
constexpr int nu_of(int r, int s)
{
  int n = 0;
  for (int c = 0; c < 3; ++c) {
    if (c < topo::nr[r] && topo::right[r][c] == s) ++n;
    if (c < topo::nl[r] && topo::left[r][c] == s) --n;
  }
  return n;
}

// The lane's view of its group.
struct Lane {
  int sub;                     // lane of the group
  unsigned base;               // LDS byte address of the cell's slice
  int gshift;                  // first lane of the group (bit position in a ballot)
  unsigned tab;                // LDS byte address of its table
  unsigned jtab;               // and of that of the exact Jacobian
};

// DDRIV3's state (WORK/IWORK): vectors by lane, scalars alike in the group,
// and the program counter of the reverse-communication form.
struct Cell {
  double yh[MAXORD + 1];         // yh[j] = YH(sub, j+1)
  double y, ywt, save1, save2, fac;
  double p[SA];                  // row `sub` of the factors: L left of the diagonal, U from it on
  double pd, prd;                // U(sub, sub) and its reciprocal (NaN where div_by cannot use it)
  int src;                       // component of a right-hand side that DGESL's interchanges bring here
  double t, h, rc, rmax, trend, told, d1, nrm;
  int nq, nwait, jtask, jstepl, nstep, work;
  int ntry, nfail, iter, pc;
  bool convrg, ier, evaljc, ntl_restart, swapped;
};

NRG_DI lds_double *slot(const Lane &ln, int i) { return at_addr(ln.base + 8u * (unsigned)i); }
// slot first + sub of the cell's slice
NRG_DI lds_double *own(const Lane &ln, int first) { return at_addr(ln.base + 8u * (unsigned)(first + ln.sub)); }
// does this lane hold a species?
NRG_DI bool holds(const Lane &ln) { return SA == G || ln.sub < SA; }
NRG_DI void count(const Lane &ln, Cell &c, int which, int n = 1) { c.work += ln.sub == which ? n : 0; }

typedef __attribute__((address_space(3))) unsigned lds_word;
NRG_DI void group_init(Lane &ln, lds_double *cells, lds_word *table, lds_word *jtable, int lane)
{
  ln.sub = lane % G;
  ln.gshift = lane & ~(G - 1);
  ln.base = (unsigned)(uintptr_t)(cells + (lane / G) * CELL_DOUBLES);
  ln.tab = (unsigned)(uintptr_t)(table + ln.sub * TABW);
  const unsigned *w = &group_table.w[0][0];
  for (int i = lane; i < G * TABW; i += WAVE) table[i] = w[i];
  ln.jtab = (unsigned)(uintptr_t)(jtable + ln.sub * JTABW);
  if (jtable)
    for (int i = lane; i < G * JTABW; i += WAVE) jtable[i] = (&jac_table.w[0][0])[i];
  if (ln.sub == 0) {
    *slot(ln, CONE) = 1.0;
    *slot(ln, CZERO) = 0.0;
    *slot(ln, CZERO + 1) = 0.0;
  }
  wave_sync();
}

// The group's bits of a ballot (bit sub).
NRG_DI unsigned bits(const Lane &ln, bool p)
{
  return (unsigned)(__ballot(p ? 1 : 0) >> ln.gshift) & ((1u << G) - 1u);
}

// Lane K's value of v in every lane of the group.
template <int K>
NRG_DI double bcast(double v)
{
  if constexpr (G == 16) return row_pass<K, 0xf>(v);
  else return row_pass<K, 0x3, 8 + K, 0xc>(v);       // a row holds two groups
}
// The largest v (>= 0) of the lanes below in the group, 0 where there is
// none: a scan within the quads, then the quads' maxima passed on.
NRG_DI double max_before(const Lane &ln, double v)
{
  double m = dpp32<0x111>(v);                        // row_shr:1
  if (G == 8) m = ln.sub >= 1 ? m : 0.0;             // a row of 16 holds two groups
  m = fmax(m, dpp32<0x90>(m));                       // quad_perm [0, 0, 1, 2]
  m = fmax(m, dpp32<0x40>(m));                       // quad_perm [0, 0, 0, 1]
  if constexpr (G == 8) {
    m = fmax(m, row_pass<3, 0x2, 11, 0x8>(m));
  } else {
    m = fmax(m, row_pass<3, 0xe>(m));
    m = fmax(m, row_pass<7, 0xc>(m));
    m = fmax(m, row_pass<11, 0x8>(m));
  }
  return m;
}

// -------------------------------------------------------------------------
// DNRM2 (slatec/dnrm2.f90:84-160) of vectors over the group's species, with
// the sums in the reference's order.  Elements without a species are 0, which
// no phase of Lawson's algorithm sees.  Its phases, for a vector without
// overflow risk: tiny components (|v| <= CUTLO) ahead of the first larger one
// are accumulated scaled by their running maximum, everything from the first
// larger one on unscaled.  HITEST keeps DDRIV3's N (all species).
// -------------------------------------------------------------------------
// All phases, one component after the other, over the N values in the group's
// exchange space (where one is unusual, or of all species).
template <int N>
NRG_DI double norm_serial(const Lane &ln)
{
  double sum = 0.0, xmax = 0.0;
  int st = 0;   // 0 = start (label 30), 1 = phase 1, 2 = phase 2, 3 = phase 4, 4 = phase 3
#pragma unroll 1
  for (int i = 0; i < N; ++i) {
    const double x = *slot(ln, CX + i), av = fabs(x);
    bool done = false;
    if (st == 0) st = av > NRM_CUTLO ? 4 : 1;
    if (st == 1) {
      if (x == 0.0) {
        done = true;
      } else if (av > NRM_CUTLO) {
        st = 4;
      } else {
        st = 2;
        xmax = av;
        const double r = x / xmax;
        sum = sum + r * r;
        done = true;
      }
    }
    if (!done && (st == 2 || st == 3)) {
      if (st == 2 && av > NRM_CUTLO) {
        sum = (sum * xmax) * xmax;
        st = 4;
      } else {
        const bool in = av <= xmax;
        const double r = (in ? x : xmax) / (in ? xmax : x);
        sum = in ? sum + r * r : 1.0 + sum * (r * r);
        xmax = in ? xmax : av;
        done = true;
      }
    }
    if (!done && st == 4) {
      if (av >= NRM_HITEST) {
        sum = (sum / x) / x;
        xmax = av;
        const double r = x / xmax;
        sum = sum + r * r;
        st = 3;
      } else {
        sum = sum + x * x;
      }
    }
  }
  wave_sync();
  return (st == 4) ? sqrt(sum) : xmax * sqrt(sum);
}

// A component that takes all phases: at or above HITEST, NaN, or so small that the
// quotients would have to be scaled, which zero is not.
NRG_DI bool unusual(const BdfConst &k, double v) { return !(fabs(v) < NRM_HITEST) || (fabs(v) < k.tiny && v != 0.0); }
// The same of NV vectors: every lane gets the norm of vector `mine`.
template <int NV>
NRG_DI double norms_serial(const Lane &ln, const double (&v)[NV], int mine)
{
  double out = 0.0;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    *own(ln, CX) = v[j];
    wave_sync();
    const double nrm = norm_serial<SA>(ln);
    out = j == mine ? nrm : out;
    wave_sync();
  }
  return out;
}

// Norms of NV vectors: every lane gets that of vector `mine`, so that the sums
// of two vectors run side by side.
//
// Most vectors have a scaled part (corrections of the major species are tiny:
// 56 to 100 % of the corrector's norms on the test fields), so there is one
// path.  Each lane knows the maximum of the tiny components before its own
// from a scan, so its quotient is formed beside the others'; only the sum runs
// in order, as sum = a + sum * b with (a, b) = (r^2, 1) below the running
// maximum, (1, r^2) at a new one and (0, 1) elsewhere.
template <int NV>
NRG_DI double norms(const Lane &ln, const BdfConst &k, const double (&v)[NV], int mine)
{
  bool over = false;
#pragma unroll
  for (int j = 0; j < NV; ++j) over = over || unusual(k, v[j]);
  wave_sync();
  if (__builtin_expect(wave_any(over), 0)) return norms_serial(ln, v, mine);
  double xmax = 0.0;
  bool none = false;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const unsigned big = bits(ln, fabs(v[j]) > NRM_CUTLO);
    const unsigned below = (big & (0u - big)) - 1u;  // the lanes ahead of the first large component
    const double av = fabs(v[j]);
    const bool ahead = ((below >> ln.sub) & 1u) != 0u;
    const bool tin = ahead && v[j] != 0.0;
    const double p = tin ? av : 0.0;
    const double before = max_before(ln, p);
    const double all = bcast<G - 1>(fmax(before, p));
    const bool grows = tin && av > before;
    // |r|: its square is what counts
    const double r = quot_raw(fmin(av, before), fmax(av, before));
    const double r2 = r * r;
    lds_double *x = at_addr(ln.base + 8u * (unsigned)(CX + 3 * G * j) + 16u * (unsigned)ln.sub);
    x[0] = tin ? (grows ? 1.0 : r2) : 0.0;
    x[1] = grows ? r2 : 1.0;
    *own(ln, CX + 3 * G * j + 2 * G) = ahead ? 0.0 : v[j] * v[j];
    xmax = j == mine ? all : xmax;
    none = j == mine ? big == 0u : none;
  }
  wave_sync();
  const lds_double *x = at_addr(ln.base + 8u * (unsigned)(CX + 3 * G * mine));
  double sum = 0.0;
#pragma unroll
  for (int i = 0; i < SA; ++i) sum = x[2 * i] + sum * x[2 * i + 1];
  sum = none ? sum : (sum * xmax) * xmax;
#pragma unroll
  for (int i = 0; i < SA; ++i) sum = sum + x[2 * G + i];
  wave_sync();
  const double s = root(sum);
  return none ? xmax * s : s;
}
// The norm of one vector: as above, but the sum passes from lane to lane (a
// broadcast per component) instead of every lane reading the terms from LDS,
// whose bandwidth the kernel runs short of first.  Component i turns the sum s
// into a + (s * b1) * b2: (a, b1, b2) as above ahead of the first large one,
// (v^2, xmax, xmax) there, (v^2, 1, 1) after it.
template <int... I>
NRG_DI double ordered_sum(double a, double b1, double b2, std::integer_sequence<int, I...>)
{
  double s = 0.0;
  ((s = bcast<I>(I == 0 ? a : a + (s * b1) * b2)), ...);
  return s;
}
NRG_DI double norm_usual(const Lane &ln, double v)
{
  const double av = fabs(v);
  const unsigned big = bits(ln, av > NRM_CUTLO);
  const unsigned first = big & (0u - big), below = first - 1u;
  const bool ahead = ((below >> ln.sub) & 1u) != 0u;
  const bool tin = ahead && v != 0.0;
  const bool here = ((first >> ln.sub) & 1u) != 0u;
  const double p = tin ? av : 0.0;
  const double before = max_before(ln, p);
  const double xmax = bcast<G - 1>(fmax(before, p));
  const bool grows = tin && av > before;
  const double r = quot_raw(fmin(av, before), fmax(av, before));
  const double r2 = r * r;
  const double a = tin ? (grows ? 1.0 : r2) : (ahead ? 0.0 : v * v);
  const double b1 = grows ? r2 : (here ? xmax : 1.0);
  const double b2 = here ? xmax : 1.0;
  const double s = root(ordered_sum(a, b1, b2, std::make_integer_sequence<int, SA>{}));
  return big == 0u ? xmax * s : s;
}
NRG_DI double norm(const Lane &ln, const BdfConst &k, double v)
{
  if (__builtin_expect(!wave_any(unusual(k, v)), 1)) return norm_usual(ln, v);
  const double one[1] = {v};
  return norms_serial<1>(ln, one, 0);
}

// -------------------------------------------------------------------------
// Mass-action right-hand side (fun, :507-536): lane sub forms the products of
// reactions sub, sub + G, ... and then adds its species' terms, two doubles of
// LDS each.  (Handing the rates around by lane broadcasts instead would take
// four times the instructions, and the VALU is what the kernel runs out of.)
// -------------------------------------------------------------------------
// words [W0, W0 + N) of a lane's table
template <int W0, int N>
NRG_DI void table_words(unsigned tab, unsigned (&w)[N])
{
  const lds_word *x = (const lds_word *)(uintptr_t)tab;
#pragma unroll
  for (int i = 0; i < N; ++i) w[i] = x[W0 + i];
}
template <int FIRST, int N>
NRG_DI double product(const Lane &ln, const unsigned (&w)[3], double k)
{
  double v = k;
  if (N > 0) v = v * *at_addr(add_half<FIRST & 1>(w[FIRST / 2], ln.base));
  if (N > 1) v = v * *at_addr(add_half<(FIRST + 1) & 1>(w[(FIRST + 1) / 2], ln.base));
  if (N > 2) v = v * *at_addr(add_half<(FIRST + 2) & 1>(w[(FIRST + 2) / 2], ln.base));
  return v;
}
template <int Q>
NRG_DI void reaction_round(const Lane &ln)
{
  const int r = Q * G + ln.sub;
  if ((Q + 1) * G <= R || r < R) {
    unsigned w[3];
    table_words<3 * Q>(ln.tab, w);
    const lds_double *k = at_addr(ln.base + 16u * (unsigned)r);
    const double fwd = product<0, round_terms(Q, 0)>(ln, w, k[0]);
    const double rev = product<3, round_terms(Q, 1)>(ln, w, k[1]);
    lds_double *x = at_addr(ln.base + 8u * CX + 24u * (unsigned)r);
    x[0] = fwd;
    x[1] = rev;
    x[2] = fwd;
  }
}
template <int... Q>
NRG_DI void reaction_rounds(const Lane &ln, std::integer_sequence<int, Q...>)
{
  (reaction_round<Q>(ln), ...);
}
NRG_DI double add_term(double zd, unsigned o)
{
  const lds_double *x = at_addr(o);
  return (zd - x[0]) + x[1];
}
NRG_DI double rhs_group(const Lane &ln, double y)
{
  unsigned w[(NTERM + 1) / 2];
  wave_sync();
  if (holds(ln)) *own(ln, CZ) = y;
  wave_sync();
  reaction_rounds(ln, std::make_integer_sequence<int, RROUNDS>{});
  table_words<OPW>(ln.tab, w);
  wave_sync();
  double zd = 0.0;
#pragma unroll
  for (int i = 0; i < NTERM; i += 2) {
    zd = add_term(zd, add_half<0>(w[i / 2], ln.base));
    if (i + 1 < NTERM) zd = add_term(zd, add_half<1>(w[i / 2], ln.base));
  }
  wave_sync();
  return zd;
}
// The whole right-hand side in one lane, at its own Z.
NRG_DI void rhs_lane(const Lane &ln, const double (&Z)[SA], double (&Zd)[SA])
{
#pragma unroll
  for (int s = 0; s < SA; ++s) Zd[s] = 0.0;
#pragma unroll
  for (int r = 0; r < R; ++r)
    rhs_reaction(r, *slot(ln, 2 * r), *slot(ln, 2 * r + 1),
                 kMSlot.v[r] >= 0 ? *slot(ln, 2 * REC_M + kMSlot.v[r]) : 0.0, Z, Zd);
}

// -------------------------------------------------------------------------
// DGEFA (slatec/dgefa.f90) with a row of the matrix to a lane.  Rows stay where
// they are until the end; pos is where LINPACK's interchanges have put the
// lane's.  Applied to whole rows they also permute L, so that DGESL can apply
// them to the right-hand side at once: every element still meets the same
// multipliers in the same order.
// -------------------------------------------------------------------------
// The largest of the group's values (NaN left out), and the smallest int.
NRG_DI double group_max(double v)
{
  v = fmax(v, dpp32<0xb1>(v));                       // quad_perm [1, 0, 3, 2]
  v = fmax(v, dpp32<0x4e>(v));                       // quad_perm [2, 3, 0, 1]
  if (G >= 8) v = fmax(v, dpp32<0x141>(v));          // row_half_mirror
  if (G >= 16) v = fmax(v, dpp32<0x140>(v));         // row_mirror
  return v;
}
NRG_DI int group_min(int v)
{
  v = min(v, __builtin_amdgcn_update_dpp(0, v, 0xb1, 0xf, 0xf, true));
  v = min(v, __builtin_amdgcn_update_dpp(0, v, 0x4e, 0xf, 0xf, true));
  if (G >= 8) v = min(v, __builtin_amdgcn_update_dpp(0, v, 0x141, 0xf, 0xf, true));
  if (G >= 16) v = min(v, __builtin_amdgcn_update_dpp(0, v, 0x140, 0xf, 0xf, true));
  return v;
}
template <int K>
NRG_DI void gefa_step(const Lane &ln, double (&a)[SA], int &pos, bool &singular)
{
  // pivot: the first of the largest in LINPACK's row order; row K itself if
  // that holds NaN, which nothing compares larger than
  const double big = group_max(pos >= K ? fabs(a[K]) : -1.0);
  const bool cand = pos >= K && (fabs(a[K]) == big || (pos == K && a[K] != a[K]));
  const int l = group_min(cand ? pos : SA);
  wave_sync();
  if (pos == l) {
#pragma unroll
    for (int i = K; i < SA; ++i) *slot(ln, CX + i) = a[i];
  }
  pos = pos == l ? K : (pos == K ? l : pos);
  wave_sync();
  const double piv = *slot(ln, CX + K);
  if (piv == 0.0) {
    singular = true;
  } else {
    // DSCAL and DAXPY, which returns at once for DA == 0 (slatec/daxpy.f90:68)
    const double t = -1.0 / piv;
    a[K] = pos > K ? t * a[K] : a[K];
#pragma unroll
    for (int i = K + 1; i < SA; ++i) {
      const double p = *slot(ln, CX + i);
      if (pos > K && p != 0.0) a[i] = a[i] + p * a[K];
    }
  }
}
template <int... K>
NRG_DI void gefa_steps(const Lane &ln, double (&a)[SA], int &pos, bool &singular,
                       std::integer_sequence<int, K...>)
{
  (gefa_step<K>(ln, a, pos, singular), ...);
}

// Factor the matrix whose column `sub` is a[]; c.ier on an exactly singular one.
NRG_DI void factor(const Lane &ln, Cell &c, const double (&a)[SA])
{
  // rows from columns
  const lds_double *x = at_addr(ln.base + 8u * CX + (unsigned)(8 * LDP) * (unsigned)(holds(ln) ? ln.sub : 0));
  double m[SA];
  wave_sync();
  if (holds(ln)) {
#pragma unroll
    for (int i = 0; i < SA; ++i) *own(ln, CX + i * LDP) = a[i];
  }
  wave_sync();
#pragma unroll
  for (int k = 0; k < SA; ++k) m[k] = x[k];
  int pos = holds(ln) ? ln.sub : -1;
  bool singular = false;
  gefa_steps(ln, m, pos, singular, std::make_integer_sequence<int, SA - 1>{});
  if (bits(ln, pos == SA - 1 && m[SA - 1] == 0.0) != 0u) singular = true;
  if (singular) c.ier = true;
  // each row, and which one it was, to the lane of its position
  wave_sync();
  if (pos >= 0) {
    lds_double *to = at_addr(ln.base + 8u * CX + (unsigned)(8 * LDP) * (unsigned)pos);
#pragma unroll
    for (int k = 0; k < SA; ++k) to[k] = m[k];
    to[SA] = __longlong_as_double((long long)ln.sub);
  }
  wave_sync();
#pragma unroll
  for (int k = 0; k < SA; ++k) c.p[k] = x[k];
  c.pd = x[holds(ln) ? ln.sub : 0];
  c.prd = fabs(c.pd) >= 0x1p-20 && fabs(c.pd) <= 0x1p40 ? recip(c.pd) : __builtin_nan("");
  c.src = (int)__double_as_longlong(x[SA]);
  wave_sync();
  c.swapped = bits(ln, holds(ln) && c.src != ln.sub) != 0u;
}

// DGESL (slatec/dgesl.f90): the lane's component of the solution.
template <int K>
NRG_DI void solve_fwd(const Lane &ln, const Cell &c, double &b)
{
  const double t = bcast<K>(b);
  if (ln.sub > K && t != 0.0) b = b + t * c.p[K];
}
// A component's sum is complete once the ones after it are through; the
// quotient by its diagonal is formed wherever it is needed.
template <bool FAST>
NRG_DI double over_diagonal(const Cell &c, double b) { return FAST ? div_by(b, c.pd, c.prd) : b / c.pd; }
template <int K, bool FAST>
NRG_DI void solve_back(const Lane &ln, const Cell &c, double &b)
{
  const double t = -bcast<K>(over_diagonal<FAST>(c, b));
  if (ln.sub < K && t != 0.0) b = b + t * c.p[K];
}
template <bool FAST, int... K>
NRG_DI void solve_steps(const Lane &ln, const Cell &c, double &b, std::integer_sequence<int, K...>)
{
  (solve_fwd<K>(ln, c, b), ...);
  (solve_back<SA - 1 - K, FAST>(ln, c, b), ...);
}
// The component of b that DGESL's interchanges bring to this lane.
NRG_DI double interchanged(const Lane &ln, const Cell &c, double b)
{
  if (wave_any(c.swapped)) {
    wave_sync();
    *own(ln, CX) = b;
    wave_sync();
    b = *slot(ln, CX + c.src);
    wave_sync();
  }
  return b;
}
// FAST: the quotients are div_by's (4 instructions of a serial chain instead of
// 11).  Where one of them is not what a division gives, its lane's component is
// unusual once it is weighted: NaN (a diagonal out of range, an overflow), or so
// small (a numerator under 2^-969 by a diagonal from 2^-20 and a weight from 2^-40
// up is under 2^-900).  cor then solves with divisions.
template <bool FAST>
NRG_DI double solve(const Lane &ln, const Cell &c, double b)
{
  solve_steps<FAST>(ln, c, b, std::make_integer_sequence<int, SA - 1>{});
  // a lane without a species keeps zeros
  return holds(ln) ? over_diagonal<FAST>(c, b) : 0.0;
}

// DDPSC (slatec/ddpsc.f90:26-38) for a compile-time order.
template <int NQ, bool ADD>
NRG_DI void psc_n(double (&yh)[MAXORD + 1])
{
#pragma unroll
  for (int j1 = 1; j1 <= NQ; ++j1)
#pragma unroll
    for (int j2 = j1; j2 <= NQ; ++j2) {
      const int j = NQ - j2 + j1;
      yh[j - 1] = ADD ? yh[j - 1] + yh[j] : yh[j - 1] - yh[j];
    }
}
template <bool ADD>
NRG_DI void psc(int nq, double (&yh)[MAXORD + 1])
{
  switch (nq) {
    case 1: psc_n<1, ADD>(yh); break;
    case 2: psc_n<2, ADD>(yh); break;
    case 3: psc_n<3, ADD>(yh); break;
    case 4: psc_n<4, ADD>(yh); break;
    default: psc_n<5, ADD>(yh); break;
  }
}

// YH(sub, col+1) read through a select chain (col in 1..MAXORD).
NRG_DI double yh_col(const Cell &c, int col)
{
  double v = opaque(c.yh[1]);
#pragma unroll
  for (int j = 2; j <= MAXORD; ++j) v = (col == j) ? opaque(c.yh[j]) : v;
  return v;
}

NRG_DI double weight(const Cell &c) { return fmax(fabs(c.y), c.ywt); }

// DDSCL (slatec/ddscl.f90:24-35).
NRG_DI void scl(Cell &c, double rh, const BdfConst &k)
{
  const double ah = fabs(c.h);
  if (c.h < 1.0)
    rh = dmin(dmin(ah * rh, ah * c.rmax), k.hmax) / ah;
  else
    rh = dmin(dmin(rh, c.rmax), k.hmax / ah);
  double r1 = 1.0;
#pragma unroll
  for (int j = 1; j <= MAXORD; ++j) {
    r1 = r1 * rh;
    // a column above NQ is written before it is read again, but for the last,
    // which keeps a SAVE1
    c.yh[j] = (j < MAXORD || c.nq == MAXORD) ? c.yh[j] * r1 : c.yh[j];
  }
  c.h = c.h * rh;
  c.rc = c.rc * rh;
}

// DDCOR, MITER = 2, IMPL = 0, IERROR = 3 (slatec/ddcor.f90:51-54,98-108); the
// norm before its division by sqrt(N).
NRG_DI double cor(const Lane &ln, Cell &c, const BdfConst &k)
{
  const double b = interchanged(ln, c, ((c.h * c.save2) - c.yh[1]) - c.save1);
  double x = solve<true>(ln, c, b), v = x / weight(c), nrm;
  if (__builtin_expect(!wave_any(unusual(k, v)), 1)) {
    nrm = norm_usual(ln, v);
  } else {
    x = solve<false>(ln, c, b);
    const double one[1] = {x / weight(c)};
    nrm = norms_serial<1>(ln, one, 0);
  }
  c.save1 = c.save1 + x;
  count(ln, c, WORK_NCORR);
  return nrm;
}

// DDNTP, K = 0 (slatec/ddntp.f90:25-32).
NRG_DI void ntp(Cell &c, double tout)
{
  c.y = yh_col(c, c.nq);
  const double r = (tout - c.t) / c.h;
#pragma unroll
  for (int j = MAXORD; j >= 1; --j) c.y = (j <= c.nq) ? c.yh[j - 1] + r * c.y : c.y;
}

NRG_DI void finish(Cell &c, int outcome) { c.pc = PC_DONE | outcome; }
NRG_DI void request_f(Cell &c, int resume) { c.pc = PC_WAIT_F | resume; }

// DDNTL up to its f call (slatec/ddntl.f90:52-63); EL/TQ are precomputed.
NRG_DI void ntl_head(Cell &c)
{
  c.ier = false;
  if (c.jtask == 0) c.rmax = 10000.0;
  c.rc = 0.0;
  c.convrg = false;
  c.trend = 1.0;
  c.nq = 1;
  c.nwait = 3;
}

// DDRIV3 init for NSTATE = 1 (slatec/ddriv3.f90:930-982): y holds C_in.
NRG_DI void bdf_init(Cell &c, double tout, const BdfConst &k)
{
  c.t = 0.0;
  double h = (tout - c.t) * (1.0 - 4.0 * k.uround);
  h = copysign(dmin(fabs(h), k.hmax), h);
  c.h = h;
  c.jtask = 0;
  c.nstep = 0;
  c.work = 0;
  c.jstepl = 0;
  c.ier = false;
  c.rc = 0.0;
  c.rmax = 0.0;
  c.trend = 0.0;
  c.nq = 1;
  c.nwait = 0;
  c.convrg = false;
  c.iter = 0;
  c.ntry = 0;
  c.nfail = 0;
  c.yh[0] = c.y;
  c.pc = PC_260;
}

// Run the cell's program until it needs f(y) (PC_WAIT_F, y set), a Jacobian
// (PC_WAIT_JAC) or is finished (PC_DONE).  On resumption after f the caller
// has put f(y) into save2.  hsign is +1 throughout (tout > 0).
//
// DDRIV3/DDSTP's control flow is laid out as stages in a fixed order, so that
// every transition taken in one pass goes forward.  Each stage's code exists
// once, is skipped by the whole wave when no group sits at it, and a group may
// pass several stages per call.
NRG_DI void advance(const Lane &ln, Cell &c, double tout, const BdfConst &k, const BdfCoef &mc)
{
  // what a stage hands to a later one of the same pass
  double ctest = 0.0, rh = 0.0;
  double px = 1.0, py = 1.0;     // argument and exponent of this lane's power
  int use = POW_FIRST;
  bool do_scale = false, rmax_after = false;
  // ---- rest of DDNTL after its f(y) (slatec/ddntl.f90:68,152-161)
  if (wave_any(c.pc == PC_NTL_F) && c.pc == PC_NTL_F) {
    count(ln, c, WORK_NFE);
    c.save1 = c.save2 / dmax(1.0, c.ywt);
    const double sum = norm(ln, k, c.save1) / k.sqrtn;
    if (sum > k.eps / fabs(c.h)) c.h = copysign(k.eps / sum, c.h);
    c.yh[1] = c.h * c.save2;
    c.fac = k.sqrt_uround;
    if (c.ntl_restart) c.rmax = 10.0;
    if (c.h == 0.0) {
      c.y = c.yh[0];
      finish(c, OUT_STEP_ZERO);
    } else {
      c.pc = PC_ATTEMPT;
    }
  }
  // ---- after f(y_pred), after a corrector f, after the Jacobian
  if (c.pc == PC_PRED_F) {
    count(ln, c, WORK_NFE);
    if (c.evaljc || c.ier) {
      c.pc = PC_WAIT_JAC | PC_JAC_DONE;
    } else {
      c.save1 = 0.0;
      c.pc = PC_CORR;
    }
  } else if (c.pc == PC_JAC_DONE) {
    if (c.ier) {
      use = POW_CONV;                                  // label 160
      c.pc = PC_RETRACT;
    } else {
      c.convrg = false;
      c.rc = 1.0;
      c.jstepl = c.nstep;
      c.save1 = 0.0;
      c.pc = PC_CORR;
    }
  } else if (c.pc == PC_CORR_F) {
    count(ln, c, WORK_NFE);
    c.pc = PC_CORR;
  }
  // ---- corrector iteration, label 130 (slatec/ddstp.f90:152-205)
  if (wave_any(c.pc == PC_CORR) && c.pc == PC_CORR) {
    c.nrm = cor(ln, c, k);
    const double d = div_by(c.nrm, k.sqrtn, mc.rsqrtn);
    if (c.iter > 0) c.trend = dmax(0.9 * c.trend, d / c.d1);
    c.d1 = d;
    ctest = dmin(2.0 * c.trend, 1.0) * d;
    if (ctest <= k.eps) {
      c.pc = PC_ERRTEST;
    } else {
      c.iter++;
      if (c.iter < 3) {
        const double l0 = el_of(mc, 1, c.nq);
        c.y = c.yh[0] + l0 * c.save1;
        request_f(c, PC_CORR_F);
      } else if (c.convrg) {                           // stale Jacobian: refresh (label 110)
        c.evaljc = true;
        c.iter = 0;
        c.y = c.yh[0];
        request_f(c, PC_PRED_F);
      } else {                                         // label 160 (:206-217)
        use = POW_CONV;
        c.pc = PC_RETRACT;
      }
    }
  }
  // ---- error test, accept, step/order selection, label 170 (:222-432)
  // A converged cell may wait here (it asks for nothing, so it re-enters on
  // the next pass unchanged) until gather_pct % of the lanes stepping in this
  // pass have arrived: the stage's code then runs once for all of them.  The
  // others always make progress, so the share is reached.
  const bool here4 = c.pc == PC_ERRTEST;
  const int n4 = __popcll(__ballot(here4 ? 1 : 0));
  const int nact = __popcll(__ballot(1));
  if (n4 > 0 && n4 * 100 >= k.gather_pct * nact && here4) {
    c.convrg = true;
    // the norm of the sum of the corrections: after one iteration it is the
    // corrector's own
    if (wave_any(c.iter > 0) && c.iter > 0) c.nrm = norm(ln, k, c.save1 / weight(c));
    if (over_tq2(mc, c.nrm, c.nq) > k.eps) {
      use = POW_ERR;                                   // (:238-289)
      c.pc = PC_RETRACT;
    } else {
      // accepted step (slatec/ddstp.f90:291-300)
      c.nstep++;
      // (EL is zero beyond NQ + 1: the columns there keep their values)
#pragma unroll
      for (int j = 1; j <= MAXORD + 1; ++j) c.yh[j - 1] = c.yh[j - 1] + el_of(mc, j, c.nq) * c.save1;
      c.y = c.yh[0];
      use = POW_FIRST;
      c.pc = PC_SCALE;
      // step-size and order selection (slatec/ddstp.f90:360-432)
      if (c.jtask == 0 || c.jtask == 2) {
        c.pc = PC_POW;
      } else if (c.nwait > 1) {
        c.nwait = c.nwait - 1;
        if (c.nwait == 1 && c.nq < k.maxord) c.yh[MAXORD] = c.save1;
      } else {
        use = POW_SELECT;
        c.pc = PC_POW;
      }
    }
  }
  // ---- retract the prediction, then the failure's step-size choice
  if (wave_any(c.pc == PC_RETRACT) && c.pc == PC_RETRACT) {
    c.t = c.told;
    psc<false>(c.nq, c.yh);
    c.pc = PC_POW;
    if (use == POW_CONV) {                           // label 160
      c.nwait = c.nq + 2;
      if (c.jtask != 0 && c.jtask != 2) c.rmax = 2.0;
    } else {                                           // error test failed (:238-289)
      c.nfail++;
      if (c.nfail < 3 || c.nq == 1) {
        if (c.jtask != 0 && c.jtask != 2) c.rmax = 2.0;
      } else {
        c.nfail = 0;                                   // restart at order 1 (:275-288)
        c.jtask = 2;
        c.y = c.yh[0];
        ntl_head(c);
        c.ntl_restart = true;
        request_f(c, PC_NTL_F);
      }
    }
  }
  // ---- the step-size candidates.  Lane 0 takes order down, lane 1 the same
  // order, the others order up (of use in lane 2): their norms, powers and
  // quotients are formed side by side.  A candidate that does not apply (order
  // 1 cannot go down, MAXORD not up, a failure does not go up) is formed from
  // whatever its vector holds and then not used.
  if (wave_any(c.pc == PC_POW) && c.pc == PC_POW) {
    const int cand = ln.sub < 2 ? ln.sub : 2;
    const double etest = over_tq2(mc, c.nrm, c.nq);
    const int kt = cand == 2 ? 2 : 0;
    const double den = mc.den[kt][c.nq - 1];
    py = mc.inv[c.nq + cand];
    double err = etest;
    const bool need = use == POW_SELECT || (use == POW_ERR && c.nq > 1);
    if (wave_any(need) && need) {
      const double w = weight(c);
      const double v[2] = {yh_col(c, c.nq) / w, (c.save1 - c.yh[MAXORD]) / w};
      const double nrm = norms<2>(ln, k, v, cand == 2 ? 1 : 0);
      const double e = nrm / den;
      err = cand == 1 ? etest : e;
    }
    px = err / k.eps;
    if (use == POW_CONV) {
      px = c.iter == 0 ? 1.0 : k.eps / ctest;
      py = 0.2;
    }
    const double pw = pow(px, py);
    // 1 / max(floor, bias * power), biases 1.3, 1.2, 1.4
    const double bias = cand == 0 ? 1.3 : cand == 1 ? 1.2 : 1.4;
    const double floor_ = use == POW_ERR ? (cand == 0 ? 1.0 : 0.0) : k.uround;
    const double rc_ = 1.0 / dmax(floor_, bias * pw);
    const double ra = bcast<0>(rc_), rb = bcast<1>(rc_), ru = bcast<2>(rc_);
    const int nq0 = c.nq;
    c.pc = PC_SCALE;
    if (use == POW_FIRST) {
      rh = rb;
      do_scale = rh > 1.0;
    } else if (use == POW_SELECT) {
      const double rh1 = (c.nq != 1) ? ra : 0.0;
      const double rh2 = rb;
      const double rh3 = (c.nq != k.maxord) ? ru : 0.0;
      if (rh1 > rh2 && rh1 >= rh3) {
        rh = rh1;
        do_scale = !(rh <= 1.0);
        if (do_scale) c.nq = c.nq - 1;
      } else if (rh2 >= rh1 && rh2 >= rh3) {
        rh = rh2;
        do_scale = !(rh <= 1.0);
      } else {
        rh = rh3;
        do_scale = !(rh <= 1.0);
        if (do_scale) {
          const double l = el_of(mc, c.nq + 1, c.nq), den = (double)(c.nq + 1);
          const int dst = c.nq + 1;
          const double newc = (c.save1 * l) / den;
#pragma unroll
          for (int j = 2; j <= MAXORD; ++j) c.yh[j] = (dst == j) ? newc : c.yh[j];
          c.nq = c.nq + 1;
        }
      }
      rmax_after = do_scale;
    } else {
      if (use == POW_CONV) {
        rh = (c.iter == 0) ? 0.3 : 0.9 * bcast<1>(pw);
      } else {
        rh = rb;
        if (c.nq > 1 && rb < ra) {
          c.nq = c.nq - 1;
          rh = ra;
        }
      }
      do_scale = true;
      if (rh * c.h == 0.0) {
        c.y = c.yh[0];
        finish(c, OUT_STEP_ZERO);
      }
    }
    if (c.nq != nq0) c.rc = (c.rc * el_of(mc, 1, c.nq)) / el_of(mc, 1, nq0);
    if (use == POW_SELECT || use == POW_ERR) c.nwait = c.nq + 2;
  }
  // ---- pending DDSCL, then the next attempt or DDRIV3's label 470
  if (wave_any(c.pc == PC_SCALE) && c.pc == PC_SCALE) {
    if (do_scale) scl(c, rh, k);
    if (rmax_after) c.rmax = 10.0;
    if (use >= POW_CONV) {
      c.pc = PC_ATTEMPT;
    } else {
      // DDSTP returned JSTATE = 1; DDRIV3 label 470 (:1371, NTASK = 1 test :1443-1449)
      c.jtask = 1;
      if (c.t < tout) {
        c.pc = PC_260;
      } else {
        ntp(c, tout);
        finish(c, OUT_OK);
      }
    }
  }
  // ---- DDRIV3 label 260: weights and guards, DDSTP entry (slatec/ddriv3.f90:1292-1351)
  if (wave_any(c.pc == PC_260) && c.pc == PC_260) {
    c.ywt = dmax(k.ewt, fabs(c.y));
    // |y_i / YWT_i| <= 1, so SUM = max(1, ||y/YWT|| / sqrt(N)) stays below 2
    // and EPS < SUM * UROUND cannot hold for EPS >= 2 * UROUND; the norm is
    // formed only when it can decide.
    bool eps_fail = false;
    if (k.eps < 2.0 * k.uround) {
      // over all species, in their order; the inert ones keep their initial concentration
      wave_sync();
      if (holds(ln)) *own(ln, CZ) = c.y;
      wave_sync();
#pragma unroll
      for (int s0 = 0; s0 < S; s0 += G) {
        const int s = s0 + ln.sub;
        if (s < S) {
          const double yv = *slot(ln, inert_species(s) ? 2 * REC_C + s : CZ + active_slot(s));
          *slot(ln, CX + s) = yv / dmax(k.ewt, fabs(yv));
        }
      }
      wave_sync();
      double sum = norm_serial<S>(ln) / k.sqrtn;
      sum = dmax(1.0, sum);
      eps_fail = k.eps < sum * k.uround;
    }
    if (eps_fail) {
      c.y = c.yh[0];
      finish(c, OUT_EPS);
    } else if (c.nstep == k.mxstep) {
      c.y = c.yh[0];
      finish(c, OUT_MXSTEP);
    } else {
      c.told = c.t;                                    // DDSTP entry (:91-106)
      c.ntry = 0;
      c.nfail = 0;
      if (c.jtask <= 0) {
        ntl_head(c);
        c.ntl_restart = false;
        request_f(c, PC_NTL_F);
      } else {
        c.pc = PC_ATTEMPT;
      }
    }
  }
  // ---- attempt, labels 100/110 (slatec/ddstp.f90:107-118)
  if (wave_any(c.pc == PC_ATTEMPT) && c.pc == PC_ATTEMPT) {
    c.ntry++;
    if (c.ntry > 50) {
      finish(c, OUT_REPEATED_FAIL);
    } else {
      count(ln, c, WORK_NATT);
      c.t = c.t + c.h;
      psc<true>(c.nq, c.yh);
      c.evaljc = (fabs(c.rc - 1.0) > 0.3) || (c.nstep >= c.jstepl + 10);
      c.iter = 0;
      c.y = c.yh[0];
      request_f(c, PC_PRED_F);
    }
  }
}

// DDPST, MITER = 2 (slatec/ddpst.f90:39-114,142-143): finite-difference
// Jacobian with adaptive increments FAC, P = I - h*l0*J and its LU.  Lane j
// perturbs species j and forms column j with a whole right-hand side of its
// own, so the columns of a cell are formed side by side.
NRG_DI void jac_fd(const Lane &ln, Cell &c, const BdfConst &k, const BdfCoef &mc)
{
  count(ln, c, WORK_NJE);
  count(ln, c, WORK_NFE, S);                         // DDPST counts N evaluations
  c.ier = false;
  const double l0 = el_of(mc, 1, c.nq);
  wave_sync();
  if (holds(ln)) {
    *own(ln, CZ) = c.y;
    *own(ln, CX) = c.save2;
  }
  wave_sync();
  const double ys = dmax(fabs(c.ywt), fabs(c.y));
  double fj = c.fac;
  double dy = fj * ys;
  while (dy == 0.0) {
    if (fj < 0.5) {
      fj = dmin(100.0 * fj, 0.5);
      dy = fj * ys;
    } else {
      dy = ys;
      break;
    }
  }
  dy = (c.nq == 1) ? copysign(dy, c.save2) : copysign(dy, c.yh[2]);
  dy = (c.y + dy) - c.y;
  const double yp = c.y + dy;
  double z[SA], f1[SA], col[SA];
#pragma unroll
  for (int q = 0; q < SA; ++q) z[q] = (q == ln.sub) ? yp : *slot(ln, CZ + q);
  rhs_lane(ln, z, f1);
  const double scale_ = ((-l0) * c.h) / dy;
  double diff = 0.0, s2m = 0.0, s1m = 0.0;
#pragma unroll
  for (int i = 0; i < SA; ++i) {
    const double s2 = *slot(ln, CX + i), d = f1[i] - s2;
    col[i] = d * scale_;
    const double di = fabs(d);
    if (i == 0 || di > diff) {
      diff = di;
      s2m = s2;
      s1m = f1[i];
    }
  }
  if (dmin(fabs(s2m), fabs(s1m)) > 0.0) {
    const double scale = dmax(fabs(s2m), fabs(s1m));
    if (diff > 0.5 * scale)
      fj = dmax(k.facmin, fj * 0.5);
    else if (k.br * scale <= diff && diff <= k.bl * scale)
      fj = dmin(fj * 2.0, 0.5);
    else if (diff < k.br * scale)
      fj = dmin(k.bp * fj, 0.5);
  }
  c.fac = fj;
#pragma unroll
  for (int i = 0; i < SA; ++i) col[i] = (i == ln.sub) ? col[i] + 1.0 : col[i];
  factor(ln, c, col);
}

// Fast mode (NRG_JAC_ANALYTIC): the iteration matrix P = I - h*l0*J with the
// exact J = d(omega)/dC of the law of mass action at the cell's fixed rate
// constants and [M] (the third-body concentration is frozen per cell, so it
// has no derivative), as DDPST forms it for a user Jacobian (MITER = 1).  No
// extra right-hand sides are evaluated; the step sequence therefore differs
// from the finite-difference (SLATEC MITER = 2) parity mode.
//
// G reactions at a time: lane i forms the derivatives of reaction q G + i by
// each of its terms, then lane j adds those by species j to its column, in the
// order of the reactions and terms.  (Every lane walking through all terms with
// its own masked in took four times the instructions.)
template <int A, int N>
NRG_DI double derivative(const double (&o)[3], double k)
{
  double d = k;
  if (N > 0 && A != 0) d = d * o[0];
  if (N > 1 && A != 1) d = d * o[1];
  if (N > 2 && A != 2) d = d * o[2];
  return d;
}
template <int N, int FIRST>
NRG_DI void operands(const Lane &ln, const unsigned (&w)[3], double (&o)[3])
{
  if (N > 0) o[0] = *at_addr(add_half<FIRST & 1>(w[FIRST / 2], ln.base));
  if (N > 1) o[1] = *at_addr(add_half<(FIRST + 1) & 1>(w[(FIRST + 1) / 2], ln.base));
  if (N > 2) o[2] = *at_addr(add_half<(FIRST + 2) & 1>(w[(FIRST + 2) / 2], ln.base));
}
template <int SIDE, int Q>
NRG_DI void side_derivatives(const Lane &ln, const unsigned (&w)[3], double k, double fac, lds_double *x)
{
  constexpr int N = round_terms(Q, SIDE), FIRST = 3 * SIDE;
  double o[3];
  operands<N, FIRST>(ln, w, o);
  if (N > 0) x[FIRST] = fac * derivative<0, N>(o, k);
  if (N > 1) x[FIRST + 1] = fac * derivative<1, N>(o, k);
  if (N > 2) x[FIRST + 2] = fac * derivative<2, N>(o, k);
}
// col += nu of reaction Rn times a derivative
template <int Rn>
NRG_DI void add_derivative(double (&col)[SA], double fd)
{
#pragma unroll
  for (int i = 0; i < SA; ++i) {
    const int nu = nu_of(Rn, kSp.full[i]);
    if (nu != 0) col[i] = col[i] + (double)nu * fd;
  }
}
template <int Rn, int N = 0>
NRG_DI void add_reaction(const Lane &ln, double (&col)[SA])
{
  if constexpr (N < most_terms(Rn)) {
    unsigned w[1];
    table_words<N * JW2 + Rn / 2>(ln.jtab, w);
    add_derivative<Rn>(col, *at_addr(add_half<Rn % 2>(w[0], ln.base)));
    add_reaction<Rn, N + 1>(ln, col);
  }
}
template <int Q, int... I>
NRG_DI void jac_round(const Lane &ln, double fac, double (&col)[SA], std::integer_sequence<int, I...>)
{
  const int r = Q * G + ln.sub;
  wave_sync();
  if ((Q + 1) * G <= R || r < R) {
    unsigned w[3];
    table_words<3 * Q>(ln.tab, w);
    const lds_double *k = at_addr(ln.base + 16u * (unsigned)r);
    lds_double *x = at_addr(ln.base + 8u * CX + 48u * (unsigned)ln.sub);
    side_derivatives<0, Q>(ln, w, k[0], fac, x);
    side_derivatives<1, Q>(ln, w, -k[1], fac, x);
  }
  wave_sync();
  (add_reaction<Q * G + I>(ln, col), ...);
}
template <int... Q>
NRG_DI void jac_rounds(const Lane &ln, double fac, double (&col)[SA], std::integer_sequence<int, Q...>)
{
  (jac_round<Q>(ln, fac, col, std::make_integer_sequence<int, ((Q + 1) * G <= R ? G : R - Q * G)>{}), ...);
}

NRG_DI void jac_exact(const Lane &ln, Cell &c, const BdfCoef &mc)
{
  count(ln, c, WORK_NJE);
  c.ier = false;
  const double fac = (-el_of(mc, 1, c.nq)) * c.h;
  wave_sync();
  if (holds(ln)) *own(ln, CZ) = c.y;
  double col[SA];
#pragma unroll
  for (int i = 0; i < SA; ++i) col[i] = 0.0;
  jac_rounds(ln, fac, col, std::make_integer_sequence<int, RROUNDS>{});
#pragma unroll
  for (int i = 0; i < SA; ++i) col[i] = (i == ln.sub) ? col[i] + 1.0 : col[i];
  factor(ln, c, col);
}

}  // namespace nrg
