// bdf_lane.h -- one cell per lane: the integrator where cells that cost alike fill
// the chip.
//
// A cell's Gear-BDF state (Nordsieck history, iteration matrix, work vectors)
// lives in VGPRs/AGPRs; its 2R rate constants live in a per-lane LDS slot.
// Every register-array index is a compile-time constant after unrolling; the
// few order- or pivot-dependent accesses are select chains.
//
// SLATEC's DDRIV3 is restated as a reverse-communication state machine
// (advance()): a lane runs until it needs a right-hand side f(y) or a
// Jacobian, then the wave evaluates f for all lanes that asked at one code
// site, or -- when enough lanes wait for one -- runs a batched
// finite-difference Jacobian + LU for those lanes (jac_batch()).  Decisions
// and arithmetic follow the reference operation by operation (this TU is
// built with -ffp-contract=off), so results agree with NRG's Fortran step to
// the rounding of the transcendental functions, and bit for bit with the
// lane groups of bdf_group.h.
//
// What bounds it: FP64 VALU issue and its latency (the state takes the whole
// register file: one wave per SIMD), and lanes that wait while others of their
// wave pass a stage.  Cells of equal cost, which stiffness order brings
// together, keep that share small; 65,536 cells fill the chip once.  The norm has
// one path for ordinary vectors instead of the walk through its phases.  Kernel
// time in stiffness order with a history: 1M flame cells 11.9 ms, 2.1M cells with
// hot kernels 3.7, 1M igniting ones 15.0.
//
// Reference: computing_module/src/current_build/chemical_kinetics_solver.f90
// (RHS :495-540, cell step :228-346) and SLATEC SDRIVE in
// computing_module/src/third_party/slatec/ (ddriv3.f90, ddstp.f90, ddntl.f90,
// ddpst.f90, ddcor.f90, ddpsc.f90, ddscl.f90, ddntp.f90, dgefa.f90,
// dgesl.f90, dnrm2.f90).
#pragma once
#include "bdf_group.h"
#include "chem_device.h"

namespace nrg {
namespace lane {

// One out-of-line copy of each transcendental for the integrator kernel,
// which calls pow a few times per step from several sites; inlined, every
// call site would carry its own 100+-instruction expansion.
__device__ __noinline__ double nl_pow(double x, double y) { return pow(x, y); }

// Three independent powers in one call: the order-selection candidates of a
// step, whose dependent chains interleave here instead of running back to back.
struct Pow3 {
  double a, b, c;
};
__device__ __noinline__ Pow3 nl_pow3(double xa, double ya, double xb, double yb, double xc, double yc)
{
  return Pow3{pow(xa, ya), pow(xb, yb), pow(xc, yc)};
}

// The lane's LDS copy (kl = recl + 2 * lane).
NRG_DI double rec_kf(const double *kl, int r) { return kl[r * 2 * WAVE]; }
NRG_DI double rec_kr(const double *kl, int r) { return kl[r * 2 * WAVE + 1]; }
NRG_DI double rec_m(const double *kl, int j) { return kl[(REC_M + j / 2) * 2 * WAVE + (j & 1)]; }
NRG_DI double rec_c(const double *kl, int s) { return kl[(REC_C + s / 2) * 2 * WAVE + (s & 1)]; }

// Rate constants and [M] from the lane's cell record in LDS (kl).
NRG_DI void rhs(const double *kl, const double (&Z)[SA], double (&Zd)[SA])
{
#pragma unroll
  for (int s = 0; s < SA; ++s) Zd[s] = 0.0;
#pragma unroll
  for (int r = 0; r < R; ++r)
    rhs_reaction(r, rec_kf(kl, r), rec_kr(kl, r), kMSlot.v[r] >= 0 ? rec_m(kl, kMSlot.v[r]) : 0.0,
                 Z, Zd);
}

// ---------------------------------------------------------------------------
// DNRM2 (slatec/dnrm2.f90:84-160): Lawson's phases as a per-element state machine.
// st: 0 = start (label 30), 1 = phase 1 (50), 2 = phase 2 (70), 3 = phase 4 (110),
//     4 = phase 3 (the DO 95 loop, unscaled sum).
// Out of line, it serves vectors with a component at or above HITEST, or NaN.
// The others go through one path (dnrm2_core): up to the first component above
// CUTLO the sum is scaled by the largest so far, from there on it is not.
// One out-of-line copy serves the call sites; the vector arrives in argument
// VGPRs.  The inert species' terms, exact zeros, are left out: in every phase
// a zero leaves SUM, XMAX and the phase as they were.  HITEST keeps DDRIV3's
// N (all species).
// ---------------------------------------------------------------------------
template <int n>
NRG_DI double dnrm2_phases(const double *x)
{
  const double cutlo = NRM_CUTLO, hitest = NRM_HITEST;
  double sum = 0.0, xmax = 0.0;
  int st = 0;
#pragma unroll
  for (int i = 0; i < n; ++i) {
    const double v = x[i], av = fabs(v);
    // the usual case first (phase 3, no overflow risk): what the state
    // machine below does for it, without walking through the other phases
    if (st == 4 && av < hitest) {
      sum = sum + v * v;
      continue;
    }
    bool done = false;
    if (st == 0) {
      if (av > cutlo) {
        st = 4;
      } else {
        st = 1;
        xmax = 0.0;
      }
    }
    if (st == 1) {
      if (v == 0.0) {
        done = true;
      } else if (av > cutlo) {
        st = 4;
      } else {
        st = 2;
        xmax = av;
        const double r = v / xmax;
        sum = sum + r * r;
        done = true;
      }
    }
    if (!done && st == 2) {
      if (av > cutlo) {
        sum = (sum * xmax) * xmax;
        st = 4;
      } else {
        if (av <= xmax) {
          const double r = v / xmax;
          sum = sum + r * r;
        } else {
          const double r = xmax / v;
          sum = 1.0 + sum * (r * r);
          xmax = av;
        }
        done = true;
      }
    }
    if (!done && st == 3) {
      if (av <= xmax) {
        const double r = v / xmax;
        sum = sum + r * r;
      } else {
        const double r = xmax / v;
        sum = 1.0 + sum * (r * r);
        xmax = av;
      }
      done = true;
    }
    if (!done && st == 4) {
      if (av >= hitest) {
        sum = (sum / v) / v;
        xmax = av;
        const double r = v / xmax;
        sum = sum + r * r;
        st = 3;
      } else {
        sum = sum + v * v;
      }
    }
  }
  return (st == 4) ? sqrt(sum) : xmax * sqrt(sum);
}

template <class... D>
__device__ __noinline__ double dnrm2_phases_vals(D... xs)
{
  const double x[sizeof...(D)] = {xs...};
  return dnrm2_phases<(int)sizeof...(D)>(x);
}
template <int... I>
NRG_DI double dnrm2_phases_seq(const double *x, std::integer_sequence<int, I...>)
{
  return dnrm2_phases_vals(x[I]...);
}

// (Components under 2^-960 count as zeros: beside a larger maximum than 2^-900
// their squares are less than half an ulp of the sum, which is 1 at least, and
// vectors that end below that take all phases.)
template <int n>
NRG_DI double dnrm2_core(const double *x)
{
  bool over = false;
#pragma unroll
  for (int i = 0; i < n; ++i) over = over || !(fabs(x[i]) < NRM_HITEST);
  if (over) return dnrm2_phases_seq(x, std::make_integer_sequence<int, n>{});
  double sum = 0.0, xmax = 0.0;
  bool scaled = true;
#pragma unroll
  for (int i = 0; i < n; ++i) {
    const double v = x[i], av = fabs(v);
    if (scaled) {
      if (av > NRM_CUTLO) {
        sum = (sum * xmax) * xmax;
        scaled = false;
      } else if (av >= 0x1p-960) {
        const bool in = av <= xmax;
        const double r = quot_raw(in ? av : xmax, in ? xmax : av), rr = r * r;
        sum = in ? sum + rr : 1.0 + sum * rr;
        xmax = in ? xmax : av;
      }
    }
    sum = scaled ? sum : sum + v * v;
  }
  if (scaled && xmax < 0x1p-900) {
    bool zero = true;
#pragma unroll
    for (int i = 0; i < n; ++i) zero = zero && x[i] == 0.0;
    if (!zero) return dnrm2_phases_seq(x, std::make_integer_sequence<int, n>{});
  }
  const double s = root(sum);
  return scaled ? xmax * s : s;
}

template <class... D>
__device__ __noinline__ double dnrm2_vals(D... xs)
{
  const double x[sizeof...(D)] = {xs...};
  return dnrm2_core<(int)sizeof...(D)>(x);
}

// Two norms in one call (independent state machines, interleaved).
struct Norm2 {
  double a, b;
};
template <class... D>
__device__ __noinline__ Norm2 dnrm2_pair_vals(D... xs)
{
  constexpr int n = (int)sizeof...(D) / 2;
  const double v[2 * n] = {xs...};
  return Norm2{dnrm2_core<n>(v), dnrm2_core<n>(v + n)};
}

template <int N, int... I>
NRG_DI double dnrm2_seq(const double (&x)[N], std::integer_sequence<int, I...>)
{
  return dnrm2_vals(x[I]...);
}

// Norm of a vector over the active species.
NRG_DI double dnrm2(const double (&x)[SA])
{
  return dnrm2_seq<SA>(x, std::make_integer_sequence<int, SA>{});
}

template <int... I>
NRG_DI Norm2 dnrm2_pair_seq(const double (&x)[SA], const double (&y)[SA], std::integer_sequence<int, I...>)
{
  return dnrm2_pair_vals(x[I]..., y[I]...);
}

// Norms of two vectors over the active species.
NRG_DI Norm2 dnrm2_pair(const double (&x)[SA], const double (&y)[SA])
{
  return dnrm2_pair_seq(x, y, std::make_integer_sequence<int, SA>{});
}

// Norm of a vector over all species.
NRG_DI double dnrm2_all(const double (&x)[S])
{
  return dnrm2_seq<S>(x, std::make_integer_sequence<int, S>{});
}

// ---------------------------------------------------------------------------
// 9x9 LU with partial pivoting (DGEFA) and solve (DGESL), column-major a[col][row].
// Row interchanges use select chains; a wave skips them when no lane pivots.
// ---------------------------------------------------------------------------
// y[i] += t * x[i] for i in [LO, SA), left alone on the lanes with `skip` set
// (DAXPY returns at once for DA == 0, slatec/daxpy.f90:68; adding 0*x is not
// the same when x is not finite or y is -0).  The wave takes the select-free
// form when no lane skips and drops the loop when every lane does; both
// happen for whole columns (a species that no rate depends on gives exact
// zeros in P and in the corrector's right-hand side).
template <int LO>
NRG_DI void daxpy_lanes(bool skip, double t, const double (&x)[SA], double (&y)[SA])
{
  if (!wave_any(!skip)) return;
  if (wave_any(skip)) {
#pragma unroll
    for (int i = LO; i < SA; ++i) y[i] = skip ? y[i] : y[i] + t * x[i];
  } else {
#pragma unroll
    for (int i = LO; i < SA; ++i) y[i] = y[i] + t * x[i];
  }
}

// As daxpy_lanes over [0, HI).
template <int HI>
NRG_DI void daxpy_head(bool skip, double t, const double (&x)[SA], double (&y)[SA])
{
  if (!wave_any(!skip)) return;
  if (wave_any(skip)) {
#pragma unroll
    for (int i = 0; i < HI; ++i) y[i] = skip ? y[i] : y[i] + t * x[i];
  } else {
#pragma unroll
    for (int i = 0; i < HI; ++i) y[i] = y[i] + t * x[i];
  }
}

template <int K>
NRG_DI void gefa_col(double (&a)[SA][SA], int (&ipvt)[SA], int &info)
{
  int l = K;
  double dmx = fabs(a[K][K]), piv = a[K][K];
#pragma unroll
  for (int i = K + 1; i < SA; ++i) {
    const double xm = fabs(a[K][i]);
    if (xm > dmx) {
      l = i;
      dmx = xm;
      piv = a[K][i];
    }
  }
  ipvt[K] = l;
  const bool zero = (piv == 0.0);
  if (zero) info = K + 1;
  const bool anyswap = wave_any(l != K);
  if (anyswap) {
#pragma unroll
    for (int i = K + 1; i < SA; ++i) a[K][i] = (l == i) ? a[K][K] : a[K][i];
    a[K][K] = piv;
  }
  // DSCAL of the column below the pivot (skipped for a zero pivot)
  const double t = -1.0 / a[K][K];
  if (wave_any(zero)) {
#pragma unroll
    for (int i = K + 1; i < SA; ++i) a[K][i] = zero ? a[K][i] : t * a[K][i];
  } else {
#pragma unroll
    for (int i = K + 1; i < SA; ++i) a[K][i] = t * a[K][i];
  }
#pragma unroll
  for (int j = K + 1; j < SA; ++j) {
    double tj = a[j][K];
    if (anyswap) {
#pragma unroll
      for (int i = K + 1; i < SA; ++i) tj = (l == i) ? a[j][i] : tj;
#pragma unroll
      for (int i = K + 1; i < SA; ++i) a[j][i] = (l == i) ? a[j][K] : a[j][i];
      a[j][K] = tj;
    }
    daxpy_lanes<K + 1>(zero || (tj == 0.0), tj, a[K], a[j]);
  }
}

template <int... K>
NRG_DI void gefa_cols(double (&a)[SA][SA], int (&ipvt)[SA], int &info, std::integer_sequence<int, K...>)
{
  (gefa_col<K>(a, ipvt, info), ...);
}

NRG_DI int gefa(double (&a)[SA][SA], int (&ipvt)[SA])
{
  int info = 0;
  gefa_cols(a, ipvt, info, std::make_integer_sequence<int, SA - 1>{});
  ipvt[SA - 1] = SA - 1;
  if (a[SA - 1][SA - 1] == 0.0) info = SA;
  return info;
}

template <int K>
NRG_DI void gesl_fwd(const double (&a)[SA][SA], const int (&ipvt)[SA], double (&b)[SA])
{
  const int l = ipvt[K];
  double t = b[K];
  if (wave_any(l != K)) {
#pragma unroll
    for (int i = K + 1; i < SA; ++i) t = (l == i) ? b[i] : t;
#pragma unroll
    for (int i = K + 1; i < SA; ++i) b[i] = (l == i) ? b[K] : b[i];
    b[K] = t;
  }
  daxpy_lanes<K + 1>(t == 0.0, t, a[K], b);
}

template <int K>
NRG_DI void gesl_back(const double (&a)[SA][SA], double (&b)[SA])
{
  b[K] = b[K] / a[K][K];
  const double t = -b[K];
  daxpy_head<K>(t == 0.0, t, a[K], b);
}

template <int... K>
NRG_DI void gesl_steps(const double (&a)[SA][SA], const int (&ipvt)[SA], double (&b)[SA],
                       std::integer_sequence<int, K...>)
{
  (gesl_fwd<K>(a, ipvt, b), ...);
  (gesl_back<SA - 1 - K>(a, b), ...);
  gesl_back<SA - 1 - (int)sizeof...(K)>(a, b);
}

NRG_DI void gesl(const double (&a)[SA][SA], const int (&ipvt)[SA], double (&b)[SA])
{
  gesl_steps(a, ipvt, b, std::make_integer_sequence<int, SA - 1>{});
}

// ---------------------------------------------------------------------------
// Gear BDF state of one cell (DDRIV3's WORK/IWORK, private to the lane) and
// the program counter of the reverse-communication form.
// ---------------------------------------------------------------------------
enum Pc : int {
  PC_260 = 0,      // DDRIV3 label 260: weights and guards, then DDSTP entry
  PC_NTL_F,        // DDNTL after its f(y)
  PC_ATTEMPT,      // DDSTP label 100: predict, then f(y_pred)
  PC_PRED_F,       // after f(y_pred) (label 110)
  PC_JAC_DONE,     // after the batched FD Jacobian + LU (DDPST)
  PC_CORR,         // label 130: corrector (DDCOR)
  PC_CORR_F,       // after f(y) of a corrector iteration
  PC_FAIL_CONV,    // label 160: corrector failure
  PC_ERRTEST,      // label 170: error test, accept, step/order selection
  PC_RETRACT,      // retract the prediction after a failed attempt
  PC_SCALE,        // apply a pending DDSCL rescale, then continue
  PC_DONE
};
enum Req : int { REQ_NONE = 0, REQ_F = 1, REQ_JAC = 2, REQ_DONE = 3 };
enum CellOutcome { OUT_OK = 0, OUT_MXSTEP = 2, OUT_STEP_ZERO = 3, OUT_REPEATED_FAIL = 4,
                   OUT_SINGULAR = 5, OUT_EPS = 6 };

struct Cell {
  double yh[MAXORD + 1][SA];   // yh[j][i] = YH(i, j+1)
  double y[SA], ywt[SA], save1[SA], save2[SA], fac[SA];
  double P[SA][SA];             // iteration matrix / LU factors, column-major
  int ipvt[SA];
  double yi[NI > 0 ? NI : 1];   // concentrations of the inert species (constant)
  double t, h, rc, rmax, trend, told, d1, ctest;
  int nq, nwait, jtask, jstepl, nstep, nfe, nje, ncorr, natt;
  int ntry, nfail, iter, pc, req, outcome;
  bool convrg, ier, evaljc, ntl_restart;
  // pending retraction / rescale (stages R and S)
  double rh, etest;
  bool fail_err, do_scale, rmax_after, after_accept;
};

// DDPSC (slatec/ddpsc.f90:26-38) for a compile-time order.
template <int NQ, bool ADD>
NRG_DI void psc_n(double (&yh)[MAXORD + 1][SA])
{
#pragma unroll
  for (int j1 = 1; j1 <= NQ; ++j1)
#pragma unroll
    for (int j2 = j1; j2 <= NQ; ++j2) {
      const int j = NQ - j2 + j1;
#pragma unroll
      for (int i = 0; i < SA; ++i) yh[j - 1][i] = ADD ? yh[j - 1][i] + yh[j][i] : yh[j - 1][i] - yh[j][i];
    }
}

template <bool ADD>
NRG_DI void psc(int nq, double (&yh)[MAXORD + 1][SA])
{
  switch (nq) {
    case 1: psc_n<1, ADD>(yh); break;
    case 2: psc_n<2, ADD>(yh); break;
    case 3: psc_n<3, ADD>(yh); break;
    case 4: psc_n<4, ADD>(yh); break;
    default: psc_n<5, ADD>(yh); break;
  }
}

// YH(:, col+1) read through a select chain (col in 1..MAXORD).
NRG_DI void yh_col(const Cell &c, int col, double (&out)[SA])
{
#pragma unroll
  for (int i = 0; i < SA; ++i) {
    double v = opaque(c.yh[1][i]);
#pragma unroll
    for (int j = 2; j <= MAXORD; ++j) v = (col == j) ? opaque(c.yh[j][i]) : v;
    out[i] = v;
  }
}

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
    const bool on = (j <= c.nq);
#pragma unroll
    for (int i = 0; i < SA; ++i) c.yh[j][i] = on ? c.yh[j][i] * r1 : c.yh[j][i];
  }
  c.h = c.h * rh;
  c.rc = c.rc * rh;
}

// DDCOR, MITER = 2, IMPL = 0, IERROR = 3 (slatec/ddcor.f90:51-54,98-108).
NRG_DI double cor(Cell &c, const BdfConst &k)
{
#pragma unroll
  for (int i = 0; i < SA; ++i) c.save2[i] = ((c.h * c.save2[i]) - c.yh[1][i]) - c.save1[i];
  gesl(c.P, c.ipvt, c.save2);
#pragma unroll
  for (int i = 0; i < SA; ++i) {
    c.save1[i] = c.save1[i] + c.save2[i];
    c.save2[i] = c.save2[i] / dmax(fabs(c.y[i]), c.ywt[i]);
  }
  c.ncorr++;
  return dnrm2(c.save2) / k.sqrtn;
}

// DDNTP, K = 0 (slatec/ddntp.f90:25-32).
NRG_DI void ntp(Cell &c, double tout)
{
  double col[SA];
  yh_col(c, c.nq, col);
#pragma unroll
  for (int i = 0; i < SA; ++i) c.y[i] = col[i];
  const double r = (tout - c.t) / c.h;
#pragma unroll
  for (int j = MAXORD; j >= 1; --j) {
    const bool on = (j <= c.nq);
#pragma unroll
    for (int i = 0; i < SA; ++i) c.y[i] = on ? c.yh[j - 1][i] + r * c.y[i] : c.y[i];
  }
}

NRG_DI void copy_yh0_to_y(Cell &c)
{
#pragma unroll
  for (int i = 0; i < SA; ++i) c.y[i] = c.yh[0][i];
}

NRG_DI void finish(Cell &c, int outcome)
{
  c.outcome = outcome;
  c.pc = PC_DONE;
  c.req = REQ_DONE;
}

NRG_DI void request_f(Cell &c, int resume)
{
  c.pc = resume;
  c.req = REQ_F;
}

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
  c.nstep = c.nfe = c.nje = c.ncorr = c.natt = 0;
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
#pragma unroll
  for (int i = 0; i < SA; ++i) c.yh[0][i] = c.y[i];
  c.pc = PC_260;
  c.req = REQ_NONE;
  c.outcome = OUT_OK;
}

// Stage guards: a lane runs a stage when it sits at that program counter and
// has not yet asked for anything in this pass; a stage's code is skipped by
// the whole wave when no lane needs it.
NRG_DI bool at(const Cell &c, int pc) { return c.req == REQ_NONE && c.pc == pc; }

// Run the cell's program until it needs f(y) (req = REQ_F, y set), a
// Jacobian (REQ_JAC) or is finished (REQ_DONE).  On REQ_F resumption the
// caller has put f(y) into save2.  hsign is +1 throughout (tout > 0).
//
// DDRIV3/DDSTP's control flow is laid out as seven stages in a fixed order,
// so that every transition taken in one pass goes forward:
//   1 DDNTL tail   2 after f / Jacobian   3 corrector (label 130)
//   4 error test, accept, step/order choice (label 170)
//   5 corrector failure (label 160)   6 DDRIV3 label 260   7 attempt (label 100)
// Each stage's code exists once; a lane may pass several stages per call.
NRG_DI void advance(Cell &c, double tout, const BdfConst &k, const BdfCoef &mc)
{
  // ---- 1: rest of DDNTL after its f(y) (slatec/ddntl.f90:68,152-161)
  if (wave_any(at(c, PC_NTL_F)) && at(c, PC_NTL_F)) {
    c.nfe++;
#pragma unroll
    for (int i = 0; i < SA; ++i) c.save1[i] = c.save2[i] / dmax(1.0, c.ywt[i]);
    const double sum = dnrm2(c.save1) / k.sqrtn;
    if (sum > k.eps / fabs(c.h)) c.h = copysign(k.eps / sum, c.h);
#pragma unroll
    for (int i = 0; i < SA; ++i) c.yh[1][i] = c.h * c.save2[i];
#pragma unroll
    for (int i = 0; i < SA; ++i) c.fac[i] = k.sqrt_uround;
    if (c.ntl_restart) c.rmax = 10.0;
    if (c.h == 0.0) {
      copy_yh0_to_y(c);
      finish(c, OUT_STEP_ZERO);
    } else {
      c.pc = PC_ATTEMPT;
    }
  }
  // ---- 2: after f(y_pred), after a corrector f, after the Jacobian
  if (wave_any(c.req == REQ_NONE && (c.pc == PC_PRED_F || c.pc == PC_JAC_DONE || c.pc == PC_CORR_F))) {
    if (at(c, PC_PRED_F)) {
      c.nfe++;
      if (c.evaljc || c.ier) {
        c.pc = PC_JAC_DONE;
        c.req = REQ_JAC;
      } else {
#pragma unroll
        for (int i = 0; i < SA; ++i) c.save1[i] = 0.0;
        c.pc = PC_CORR;
      }
    } else if (at(c, PC_JAC_DONE)) {
      if (c.ier) {
        c.pc = PC_FAIL_CONV;
      } else {
        c.convrg = false;
        c.rc = 1.0;
        c.jstepl = c.nstep;
#pragma unroll
        for (int i = 0; i < SA; ++i) c.save1[i] = 0.0;
        c.pc = PC_CORR;
      }
    } else if (at(c, PC_CORR_F)) {
      c.nfe++;
      c.pc = PC_CORR;
    }
  }
  // ---- 3: corrector iteration, label 130 (slatec/ddstp.f90:152-205)
  if (wave_any(at(c, PC_CORR)) && at(c, PC_CORR)) {
    const double d = cor(c, k);
    if (c.iter > 0) c.trend = dmax(0.9 * c.trend, d / c.d1);
    c.d1 = d;
    c.ctest = dmin(2.0 * c.trend, 1.0) * d;
    if (c.ctest <= k.eps) {
      c.pc = PC_ERRTEST;
    } else {
      c.iter++;
      if (c.iter < 3) {
        const double l0 = el_of(mc, 1, c.nq);
#pragma unroll
        for (int i = 0; i < SA; ++i) c.y[i] = c.yh[0][i] + l0 * c.save1[i];
        request_f(c, PC_CORR_F);
      } else if (c.convrg) {                           // stale Jacobian: refresh (label 110)
        c.evaljc = true;
        c.iter = 0;
        copy_yh0_to_y(c);
        request_f(c, PC_PRED_F);
      } else {
        c.pc = PC_FAIL_CONV;
      }
    }
  }
  // ---- 4: error test, accept, step/order selection, label 170 (:222-432)
  // A converged lane may wait here (it asks for nothing, so it re-enters on
  // the next pass unchanged) until gather_pct % of the lanes stepping in this
  // pass have arrived: the stage's code then runs once for all of them.  The
  // others always make progress, so the share is reached.
  const bool here4 = at(c, PC_ERRTEST);
  const int n4 = __popcll(__ballot(here4 ? 1 : 0));
  const int nact = __popcll(__ballot(1));
  if (n4 > 0 && n4 * 100 >= k.gather_pct * nact && here4) {
    c.convrg = true;
#pragma unroll
    for (int i = 0; i < SA; ++i) c.save2[i] = c.save1[i] / dmax(fabs(c.y[i]), c.ywt[i]);
    const double etest = over_tq(mc, dnrm2(c.save2), 2, c.nq);
    c.etest = etest;
    if (etest > k.eps) {
      c.fail_err = true;                               // -> stage R (:238-289)
      c.pc = PC_RETRACT;
    } else {
      // accepted step (slatec/ddstp.f90:291-300)
      c.nstep++;
#pragma unroll
      for (int j = 1; j <= MAXORD + 1; ++j) {
        if (j <= c.nq + 1) {
          const double e = el_of(mc, j, c.nq);
#pragma unroll
          for (int i = 0; i < SA; ++i) c.yh[j - 1][i] = c.yh[j - 1][i] + e * c.save1[i];
        }
      }
      copy_yh0_to_y(c);
      c.do_scale = false;
      c.rmax_after = false;
      c.after_accept = true;
      // step-size and order selection (slatec/ddstp.f90:360-432)
      if (c.jtask == 0 || c.jtask == 2) {
        const double rh = 1.0 / dmax(k.uround, 1.2 * nl_pow(etest / k.eps, mc.inv[c.nq + 1]));
        c.rh = rh;
        c.do_scale = rh > 1.0;
      } else if (c.nwait > 1) {
        c.nwait = c.nwait - 1;
        if (c.nwait == 1 && c.nq < k.maxord) {
#pragma unroll
          for (int i = 0; i < SA; ++i) c.yh[MAXORD][i] = c.save1[i];
        }
      } else {
        // The three candidates (order down, same, up) are independent: both
        // norms come from one call and the three powers from another.  A
        // candidate that does not apply (order 1 cannot go down, MAXORD not
        // up) is formed from whatever its vector holds and then not used.
        double dn[SA], up[SA];
        yh_col(c, c.nq, dn);
#pragma unroll
        for (int i = 0; i < SA; ++i) {
          const double w = dmax(fabs(c.y[i]), c.ywt[i]);
          dn[i] = dn[i] / w;
          up[i] = (c.save1[i] - c.yh[MAXORD][i]) / w;
        }
        const Norm2 nr = dnrm2_pair(dn, up);
        const double erdn = over_tq(mc, nr.a, 1, c.nq);
        const double erup = over_tq(mc, nr.b, 3, c.nq);
        const Pow3 pw = nl_pow3(erdn / k.eps, mc.inv[c.nq], etest / k.eps,
                                mc.inv[c.nq + 1], erup / k.eps, mc.inv[c.nq + 2]);
        const double rh1 = (c.nq != 1) ? 1.0 / dmax(k.uround, 1.3 * pw.a) : 0.0;
        const double rh2 = 1.0 / dmax(k.uround, 1.2 * pw.b);
        const double rh3 = (c.nq != k.maxord) ? 1.0 / dmax(k.uround, 1.4 * pw.c) : 0.0;
        double rh;
        bool change = true;
        if (rh1 > rh2 && rh1 >= rh3) {
          rh = rh1;
          if (rh <= 1.0) {
            change = false;
          } else {
            c.nq = c.nq - 1;
            c.rc = (c.rc * el_of(mc, 1, c.nq)) / el_of(mc, 1, c.nq + 1);
          }
        } else if (rh2 >= rh1 && rh2 >= rh3) {
          rh = rh2;
          if (rh <= 1.0) change = false;
        } else {
          rh = rh3;
          if (rh <= 1.0) {
            change = false;
          } else {
            const double e = el_of(mc, c.nq + 1, c.nq);
            const double den = (double)(c.nq + 1);
            const int dst = c.nq + 1;
            double newc[SA];
#pragma unroll
            for (int i = 0; i < SA; ++i) newc[i] = (c.save1[i] * e) / den;
#pragma unroll
            for (int j = 2; j <= MAXORD; ++j) {
#pragma unroll
              for (int i = 0; i < SA; ++i) c.yh[j][i] = (dst == j) ? newc[i] : c.yh[j][i];
            }
            c.nq = c.nq + 1;
            c.rc = (c.rc * el_of(mc, 1, c.nq)) / el_of(mc, 1, c.nq - 1);
          }
        }
        c.rh = rh;
        c.do_scale = change;
        c.rmax_after = change;
        c.nwait = c.nq + 2;
      }
      c.pc = PC_SCALE;
    }
  }
  // ---- 5: corrector failure, label 160 (slatec/ddstp.f90:206-217)
  if (wave_any(at(c, PC_FAIL_CONV)) && at(c, PC_FAIL_CONV)) {
    c.fail_err = false;
    c.pc = PC_RETRACT;
  }
  // ---- R: retract the prediction, then the failure's step-size choice
  if (wave_any(at(c, PC_RETRACT)) && at(c, PC_RETRACT)) {
    c.t = c.told;
    psc<false>(c.nq, c.yh);
    c.after_accept = false;
    c.rmax_after = false;
    if (!c.fail_err) {                                 // label 160
      c.nwait = c.nq + 2;
      if (c.jtask != 0 && c.jtask != 2) c.rmax = 2.0;
      const double rh = (c.iter == 0) ? 0.3 : 0.9 * nl_pow(k.eps / c.ctest, 0.2);
      if (rh * c.h == 0.0) {
        copy_yh0_to_y(c);
        finish(c, OUT_STEP_ZERO);
      } else {
        c.rh = rh;
        c.do_scale = true;
        c.pc = PC_SCALE;
      }
    } else {                                           // error test failed (:238-289)
      c.nfail++;
      if (c.nfail < 3 || c.nq == 1) {
        if (c.jtask != 0 && c.jtask != 2) c.rmax = 2.0;
        const double rh2 = 1.0 / (1.2 * nl_pow(c.etest / k.eps, mc.inv[c.nq + 1]));
        double rh = rh2;
        if (c.nq > 1) {
          double col[SA];
          yh_col(c, c.nq, col);
#pragma unroll
          for (int i = 0; i < SA; ++i) c.save2[i] = col[i] / dmax(fabs(c.y[i]), c.ywt[i]);
          const double erdn = over_tq(mc, dnrm2(c.save2), 1, c.nq);
          const double rh1 = 1.0 / dmax(1.0, 1.3 * nl_pow(erdn / k.eps, mc.inv[c.nq]));
          if (rh2 < rh1) {
            c.nq = c.nq - 1;
            c.rc = (c.rc * el_of(mc, 1, c.nq)) / el_of(mc, 1, c.nq + 1);
            rh = rh1;
          }
        }
        c.nwait = c.nq + 2;
        if (rh * c.h == 0.0) {
          copy_yh0_to_y(c);
          finish(c, OUT_STEP_ZERO);
        } else {
          c.rh = rh;
          c.do_scale = true;
          c.pc = PC_SCALE;
        }
      } else {
        c.nfail = 0;                                   // restart at order 1 (:275-288)
        c.jtask = 2;
        copy_yh0_to_y(c);
        ntl_head(c);
        c.ntl_restart = true;
        request_f(c, PC_NTL_F);
      }
    }
  }
  // ---- S: pending DDSCL, then the next attempt or DDRIV3's label 470
  if (wave_any(at(c, PC_SCALE)) && at(c, PC_SCALE)) {
    if (c.do_scale) scl(c, c.rh, k);
    if (c.rmax_after) c.rmax = 10.0;
    if (!c.after_accept) {
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
  // ---- 6: DDRIV3 label 260: weights and guards, DDSTP entry (slatec/ddriv3.f90:1292-1351)
  if (wave_any(at(c, PC_260)) && at(c, PC_260)) {
#pragma unroll
    for (int i = 0; i < SA; ++i) c.ywt[i] = dmax(k.ewt, fabs(c.y[i]));
    // |y_i / YWT_i| <= 1, so SUM = max(1, ||y/YWT|| / sqrt(N)) stays below 2
    // and EPS < SUM * UROUND cannot hold for EPS >= 2 * UROUND; the norm is
    // formed only when it can decide (its SAVE2 is dead: the next f overwrites it).
    bool eps_fail = false;
    if (k.eps < 2.0 * k.uround) {
      double v[S];
#pragma unroll
      for (int sp = 0; sp < S; ++sp) {
        if (kSp.act[sp] >= 0) {
          v[sp] = c.y[kSp.act[sp]] / c.ywt[kSp.act[sp]];
        } else {
          const double yv = c.yi[kSp.islot[sp]];
          v[sp] = yv / dmax(k.ewt, fabs(yv));
        }
      }
      double sum = dnrm2_all(v) / k.sqrtn;
      sum = dmax(1.0, sum);
      eps_fail = k.eps < sum * k.uround;
    }
    if (eps_fail) {
      copy_yh0_to_y(c);
      finish(c, OUT_EPS);
    } else if (c.nstep == k.mxstep) {
      copy_yh0_to_y(c);
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
  // ---- 7: attempt, labels 100/110 (slatec/ddstp.f90:107-118)
  if (wave_any(at(c, PC_ATTEMPT)) && at(c, PC_ATTEMPT)) {
    c.ntry++;
    if (c.ntry > 50) {
      finish(c, OUT_REPEATED_FAIL);
    } else {
      c.natt++;
      c.t = c.t + c.h;
      psc<true>(c.nq, c.yh);
      c.evaljc = (fabs(c.rc - 1.0) > 0.3) || (c.nstep >= c.jstepl + 10);
      c.iter = 0;
      copy_yh0_to_y(c);
      request_f(c, PC_PRED_F);
    }
  }
}

// DDPST, MITER = 2 (slatec/ddpst.f90:39-114,142-143) for the lanes with
// `mine` set: finite-difference Jacobian with adaptive increments FAC,
// P = I - h*l0*J and its LU.  The column loop is unrolled: with a static
// column index the gathers of y_j, YWT_j, FAC_j and the scatter of the column
// into P are plain register moves instead of select chains over all nine
// columns (measured: 11-18 % less time per step than one shared loop body,
// despite nine RHS copies).
NRG_DI void jac_batch(Cell &c, bool mine, const BdfConst &k, const BdfCoef &mc, const double *kl)
{
  if (mine) {
    c.nje++;
    c.ier = false;
  }
  const double l0 = mine ? el_of(mc, 1, c.nq) : 0.0;
#pragma unroll
  for (int j = 0; j < SA; ++j) {
    double ywj = 0.0, yj = 0.0, fj = 0.0, s2j = 0.0, yh2j = 0.0;
#pragma unroll
    for (int q = 0; q < SA; ++q) {
      const bool hit = (q == j);
      ywj = hit ? opaque(c.ywt[q]) : ywj;
      yj = hit ? opaque(c.y[q]) : yj;
      fj = hit ? opaque(c.fac[q]) : fj;
      s2j = hit ? opaque(c.save2[q]) : s2j;
      yh2j = hit ? opaque(c.yh[2][q]) : yh2j;
    }
    double f1[SA];
    if (mine) {
      const double ys = dmax(fabs(ywj), fabs(yj));
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
      dy = (c.nq == 1) ? copysign(dy, s2j) : copysign(dy, yh2j);
      dy = (yj + dy) - yj;
      const double yp = yj + dy;
#pragma unroll
      for (int q = 0; q < SA; ++q) c.y[q] = (q == j) ? yp : c.y[q];
      rhs(kl, c.y, f1);
#pragma unroll
      for (int q = 0; q < SA; ++q) c.y[q] = (q == j) ? yj : c.y[q];
      const double factor = ((-l0) * c.h) / dy;
      double col[SA];
#pragma unroll
      for (int i = 0; i < SA; ++i) col[i] = (f1[i] - c.save2[i]) * factor;
      double diff = fabs(c.save2[0] - f1[0]);
      double s2m = c.save2[0], s1m = f1[0];
#pragma unroll
      for (int i = 1; i < SA; ++i) {
        const double di = fabs(c.save2[i] - f1[i]);
        if (di > diff) {
          diff = di;
          s2m = c.save2[i];
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
#pragma unroll
      for (int q = 0; q < SA; ++q) {
        const bool hit = (q == j);
        c.fac[q] = hit ? fj : c.fac[q];
#pragma unroll
        for (int i = 0; i < SA; ++i) c.P[q][i] = hit ? col[i] : c.P[q][i];
      }
    }
  }
  if (mine) {
    c.nfe += S;                                        // DDPST counts N evaluations
#pragma unroll
    for (int i = 0; i < SA; ++i) c.P[i][i] = c.P[i][i] + 1.0;
  }
  // DGEFA for the lanes of the batch (the pivot ballots inside see only them)
  if (mine) {
    if (gefa(c.P, c.ipvt) != 0) c.ier = true;
  }
}

// Fast mode (NRG_JAC_ANALYTIC): the iteration matrix P = I - h*l0*J with the
// exact J = d(omega)/dC of the law of mass action at the cell's fixed rate
// constants and [M] (the third-body concentration is frozen per cell, so it
// has no derivative), as DDPST forms it for a user Jacobian (MITER = 1).  No
// extra right-hand sides are evaluated; the step sequence therefore differs
// from the finite-difference (SLATEC MITER = 2) parity mode.
NRG_DI void jac_analytic(Cell &c, bool mine, const BdfCoef &mc, const double *kl)
{
  if (!mine) return;
  c.nje++;
  c.ier = false;
  const double fac = (-el_of(mc, 1, c.nq)) * c.h;
#pragma unroll
  for (int q = 0; q < SA; ++q)
#pragma unroll
    for (int i = 0; i < SA; ++i) c.P[q][i] = 0.0;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const double m = kMSlot.v[r] >= 0 ? rec_m(kl, kMSlot.v[r]) : 0.0;
#pragma unroll
    for (int side = 0; side < 2; ++side) {
      const int n = side == 0 ? topo::nl[r] : topo::nr[r];
      const double k = side == 0 ? rec_kf(kl, r) : -rec_kr(kl, r);
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        const int sa = side == 0 ? topo::left[r][a] : topo::right[r][a];
        if (a >= n || sa == S) continue;
        // d/dC_sa of k * prod_terms: the product of the other terms
        double d = k;
#pragma unroll
        for (int b = 0; b < 3; ++b) {
          const int sb = side == 0 ? topo::left[r][b] : topo::right[r][b];
          if (b < n && b != a) d = d * (sb == S ? m : c.y[act_of(sb)]);
        }
        const double fd = fac * d;
#pragma unroll
        for (int i = 0; i < SA; ++i) {
          const int nu = nu_of(r, kSp.full[i]);
          if (nu != 0) c.P[act_of(sa)][i] = c.P[act_of(sa)][i] + (double)nu * fd;
        }
      }
    }
  }
#pragma unroll
  for (int i = 0; i < SA; ++i) c.P[i][i] = c.P[i][i] + 1.0;
  if (gefa(c.P, c.ipvt) != 0) c.ier = true;
}

}  // namespace lane
}  // namespace nrg
