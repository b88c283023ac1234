// chem_device.h -- thermochemistry, rate constants and mass action of the
// gfx950 chemistry step, one cell per lane (the integrators: bdf_group.h, bdf_lane.h).
//
// The mechanism's numeric coefficients are one LDS copy per block.  Every
// register-array index is a compile-time constant after unrolling.  Arithmetic
// follows the reference operation by operation (this TU is built with
// -ffp-contract=off), so results agree with NRG's Fortran step to the rounding
// of the transcendental functions.
//
// Reference: computing_module/src/current_build/chemical_kinetics_solver.f90
// (rates :360-493, RHS :495-540, cell step :228-346).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <utility>

// the reaction topology these kernels are built for (one build per topology)
#ifndef NRG_TOPOLOGY_HEADER
#define NRG_TOPOLOGY_HEADER "topology_keromnes.h"
#endif
#include NRG_TOPOLOGY_HEADER

#define NRG_DI __device__ __forceinline__

namespace nrg {

constexpr int S = topo::S;
constexpr int R = topo::R;
constexpr int MAXORD = 5;
constexpr int WAVE = 64;

constexpr double R_GAS_J = 8.31446261815324;   // package_library/src/global_data.f90:36
constexpr double T_REF = 298.15;               // :38
constexpr double T_CEIL = 6000.0;              // :44

// Mechanism coefficients, staged once per block in LDS.  Quotients by
// constants that the reference evaluates per call (a_i/i, (-E)/R_u, P_atm/R_u)
// are precomputed on the host with the same single IEEE division.
struct MechCoef {
  double A[R], beta[R], A_low[R], beta_low[R];
  double mE_R[R], mElow_R[R];    // (-E_act)/R_u, (-E_act_low)/R_u
  double troe[4][R];             // alpha, T***, T*, T**
  double one_m_alpha[R];         // 1 - alpha
  double eff[R][S];              // enhanced efficiencies
  double a[S][2][7];             // NASA-7 x R_u; [s][set][i], set 1 = T >= 1000 K
  double hdiv[S][2][5];          // a5/5, a4/4, a3/3, a2/2, a1/1
  double sdiv[S][2][3];          // a5/4, a4/3, a3/2
  double W[S];                   // molar masses
  double h_ref[S];               // h_s(T_ref), T_ref = 298.15 K
  double el[MAXORD][MAXORD + 1]; // el[nq-1][j-1] = EL(j, nq)   (slatec/ddcst.f90, MINT = 2)
  double tq[MAXORD][3];          // tq[nq-1][k-1] = TQ(k, nq)
  double patm_r;                 // P_atm / R_u
  double lnA[R], lnA_low[R];     // ln A, ln A_low (the explicit-rate screen's exponents)
  double ln_patm_r;              // ln(P_atm / R_u)
};

// The part of the mechanism the integrator kernel reads (one LDS copy per block).
struct BdfCoef {
  double el[MAXORD][MAXORD + 1];
  double den[3][MAXORD];         // den[k-1][nq-1] = TQ(k, nq) * sqrt(N)
  double rsqrtn, rden2[MAXORD];  // what div_by takes of sqrt(N) and of den[1]
  double inv[8];                 // 1 / n
  double W[S];
  double h_ref[S];
};

// Integrator constants of one call (reference literals + D1MACH-derived values).
struct BdfConst {
  double eps, ewt, hmax, uround, sqrtn, sqrt_uround;
  double tiny;                   // weighted components below it take DNRM2's phases one by one
  double br, bl, bp, facmin;     // u**.875, u**.75, u**-.15, u**.78 (slatec/ddpst.f90:54-57)
  double t_gate;
  int mxstep, maxord;
  int gather_pct;
  int refill_idle;               // persistent form: idle lanes (of 64) that trigger a refill
};

NRG_DI double dmax(double a, double b) { return (a >= b) ? a : b; }
NRG_DI double dmin(double a, double b) { return (a <= b) ? a : b; }

// Math for the rate-constant kernel, where inlining is the better trade.
// Cases whose IEEE result is exact skip the expansion: pow(x, +-0) = 1,
// pow(x, 1) = x, exp(+-0) = 1; exp(x) rounds to 1 for |x| < 2^-54 and to +0
// below -746 (under half the least subnormal).  The mechanism's zero
// temperature exponents and activation energies and its disabled Troe terms
// (T*** = 0, T* = T** = 1e30) hit them for every cell alike.
struct InlineMath {
  static NRG_DI double pow_(double x, double y)
  {
    if (y == 0.0) return 1.0;
    if (y == 1.0) return x;
    return pow(x, y);
  }
  static NRG_DI double exp_(double x)
  {
    if (fabs(x) < 0x1p-60) return 1.0;
    if (x < -746.0) return 0.0;
    return exp(x);
  }
  static NRG_DI double log_(double x) { return log(x); }
  static NRG_DI double log10_(double x) { return log10(x); }
  // x / T and x / R_u, as the reference divides
  static NRG_DI double over_T(double x, double T) { return x / T; }
  static NRG_DI double over_R(double x) { return x / R_GAS_J; }
  // k_r = k_f / K_c with K_c = exp(lnKp) * x**d_nu (d_nu = 0: pow(x, 0) = 1 exactly)
  static NRG_DI double reverse_(double kf, double lnKp, double x, double d_nu)
  {
    const double Kp = exp_(lnKp);
    const double Kc = (d_nu == 0.0) ? Kp * 1.0 : Kp * pow_(x, d_nu);
    return kf / Kc;
  }
  // A T^b exp(mE_R / T), in the reference's order of operations
  static NRG_DI double arrh_(double A, double b, double mE_R, double T)
  {
    return (A * pow_(T, b)) * exp_(mE_R / T);
  }
};

// Cheaper transcendentals for estimates that no parity path depends on (the
// surrogate gate's rate-consistency test): x^y as exp(y ln x) on positive x,
// so ln T and ln(P_atm/(R_u T)) are computed once per cell and shared by every
// reaction instead of a full pow per rate constant, and an Arrhenius term as
// one exp.  Relative error ~1e-15 for the exponents of a mechanism
// (|y ln x| < 50).
struct EstimateMath {
  static NRG_DI double pow_(double x, double y)
  {
    if (y == 0.0) return 1.0;
    if (y == 1.0) return x;
    if (y == -1.0) return 1.0 / x;
    return exp(y * log(x));
  }
  static NRG_DI double exp_(double x) { return exp(x); }
  static NRG_DI double log_(double x) { return log(x); }
  static NRG_DI double log10_(double x) { return log10(x); }
  // divisions by T and R_u as products with one reciprocal per cell (1/T is
  // the same expression at every call, formed once) and a constant
  static NRG_DI double over_T(double x, double T) { return x * (1.0 / T); }
  static NRG_DI double over_R(double x) { return x * (1.0 / R_GAS_J); }
  // k_f / K_c as k_f exp(-lnKp) x**(-d_nu): no division
  static NRG_DI double reverse_(double kf, double lnKp, double x, double d_nu)
  {
    return kf * exp(-lnKp) * ((d_nu == 0.0) ? 1.0 : pow_(x, -d_nu));
  }
  static NRG_DI double arrh_(double A, double b, double mE_R, double T)
  {
    return A * exp(b * log(T) + mE_R * (1.0 / T));
  }
};

// A value pinned in a VGPR.  Select chains over register arrays go through it,
// so the optimiser cannot turn "select between loads" into one load through a
// selected address (which would keep the whole array in private memory).
NRG_DI double opaque(double x)
{
  asm("" : "+v"(x));
  return x;
}

// ---------------------------------------------------------------------------
// Compile-time facts about the topology
// ---------------------------------------------------------------------------
// Does fun (chemical_kinetics_solver.f90:509-527) multiply by [M] for reaction r?
constexpr bool m_in_rhs(int r)
{
  for (int c = 0; c < 3; ++c)
    if (c < topo::nl[r] && topo::left[r][c] == S) return true;
  for (int c = 0; c < 3; ++c)
    if (c < topo::nr[r] && topo::right[r][c] == S) return true;
  return false;
}
constexpr int m_slot(int r)
{
  int k = 0;
  for (int q = 0; q < r; ++q) k += m_in_rhs(q) ? 1 : 0;
  return m_in_rhs(r) ? k : -1;
}
struct MSlotTable {
  int v[R];
};
constexpr MSlotTable make_mslot()
{
  MSlotTable t{};
  for (int r = 0; r < R; ++r) t.v[r] = m_slot(r);
  return t;
}
constexpr MSlotTable kMSlot = make_mslot();   // [M] register slot of reaction r, or -1
constexpr int count_m()
{
  int k = 0;
  for (int r = 0; r < R; ++r) k += m_in_rhs(r) ? 1 : 0;
  return k;
}
constexpr int NM = count_m() > 0 ? count_m() : 1;
// [M] needed at setup: third-body and fall-off reactions.
constexpr bool uses_m(int r)
{
  return topo::rtype[r] == 1 || topo::rtype[r] == 2 || topo::rtype[r] == 3 ||
         topo::rtype[r] == 6 || topo::rtype[r] == 7;
}

// Cell record: what rates_kernel hands the integrator for integrated cell
// t of a chunk of nrec positions, as pairs of doubles (16 bytes: one lane's
// share of a direct HBM -> LDS load, global_load_lds_dwordx4).
//   pairs [0, R)             (k_f(r), k_r(r))
//   pairs [REC_M, REC_C)     [M] slots 2j, 2j+1
//   pairs [REC_C, REC_PAIRS) C_s (mol/m^3) at slot s, then the cell's inner index
//                            (its bits) at slot S
// In HBM pair p of record t sits at rec[2 (p nrec + t)] (pair-major: the
// rate kernel's waves write 1 KiB runs); the integrator keeps a cell's copy in
// LDS, pair p at doubles 2p, 2p+1 of the cell's slice.
constexpr int REC_M = R;
constexpr int REC_C = REC_M + (NM + 1) / 2;
constexpr int REC_PAIRS = REC_C + (S + 2) / 2;
constexpr int REC_CELL = S;
// Offset (doubles) of slot j of the pairs starting at pair p0, position 0.
NRG_DI long long rec_slot(int p0, int j, long long nrec)
{
  return 2 * ((long long)(p0 + j / 2) * nrec) + (j & 1);
}
// Species that no reaction consumes or produces (N2 in H2-air) enter only
// through the third-body concentrations, which are fixed per cell.  For them
// f_s = 0 and no f_i depends on y_s, so under DDRIV3 every correction, every
// YH column beyond the first and every norm term of theirs is an exact zero
// (Lawson's norm passes zeros through unchanged) and their row and column of
// P are those of the identity (the LU and the solves of the other species do
// not see them).  The integrator state therefore holds the SA active species;
// an inert species keeps its initial concentration.
constexpr bool reacts(int s)
{
  for (int r = 0; r < R; ++r)
    for (int c = 0; c < 3; ++c)
      if ((c < topo::nl[r] && topo::left[r][c] == s) || (c < topo::nr[r] && topo::right[r][c] == s))
        return true;
  return false;
}
constexpr int count_active()
{
  int n = 0;
  for (int s = 0; s < S; ++s) n += reacts(s) ? 1 : 0;
  return n;
}
constexpr int SA = count_active();
constexpr int NI = S - SA;
struct SpeciesMap {
  int act[S];                    // active slot of species s, or -1
  int full[SA];                  // species of active slot a
  int islot[S];                  // inert slot of species s, or -1
  int inert[NI > 0 ? NI : 1];    // species of inert slot i
};
constexpr SpeciesMap make_species_map()
{
  SpeciesMap m{};
  int a = 0, i = 0;
  for (int s = 0; s < S; ++s) {
    m.act[s] = -1;
    m.islot[s] = -1;
    if (reacts(s)) {
      m.act[s] = a;
      m.full[a++] = s;
    } else {
      m.islot[s] = i;
      m.inert[i++] = s;
    }
  }
  return m;
}
constexpr SpeciesMap kSp = make_species_map();
constexpr int act_of(int s) { return (s >= 0 && s < S && kSp.act[s] >= 0) ? kSp.act[s] : 0; }

// ---------------------------------------------------------------------------
// NASA-7 thermochemistry (thermophysical_properties_class.f90:225-300)
// ---------------------------------------------------------------------------
NRG_DI double clip_t(double T) { return dmin(T, T_CEIL); }

template <class M = InlineMath>
NRG_DI double h_molar(const MechCoef &mc, double T, int s)
{
  const double temp = clip_t(T);
  const int set = (temp >= 1000.0) ? 1 : 0;
  const double *d = mc.hdiv[s][set];
  double hs = d[0];
  hs = hs * temp + d[1];
  hs = hs * temp + d[2];
  hs = hs * temp + d[3];
  hs = hs * temp + d[4];
  hs = hs + M::over_T(mc.a[s][set][5], temp);
  return hs * temp;
}

template <class M = InlineMath>
NRG_DI double s_molar(const MechCoef &mc, double T, int s)
{
  const double temp = clip_t(T);
  const int set = (temp >= 1000.0) ? 1 : 0;
  const double *d = mc.sdiv[s][set];
  const double *a = mc.a[s][set];
  double sm = d[0];
  sm = sm * temp + d[1];
  sm = sm * temp + d[2];
  sm = sm * temp + a[1];
  return (sm * temp + a[6]) + a[0] * M::log_(temp);
}

NRG_DI double cp_molar(const MechCoef &mc, double T, int s)
{
  const double temp = clip_t(T);
  const double *a = mc.a[s][(temp >= 1000.0) ? 1 : 0];
  double cp = a[4];
  cp = cp * temp + a[3];
  cp = cp * temp + a[2];
  cp = cp * temp + a[1];
  cp = cp * temp + a[0];
  return cp;
}

NRG_DI double e_molar(const MechCoef &mc, double T, int s)
{
  return h_molar(mc, T, s) - R_GAS_J * T;   // unclipped T (:298)
}

// ---------------------------------------------------------------------------
// Rate constants (chemical_kinetics_solver.f90:360-493) of one cell, written
// into its cell record (below): k_f(r) and k_r(r) as pair r, and [M] of the
// reactions whose RHS term uses it (:235-248) in the [M] pairs.
// ---------------------------------------------------------------------------
// Reactions [R0, R1) only (their k_f, k_r and [M] slots).
// k_f, k_r and [M] of reaction r at T (already capped at 1e4 K), from the
// species' entropies sv and enthalpies hv at T (:394-485).
template <class M>
NRG_DI void reaction_k(const MechCoef &mc, double T, const double (&sv)[S], const double (&hv)[S],
                       const double (&C)[S], int r, double &kf_out, double &kr_out, double &m_out)
{
  double m = 0.0;
  if (uses_m(r)) {
#pragma unroll
    for (int s = 0; s < S; ++s) m = m + C[s] * mc.eff[r][s];
  }
  double d_s = 0.0, d_h = 0.0;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const int sp = topo::right[r][c];
    if (c < topo::nr[r] && sp != S) {
      d_s = d_s + sv[sp < S ? sp : 0];
      d_h = d_h + hv[sp < S ? sp : 0];
    }
  }
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const int sp = topo::left[r][c];
    if (c < topo::nl[r] && sp != S) {
      d_s = d_s - sv[sp < S ? sp : 0];
      d_h = d_h - hv[sp < S ? sp : 0];
    }
  }
  const double d_nu = (double)(topo::nr[r] - topo::nl[r]);
  const int rt = topo::rtype[r];
  double kf = 0.0, kr = 0.0;
  if (rt == 0 || rt == 1 || rt == 5 || rt == 6) {
    kf = M::arrh_(mc.A[r], mc.beta[r], mc.mE_R[r], T);
  } else if (rt == 2 || rt == 7) {
    const double k0 = M::arrh_(mc.A_low[r], mc.beta_low[r], mc.mElow_R[r], T);
    const double kinf = M::arrh_(mc.A[r], mc.beta[r], mc.mE_R[r], T);
    const double pr = (k0 * m) / kinf;
    kf = kinf * (pr / (1.0 + pr));
  } else if (rt == 3) {
    // (A T^b) exp(-E/RT): the product the reference forms after its two exps
    const double k0 = M::arrh_(mc.A_low[r], mc.beta_low[r], mc.mElow_R[r], T);
    const double kinf = M::arrh_(mc.A[r], mc.beta[r], mc.mE_R[r], T);
    const double pr = (k0 * m) / kinf;
    const double fcent = (mc.one_m_alpha[r] * M::exp_(-(T / mc.troe[1][r])) +
                          mc.troe[0][r] * M::exp_(-(T / mc.troe[2][r]))) +
                         M::exp_(-M::over_T(mc.troe[3][r], T));
    const double lf = M::log10_(fcent);
    const double c = -0.4 - 0.67 * lf;
    const double n = 0.75 - 1.27 * lf;
    const double d = 0.14;
    double blend;
    if (pr != 0.0) {
      const double lp = M::log10_(pr);
      const double x = (lp + c) / (n - d * (lp + c));
      blend = M::pow_(fcent, 1.0 / (1.0 + x * x));
    } else {
      blend = M::pow_(fcent, -1.0 / d);
    }
    kf = (kinf * (pr / (1.0 + pr))) * blend;
  }
  if (rt == 0 || rt == 1 || rt == 2 || rt == 3) {
    // K_c = K_p * ((P_atm/R_u)/T)**d_nu, K_p = exp(dS/R - dH/(R T))
    kr = M::reverse_(kf, M::over_R(d_s) - M::over_T(M::over_R(d_h), T), M::over_T(mc.patm_r, T), d_nu);
  }
  kf_out = kf;
  kr_out = kr;
  m_out = m;
}

template <class M, int R0 = 0, int R1 = R>
NRG_DI void rate_constants(const MechCoef &mc, double Tin, const double (&C)[S], double *rec,
                           long long nrec)
{
  const double T = dmin(Tin, 10000.0);
  double sv[S], hv[S];
#pragma unroll
  for (int c = 0; c < S; ++c) {
    sv[c] = s_molar<M>(mc, T, c);
    hv[c] = h_molar(mc, T, c);
  }
#pragma unroll
  for (int r = R0; r < R1; ++r) {
    double kf, kr, m;
    reaction_k<M>(mc, T, sv, hv, C, r, kf, kr, m);
    if (uses_m(r) && kMSlot.v[r] >= 0) rec[rec_slot(REC_M, kMSlot.v[r], nrec)] = m;
    *reinterpret_cast<double2 *>(rec + rec_slot(r, 0, nrec)) = make_double2(kf, kr);
  }
}

// ---------------------------------------------------------------------------
// Mass-action right-hand side, the accumulation order of fun (:507-536), on
// the active species (an inert species' f is zero).
// ---------------------------------------------------------------------------
// Mass-action contribution of reaction r (:520-535) with rate constants kf,
// kr and third-body concentration m.
NRG_DI void rhs_reaction(int r, double kf, double kr, double m, const double (&Z)[SA], double (&Zd)[SA])
{
  double fwd = kf;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const int sp = topo::left[r][c];
    if (c < topo::nl[r]) fwd = fwd * ((sp == S) ? m : Z[act_of(sp)]);
  }
  double rev = kr;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const int sp = topo::right[r][c];
    if (c < topo::nr[r]) rev = rev * ((sp == S) ? m : Z[act_of(sp)]);
  }
#pragma unroll
  for (int a = 0; a < SA; ++a) {
    const int s = kSp.full[a];
#pragma unroll
    for (int c = 0; c < 3; ++c)
      if (c < topo::nl[r] && topo::left[r][c] == s) Zd[a] = (Zd[a] - fwd) + rev;
#pragma unroll
    for (int c = 0; c < 3; ++c)
      if (c < topo::nr[r] && topo::right[r][c] == s) Zd[a] = (Zd[a] - rev) + fwd;
  }
}

// Species (bit s = species s) on one side of reaction r, third body left out.
constexpr unsigned side_mask(int r, int side)
{
  unsigned m = 0;
  for (int c = 0; c < 3; ++c) {
    const int sp = side ? topo::right[r][c] : topo::left[r][c];
    const int n = side ? topo::nr[r] : topo::nl[r];
    if (c < n && sp >= 0 && sp < S) m |= 1u << sp;
  }
  return m;
}
constexpr bool has_reverse(int r)
{
  return topo::rtype[r] == 0 || topo::rtype[r] == 1 || topo::rtype[r] == 2 || topo::rtype[r] == 3;
}
static_assert(S <= 32, "species masks are 32-bit");

// The part of omega(C, T) of the active species that reactions [R0, R1)
// contribute, with the rate constants computed one reaction at a time (no
// array of all k_f, k_r is held).  A reaction whose left side holds a species
// the cell does not contain has a zero forward rate, and likewise for the
// right side and the reverse rate; when both are zero for every lane of the
// wave, the reaction adds nothing and is skipped (fresh gas, whose radicals
// are exact zeros, needs a handful of the reactions).
template <class Mth, int R0 = 0, int R1 = R>
NRG_DI void explicit_rates(const MechCoef &mc, double Tin, const double (&C)[S], double (&Zd)[SA])
{
  const double T = dmin(Tin, 10000.0);
  double sv[S], hv[S], Z[SA];
  unsigned absent = 0;
#pragma unroll
  for (int c = 0; c < S; ++c) {
    sv[c] = s_molar<Mth>(mc, T, c);
    hv[c] = h_molar<Mth>(mc, T, c);
    absent |= (C[c] == 0.0) ? 1u << c : 0u;
  }
#pragma unroll
  for (int i = 0; i < SA; ++i) {
    Z[i] = C[kSp.full[i]];
    Zd[i] = 0.0;
  }
#pragma unroll
  for (int r = R0; r < R1; ++r) {
    const bool fwd = (absent & side_mask(r, 0)) == 0;
    const bool rev = has_reverse(r) && (absent & side_mask(r, 1)) == 0;
    if (__any((fwd || rev) ? 1 : 0)) {
      double kf, kr, m;
      reaction_k<Mth>(mc, T, sv, hv, C, r, kf, kr, m);
      rhs_reaction(r, kf, kr, m, Z, Zd);
    }
  }
}

}  // namespace nrg
