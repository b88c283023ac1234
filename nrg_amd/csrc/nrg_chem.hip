// nrg_chem.hip -- kernels and entry points of the gfx950 chemistry step for
// one reaction topology.
//
// Entry points are declared in include/nrg_chem.h; each replaces a piece of
// NRG's chemical_kinetics_solver (computing_module/src/current_build/
// chemical_kinetics_solver.f90) or of the split-step closure the flow solvers
// apply after it.  All device work runs on the handle's stream.
//
// The kernels unroll the mechanism's reaction lists at compile time, so this
// file is built once per topology (the Makefile sets NRG_TOPOLOGY_HEADER,
// NRG_TOPO_NS, NRG_TOPO_OPS_FN, NRG_TOPO_NAME and NRG_TOPO_PRIMARY).  Each build
// lives in its own namespace and hands its entry points to the C-ABI
// (nrg_api.cpp) as a table (topo_api.h); nrg_chem_create picks the table whose
// topology the mechanism has.
//
// NRG_PART splits a build into objects: 1 = everything but the integrator
// kernels' bodies, 2 = the lane-group integrator alone, 3 = the one-cell-per-lane
// integrator alone (so that they can be compiled with options of their own);
// 0 (default) = all in one.  With NRG_PART 2, NRG_BDF_JAC selects the kernel's
// instantiation: 1 = finite-difference Jacobian, 2 = analytic, unset = both.
#ifndef NRG_PART
#define NRG_PART 0
#endif
#ifndef NRG_TOPO_NS
#define NRG_TOPO_NS nrg_topo_keromnes
#define NRG_TOPO_OPS_FN nrg_topo_ops_keromnes
#define NRG_TOPO_NAME "KEROMNES"
#define NRG_TOPO_PRIMARY 1
#endif
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <new>
#include <vector>

#include "../../include/nrg_chem.h"
#include "../../include/nrg_low_mach.h"
#include "../../include/nrg_surrogate.h"
#include "bdf_group.h"
#include "bdf_lane.h"
#include "chem_device.h"
#include "mlp_internal.h"
#include "nrg_common.h"
#include "topo_api.h"

using namespace nrg;

// nothing of this build is exported: the C-ABI reaches it through its table
#pragma GCC visibility push(hidden)
namespace NRG_TOPO_NS {

// This build's handle; the C-ABI sees it only as an opaque pointer.
struct nrg_chem_handle;
typedef nrg_chem_handle nrg_chem_t;
void nrg_chem_destroy(nrg_chem_t *h);
int nrg_chem_table_step_dev(nrg_chem_t *h, const nrg_grid *grid, double dt, const double *T,
                            const double *p, const double *rho, const double *const *Y,
                            const int8_t *bc, double *const *Y_prod, double *const *Y_prod2,
                            double *E_f_prod, int32_t *cell_status, nrg_chem_stats *stats);

namespace kern {

// Field addressing of one call (Fortran column-major with ghost layers).
struct GridIdx {
  int lo0, lo1, lo2;
  int nx, ny;                 // allocated extents in dims 1, 2
  int ilo0, ilo1, ilo2;       // inner lower bounds
  int ix, iy, iz;             // inner extents
  int idx32;                  // 1: inner indices and allocation offsets below 2^31 (32-bit division)
  long long ninner;
  long long pad0, pad1;       // allocation offsets [pad0, pad1) holding every inner cell; pad0 % 64 == 0
};

// Is allocation offset p an inner cell (not a ghost)?
NRG_DI bool inner_at(const GridIdx &g, long long p)
{
  long long i, j, k;
  if (g.idx32) {
    const unsigned pu = (unsigned)p, nx = (unsigned)g.nx, ny = (unsigned)g.ny;
    const unsigned r = pu / nx;
    i = pu - r * nx;
    j = r % ny;
    k = r / ny;
  } else {
    const long long r = p / g.nx;
    i = p - r * g.nx;
    j = r % g.ny;
    k = r / g.ny;
  }
  return (unsigned long long)(i - (g.ilo0 - g.lo0)) < (unsigned long long)g.ix &&
         (unsigned long long)(j - (g.ilo1 - g.lo1)) < (unsigned long long)g.iy &&
         (unsigned long long)(k - (g.ilo2 - g.lo2)) < (unsigned long long)g.iz;
}

// The aligned walk: thread t of the launch takes allocation offset pad0 + t,
// from the 64-cell slice of the first inner cell to the last inner cell, and
// skips ghost cells.  With ghost layers a row of inner cells starts off a cache
// line; walking inner cells in order would make every wave touch one more line
// per field.  One offset per thread: a grid-stride loop here let the compiler
// hoist the LDS-staged mechanism into registers (closure 72 -> 169 VGPRs) and
// was slower for every kernel that uses it.
template <class F>
NRG_DI void at_inner_cell(const GridIdx &g, F &&f)
{
  const long long off = g.pad0 + (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (off < g.pad1 && inner_at(g, off)) f(off);
}

NRG_DI long long cell_offset(const GridIdx &g, long long q)
{
  long long i, j, kk;
  if (g.idx32) {
    const unsigned qu = (unsigned)q, ix = (unsigned)g.ix, iy = (unsigned)g.iy;
    const unsigned r = qu / ix;
    i = (long long)(qu - r * ix) + g.ilo0;
    j = (long long)(r % iy) + g.ilo1;
    kk = (long long)(r / iy) + g.ilo2;
  } else {
    i = q % g.ix + g.ilo0;
    j = (q / g.ix) % g.iy + g.ilo1;
    kk = q / ((long long)g.ix * g.iy) + g.ilo2;
  }
  return (i - g.lo0) + (long long)g.nx * ((j - g.lo1) + (long long)g.ny * (kk - g.lo2));
}

struct StepArgs {
  GridIdx g;
  double dt;
  BdfConst k;
  const MechCoef *mech;
  const double *T, *rho;
  const double *Y[S];
  const int8_t *bc;
  double *Yp[S], *Yp2[S];
  double *Efp;
  int32_t *status;
  int32_t *nstep, *nfe, *nje;          // optional per-cell work counters
  unsigned long long *acc;              // [16] work/status accumulators
  unsigned long long *queue;            // next unclaimed cell of the chunk (persistent form)
  int jac_pct;                          // run a Jacobian batch when >= this % of pending lanes want one
  const double *rates;                  // cell records of the chunk's positions (REC_PAIRS pairs each)
  double *rates_out;                    // same buffer, written by rates_kernel
  long long base, nchunk;               // this launch covers queue positions [base, base+nchunk)
  const int32_t *list;                  // NULL: position t is inner cell t; else inner cell list[t]
  int32_t *hist;                        // optional: each inner cell's work (hist_code), for ordering
  int cpw;                              // cells a wave of the integrator holds at a time
  // How many of the launch's positions are integrated: in stiffness order, whose
  // gated cells come last, from the npos positions and the gated ones among them;
  // else rates_kernel counts them in *live and gives them the records [0, *live).
  const unsigned long long *gated;
  unsigned long long *live;
  long long npos;
};

NRG_DI long long live_records(const StepArgs &a)
{
  if (!a.gated) return (long long)*a.live;
  const long long n = a.npos - (long long)*a.gated - a.base;
  return n < 0 ? 0 : n < a.nchunk ? n : a.nchunk;
}

// Inner cell (inner-loop order) at position base + t of the launch's queue.
// The 64-bit form alone: the integrator kernel's one call (at a refill) keeps
// its register allocation without the second path.
NRG_DI long long cell_offset_wide(const GridIdx &g, long long q)
{
  const long long i = q % g.ix + g.ilo0;
  const long long j = (q / g.ix) % g.iy + g.ilo1;
  const long long kk = q / ((long long)g.ix * g.iy) + g.ilo2;
  return (i - g.lo0) + (long long)g.nx * ((j - g.lo1) + (long long)g.ny * (kk - g.lo2));
}

// A store of the passes over all fields that HBM bounds; with STREAM, past the
// caches, which pays where such a pass touches more than the 256 MB memory-side
// cache holds before anything is read again (streams()).  Waves write whole
// 64-cell slices (a line written in parts costs more so: the table step with its
// gated cells' stores apart 142 us, together 127).
template <bool STREAM, class V, class W>
NRG_DI void put(V *p, W v)
{
  if (STREAM)
    __builtin_nontemporal_store((V)v, p);
  else
    *p = (V)v;
}

NRG_DI long long cell_of(const StepArgs &a, long long t)
{
  return a.list ? (long long)a.list[a.base + t] : a.base + t;
}

// Block-wide staging of the mechanism coefficients into LDS: each thread
// issues its loads (up to 4) before the first store, so a block waits for one
// round trip to memory instead of one per element it copies.
NRG_DI void stage_mech(MechCoef &dst, const MechCoef *src)
{
  const double *s = reinterpret_cast<const double *>(src);
  double *d = reinterpret_cast<double *>(&dst);
  constexpr int n = sizeof(MechCoef) / sizeof(double);
  constexpr int K = 4;
  const int stride = blockDim.x;
  for (int i0 = threadIdx.x; i0 < n; i0 += K * stride) {
    double v[K];
#pragma unroll
    for (int k = 0; k < K; ++k) v[k] = (i0 + k * stride < n) ? s[i0 + k * stride] : 0.0;
#pragma unroll
    for (int k = 0; k < K; ++k)
      if (i0 + k * stride < n) d[i0 + k * stride] = v[k];
  }
  __syncthreads();
}

NRG_DI void stage_bdf(BdfCoef &dst, const MechCoef *src, double sqrtn)
{
  for (int i = threadIdx.x; i < MAXORD * (MAXORD + 1); i += blockDim.x)
    (&dst.el[0][0])[i] = (&src->el[0][0])[i];
  for (int i = threadIdx.x; i < 3 * MAXORD; i += blockDim.x) {
    const double d = src->tq[i % MAXORD][i / MAXORD] * sqrtn;
    (&dst.den[0][0])[i] = d;
    if (i / MAXORD == 1) dst.rden2[i % MAXORD] = recip(d);
  }
  if (threadIdx.x == 0) dst.rsqrtn = recip(sqrtn);
  if (threadIdx.x < 8) dst.inv[threadIdx.x] = 1.0 / (double)(int)threadIdx.x;
  for (int i = threadIdx.x; i < S; i += blockDim.x) {
    dst.W[i] = src->W[i];
    dst.h_ref[i] = src->h_ref[i];
  }
  __syncthreads();
}

// What a step records of a cell for the next one's order: its steps and, above
// them, its right-hand sides (0 if gated).
constexpr int HIST_FE_SHIFT = 16, HIST_STEPS = (1 << HIST_FE_SHIFT) - 1;
NRG_DI int32_t hist_code(int nstep, int nfe) { return min(nstep, HIST_STEPS) | (min(nfe, 0x7fff) << HIST_FE_SHIFT); }

// accumulator slots
enum { ACC_INTEG = 0, ACC_NSTEP, ACC_NFE, ACC_NJE, ACC_NCORR, ACC_NATT, ACC_NSTEP_MAX, ACC_NFE_MAX,
       ACC_STATUS0,     // ACC_STATUS0 + NRG_CELL_* (8 slots)
       ACC_QUEUE0 = 16, // one queue head per chunk
       MAX_CHUNKS = 48,
       ACC_LIVE0 = ACC_QUEUE0 + MAX_CHUNKS,   // and one count of integrated cells
       ACC_SLOTS = ACC_LIVE0 + MAX_CHUNKS };

// Zero the work accumulators and the queue head (a kernel, so the launch
// sequence can be captured in a graph without memset nodes).
#if NRG_PART < 2
__global__ void reset_kernel(unsigned long long *acc, int n)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) acc[i] = 0ull;
}
#endif

// Load one cell and set it up (chemical_kinetics_solver.f90:228-265): the
// group's lanes copy cell record t (rates_kernel) from HBM to the cell's slice of
// LDS, all loads in one round trip.
NRG_DI void start_cell(const StepArgs &a, long long t, Cell &c, const Lane &ln)
{
  const double *src = a.rates + 2 * t;
  constexpr int K = (REC_PAIRS + G - 1) / G;
  double2 v[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int p = k * G + ln.sub;
    if ((k + 1) * G <= REC_PAIRS || p < REC_PAIRS)
      v[k] = *reinterpret_cast<const double2 *>(src + 2 * (long long)p * a.nchunk);
  }
  wave_sync();
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int p = k * G + ln.sub;
    if ((k + 1) * G <= REC_PAIRS || p < REC_PAIRS) {
      *slot(ln, 2 * p) = v[k].x;
      *slot(ln, 2 * p + 1) = v[k].y;
    }
  }
  wave_sync();
  c.y = holds(ln) ? *slot(ln, 2 * REC_C + slot_species(ln.sub)) : 0.0;
  bdf_init(c, a.dt, a.k);
}

#if NRG_PART < 2
// Cell records of the chunk's positions: the gate (:224-227) and the outputs of the
// cells it closes (:341-346), and for every integrated cell its concentrations (:228-233), rate constants and [M]
// (:235-252, 360-493), kept apart from the integrator so its ~80
// transcendentals run coherently.  A block covers
// RATES_CELLS cells RATES_GROUPS times: the waves of group g compute
// reactions [g R / G, (g+1) R / G) (a wave-uniform split, so each wave's code
// and registers cover a part of the mechanism: occupancy 4 instead of 1-2).
#ifndef RATES_GROUPS
#define RATES_GROUPS 2
#endif
constexpr int RATES_CELLS = 256 / RATES_GROUPS;

__global__ void __launch_bounds__(256) rates_kernel(StepArgs a)
{
  __shared__ MechCoef mc;
  stage_mech(mc, a.mech);
  const int grp = __builtin_amdgcn_readfirstlane(threadIdx.x / RATES_CELLS);   // wave-uniform
  const long long t = (long long)blockIdx.x * RATES_CELLS + (threadIdx.x % RATES_CELLS);
  const bool in = t < a.nchunk;
  long long q = 0, off = 0, record = t;
  double T = 0.0;
  bool live = false;
  if (in) {
    q = cell_of(a, t);
    off = cell_offset(a.g, q);
    T = a.T[off];
    live = T >= a.k.t_gate && (!a.bc || a.bc[off] == 0);
  }
  if (!a.gated) {
    // the block's integrated cells take the next records (one atomic a block)
    constexpr int WAVES = RATES_CELLS / WAVE;
    __shared__ unsigned long long first;
    __shared__ int count[WAVES];
    const unsigned long long mask = __ballot(live ? 1 : 0);
    const int w = threadIdx.x % RATES_CELLS / WAVE;
    if (grp == 0 && threadIdx.x % WAVE == 0) count[w] = __popcll(mask);
    __syncthreads();
    int before = __popcll(mask & ((1ull << (threadIdx.x % WAVE)) - 1ull)), all = 0;
    for (int i = 0; i < WAVES; ++i) {
      before += i < w ? count[i] : 0;
      all += count[i];
    }
    if (threadIdx.x == 0 && all) first = atomicAdd(a.live, (unsigned long long)all);
    __syncthreads();
    record = (long long)first + before;
  }
  if (!live) {
    if (in && grp == 0) {
#pragma unroll
      for (int s = 0; s < S; ++s) a.Yp[s][off] = 0.0;
      a.Efp[off] = 0.0;
      if (a.status) a.status[off] = NRG_CELL_GATED;
      if (a.nstep) {
        a.nstep[q] = 0;
        a.nfe[q] = 0;
        a.nje[q] = 0;
      }
      if (a.hist) a.hist[q] = 0;
    }
    return;
  }
  double *out = a.rates_out + 2 * record;
  const double rho = a.rho[off];
  double C[S];
#pragma unroll
  for (int s = 0; s < S; ++s) C[s] = (a.Y[s][off] * rho) / mc.W[s];
  constexpr int G = RATES_GROUPS;
  static_assert(G == 1 || G == 2 || G == 4, "RATES_GROUPS must be 1, 2 or 4");
  if (G == 1 || grp == 0)
    rate_constants<InlineMath, 0, R / G>(mc, T, C, out, a.nchunk);
  else if (G == 2 || grp == 1)
    rate_constants<InlineMath, R / G, 2 * R / G>(mc, T, C, out, a.nchunk);
  else if (grp == 2)
    rate_constants<InlineMath, 2 * R / G, 3 * R / G>(mc, T, C, out, a.nchunk);
  else
    rate_constants<InlineMath, 3 * R / G, R>(mc, T, C, out, a.nchunk);
  // the concentrations and the cell's index, written last (stored ahead of the
  // rate constants, they doubled the kernel's registers: occupancy 4 -> 2)
  if (grp == 0) {
#pragma unroll
    for (int j = 0; j <= REC_CELL; j += 2) {
      const double lo = j < S ? C[j] : __longlong_as_double(q);
      const double hi = j + 1 < S ? C[j + 1] : (j + 1 == REC_CELL ? __longlong_as_double(q) : 0.0);
      *reinterpret_cast<double2 *>(out + rec_slot(REC_C, j, a.nchunk)) = make_double2(lo, hi);
    }
  }
}

#endif

// Output assembly (:318-340) once the cell's DDRIV3 has returned, a species to
// a lane, and the cell's work and status counts (tally, in LDS).
NRG_DI void finish_cell(const StepArgs &a, const BdfCoef &mc, const Cell &c, const Lane &ln,
                        unsigned long long *tally)
{
  wave_sync();
  if (holds(ln)) *own(ln, CZ) = c.y;
  wave_sync();
  const long long q = __double_as_longlong(*slot(ln, 2 * REC_C + REC_CELL));
  const long long off = cell_offset(a.g, q);
#pragma unroll
  for (int s0 = 0; s0 < S; s0 += G) {
    const int s = s0 + ln.sub;
    if (s < S) {
      // the initial concentration as rates_kernel recorded it
      const double cin = *slot(ln, 2 * REC_C + s);
      const double ys = inert_species(s) ? cin : *slot(ln, CZ + active_slot(s));
      const double dc = ys - cin;
      a.Yp[s][off] = (dc * mc.W[s]) / a.dt;
      a.Yp2[s][off] = dc;
      *slot(ln, CX + s) = (mc.h_ref[s] * dc) / a.dt;
    }
  }
  wave_sync();
  const int out = c.pc & 15;
  const int status = (out == OUT_OK) ? NRG_CELL_OK
                   : (out == OUT_MXSTEP || out == OUT_EPS) ? NRG_CELL_MXSTEP
                   : (out == OUT_STEP_ZERO) ? NRG_CELL_STEP_ZERO
                   : (out == OUT_REPEATED_FAIL) ? NRG_CELL_REPEATED_FAIL
                   : NRG_CELL_SINGULAR;
  if (ln.sub == 0) {
    double ef = 0.0;
#pragma unroll
    for (int s = 0; s < S; ++s) ef = ef - *slot(ln, CX + s);
    a.Efp[off] = ef;
    if (a.status) a.status[off] = status;
    if (a.nstep) a.nstep[q] = c.nstep;
    if (a.hist) a.hist[q] = hist_code(c.nstep, c.work);   // lane 0's counter: NFE
    atomicAdd(&tally[ACC_STATUS0 + status], 1ull);
  }
  if (a.nstep && ln.sub == WORK_NFE) a.nfe[q] = c.work;
  if (a.nstep && ln.sub == WORK_NJE) a.nje[q] = c.work;
  // the work counters, each added by the lane that holds it, and the others
  static_assert(ACC_NJE == ACC_NFE + WORK_NJE && ACC_NCORR == ACC_NFE + WORK_NCORR &&
                ACC_NATT == ACC_NFE + WORK_NATT && WORK_NFE == 0 && G >= 4, "a counter to a lane");
  const int nfe = __shfl(c.work, ln.gshift + WORK_NFE, WAVE);
  if (ln.sub < 4) {
    atomicAdd(&tally[ACC_NFE + ln.sub], (unsigned long long)c.work);
    if (ln.sub < 2)
      atomicAdd(&tally[ln.sub == 0 ? ACC_INTEG : ACC_NSTEP], ln.sub == 0 ? 1ull : (unsigned long long)c.nstep);
    else
      atomicMax(&tally[ln.sub == 2 ? ACC_NSTEP_MAX : ACC_NFE_MAX], (unsigned long long)(ln.sub == 2 ? c.nstep : nfe));
  }
  wave_sync();
}

// A wave's counts into the launch's: one atomic per counter.
NRG_DI void flush_tally(unsigned long long *acc, const unsigned long long *tally, int lane)
{
  wave_sync();
  if (lane < ACC_QUEUE0 && tally[lane]) {
    if (lane == ACC_NSTEP_MAX || lane == ACC_NFE_MAX)
      atomicMax(&acc[lane], tally[lane]);
    else
      atomicAdd(&acc[lane], tally[lane]);
  }
}

// One chemistry step (solve_chemical_kinetics, :224-346), a cell to a group of
// G lanes (bdf_group.h).  A resident grid of one-wave blocks; each wave holds up
// to a.cpw cells and takes the next unclaimed ones of the chunk's queue (one
// atomic per wave per refill) once k.refill_idle of its 64 lanes (in proportion
// where it holds fewer cells) are idle, or all are.
// Each pass evaluates f for the cells that asked for it and, when at least
// jac_pct % of the pending cells wait for a Jacobian or nothing else is
// pending, forms and factors the waiting cells' iteration matrices.
//
// Idle lanes that trigger a refill.  In stiffness order a wave's cells cost
// alike and are best started together (256 x 4096 flame cells: 17.8 ms, 22.4
// with 32, 26.0 with 8); in natural order a long cell would keep the others'
// lanes idle (262,144 cells of an igniting mixture: 12.1 ms with 64, 9.0 with
// 32, 8.0 with 8, but flame fronts and hot kernels want more: 22.0, 23.5, 24.2
// and 6.7, 6.4, 9.1), except where the last call has counted that the grid's cells
// cost alike (plan): they are started together as well.
constexpr int REFILL_IDLE_ORDERED = 63, REFILL_IDLE_NATURAL = 32;

// Resident waves per SIMD the register budget is sized for (168 registers at
// three, 256 at two): a group of 8 lanes needs 166, one of 16 up to 213 without
// spills, and spilling costs more than the third wave gives.
constexpr int BDF_WAVES = G == 8 ? 3 : 2;
template <bool ANALYTIC>
__global__ void __launch_bounds__(WAVE) __attribute__((amdgpu_waves_per_eu(BDF_WAVES)))
chem_bdf_kernel(StepArgs a)
#if NRG_PART == 1 || NRG_PART == 3
;   // defined in the integrator part of this build
extern template __global__ void chem_bdf_kernel<false>(StepArgs);
extern template __global__ void chem_bdf_kernel<true>(StepArgs);
#else
{
  __shared__ BdfCoef mc;
  __shared__ __align__(16) double cells[CPW * CELL_DOUBLES];   // the cells' slices
  __shared__ __align__(16) unsigned table[G * TABW];
  __shared__ __align__(16) unsigned jtable[ANALYTIC ? G * JTABW : 4];
  __shared__ unsigned long long tally[ACC_QUEUE0];             // the wave's share of acc
  const int lane = threadIdx.x;
  if (lane < ACC_QUEUE0) tally[lane] = 0ull;
  stage_bdf(mc, a.mech, a.k.sqrtn);
  Lane ln;
  group_init(ln, (lds_double *)cells, (lds_word *)table, ANALYTIC ? (lds_word *)jtable : nullptr, lane);
  Cell c;
  c.pc = PC_IDLE;
  const int grp = lane / G;
  const long long limit = live_records(a);
  if (blockIdx.x == 0 && lane == 0) tally[ACC_STATUS0 + NRG_CELL_GATED] = (unsigned long long)(a.nchunk - limit);
  bool exhausted = grp >= a.cpw;
  for (;;) {
    bool need = c.pc >= PC_DONE && !exhausted;
    if (wave_any(c.pc < PC_DONE) && __popcll(__ballot(need ? 1 : 0)) * CPW < a.k.refill_idle * a.cpw)
      need = false;
    while (wave_any(need)) {
      const unsigned long long mask = __ballot(need ? 1 : 0);
      const int leader = __ffsll((long long)mask) - 1;
      unsigned long long base = 0;
      if (lane == leader) base = atomicAdd(a.queue, (unsigned long long)(__popcll(mask) / G));
      base = __shfl(base, leader, WAVE);
      if (need) {
        const long long t =
            (long long)(base + (unsigned long long)(__popcll(mask & ((1ull << ln.gshift) - 1ull)) / G));
        if (t >= limit)
          exhausted = true;
        else
          start_cell(a, t, c, ln);
      }
      need = need && c.pc >= PC_DONE && !exhausted;
    }
    if (!wave_any(c.pc < PC_DONE)) break;
    const bool wantj = (c.pc & PC_WAIT_JAC) != 0, wantf = (c.pc & PC_WAIT_F) != 0;
    const int nj = __popcll(__ballot(wantj ? 1 : 0));
    const int nf = __popcll(__ballot(wantf ? 1 : 0));
    const bool run_jac = nj > 0 && (nf == 0 || nj * 100 >= a.jac_pct * (nj + nf));
    if (wantf) {
      c.save2 = rhs_group(ln, c.y);
      c.pc &= 15;
    }
    if (run_jac && wantj) {
      if (ANALYTIC)
        jac_exact(ln, c, mc);
      else
        jac_fd(ln, c, a.k, mc);
      c.pc &= 15;
    }
    if (c.pc < PC_WAIT_F) advance(ln, c, a.dt, a.k, mc);
    if ((c.pc & PC_DONE) && c.pc != PC_IDLE) {
      finish_cell(a, mc, c, ln, tally);
      c.pc = PC_IDLE;
    }
  }
  flush_tally(a.acc, tally, lane);
}
#endif

// ---------------------------------------------------------------------------
// The same step with one cell per lane (bdf_lane.h), where a launch's cells fill the
// chip so (lane_launch), for the topologies whose state fits the register file.
// ---------------------------------------------------------------------------
constexpr bool LANE_KERNEL = SA <= 10;
constexpr int LANE_WAVES_PER_CU = 4;   // one to a SIMD: it takes the whole register file
#if NRG_PART == 0 || NRG_PART == 3
typedef __attribute__((address_space(3))) void lds_void;

// Load one cell and set it up (chemical_kinetics_solver.f90:228-265).  The
// cell record t (rates_kernel) goes from HBM straight into the lane's LDS slots
// (recl: the block's record array, kl: this lane's view of it): one round trip, no
// registers in between.
NRG_DI void start_cell(const StepArgs &a, long long t, long long &q, long long &off, lane::Cell &c,
                       lds_double *recl, const double *kl)
{
  const double *src = a.rates + 2 * t;
#pragma unroll
  for (int p = 0; p < REC_PAIRS; ++p)
    __builtin_amdgcn_global_load_lds((const void *)(src + 2 * (long long)p * a.nchunk),
                                     (lds_void *)(recl + 2 * p * WAVE), 16, 0, 0);   // M0: LDS address
  // a direct load's data is in LDS once vmcnt has counted it
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  q = __double_as_longlong(lane::rec_c(kl, REC_CELL));
  off = cell_offset_wide(a.g, q);
#pragma unroll
  for (int s = 0; s < S; ++s) {
    if (kSp.act[s] >= 0)
      c.y[kSp.act[s]] = lane::rec_c(kl, s);
    else
      c.yi[kSp.islot[s]] = lane::rec_c(kl, s);
  }
  lane::bdf_init(c, a.dt, a.k);
}

// A lane's counts of its finished cells.  (In registers: cells of equal cost
// finish together, and 64 atomics to one LDS word take as many turns; 2.1M
// cells with hot kernels 5.44 ms so, 4.85 here.)
struct LaneTally {
  unsigned integrated = 0;
  unsigned long long nstep = 0, nfe = 0, nje = 0, ncorr = 0, natt = 0;
  int nstep_max = 0, nfe_max = 0;
};

// Output assembly (:318-340) once the cell's DDRIV3 has returned, and its
// counts (a failure's straight into the wave's).
NRG_DI void finish_cell(const StepArgs &a, const BdfCoef &mc, long long q, long long off,
                        const lane::Cell &c, const double *kl, LaneTally &tl, unsigned long long *tally)
{
  double ef = 0.0;
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const double cin = lane::rec_c(kl, s);   // the initial concentration as rates_kernel recorded it
    const double ys = (kSp.act[s] >= 0) ? c.y[kSp.act[s]] : c.yi[kSp.islot[s]];
    const double dc = ys - cin;
    a.Yp[s][off] = (dc * mc.W[s]) / a.dt;
    a.Yp2[s][off] = dc;
    ef = ef - (mc.h_ref[s] * dc) / a.dt;
  }
  a.Efp[off] = ef;
  const int status = (c.outcome == lane::OUT_OK) ? NRG_CELL_OK
                   : (c.outcome == lane::OUT_MXSTEP || c.outcome == lane::OUT_EPS) ? NRG_CELL_MXSTEP
                   : (c.outcome == lane::OUT_STEP_ZERO) ? NRG_CELL_STEP_ZERO
                   : (c.outcome == lane::OUT_REPEATED_FAIL) ? NRG_CELL_REPEATED_FAIL
                   : NRG_CELL_SINGULAR;
  if (a.status) a.status[off] = status;
  if (a.nstep) {
    a.nstep[q] = c.nstep;
    a.nfe[q] = c.nfe;
    a.nje[q] = c.nje;
  }
  if (a.hist) a.hist[q] = hist_code(c.nstep, c.nfe);
  if (status != NRG_CELL_OK) atomicAdd(&tally[ACC_STATUS0 + status], 1ull);
  tl.integrated += 1;
  tl.nstep += c.nstep;
  tl.nfe += c.nfe;
  tl.nje += c.nje;
  tl.ncorr += c.ncorr;
  tl.natt += c.natt;
  tl.nstep_max = max(tl.nstep_max, c.nstep);
  tl.nfe_max = max(tl.nfe_max, c.nfe);
}
#endif

// A resident grid of one-wave blocks; once k.refill_idle lanes of a wave have
// finished (or all have), they take the next unclaimed cells from a.queue (one
// atomic per wave per refill).  Each pass either evaluates f for the lanes that
// asked, or -- when at least jac_pct % of the pending lanes wait for a Jacobian,
// or nothing else is pending -- forms and factors the iteration matrices of the
// waiting lanes.
template <bool ANALYTIC>
__global__ void __launch_bounds__(WAVE) __attribute__((amdgpu_waves_per_eu(1)))
chem_bdf_lane_kernel(StepArgs a)
#if NRG_PART == 1 || NRG_PART == 2
;   // defined in a part of its own
extern template __global__ void chem_bdf_lane_kernel<false>(StepArgs);
extern template __global__ void chem_bdf_lane_kernel<true>(StepArgs);
#else
{
  __shared__ BdfCoef mc;
  __shared__ __align__(16) double recl[2 * REC_PAIRS * WAVE];   // the lanes' cell records
  __shared__ unsigned long long tally[ACC_QUEUE0];              // the wave's share of acc
  static_assert(4 * (sizeof(BdfCoef) + sizeof recl + sizeof tally) <= 160 * 1024, "four blocks to a CU");
  const int lane = threadIdx.x;
  if (lane < ACC_QUEUE0) tally[lane] = 0ull;
  stage_bdf(mc, a.mech, a.k.sqrtn);
  const double *kl = recl + 2 * lane;
  lds_double *recl_lds = (lds_double *)recl;   // the array's LDS address (direct loads' M0)
  const long long limit = live_records(a);
  if (blockIdx.x == 0 && lane == 0) tally[ACC_STATUS0 + NRG_CELL_GATED] = (unsigned long long)(a.nchunk - limit);
  lane::Cell c;
  c.req = lane::REQ_DONE;
  long long q = -1, off = 0;
  LaneTally tl;
  bool have = false, exhausted = false;
  for (;;) {
    // refill in batches: new cells start together, so the wave's lanes stay
    // near the same stage (refilling every pass measured 30 % slower)
    bool need = !have && !exhausted;
    if (wave_any(have) && __popcll(__ballot(need ? 1 : 0)) < a.k.refill_idle) need = false;
    while (wave_any(need)) {
      const unsigned long long mask = __ballot(need ? 1 : 0);
      const int leader = __ffsll((long long)mask) - 1;
      unsigned long long base = 0;
      if (lane == leader) base = atomicAdd(a.queue, (unsigned long long)__popcll(mask));
      base = __shfl(base, leader, WAVE);
      if (need) {
        const long long t = (long long)(base + (unsigned long long)__popcll(mask & ((1ull << lane) - 1ull)));
        if (t >= limit) {
          exhausted = true;
        } else {
          start_cell(a, t, q, off, c, recl_lds, kl);
          have = true;
        }
      }
      need = !have && !exhausted;
    }
    if (!wave_any(have)) break;
    const bool wantj = have && c.req == lane::REQ_JAC;
    const bool wantf = have && c.req == lane::REQ_F;
    const int nj = __popcll(__ballot(wantj ? 1 : 0));
    const int nf = __popcll(__ballot(wantf ? 1 : 0));
    const bool run_jac = nj > 0 && (nf == 0 || nj * 100 >= a.jac_pct * (nj + nf));
    if (run_jac) {
      if (ANALYTIC)
        lane::jac_analytic(c, wantj, mc, kl);
      else
        lane::jac_batch(c, wantj, a.k, mc, kl);
    }
    else if (wantf)
      lane::rhs(kl, c.y, c.save2);
    if (have && (c.req == lane::REQ_NONE || (run_jac ? wantj : wantf))) {
      c.req = lane::REQ_NONE;
      lane::advance(c, a.dt, a.k, mc);
    }
    if (have && c.req == lane::REQ_DONE) {
      finish_cell(a, mc, q, off, c, kl, tl, tally);
      have = false;
    }
  }
  atomicAdd(&tally[ACC_INTEG], (unsigned long long)tl.integrated);
  atomicAdd(&tally[ACC_NSTEP], tl.nstep);
  atomicAdd(&tally[ACC_NFE], tl.nfe);
  atomicAdd(&tally[ACC_NJE], tl.nje);
  atomicAdd(&tally[ACC_NCORR], tl.ncorr);
  atomicAdd(&tally[ACC_NATT], tl.natt);
  atomicMax(&tally[ACC_NSTEP_MAX], (unsigned long long)tl.nstep_max);
  atomicMax(&tally[ACC_NFE_MAX], (unsigned long long)tl.nfe_max);
  wave_sync();
  if (lane == 0) {
    unsigned long long failed = 0;
    for (int s = 0; s < 6; ++s) failed += (s == NRG_CELL_OK || s == NRG_CELL_GATED) ? 0ull : tally[ACC_STATUS0 + s];
    tally[ACC_STATUS0 + NRG_CELL_OK] = tally[ACC_INTEG] - failed;
  }
  flush_tally(a.acc, tally, lane);
}
#endif

#if NRG_PART == 2 || NRG_PART == 3
// The integrator parts end here: their kernels, compiled with their own
// options (the Makefile), and nothing else.
#if NRG_PART == 3
template __global__ void chem_bdf_lane_kernel<false>(StepArgs);
template __global__ void chem_bdf_lane_kernel<true>(StepArgs);
#endif
#if NRG_PART == 2 && (!defined(NRG_BDF_JAC) || NRG_BDF_JAC == 1)
template __global__ void chem_bdf_kernel<false>(StepArgs);
#endif
#if NRG_PART == 2 && (!defined(NRG_BDF_JAC) || NRG_BDF_JAC == 2)
template __global__ void chem_bdf_kernel<true>(StepArgs);
#endif
}  // namespace kern
}  // namespace NRG_TOPO_NS
#pragma GCC visibility pop
#else

// ---------------------------------------------------------------------------
// Split-step closure and EOS (cabaret_solver.f90:3316-3318,3386-3416;
// table_approximated_real_gas.f90:410-440; thermophysical_properties_class.f90:409-452)
// ---------------------------------------------------------------------------
struct ClosureArgs {
  GridIdx g;
  double dt;
  int apply_sources;                    // 0: EOS only
  int ndim;
  const MechCoef *mech;
  const double *rho;
  const double *v[3];
  const double *Efp;
  const double *Yp[S];
  const int8_t *bc;
  double *E_f;
  double *Y[S];
  double *T, *p;
};

NRG_DI double calculate_temperature(const MechCoef &mc, double T, double e_i, const double (&X)[S])
{
  const double eps = (double)1e-08f;
  double temp = clip_t(T);
  double h_const = 0.0;
#pragma unroll
  for (int s = 0; s < S; ++s) h_const = h_const + mc.h_ref[s] * X[s];
  double cp = 0.0;
#pragma unroll
  for (int s = 0; s < S; ++s) cp = cp + cp_molar(mc, temp, s) * X[s];
  for (int iter = 1; iter <= 1000; ++iter) {
    double e = 0.0;
#pragma unroll
    for (int s = 0; s < S; ++s) e = e + e_molar(mc, temp, s) * X[s];
    const double e_int = e - h_const;
    const double residual = (e_i - e_int) / cp;
    temp = temp + residual;
    if (fabs(residual) < eps) break;
  }
  return temp;
}

template <bool STREAM>
__global__ void __launch_bounds__(256) closure_kernel(ClosureArgs a)
{
  __shared__ MechCoef mc;
  stage_mech(mc, a.mech);
  at_inner_cell(a.g, [&](long long off) {
    if (a.bc && a.bc[off] != 0) return;
    const double rho = a.rho[off];
    double Ef = a.E_f[off];
    double y[S];
    if (a.apply_sources) {
      const double efp = 0.0 + a.Efp[off] * a.dt;
      Ef = Ef + efp / rho;
      double sum = 0.0;
#pragma unroll
      for (int s = 0; s < S; ++s) {
        const double ypr = 0.0 + a.Yp[s][off] * a.dt;
        y[s] = a.Y[s][off] + ypr / rho;
        sum = sum + y[s];
      }
#pragma unroll
      for (int s = 0; s < S; ++s) y[s] = dmax(y[s], 0.0) / sum;
      put<STREAM>(&a.E_f[off], Ef);
#pragma unroll
      for (int s = 0; s < S; ++s) put<STREAM>(&a.Y[s][off], y[s]);
    } else {
#pragma unroll
      for (int s = 0; s < S; ++s) y[s] = a.Y[s][off];
    }
    double e_i = Ef;
    for (int d = 0; d < a.ndim; ++d) {
      const double vd = a.v[d][off];
      e_i = e_i - 0.5 * (vd * vd);
    }
    double avg = 0.0;
#pragma unroll
    for (int s = 0; s < S; ++s) avg = avg + y[s] / mc.W[s];
    const double wmix = 1.0 / avg;
    double X[S];
#pragma unroll
    for (int s = 0; s < S; ++s) X[s] = (y[s] / mc.W[s]) * wmix;
    e_i = e_i * wmix;
    const double Tn = calculate_temperature(mc, a.T[off], e_i, X);
    put<STREAM>(&a.T[off], Tn);
    if (a.p) put<STREAM>(&a.p[off], ((Tn * rho) * R_GAS_J) / wmix);
  });
}

struct EnergyArgs {
  GridIdx g;
  int ndim;
  const MechCoef *mech;
  const double *T;
  const double *Y[S];
  const double *v[3];
  double *E_f;
};

__global__ void __launch_bounds__(256) energy_kernel(EnergyArgs a)
{
  __shared__ MechCoef mc;
  stage_mech(mc, a.mech);
  const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= a.g.ninner) return;
  const long long off = cell_offset(a.g, q);
  double y[S], X[S], avg = 0.0;
#pragma unroll
  for (int s = 0; s < S; ++s) {
    y[s] = a.Y[s][off];
    avg = avg + y[s] / mc.W[s];
  }
  const double wmix = 1.0 / avg;
#pragma unroll
  for (int s = 0; s < S; ++s) X[s] = (y[s] / mc.W[s]) * wmix;
  const double T = a.T[off];
  double e = 0.0, hc = 0.0;
#pragma unroll
  for (int s = 0; s < S; ++s) e = e + e_molar(mc, T, s) * X[s];
#pragma unroll
  for (int s = 0; s < S; ++s) hc = hc + mc.h_ref[s] * X[s];
  double Ef = (e - hc) / wmix;
  for (int d = 0; d < a.ndim; ++d) {
    const double vd = a.v[d][off];
    Ef = Ef + 0.5 * (vd * vd);
  }
  a.E_f[off] = Ef;
}

// ---------------------------------------------------------------------------
// Table-approximated chemistry (chemical_kinetics_solver.f90:250-346 with
// ODE_solver = 'table_approximated', interpolate_chemical_kinetics :650-685):
// the "concentrations" are the mass fractions themselves, replaced by the
// table's dC(T) interpolated linearly in T (the last bracketing interval
// wins; below the table 0, above it the last row); then Y_prod = C_out*W/dt,
// Y_prod2 = C_out - Y, E_f_prod = -sum_s h_s(T_ref)*C_out/dt.
// ---------------------------------------------------------------------------
struct TableArgs {
  GridIdx g;
  double dt, t_gate;
  const MechCoef *mech;
  const double *T;
  const double *Y[S];
  const int8_t *bc;
  double *Yp[S], *Yp2[S];
  double *Efp;
  int32_t *status;
  const double *table;      // T_t[rows], dC_t[S][rows]
  int rows;
  int ascending;            // T_t strictly increasing: bisection finds the same interval
  unsigned long long *acc;  // [0] integrated cells
};

// The interval the reference's scan ends on (the last i with
// T_t[i] <= T <= T_t[i+1]), or -1 if none.  For a strictly increasing table
// that is the largest i with T_t[i] <= T, capped at rows-2 (T on a node k
// sits in intervals k-1 and k; k wins), so bisection gives it in log2(rows)
// probes.  Any other table is scanned in full.
__device__ __forceinline__ int table_interval(const double *Tt, int rows, int ascending, double T)
{
  if (ascending) {
    if (!(T >= Tt[0] && T <= Tt[rows - 1])) return -1;
    int lo = 0, hi = rows - 1;      // Tt[lo] <= T; the answer lies in [lo, hi]
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (Tt[mid] <= T) lo = mid;
      else hi = mid - 1;
    }
    return lo < rows - 1 ? lo : rows - 2;
  }
  int last = -1;
  for (int i = 0; i + 1 < rows; ++i)
    if (T >= Tt[i] && T <= Tt[i + 1]) last = i;
  return last;
}

constexpr int TABLE_THREADS = 256;
constexpr int TABLE_LDS_BYTES = 32768;        // a table up to this size is staged in LDS

// A grid of as many blocks as fit on the CUs strides over the cells, so the
// table is staged into LDS once per block (not once per 256 cells) and the
// integrated-cell count takes one global atomic per block.
template <bool TAB_LDS, bool STREAM>
__global__ void __launch_bounds__(TABLE_THREADS) table_kernel(TableArgs a)
{
  extern __shared__ double tab_lds[];         // T_t[rows], dC_t[S][rows] when TAB_LDS
  __shared__ double W[S], href[S];
  __shared__ unsigned long long n_integ;
  if (threadIdx.x < S) {
    W[threadIdx.x] = a.mech->W[threadIdx.x];
    href[threadIdx.x] = a.mech->h_ref[threadIdx.x];
  }
  if (threadIdx.x == 0) n_integ = 0;
  if (TAB_LDS)
    for (int k = threadIdx.x; k < (S + 1) * a.rows; k += TABLE_THREADS) tab_lds[k] = a.table[k];
  __syncthreads();
  const double *Tt = TAB_LDS ? tab_lds : a.table;
  const double *dC = Tt + a.rows;
  unsigned long long cnt = 0;
  const long long stride = (long long)gridDim.x * TABLE_THREADS;
  // Waves walk the allocation in 64-cell slices aligned with it (from the
  // first inner cell's slice to the last inner cell) and skip ghost cells:
  // with ghost layers a row of inner cells starts off a cache line, and
  // walking inner cells would make every wave touch one line more per field.
  for (long long off = a.g.pad0 + (long long)blockIdx.x * TABLE_THREADS + threadIdx.x; off < a.g.pad1; off += stride) {
    if (!inner_at(a.g, off)) continue;
    const double T = a.T[off];
    const int8_t bcv = a.bc ? a.bc[off] : (int8_t)0;
    const bool run = T >= a.t_gate && bcv == 0;
    double c[S], ef = 0.0;
#pragma unroll
    for (int s = 0; s < S; ++s) c[s] = 0.0;
    if (run) {
      ++cnt;
      double cin[S];
#pragma unroll
      for (int s = 0; s < S; ++s) c[s] = cin[s] = a.Y[s][off];
      const int i = table_interval(Tt, a.rows, a.ascending, T);
      if (i >= 0) {
        const double t0 = Tt[i], t1 = Tt[i + 1], up = t1 - t0, dn = t0 - t1;
#pragma unroll
        for (int s = 0; s < S; ++s)
          c[s] = (dC[s * a.rows + i + 1] * (T - t0)) / up +
                 (dC[s * a.rows + i] * (T - t1)) / dn;
      }
      if (T < Tt[0]) {
#pragma unroll
        for (int s = 0; s < S; ++s) c[s] = 0.0;
      }
      if (T > Tt[a.rows - 1]) {
#pragma unroll
        for (int s = 0; s < S; ++s) c[s] = dC[s * a.rows + a.rows - 1];
      }
#pragma unroll
      for (int s = 0; s < S; ++s) {
        put<STREAM>(&a.Yp2[s][off], c[s] - cin[s]);
        ef = ef - (href[s] * c[s]) / a.dt;
        c[s] = (c[s] * W[s]) / a.dt;
      }
    }
    // what gated cells have too, for the whole slice at once
#pragma unroll
    for (int s = 0; s < S; ++s) put<STREAM>(&a.Yp[s][off], c[s]);
    put<STREAM>(&a.Efp[off], ef);
    if (a.status) put<STREAM>(&a.status[off], run ? NRG_CELL_OK : NRG_CELL_GATED);
  }
  if (cnt) atomicAdd(&n_integ, cnt);
  __syncthreads();
  if (threadIdx.x == 0 && n_integ) atomicAdd(a.acc, n_integ);
}

// ---------------------------------------------------------------------------
// Low-Mach (FDS) coupling (fds_low_mach_solver.f90, table_approximated_real_gas.
// f90:570-677).  Per-cell, HBM-bound; one thread per offset of the aligned
// walk, the mechanism staged in LDS per block.
// ---------------------------------------------------------------------------
constexpr int LM_THREADS = 256;

struct LowMachEosArgs {
  GridIdx g;
  double dt;
  int predictor, ndim;
  const MechCoef *mech;
  const double *rho, *Y[S], *v[3], *dp;
  const int8_t *bc;
  double *p_stat, *p_stat_old, *T, *mmm;
  double *p, *cp, *gamma, *h_s, *v_s, *e_i, *E_f;   // optional
};

template <bool STREAM>
__global__ void __launch_bounds__(LM_THREADS) low_mach_eos_kernel(LowMachEosArgs a)
{
  __shared__ MechCoef mc;
  stage_mech(mc, a.mech);
  at_inner_cell(a.g, [&](long long off) {
    if (a.bc && a.bc[off] != 0) return;
    double X[S], avg = 0.0;
#pragma unroll
    for (int s = 0; s < S; ++s) {
      X[s] = a.Y[s][off];
      avg = avg + X[s] / mc.W[s];
    }
    const double W = 1.0 / avg;
    put<STREAM>(&a.mmm[off], W);
#pragma unroll
    for (int s = 0; s < S; ++s) X[s] = (X[s] * W) / mc.W[s];
    double ps;
    if (a.predictor) {
      const double p0 = a.p_stat[off];
      put<STREAM>(&a.p_stat_old[off], p0);
      ps = p0 + a.dp[off] * a.dt;
    } else {
      ps = 0.5 * ((a.p_stat[off] + a.p_stat_old[off]) + a.dp[off] * a.dt);
    }
    put<STREAM>(&a.p_stat[off], ps);
    const double rho = a.rho[off];
    const double T = ((ps / rho) / R_GAS_J) * W;
    put<STREAM>(&a.T[off], T);
    double cp = 0.0;
#pragma unroll
    for (int s = 0; s < S; ++s) cp = cp + cp_molar(mc, T, s) * X[s];
    const double g = cp / (cp - R_GAS_J);
    if (a.gamma) put<STREAM>(&a.gamma[off], g);
    if (a.h_s) {
      double hT = 0.0, h0 = 0.0;
#pragma unroll
      for (int s = 0; s < S; ++s) hT = hT + h_molar(mc, T, s) * X[s];
#pragma unroll
      for (int s = 0; s < S; ++s) h0 = h0 + mc.h_ref[s] * X[s];
      put<STREAM>(&a.h_s[off], (hT - h0) / W);
    }
    if (a.cp) put<STREAM>(&a.cp[off], cp);
    if (a.p) put<STREAM>(&a.p[off], ps);
    if (a.v_s) put<STREAM>(&a.v_s[off], sqrt((g * ps) / rho));
    const double ei = (ps / rho) / (g - 1.0);
    if (a.e_i) put<STREAM>(&a.e_i[off], ei);
    if (a.E_f && a.ndim > 0) {
      const double vd = a.v[a.ndim - 1][off];
      put<STREAM>(&a.E_f[off], ei + 0.5 * (vd * vd));
    }
  });
}

struct LowMachSpeciesArgs {
  GridIdx g;
  double dt;
  int corrector;
  const double *rho_a, *Y_a[S], *rho_b, *Y_b[S];
  const double *rhs[S], *Yd[S], *Yc[S];   // rhs[0], Yd[0], Yc[0] NULL: term absent
  const int8_t *bc;
  double *rho_out, *Y_out[S];
};

template <bool STREAM>
__global__ void __launch_bounds__(LM_THREADS) low_mach_species_kernel(LowMachSpeciesArgs a)
{
  at_inner_cell(a.g, [&](long long off) {
    if (a.bc && a.bc[off] != 0) return;
    double r[S];
    const double ra = a.rho_a[off];
    const double rb = a.corrector ? a.rho_b[off] : 0.0;
#pragma unroll
    for (int s = 0; s < S; ++s) {
      const double f = a.rhs[0] ? a.rhs[s][off] : 0.0;
      if (!a.corrector) {
        r[s] = ra * a.Y_a[s][off] + f * a.dt;
        if (a.Yd[0]) r[s] = r[s] + a.Yd[s][off] * a.dt;
        if (a.Yc[0]) r[s] = r[s] + a.Yc[s][off] * a.dt;
      } else {
        r[s] = 0.5 * (ra * a.Y_a[s][off] + rb * a.Y_b[s][off]) + f * (0.5 * a.dt);
        if (a.Yd[0]) r[s] = r[s] + (0.5 * a.Yd[s][off]) * a.dt;
        if (a.Yc[0]) r[s] = r[s] + (0.5 * a.Yc[s][off]) * a.dt;
      }
    }
    double sum = 0.0;
#pragma unroll
    for (int s = 0; s < S; ++s) {
      r[s] = dmax(r[s], 0.0);
      sum = sum + r[s];
    }
    if (sum > DBL_MIN) {
      put<STREAM>(&a.rho_out[off], sum);
#pragma unroll
      for (int s = 0; s < S; ++s) put<STREAM>(&a.Y_out[s][off], r[s] / sum);
    }
  });
}

struct LowMachDivArgs {
  GridIdx g;
  const MechCoef *mech;
  const double *rho, *T, *Y[S], *mmm, *Efc, *Yc[S];
  const int8_t *bc;
  double *div;
};

// (The fields' loads are issued before the mechanism is staged, so that a block
// waits for memory once: 2.0M cells 110 -> 98 us.)
template <bool STREAM>
__global__ void __launch_bounds__(LM_THREADS) low_mach_div_kernel(LowMachDivArgs a)
{
  __shared__ MechCoef mc;
  const long long off = a.g.pad0 + (long long)blockIdx.x * LM_THREADS + threadIdx.x;
  const bool in = off < a.g.pad1 && inner_at(a.g, off);
  int8_t bc = 0;
  double W = 1.0, rho = 1.0, T = 1.0, d = 0.0, Y[S] = {}, Yc[S] = {};
  if (in) {
    if (a.bc) bc = a.bc[off];
    W = a.mmm[off];
    rho = a.rho[off];
    T = a.T[off];
    d = d + a.Efc[off];
#pragma unroll
    for (int s = 0; s < S; ++s) Y[s] = a.Y[s][off];
#pragma unroll
    for (int s = 0; s < S; ++s) Yc[s] = a.Yc[s][off];
  }
  stage_mech(mc, a.mech);
  if (!in || bc != 0) return;
  double cp = 0.0;
#pragma unroll
  for (int s = 0; s < S; ++s) cp = cp + cp_molar(mc, T, s) * ((Y[s] * W) / mc.W[s]);
  const double heat = ((rho * cp) * T) / W;
  d = d / heat;
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const double hs = (h_molar(mc, T, s) - mc.h_ref[s]) / mc.W[s];
    d = d + (((W / mc.W[s]) / rho) - hs / heat) * Yc[s];
  }
  put<STREAM>(&a.div[off], d);
}

// ---------------------------------------------------------------------------
// Stiffness-ordered queue: bin the inner cells by expected cost, most
// expensive bin first.  A block bins a contiguous run of cells (one
// global atomic per bin and block); within a bin, the cells of a run come in
// roughly increasing index order.
// ---------------------------------------------------------------------------
// Bins by steps, and of each by right-hand sides (modulo): a wave's lanes wait for
// each other wherever their paths through the integrator part, and cells that
// took as many right-hand sides in as many steps mostly took the same path (256^3
// hot kernels: 65 % of the lanes busy per instruction by steps alone, 71 % so).  One cell
// per lane, by steps / 16 / 64 bins of each: 2.1M cells with hot kernels 4.85 / 3.73 /
// 3.69 ms, 1M flame cells 14.6 / 12.2 / 11.9, 1M igniting 17.3 / 15.7 / 14.9.  (By a hash
// of the path instead: 3.73, 11.4, 16.0.)  Placing 16.7M cells costs 0.26 ms, 0.10 with 64 bins.
constexpr int NBIN_STEP = 64, NBIN_FE = 64;
constexpr int NBIN = NBIN_STEP * NBIN_FE;
constexpr int BIN_THREADS = 256;
constexpr int BIN_RUN_MAX = 32;       // cells a thread takes, at most

struct BinArgs {
  GridIdx g;
  const double *T;
  const int8_t *bc;
  double t_gate;
  const int32_t *hist;              // hist_code of the previous call, or NULL (use T)
  unsigned long long *count;        // [NBIN]
  unsigned long long *cursor;       // [NBIN] cells of each bin placed
  const int32_t *in_list;           // cells to order (NULL: all inner cells 0..npos-1)
  long long npos;                   // number of cells to order
  int32_t *list;                    // [npos] the ordered cells
  int run;                          // cells a thread takes
};

// 0 = gated (no integration); otherwise grows with the expected cost.
NRG_DI int cost_bin(const BinArgs &a, long long q)
{
  const long long off = cell_offset(a.g, q);
  const int8_t b = a.bc ? a.bc[off] : (int8_t)0;
  const double T = a.T[off];
  if (!(T >= a.t_gate && b == 0)) return 0;
  if (a.hist) {
    const int code = a.hist[q], n = code & HIST_STEPS, fe = code >> HIST_FE_SHIFT;
    const int k = n <= 31 ? n : 31 + (n - 28) / 4;     // unit bins to 31 steps, then 4-step bins
    return (1 + min(NBIN_STEP - 2, k)) * NBIN_FE + fe % NBIN_FE;
  }
  const double x = (T - a.t_gate) * (1.0 / 50.0);                     // first call: 50 K bins
  return (1 + (x < (double)(NBIN_STEP - 2) ? (int)x : NBIN_STEP - 2)) * NBIN_FE;
}

// Histogram of the block's run into LDS.
NRG_DI void bin_histogram(const BinArgs &a, unsigned int *h)
{
  for (int b = threadIdx.x; b < NBIN; b += BIN_THREADS) h[b] = 0u;
  __syncthreads();
  const long long p0 = (long long)blockIdx.x * a.run * BIN_THREADS + threadIdx.x;
  for (int k = 0; k < a.run; ++k) {
    const long long p = p0 + (long long)k * BIN_THREADS;
    if (p < a.npos) atomicAdd(&h[cost_bin(a, a.in_list ? (long long)a.in_list[p] : p)], 1u);
  }
  __syncthreads();
}

__global__ void __launch_bounds__(BIN_THREADS) bin_count_kernel(BinArgs a)
{
  __shared__ unsigned int h[NBIN];
  bin_histogram(a, h);
  for (int b = threadIdx.x; b < NBIN; b += BIN_THREADS)
    if (h[b]) atomicAdd(&a.count[b], (unsigned long long)h[b]);
}

// Each block claims its bins' slots with one atomic per bin, behind the cells of
// the more expensive bins, then places its run's cells (same run as
// bin_count_kernel, binned again).  A thread has 16 bins: one claim after the other, each
// waited for, took 54 us of a list of 84,000 cells (12 now), 194 of 545,400 igniting
// cells (33) and 326 of 16.7M with hot kernels (261).
__global__ void __launch_bounds__(BIN_THREADS) bin_scatter_kernel(BinArgs a)
{
  __shared__ unsigned int h[NBIN];
  __shared__ unsigned long long base[NBIN], sums[BIN_THREADS / WAVE];
  bin_histogram(a, h);
  // cells of the more expensive bins: each thread's bins, then the threads after it
  constexpr int PER = NBIN / BIN_THREADS;
  static_assert(NBIN % BIN_THREADS == 0, "bins to a thread");
  const int b0 = threadIdx.x * PER, lane = threadIdx.x & (WAVE - 1), w = threadIdx.x / WAVE;
  unsigned long long cells[PER], claim[PER], mine = 0;
#pragma unroll
  for (int k = 0; k < PER; ++k) cells[k] = a.count[b0 + k];
  // the claims, all under way before the first is waited for (neighbouring threads take
  // neighbouring bins: those that a run fills lie together)
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int b = k * BIN_THREADS + threadIdx.x;
    claim[k] = h[b] ? atomicAdd(&a.cursor[b], (unsigned long long)h[b]) : 0ull;
  }
#pragma unroll
  for (int k = 0; k < PER; ++k) mine += cells[k];
  unsigned long long after = mine;
  for (int d = 1; d < WAVE; d <<= 1) {
    const unsigned long long v = __shfl_down(after, d, WAVE);
    after += lane + d < WAVE ? v : 0ull;
  }
  if (lane == 0) sums[w] = after;
  __syncthreads();
  for (int k = w + 1; k < BIN_THREADS / WAVE; ++k) after += sums[k];
  after -= mine;
#pragma unroll
  for (int k = PER - 1; k >= 0; --k) {
    base[b0 + k] = after;
    after += cells[k];
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int b = k * BIN_THREADS + threadIdx.x;
    base[b] += claim[k];
    h[b] = 0u;
  }
  __syncthreads();
  const long long p0 = (long long)blockIdx.x * a.run * BIN_THREADS + threadIdx.x;
  for (int k = 0; k < a.run; ++k) {
    const long long p = p0 + (long long)k * BIN_THREADS;
    if (p < a.npos) {
      const long long q = a.in_list ? (long long)a.in_list[p] : p;
      const int b = cost_bin(a, q);
      const unsigned int rank = atomicAdd(&h[b], 1u);
      a.list[base[b] + rank] = (int32_t)q;
    }
  }
}

// ---------------------------------------------------------------------------
// Learned step: features -> network -> gate -> FP64 fallback list
// ---------------------------------------------------------------------------
constexpr int NIN = S + 3, NOUT = S + 1;

enum { SUR_FALLBACK = 0, SUR_ACCEPT, SUR_GATED, SUR_R_DOMAIN, SUR_R_ELEM, SUR_R_NEG, SUR_R_ENERGY,
       SUR_R_CONF, SUR_R_RATE, SUR_FROZEN, SUR_CAND, SUR_RECHECK, SUR_SLOTS = 12 };
constexpr int SUR_NREASONS = SUR_R_RATE - SUR_R_DOMAIN + 1;

struct SurArgs {
  GridIdx g;
  double dt, t_gate;
  const MechCoef *mech;
  const double *T, *p, *rho;
  const double *Y[S];
  const int8_t *bc;
  float in_shift[NIN], in_scale[NIN], out_shift[NOUT], out_scale[NOUT];
  float y_floor;
  double t_min, t_max, p_min, p_max;
  int dt_ok;
  double elem_tol, elem_floor, y_neg_tol, energy_tol, dT_max, dT_freeze, dY_freeze, rate_tol;
  int ne;
  double E[NRG_SUR_MAX_ELEMENTS][S];
  const int32_t *cand;        // NULL: position p is inner cell p; else inner cell cand[p]
  long long npos;             // positions the network, rate check and gate visit
  int32_t *screen_out;        // the screen: where the cells it does not freeze go
  int screen_slot;            // ... and the counter that numbers them (SUR_CAND, SUR_FALLBACK)
  int screen_fp64;            // 1: the FP64 estimate decides every live cell
  int32_t *recheck;           // cells screen_kernel leaves to rate_screen_kernel ...
  const unsigned long long *recheck_n;   // ... and their number (acc[SUR_RECHECK])
  bf16 *X;                    // npos x MLP_IN_PAD
  const float *Ypred;         // npos x NOUT
  double *Yp[S], *Yp2[S];
  double *Efp;
  int32_t *status;
  int32_t *list;              // fallback cells (inner index)
  int8_t *rate_bad;           // per inner cell: 1 = the rate-consistency test failed
  unsigned long long *acc;    // SUR_* counters
};

NRG_DI bool gated_cell(const SurArgs &a, long long off)
{
  const int8_t bcv = a.bc ? a.bc[off] : (int8_t)0;
  return !(a.T[off] >= a.t_gate && bcv == 0);
}

__global__ void __launch_bounds__(256) featurize_kernel(SurArgs a)
{
  const long long pos = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (pos >= a.npos) return;
  const long long q = a.cand ? (long long)a.cand[pos] : pos;
  const long long off = cell_offset(a.g, q);
  bf16 *x = a.X + pos * MLP_IN_PAD;
  float f[MLP_IN_PAD];
#pragma unroll
  for (int i = 0; i < MLP_IN_PAD; ++i) f[i] = 0.0f;
  if (gated_cell(a, off)) {
    // the FP64 step's handling of a skipped cell (chemical_kinetics_solver.f90:341-346)
#pragma unroll
    for (int s = 0; s < S; ++s) a.Yp[s][off] = 0.0;
    a.Efp[off] = 0.0;
    if (a.status) a.status[off] = NRG_CELL_GATED;
  } else {
    f[0] = (float)a.T[off];
    f[1] = (float)log(a.p[off]);
#pragma unroll
    for (int s = 0; s < S; ++s) f[2 + s] = logf((float)a.Y[s][off] + a.y_floor);
    f[S + 2] = (float)log(a.dt);
#pragma unroll
    for (int i = 0; i < NIN; ++i) f[i] = (f[i] - a.in_shift[i]) * a.in_scale[i];
  }
#pragma unroll
  for (int i = 0; i < MLP_IN_PAD; ++i) x[i] = (bf16)f[i];
}

// Solve the n x n system M z = b in place (n <= 4, partial pivoting).  Loops
// run to the compile-time bound with n as a predicate, so M and b stay in
// registers (row swaps are selects).
NRG_DI bool small_solve(double (&M)[NRG_SUR_MAX_ELEMENTS][NRG_SUR_MAX_ELEMENTS],
                        double (&b)[NRG_SUR_MAX_ELEMENTS], int n)
{
  constexpr int NE = NRG_SUR_MAX_ELEMENTS;
  bool ok = true;
#pragma unroll
  for (int k = 0; k < NE; ++k) {
    if (k >= n) break;
    int piv = k;
    double best = fabs(M[k][k]);
#pragma unroll
    for (int i = k + 1; i < NE; ++i)
      if (i < n && fabs(M[i][k]) > best) {
        piv = i;
        best = fabs(M[i][k]);
      }
    if (best == 0.0) ok = false;
#pragma unroll
    for (int i = k + 1; i < NE; ++i) {
      const bool sw = (piv == i);
#pragma unroll
      for (int j = 0; j < NE; ++j) {
        const double t = M[k][j];
        M[k][j] = sw ? M[i][j] : M[k][j];
        M[i][j] = sw ? t : M[i][j];
      }
      const double t = b[k];
      b[k] = sw ? b[i] : b[k];
      b[i] = sw ? t : b[i];
    }
#pragma unroll
    for (int i = k + 1; i < NE; ++i) {
      if (i >= n) break;
      const double f = M[i][k] / M[k][k];
#pragma unroll
      for (int j = k; j < NE; ++j) M[i][j] -= f * M[k][j];
      b[i] -= f * b[k];
    }
  }
#pragma unroll
  for (int k = NE - 1; k >= 0; --k) {
    if (k >= n) continue;
    double s = b[k];
#pragma unroll
    for (int j = k + 1; j < NE; ++j)
      if (j < n) s -= M[k][j] * b[j];
    b[k] = s / M[k][k];
  }
  return ok;
}

// The per-reason counts are summed per block in LDS and added to the global
// counters once per block.
// The rate-consistency test of the gate, in a kernel of its own (the gate
// kernel's registers leave no room for the rate constants).  For every live
// cell the answer the gate would give before its conservation checks (the
// network's increment, or zero for a cell it freezes) is compared with the
// explicit estimate of the step, C_s(t+dt) - C_s = omega_s(C, T) dt, from the
// FP64 rate constants (EstimateMath transcendentals) and mass action at the
// cell's own state;
// rate_bad[q] = 1 where some active species differs by more than rate_tol in
// mass fraction.  As in rates_kernel, waves 0-1 and 2-3 of a block take the
// two halves of the reactions for the same 128 cells (one half per thread
// fits in half the registers) and add their parts of omega in LDS.
constexpr int RCHECK_CELLS = 128;

__global__ void __launch_bounds__(256) rate_check_kernel(SurArgs a)
{
  __shared__ MechCoef mc;
  __shared__ double part[RCHECK_CELLS][SA];
  stage_mech(mc, a.mech);
  const int group = __builtin_amdgcn_readfirstlane(threadIdx.x / RCHECK_CELLS);
  const int local = threadIdx.x % RCHECK_CELLS;
  const long long pos = (long long)blockIdx.x * RCHECK_CELLS + local;
  const long long q = pos < a.npos ? (a.cand ? (long long)a.cand[pos] : pos) : 0;
  const long long off = pos < a.npos ? cell_offset(a.g, q) : 0;
  const bool live = pos < a.npos && !gated_cell(a, off);
  double y[S], C[S], Zd[SA];
  double rho = 1.0;
  if (live) {
    rho = a.rho[off];
#pragma unroll
    for (int s = 0; s < S; ++s) {
      y[s] = a.Y[s][off];
      C[s] = (y[s] * rho) / mc.W[s];
    }
    if (group == 0) explicit_rates<EstimateMath, 0, R / 2>(mc, a.T[off], C, Zd);
    else explicit_rates<EstimateMath, R / 2, R>(mc, a.T[off], C, Zd);
    if (group == 1) {
#pragma unroll
      for (int i = 0; i < SA; ++i) part[local][i] = Zd[i];
    }
  }
  __syncthreads();
  if (group != 0 || pos >= a.npos) return;
  int8_t bad = 0;
  if (live) {
    const float *yp = a.Ypred + pos * NOUT;
    const double dT = (double)yp[0] * a.out_scale[0] + a.out_shift[0];
    double dy[S], dymax = 0.0;
#pragma unroll
    for (int s = 0; s < S; ++s) {
      dy[s] = (double)yp[1 + s] * a.out_scale[1 + s] + a.out_shift[1 + s];
      dymax = fmax(dymax, fabs(dy[s]));
    }
    const bool frozen = a.dT_freeze > 0.0 && fabs(dT) <= a.dT_freeze && dymax <= a.dY_freeze;
#pragma unroll
    for (int i = 0; i < SA; ++i) {
      const int s = kSp.full[i];
      const double est = (((Zd[i] + part[local][i]) * a.dt) * mc.W[s]) / rho;
      if (!(fabs(est - (frozen ? 0.0 : dy[s])) <= a.rate_tol)) bad = 1;
    }
  }
  a.rate_bad[pos] = bad;
}

// The explicit-rate screen: the learned step's freeze test without the
// network.  For every live cell it forms the explicit estimate of the step,
// dY_s = omega_s(C, T) dt W_s / rho (rate constants and mass action as in
// rate_check_kernel), and the temperature change that estimate implies at the
// cell's frozen cv, dT = -(sum_s e_s(T) dY_s / W_s) / cv with
// cv = sum_s (Y_s / W_s)(cp_s(T) - R).  A cell with every |dY_s| <= dY_freeze
// and |dT| <= dT_freeze is taken as inert and gets the zero increment (the FP64
// step's outputs for a cell whose concentrations do not change).  Every other
// live cell is appended to screen_out: the network's candidates, or, for the
// method without the network, the FP64 fallback list.  Gated cells get the
// FP64 step's outputs for a skipped cell (chemical_kinetics_solver.f90:341-346).
//
// Two kernels share the work, and the decision is always the one the FP64
// estimate gives.  screen_kernel visits every inner cell and evaluates the
// estimate with FP64 exponents and FP32 exponentials (the transcendentals
// that make up most of the FP64 estimate's cost), carrying a bound on its
// distance from the FP64 estimate.  Where the bound settles the decision it
// decides; the other live cells go to a list, which rate_screen_kernel then
// decides with the FP64 estimate itself.

NRG_DI void freeze_outputs(const SurArgs &a, long long off)
{
#pragma unroll
  for (int s = 0; s < S; ++s) {
    a.Yp[s][off] = 0.0;
    a.Yp2[s][off] = 0.0;
  }
  a.Efp[off] = 0.0;
  if (a.status) a.status[off] = NRG_CELL_SURROGATE;
}

// Appends the wave's lanes with `take` to out[] at the counter *ctr.
NRG_DI void wave_append(bool take, int lane, long long q, int32_t *out, unsigned long long *ctr)
{
  const unsigned long long mask = __ballot(take ? 1 : 0);
  if (!mask) return;
  const int leader = __ffsll((long long)mask) - 1;
  unsigned long long base = 0;
  if (lane == leader) base = atomicAdd(ctr, (unsigned long long)__popcll(mask));
  base = __shfl(base, leader, WAVE);
  if (take) out[base + __popcll(mask & ((1ull << lane) - 1ull))] = (int32_t)q;
}

// The FP64 decision on the cells screen_kernel lists (recheck[0, *recheck_n)).
// Waves 0-1 and 2-3 of a block take the two halves of the reactions for the
// same 128 cells, as in rate_check_kernel; blocks stride over the list.
__global__ void __launch_bounds__(256) rate_screen_kernel(SurArgs a)
{
  const long long npos = (long long)*a.recheck_n;
  if ((long long)blockIdx.x * RCHECK_CELLS >= npos) return;   // the whole block
  __shared__ MechCoef mc;
  __shared__ double part[RCHECK_CELLS][SA];
  __shared__ double rW[S];   // 1 / W_s: the estimate multiplies where the step divides
  __shared__ unsigned long long blk[SUR_SLOTS];
  if (threadIdx.x < SUR_SLOTS) blk[threadIdx.x] = 0ull;
  if (threadIdx.x < S) rW[threadIdx.x] = 1.0 / a.mech->W[threadIdx.x];
  stage_mech(mc, a.mech);
  const int group = __builtin_amdgcn_readfirstlane(threadIdx.x / RCHECK_CELLS);
  const int lane = threadIdx.x & (WAVE - 1);
  const int local = threadIdx.x % RCHECK_CELLS;
  for (long long p0 = (long long)blockIdx.x * RCHECK_CELLS; p0 < npos;
       p0 += (long long)gridDim.x * RCHECK_CELLS) {
    // the coefficients in LDS are read where they are used, not held in
    // registers across the loop
    asm volatile("" ::: "memory");
    const long long pos = p0 + local;
    const bool live = pos < npos;   // listed cells are live
    const long long q = live ? (long long)a.recheck[pos] : 0;
    const long long off = live ? cell_offset(a.g, q) : 0;
    double C[S], Zd[SA];
    double rho = 1.0, T = 0.0;
    if (live) {
      rho = a.rho[off];
      T = a.T[off];
#pragma unroll
      for (int s = 0; s < S; ++s) C[s] = (a.Y[s][off] * rho) * rW[s];
      if (group == 0) explicit_rates<EstimateMath, 0, R / 2>(mc, T, C, Zd);
      else explicit_rates<EstimateMath, R / 2, R>(mc, T, C, Zd);
      if (group == 1) {
#pragma unroll
        for (int i = 0; i < SA; ++i) part[local][i] = Zd[i];
      }
    }
    __syncthreads();
    if (group == 0) {
      bool frozen = false;
      if (live) {
        double dymax = 0.0, de = 0.0, cv = 0.0;
        const double rrho = 1.0 / rho;
#pragma unroll
        for (int i = 0; i < SA; ++i) {
          const int s = kSp.full[i];
          const double est = (((Zd[i] + part[local][i]) * a.dt) * mc.W[s]) * rrho;
          dymax = fmax(dymax, fabs(est));
          de += e_molar(mc, T, s) * (est * rW[s]);
        }
#pragma unroll
        for (int s = 0; s < S; ++s) cv += (C[s] * rrho) * (cp_molar(mc, T, s) - R_GAS_J);
        const double dT = -de / cv;
        frozen = a.dT_freeze > 0.0 && dymax <= a.dY_freeze && fabs(dT) <= a.dT_freeze;
        if (frozen) freeze_outputs(a, off);
      }
      wave_append(live && !frozen, lane, q, a.screen_out, &a.acc[a.screen_slot]);
      const unsigned long long c_frz = __popcll(__ballot(live && frozen ? 1 : 0));
      if (lane == 0 && c_frz) {
        atomicAdd(&blk[SUR_ACCEPT], c_frz);
        atomicAdd(&blk[SUR_FROZEN], c_frz);
      }
    }
    __syncthreads();   // part[] is rewritten by the next slice
  }
  if (threadIdx.x < SUR_SLOTS && (int)threadIdx.x != a.screen_slot && blk[threadIdx.x])
    atomicAdd(&a.acc[threadIdx.x], blk[threadIdx.x]);
}

// ln x for x > 0 (normal or subnormal): frexp's exponent plus an FP32 log2 of
// the mantissa m in [0.5, 1).  Rounding m to FP32 moves log2 m by at most
// 2^-24 / ln 2 and log2f is within 2 ulp (2^-23 on [-1, 0]), so
// |ln_m32(x) - ln x| < 2^-22, bounded below by SCR_LN_ERR.
constexpr double SCR_LN_ERR = 0x1p-20;
constexpr double SCR_LN2 = 0.69314718055994530942;
constexpr double SCR_LOG2E = 1.4426950408889634074;
constexpr double SCR_LN10 = 2.30258509299404568402;

NRG_DI double ln_m32(double x)
{
  int e;
  const double m = frexp(x, &e);
  return ((double)e + (double)log2f((float)m)) * SCR_LN2;
}

// v = e^x as FP32 exp2 of an FP64 exponent x that is within ex of the exact
// one, and err, a bound on |v - e^x_exact|: rounding x log2(e) to FP32 moves
// the value by at most |x| 2^-24 relative and exp2f is within 2 ulp (2^-22),
// here taken as 2^-23 |x| and 2^-21; e^ex - 1 <= 1.01 ex for ex <= 0.01; and
// FP32 results below its normal range add at most 2^-125 (exponents below
// -100 give the value 0 with that bound).  Returns false where the value
// overflows FP32, is NaN, or the bound exceeds 1 %.
NRG_DI bool exp_term(double x, double ex, double &v, double &err)
{
  if (x == -INFINITY) {   // a zero rate constant or third-body concentration
    v = 0.0;
    err = 0.0;
    return true;
  }
  if (x < -100.0) {       // below FP32's range: e^(x + ex) < e^-99 < 2^-125 for ex <= 1
    v = 0.0;
    err = 0x1p-125;
    return ex <= 1.0;
  }
  const double rel = ex + fabs(x) * 0x1p-23 + 0x1p-21;
  const float y = exp2f((float)(x * SCR_LOG2E));
  v = (double)y;
  err = rel * 1.01 * v + 0x1p-125;
  return y <= 3.0e38f && rel <= 0.01;
}

// Stoichiometry of species s in reaction r: right minus left count, and the
// number of times it appears (the bound adds a term's error once per
// appearance, as the right-hand side adds the term).
constexpr int nu_net(int r, int s)
{
  int n = 0;
  for (int c = 0; c < 3; ++c) {
    if (c < topo::nr[r] && topo::right[r][c] == s) ++n;
    if (c < topo::nl[r] && topo::left[r][c] == s) --n;
  }
  return n;
}
constexpr int nu_occ(int r, int s)
{
  int n = 0;
  for (int c = 0; c < 3; ++c) {
    if (c < topo::nr[r] && topo::right[r][c] == s) ++n;
    if (c < topo::nl[r] && topo::left[r][c] == s) ++n;
  }
  return n;
}

// Screen estimate of one cell: FP64 exponents (ln k_f, ln K_p, ln [M], ln C
// from ln_m32) and FP32 exponentials.  acc[i] = sum over the reactions of
// nu (F - B) for active species i, bnd[i] a bound on its distance from the
// FP64 estimate's sum.  The reactions' arithmetic follows reaction_k (rate
// constants, chemical_kinetics_solver.f90:394-485) and rhs_reaction (mass
// action, :507-536) in logarithms:
//   ln k_f = ln A + b ln T - E/(R T)
//   fall-off: ln k_f = ln k_inf - ln(1 + 1/P_r) [+ ln F for Troe, with
//             ln F = ln F_cent / (1 + x^2)], ln P_r = ln k_0 + ln [M] - ln k_inf
//   ln k_r = ln k_f - ln K_p + d_nu ln(R_u T / P_atm)
// Returns false (the FP64 path decides the cell) where a term leaves FP32's
// range, a bound exceeds 1 % or a quantity the logarithms need is not
// positive (a negative concentration or [M], a Troe denominator near zero).
NRG_DI bool screen_estimate(const MechCoef &mc, double Tin, const double (&C)[S], double (&acc)[SA],
                            double (&bnd)[SA], double (&H)[S])
{
  const double T = dmin(Tin, 10000.0);
  const double lnT = log(T), rT = 1.0 / T;
  const double ln_x = mc.ln_patm_r - lnT;   // ln(P_atm / (R_u T))
  bool ok = true;
  double lnC[S], G[S];                    // G_s = s_s/R - h_s/(R T): ln K_p = sum nu G
  unsigned absent = 0;
#pragma unroll
  for (int s = 0; s < S; ++s) {
    ok = ok && C[s] >= 0.0;
    absent |= (C[s] == 0.0) ? 1u << s : 0u;
    lnC[s] = C[s] > 0.0 ? ln_m32(C[s]) : 0.0;
    H[s] = h_molar<EstimateMath>(mc, T, s);
    G[s] = s_molar<EstimateMath>(mc, T, s) * (1.0 / R_GAS_J) - (H[s] * (1.0 / R_GAS_J)) * rT;
    // each species' values are formed here, in turn: left to the compiler,
    // every species' coefficients were loaded at once (twice the registers)
    asm volatile("" : "+v"(G[s]), "+v"(lnC[s]), "+v"(H[s]));
  }
#pragma unroll
  for (int i = 0; i < SA; ++i) {
    acc[i] = 0.0;
    bnd[i] = 0.0;
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const bool fwd = (absent & side_mask(r, 0)) == 0;
    const bool rev = has_reverse(r) && (absent & side_mask(r, 1)) == 0;
    if (!__any((fwd || rev) ? 1 : 0)) continue;
    const int rt = topo::rtype[r];
    double m = 0.0, lm = 0.0;
    if (uses_m(r)) {
#pragma unroll
      for (int s = 0; s < S; ++s) m = m + C[s] * mc.eff[r][s];
      lm = m > 0.0 ? ln_m32(m) : -INFINITY;
    }
    // ln k_f and a bound on its error
    // (rok: this reaction's checks, which matter only where the cell has a
    // term of it)
    double lkf = mc.lnA[r] + mc.beta[r] * lnT + mc.mE_R[r] * rT, ekf = 0.0;
    bool rok = true;
    if (rt == 2 || rt == 3 || rt == 7) {
      const double lk0 = mc.lnA_low[r] + mc.beta_low[r] * lnT + mc.mElow_R[r] * rT;
      // P_r = 0 ([M] = 0: every efficiency of the cell's species zero, or
      // k_0 = 0): k_f = k_inf * 0 * F = 0 exactly in the FP64 estimate too
      const bool zero_pr = m == 0.0 || lk0 == -INFINITY;
      const double lpr = zero_pr ? 0.0 : lk0 + lm - lkf;
      rok = m >= 0.0 && lpr > -1e4 && lpr < 1e4;
      // ln(P_r / (1 + P_r)) = -softplus(-ln P_r) in FP32: the argument's
      // rounding, expf and log1pf (2 ulp each) and the sum stay within
      // (|ln P_r| + 1) 2^-23 + 2^-21; ln [M] adds SCR_LN_ERR
      const float z = (float)(-lpr);
      const float sp = z > 0.0f ? z + log1pf(expf(-z)) : log1pf(expf(z));
      lkf = lkf - (double)sp;
      ekf = SCR_LN_ERR + (fabs(lpr) + 1.0) * 0x1p-23 + 0x1p-21;
      if (rt == 3) {
        double e1, e2, e3, r1, r2, r3;
        rok = exp_term(-(T / mc.troe[1][r]), 0.0, e1, r1) && rok;
        rok = exp_term(-(T / mc.troe[2][r]), 0.0, e2, r2) && rok;
        rok = exp_term(-(mc.troe[3][r] * rT), 0.0, e3, r3) && rok;
        const double fcent = (mc.one_m_alpha[r] * e1 + mc.troe[0][r] * e2) + e3;
        const double efc = fabs(mc.one_m_alpha[r]) * r1 + fabs(mc.troe[0][r]) * r2 + r3;
        // (with P_r = 0 the FP64 estimate multiplies 0 by F_cent^(-1/0.14),
        // finite for F_cent above 1e-40)
        rok = rok && fcent > 0.0 && efc <= 0.001 * fcent && (!zero_pr || fcent > 1e-40);
        const double lnfc = ln_m32(fcent > 0.0 ? fcent : 1.0);
        const double elnfc = SCR_LN_ERR + 1.01 * efc / (fcent > 0.0 ? fcent : 1.0);
        const double lf = lnfc * (1.0 / SCR_LN10);
        const double cc = -0.4 - 0.67 * lf, nn = 0.75 - 1.27 * lf;
        const double nume = lpr * (1.0 / SCR_LN10) + cc;
        const double den = nn - 0.14 * nume;
        const double xx = nume / den;
        // perturbations of the numerator and denominator of x from ln [M]
        // and ln F_cent, and the resulting bound on |x - x_FP64|; the
        // derivative of 1 / (1 + x^2) is at most 0.65 in magnitude
        const double elf = elnfc * (1.0 / SCR_LN10);
        const double dnum = SCR_LN_ERR * (1.0 / SCR_LN10) + 0.67 * elf;
        const double dden = 1.27 * elf + 0.14 * dnum;
        rok = rok && (zero_pr || (fabs(den) > 0.0625 && fabs(den) > 2.0 * dden));
        const double adn = fabs(den) > 2.0 * dden ? fabs(den) : 1.0;
        const double exx = (dnum * adn + fabs(nume) * dden) / (adn * (adn - dden));
        lkf = lkf + lnfc / (1.0 + xx * xx);
        ekf = ekf + fabs(lnfc) * 0.65 * exx + elnfc;
      }
      if (zero_pr) lkf = -INFINITY;
    }
    // forward and reverse terms of the mass action
    double xf = lkf, ef = ekf;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const int sp = topo::left[r][c];
      if (c < topo::nl[r]) {
        xf = xf + ((sp == S) ? lm : lnC[sp < S ? sp : 0]);
        ef = ef + SCR_LN_ERR;
      }
    }
    ok = ok && (rok || !(fwd || rev));
    double F = 0.0, eF = 0.0;
    if (fwd) ok = exp_term(xf, ef, F, eF) && ok;
    double B = 0.0, eB = 0.0;
    if (has_reverse(r)) {
      double lnKp = 0.0;
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const int sp = topo::right[r][c];
        if (c < topo::nr[r] && sp != S) lnKp = lnKp + G[sp < S ? sp : 0];
      }
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const int sp = topo::left[r][c];
        if (c < topo::nl[r] && sp != S) lnKp = lnKp - G[sp < S ? sp : 0];
      }
      const double d_nu = (double)(topo::nr[r] - topo::nl[r]);
      double xb = (lkf - lnKp) - d_nu * ln_x, eb = ekf;
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const int sp = topo::right[r][c];
        if (c < topo::nr[r]) {
          xb = xb + ((sp == S) ? lm : lnC[sp < S ? sp : 0]);
          eb = eb + SCR_LN_ERR;
        }
      }
      if (rev) ok = exp_term(xb, eb, B, eB) && ok;
    }
#pragma unroll
    for (int i = 0; i < SA; ++i) {
      const int s = kSp.full[i];
      if (nu_net(r, s) != 0) acc[i] = acc[i] + (double)nu_net(r, s) * (F - B);
      if (nu_occ(r, s) != 0) bnd[i] = bnd[i] + (double)nu_occ(r, s) * (eF + eB);
    }
  }
  return ok;
}

enum { SCR_FROZEN = 0, SCR_PASS = 1, SCR_RECHECK = 2 };   // screen_kernel's outcome for a live cell

// The screen over every inner cell (a block per 256 cells, one cell per
// thread; a loop over slices would hold the expansions' FP64 constants in
// registers across it and halve the resident waves).  Outcomes: gated, frozen, passed on (screen_out), or
// listed for rate_screen_kernel (recheck).  With screen_fp64 every live cell
// is listed, so the FP64 estimate decides every cell.
__global__ void __launch_bounds__(256) screen_kernel(SurArgs a)
{
  __shared__ MechCoef mc;
  __shared__ double rW[S];
  __shared__ unsigned long long blk[SUR_SLOTS];
  if (threadIdx.x < SUR_SLOTS) blk[threadIdx.x] = 0ull;
  if (threadIdx.x < S) rW[threadIdx.x] = 1.0 / a.mech->W[threadIdx.x];
  stage_mech(mc, a.mech);
  const int lane = threadIdx.x & (WAVE - 1);
  const long long n = a.g.ninner;
  const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const bool valid = q < n;
  const long long off = valid ? cell_offset(a.g, q) : 0;
  // every input in one round trip to memory (the loads do not wait for the
  // gate test, as in gated_cell)
  double T = 0.0, rho = 1.0, y[S];
  int8_t bcv = 0;
  if (valid) {
    T = a.T[off];
    bcv = a.bc ? a.bc[off] : (int8_t)0;
    rho = a.rho[off];
#pragma unroll
    for (int s = 0; s < S; ++s) y[s] = a.Y[s][off];
  }
  const bool gated = valid && !(T >= a.t_gate && bcv == 0);
  const bool live = valid && !gated;
  int outcome = SCR_PASS;
  if (live) {
    double C[S], acc[SA], bnd[SA], H[S];
#pragma unroll
    for (int s = 0; s < S; ++s) C[s] = (y[s] * rho) * rW[s];
    const bool ok = screen_estimate(mc, T, C, acc, bnd, H);
    // the decision with the FP64 estimate's expressions, each side of each
    // threshold taken only where the bound puts the FP64 estimate there too
    const double rrho = 1.0 / rho;
    bool in = true, out = false;
    double de = 0.0, bde = 0.0, dabs = 0.0, cv = 0.0;
#pragma unroll
    for (int i = 0; i < SA; ++i) {
      const int s = kSp.full[i];
      const double est = ((acc[i] * a.dt) * mc.W[s]) * rrho;
      const double b = (((bnd[i] * a.dt) * mc.W[s]) * rrho) * (1.0 + 0x1p-40);
      in = in && fabs(est) + b <= a.dY_freeze;
      out = out || fabs(est) - b > a.dY_freeze;
      // e_s as e_molar forms it, from h_s with a5 * (1/T) where h_molar
      // divides: within 2^-50 (|a5| + |h_s|) of the FP64 estimate's e_s
      const double e = H[s] - R_GAS_J * T;
      de += e * (est * rW[s]);
      bde += fabs(e) * (b * rW[s]);
      const double ea = fabs(e) + 0x1p-10 * (fabs(mc.a[s][0][5]) + fabs(mc.a[s][1][5]) + fabs(H[s]));
      dabs += ea * ((fabs(est) + b) * rW[s]);
      asm volatile("" : "+v"(de), "+v"(bde), "+v"(dabs));   // in turn, as in screen_estimate
    }
#pragma unroll
    for (int s = 0; s < S; ++s) {
      cv += (C[s] * rrho) * (cp_molar(mc, T, s) - R_GAS_J);
      asm volatile("" : "+v"(cv));
    }
    // bT bounds |dT - dT_FP64|: the bounds on the estimates, the two e_s
    // and the FP64 roundings of both sums (dabs)
    const double dT = -de / cv;
    const double bT = (bde + dabs * 0x1p-40) / cv + fabs(dT) * 0x1p-40;
    const bool sane = ok && cv > 0.0 && bT < INFINITY && fabs(dT) < INFINITY;
    in = in && fabs(dT) + bT <= a.dT_freeze;
    out = out || fabs(dT) - bT > a.dT_freeze;
    outcome = (!sane || a.screen_fp64) ? SCR_RECHECK : out ? SCR_PASS : in ? SCR_FROZEN : SCR_RECHECK;
    if (outcome == SCR_FROZEN) freeze_outputs(a, off);
  }
  if (gated) {
#pragma unroll
    for (int s = 0; s < S; ++s) a.Yp[s][off] = 0.0;
    a.Efp[off] = 0.0;
    if (a.status) a.status[off] = NRG_CELL_GATED;
  }
  wave_append(live && outcome == SCR_PASS, lane, q, a.screen_out, &a.acc[a.screen_slot]);
  wave_append(live && outcome == SCR_RECHECK, lane, q, a.recheck, &a.acc[SUR_RECHECK]);
  const unsigned long long c_frz = __popcll(__ballot(live && outcome == SCR_FROZEN ? 1 : 0));
  const unsigned long long c_gat = __popcll(__ballot(gated ? 1 : 0));
  if (lane == 0) {
    if (c_frz) {
      atomicAdd(&blk[SUR_ACCEPT], c_frz);
      atomicAdd(&blk[SUR_FROZEN], c_frz);
    }
    if (c_gat) atomicAdd(&blk[SUR_GATED], c_gat);
  }
  __syncthreads();
  if (threadIdx.x < SUR_SLOTS && (int)threadIdx.x != a.screen_slot && (int)threadIdx.x != SUR_RECHECK &&
      blk[threadIdx.x])
    atomicAdd(&a.acc[threadIdx.x], blk[threadIdx.x]);
}

template <bool RATE>
__global__ void __launch_bounds__(256) gate_kernel(SurArgs a)
{
  __shared__ MechCoef mc;
  __shared__ unsigned long long blk[SUR_SLOTS];
  if (threadIdx.x < SUR_SLOTS) blk[threadIdx.x] = 0ull;
  stage_mech(mc, a.mech);
  const int lane = threadIdx.x & (WAVE - 1);
  const long long pos = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const bool valid = pos < a.npos;
  const long long q = valid ? (a.cand ? (long long)a.cand[pos] : pos) : 0;
  const long long off = valid ? cell_offset(a.g, q) : 0;
  const bool gated = valid && gated_cell(a, off);
  const bool live = valid && !gated;
  int reason = 0;   // 0 accept, else SUR_R_*
  if (live) {
    const double T = a.T[off], p = a.p[off], rho = a.rho[off];
    double y[S], dy[S];
#pragma unroll
    for (int s = 0; s < S; ++s) y[s] = a.Y[s][off];
    const float *yp = a.Ypred + pos * NOUT;
    const double dT = (double)yp[0] * a.out_scale[0] + a.out_shift[0];
    bool finite = isfinite(dT);
#pragma unroll
    for (int s = 0; s < S; ++s) {
      dy[s] = (double)yp[1 + s] * a.out_scale[1 + s] + a.out_shift[1 + s];
      finite = finite && isfinite(dy[s]);
    }
    bool frozen = false;
    if (!finite || !(T >= a.t_min && T <= a.t_max && p >= a.p_min && p <= a.p_max) || !a.dt_ok) {
      reason = SUR_R_DOMAIN;
    } else {
      double dymax = 0.0;
#pragma unroll
      for (int s = 0; s < S; ++s) dymax = fmax(dymax, fabs(dy[s]));
      frozen = a.dT_freeze > 0.0 && fabs(dT) <= a.dT_freeze && dymax <= a.dY_freeze;
      if (!frozen && !(fabs(dT) <= a.dT_max)) reason = SUR_R_CONF;
      if (RATE && reason == 0 && a.rate_bad[pos]) {
        frozen = false;
        reason = SUR_R_RATE;
      }
    }
    if (frozen) {
      // inert: the FP64 step's outputs for a cell whose concentrations do not change
#pragma unroll
      for (int s = 0; s < S; ++s) {
        a.Yp[s][off] = 0.0;
        a.Yp2[s][off] = 0.0;
      }
      a.Efp[off] = 0.0;
      if (a.status) a.status[off] = NRG_CELL_SURROGATE;
    }
    if (frozen) reason = -1;
    // element balance of the raw increment: sum_s E_es dY_s / W_s  [mol/kg]
    double res[NRG_SUR_MAX_ELEMENTS] = {0.0, 0.0, 0.0, 0.0};
    double d[S];
    if (reason == 0) {
#pragma unroll
      for (int e = 0; e < NRG_SUR_MAX_ELEMENTS; ++e) {
        if (e >= a.ne) break;
        double r = 0.0, sc = 0.0;
#pragma unroll
        for (int s = 0; s < S; ++s) {
          r += a.E[e][s] * dy[s] / mc.W[s];
          sc += a.E[e][s] * fabs(dy[s]) / mc.W[s];
        }
        res[e] = r;
        if (fabs(r) > a.elem_tol * sc + a.elem_floor) reason = SUR_R_ELEM;
      }
    }
    if (reason == 0) {
      // project onto sum_s E_es dY_s / W_s = 0, weighting the correction by |dY_s|
      double M[NRG_SUR_MAX_ELEMENTS][NRG_SUR_MAX_ELEMENTS] = {};
#pragma unroll
      for (int s = 0; s < S; ++s) d[s] = fabs(dy[s]) + 1e-12;
#pragma unroll
      for (int e = 0; e < NRG_SUR_MAX_ELEMENTS; ++e)
#pragma unroll
        for (int f = 0; f < NRG_SUR_MAX_ELEMENTS; ++f) {
          if (e >= a.ne || f >= a.ne) continue;
          double m = 0.0;
#pragma unroll
          for (int s = 0; s < S; ++s) m += a.E[e][s] * a.E[f][s] * d[s] / (mc.W[s] * mc.W[s]);
          M[e][f] = m;
        }
      if (small_solve(M, res, a.ne)) {
#pragma unroll
        for (int s = 0; s < S; ++s) {
          double c = 0.0;
#pragma unroll
          for (int e = 0; e < NRG_SUR_MAX_ELEMENTS; ++e)
            if (e < a.ne) c += a.E[e][s] * res[e];
          dy[s] -= d[s] * c / mc.W[s];
        }
      }
#pragma unroll
      for (int s = 0; s < S; ++s)
        if (y[s] + dy[s] < -a.y_neg_tol) reason = SUR_R_NEG;
    }
    double dc[S], efp = 0.0;
    if (reason == 0) {
      // chemistry sources of the projected increment, as the FP64 step writes them
#pragma unroll
      for (int s = 0; s < S; ++s) {
        dc[s] = (rho * dy[s]) / mc.W[s];
        efp = efp - (mc.h_ref[s] * dc[s]) / a.dt;
      }
      // energy: E_f(T, Y), source application and e->T, as nrg_chem_closure_dev
      double avg = 0.0, X[S], e0 = 0.0, hc = 0.0;
#pragma unroll
      for (int s = 0; s < S; ++s) avg = avg + y[s] / mc.W[s];
      double wmix = 1.0 / avg;
#pragma unroll
      for (int s = 0; s < S; ++s) X[s] = (y[s] / mc.W[s]) * wmix;
#pragma unroll
      for (int s = 0; s < S; ++s) {
        e0 = e0 + e_molar(mc, T, s) * X[s];
        hc = hc + mc.h_ref[s] * X[s];
      }
      const double Ef = (e0 - hc) / wmix + (0.0 + efp * a.dt) / rho;
      double y1[S], sum = 0.0;
#pragma unroll
      for (int s = 0; s < S; ++s) {
        y1[s] = y[s] + (0.0 + ((rho * dy[s]) / a.dt) * a.dt) / rho;
        sum = sum + y1[s];
      }
      avg = 0.0;
#pragma unroll
      for (int s = 0; s < S; ++s) {
        y1[s] = dmax(y1[s], 0.0) / sum;
        avg = avg + y1[s] / mc.W[s];
      }
      wmix = 1.0 / avg;
#pragma unroll
      for (int s = 0; s < S; ++s) X[s] = (y1[s] / mc.W[s]) * wmix;
      const double T1 = calculate_temperature(mc, T, Ef * wmix, X);
      if (!(fabs(dT - (T1 - T)) <= a.energy_tol)) reason = SUR_R_ENERGY;
    }
    if (reason == 0) {
#pragma unroll
      for (int s = 0; s < S; ++s) {
        a.Yp[s][off] = (dc[s] * mc.W[s]) / a.dt;
        a.Yp2[s][off] = dc[s];
      }
      a.Efp[off] = efp;
      if (a.status) a.status[off] = NRG_CELL_SURROGATE;
    }
  }
  const bool rej = live && reason > 0;
  const unsigned long long mask = __ballot(rej ? 1 : 0);
  if (mask) {
    const int leader = __ffsll((long long)mask) - 1;
    unsigned long long base = 0;
    if (lane == leader) base = atomicAdd(&a.acc[SUR_FALLBACK], (unsigned long long)__popcll(mask));
    base = __shfl(base, leader, WAVE);
    if (rej) a.list[base + __popcll(mask & ((1ull << lane) - 1ull))] = (int32_t)q;
  }
  const unsigned long long c_acc = __popcll(__ballot(live && reason <= 0 ? 1 : 0));
  const unsigned long long c_frz = __popcll(__ballot(live && reason < 0 ? 1 : 0));
  const unsigned long long c_gat = __popcll(__ballot(gated ? 1 : 0));
  unsigned long long c_r[SUR_NREASONS];
#pragma unroll
  for (int i = 0; i < SUR_NREASONS; ++i)
    c_r[i] = __popcll(__ballot(rej && reason == SUR_R_DOMAIN + i ? 1 : 0));
  if (lane == 0) {
    atomicAdd(&blk[SUR_ACCEPT], c_acc);
    atomicAdd(&blk[SUR_GATED], c_gat);
    atomicAdd(&blk[SUR_FROZEN], c_frz);
#pragma unroll
    for (int i = 0; i < SUR_NREASONS; ++i) atomicAdd(&blk[SUR_R_DOMAIN + i], c_r[i]);
  }
  __syncthreads();
  if (threadIdx.x < SUR_SLOTS && threadIdx.x != SUR_FALLBACK && blk[threadIdx.x])
    atomicAdd(&a.acc[threadIdx.x], blk[threadIdx.x]);
}

}  // namespace kern
using namespace kern;

// ===========================================================================
// Scratch of nrg_chem_step_dev_noalloc: the work accumulators and queue heads
// (ACC_SLOTS words, padded to 1024 bytes), then the cell records of one chunk
// of NRG_NOALLOC_CHUNK_CELLS cells.  One copy per device, held until the
// process ends.  Host code reaches it only through the per-device address
// hipGetSymbolAddress returned (g_noalloc_scratch), never through its name.
// ===========================================================================
constexpr size_t NOALLOC_ACC_BYTES = 1024;
#if NRG_TOPO_PRIMARY
static_assert(ACC_SLOTS * sizeof(unsigned long long) <= NOALLOC_ACC_BYTES, "accumulators");
static_assert(NOALLOC_ACC_BYTES + (size_t)NRG_NOALLOC_CHUNK_CELLS * REC_PAIRS * 2 * sizeof(double) <=
                  (size_t)NRG_NOALLOC_SCRATCH_BYTES, "cell records of one chunk");
static_assert((long long)NRG_NOALLOC_MAX_CELLS <= (long long)MAX_CHUNKS * NRG_NOALLOC_CHUNK_CELLS,
              "one queue head per chunk");
// (one build of the library holds the array; the others refuse the no-alloc entry point)
static __device__ __align__(256) unsigned char scratch[NRG_NOALLOC_SCRATCH_BYTES];
#endif

// ===========================================================================
// Host side
// ===========================================================================
// What a captured step graph depends on: its kernel arguments and the queue set-up.
struct StepKey {
  StepArgs args;
  const double *rates;         // buffer the graph's kernels write (reallocated when it grows)
  int use_hist, form;
  long long chunk_max;
  long long persistent_blocks; // the integrator's grid (the autotuner may change it alone)
  int jacobian;                // NRG_JAC_* and which chunks go one cell to a lane: the
  unsigned long long lanes;    // integrator kernels the graph launches
};

// What a handle's previous call on a grid counted, and what it led to (plan).
struct Seen {
  bool valid = false, alike = false;
  GridIdx g{};
  long long cells = 0, nfe_max = 0;
  double nfe = 0.0, nstep = 0.0;
  unsigned long long lanes = 0;
};

// Pinned memory for the host-pointer entry points' fields, at most (102,000 cells of
// KEROMNES); a handle holds what its largest call up to that has needed, and grows it
// by half at least, as pinning takes ~0.3 ms a MiB.
constexpr size_t STAGE_PINNED_MAX = 24u << 20;

struct nrg_chem_handle {
  int device = 0;
  hipStream_t stream = nullptr;
  MechCoef host_mech{};
  MechCoef *dev_mech = nullptr;
  BdfConst k{};
  nrg_chem_opts opts{};
  unsigned long long *dev_acc = nullptr;   // [16] accumulators + [1] queue head
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  int form = NRG_FORM_PLAIN;
  int jac_pct = 50;
  bool refill_auto = true;                 // the caller has set no refill threshold
  int persistent_blocks = 0;               // resident one-wave blocks of the integrator
  int lane_blocks = 0;                     // and of its one-cell-per-lane form
  // staging for the host-pointer entry point: device, and pinned host memory for small fields
  void *stage = nullptr, *pinned = nullptr;
  size_t stage_bytes = 0, pinned_bytes = 0;
  unsigned long long *acc_host = nullptr;  // pinned: counters on their way back (or NULL)
  // cell records of one chunk: REC_PAIRS pairs of doubles per position
  double *rates = nullptr;
  long long rates_cells = 0;
  long long chunk_max = 1ll << 23;
  // learned step: features, network outputs, fallback list, counters
  hipEvent_t ev2 = nullptr, ev3 = nullptr;
  nrg::bf16 *sur_X = nullptr;
  float *sur_Y = nullptr;
  int32_t *sur_list = nullptr;
  int32_t *sur_cand = nullptr;             // cells the explicit-rate screen hands to the network
  int32_t *sur_recheck = nullptr;          // cells its FP32 pass leaves to the FP64 estimate
  int8_t *sur_rate_bad = nullptr;
  long long recheck_blocks = 0;            // resident blocks of rate_screen_kernel
  unsigned long long *sur_acc = nullptr;
  long long sur_cells = 0;
  // stiffness-ordered queue
  int order = NRG_ORDER_NATURAL;
  int32_t *order_list = nullptr;
  int32_t *hist = nullptr;
  unsigned long long *bins = nullptr;      // count[NBIN], cursor[NBIN]
  long long order_cells = 0;
  Seen seen_step, seen_fallback;           // steps, and fallbacks of the learned step
  bool hist_valid = false;
  GridIdx hist_grid{};
  // table-approximated mode: T_t[rows], then dC_t[S][rows]
  double *table = nullptr;
  int table_rows = 0;
  int table_ascending = 0;
  int num_cu = 1;
  // step graph (opts.use_graph)
  bool use_graph = false;
  hipGraphExec_t graph_exec = nullptr;
  StepKey graph_key{};
  long long graph_captures = 0;
};

namespace {

// Gear coefficient tables EL, TQ for MINT = 2 (slatec/ddcst.f90:39-86): the
// l-vectors of the BDF formulas of orders 1..5, normalised by l1.
void gear_tables(double el[MAXORD][MAXORD + 1], double tq[MAXORD][3])
{
  double E[14][13] = {};      // E[i][j] = EL(i, j), 1-based
  double fact[13] = {};
  fact[1] = 1.0;
  for (int i = 2; i <= MAXORD; ++i) fact[i] = (double)i * fact[i - 1];
  E[1][1] = 1.0;
  E[2][1] = 1.0;
  for (int j = 2; j <= MAXORD; ++j) {
    E[1][j] = fact[j];
    for (int i = 2; i <= j; ++i) E[i][j] = (double)j * E[i][j - 1] + E[i - 1][j - 1];
    E[j + 1][j] = 1.0;
  }
  double harm = 1.0;
  for (int j = 2; j <= MAXORD; ++j) {
    harm = harm + 1.0 / (double)j;
    for (int i = 1; i <= j + 1; ++i) E[i][j] = E[i][j] / (fact[j] * harm);
  }
  for (int nq = 1; nq <= MAXORD; ++nq) {
    for (int j = 1; j <= MAXORD + 1; ++j) el[nq - 1][j - 1] = E[j][nq];
    tq[nq - 1][0] = (nq > 1) ? 1.0 / fact[nq - 1] : 0.0;
    tq[nq - 1][1] = (double)(nq + 1) / E[1][nq];
    tq[nq - 1][2] = (double)(nq + 2) / E[1][nq];
  }
}

int build_mech(const nrg_chem_mech *m, MechCoef &mc)
{
  if (!m) return set_error(NRG_CHEM_E_ARG, "mech is NULL");
  if (m->species_number != S || m->reactions_number != R)
    return set_error(NRG_CHEM_E_MECH, "compiled for S=%d R=%d, got S=%d R=%d", S, R,
                     m->species_number, m->reactions_number);
  if (!m->reactions_type || !m->chemical_coeffs || !m->A || !m->beta || !m->E_act || !m->A_low ||
      !m->beta_low || !m->E_act_low || !m->Troe_coeffs || !m->enhanced_efficiencies ||
      !m->a_coeffs || !m->molar_masses)
    return set_error(NRG_CHEM_E_ARG, "mechanism array pointer is NULL");
  for (int r = 0; r < R; ++r)
    if (m->reactions_type[r] != topo::rtype[r])
      return set_error(NRG_CHEM_E_MECH, "reaction %d has type %d, kernels compiled for %d", r + 1,
                       m->reactions_type[r], topo::rtype[r]);
  for (int i = 0; i < 8 * R; ++i)
    if (m->chemical_coeffs[i] != topo::chemical_coeffs[i])
      return set_error(NRG_CHEM_E_MECH, "chemical_coeffs differ from the compiled topology at %d", i);
  for (int s = 0; s < S; ++s)
    if (!(m->molar_masses[s] > 0.0))
      return set_error(NRG_CHEM_E_MECH, "molar mass of species %d is not positive", s + 1);
  std::memset(&mc, 0, sizeof(mc));
  for (int r = 0; r < R; ++r) {
    mc.A[r] = m->A[r];
    mc.beta[r] = m->beta[r];
    mc.A_low[r] = m->A_low[r];
    mc.beta_low[r] = m->beta_low[r];
    mc.mE_R[r] = (-m->E_act[r]) / R_GAS_J;
    mc.mElow_R[r] = (-m->E_act_low[r]) / R_GAS_J;
    for (int q = 0; q < 4; ++q) mc.troe[q][r] = m->Troe_coeffs[r + R * q];
    mc.one_m_alpha[r] = 1.0 - mc.troe[0][r];
    for (int s = 0; s < S; ++s) mc.eff[r][s] = m->enhanced_efficiencies[r + R * s];
  }
  for (int s = 0; s < S; ++s) {
    for (int set = 0; set < 2; ++set) {
      const double *a = m->a_coeffs + 14 * s + 7 * set;
      for (int i = 0; i < 7; ++i) mc.a[s][set][i] = a[i];
      mc.hdiv[s][set][0] = a[4] / 5.0;
      mc.hdiv[s][set][1] = a[3] / 4.0;
      mc.hdiv[s][set][2] = a[2] / 3.0;
      mc.hdiv[s][set][3] = a[1] / 2.0;
      mc.hdiv[s][set][4] = a[0] / 1.0;
      mc.sdiv[s][set][0] = a[4] / 4.0;
      mc.sdiv[s][set][1] = a[3] / 3.0;
      mc.sdiv[s][set][2] = a[2] / 2.0;
    }
    mc.W[s] = m->molar_masses[s];
  }
  // h_s(T_ref): low-T set (T_ref < 1000 K), same Horner order as the kernel.
  for (int s = 0; s < S; ++s) {
    const double t = T_REF;
    const double *d = mc.hdiv[s][0];
    double hs = d[0];
    for (int i = 1; i < 5; ++i) hs = hs * t + d[i];
    hs = hs + mc.a[s][0][5] / t;
    mc.h_ref[s] = hs * t;
  }
  gear_tables(mc.el, mc.tq);
  mc.patm_r = 101325.0 / R_GAS_J;
  for (int r = 0; r < R; ++r) {
    mc.lnA[r] = std::log(mc.A[r]);
    mc.lnA_low[r] = std::log(mc.A_low[r]);
  }
  mc.ln_patm_r = std::log(mc.patm_r);
  return NRG_CHEM_OK;
}

BdfConst make_const(const nrg_chem_opts &o)
{
  BdfConst k{};
  k.eps = o.eps;
  k.ewt = o.ewt;
  k.hmax = o.hmax;
  k.uround = 2.220446049250313080847e-16;        // epsilon(1d0)
  k.sqrtn = std::sqrt((double)S);
  // with weights under 2^-40 every component (solve, bdf_group.h)
  k.tiny = o.ewt >= 0x1p-40 ? 0x1p-900 : INFINITY;
  k.sqrt_uround = std::sqrt(k.uround);
  k.br = std::pow(k.uround, 0.875);
  k.bl = std::pow(k.uround, 0.75);
  k.bp = std::pow(k.uround, -0.15);
  k.facmin = std::pow(k.uround, 0.78);
  k.t_gate = o.t_gate;
  k.mxstep = o.mxstep;
  k.maxord = std::min(o.mxord, MAXORD);
  k.gather_pct = o.errtest_gather_pct;
  k.refill_idle = o.refill_min_idle > 0                ? o.refill_min_idle
                  : o.cell_order == NRG_ORDER_STIFFNESS ? REFILL_IDLE_ORDERED
                                                        : REFILL_IDLE_NATURAL;
  return k;
}

int make_grid(const nrg_grid *grid, GridIdx &g)
{
  if (!grid) return set_error(NRG_CHEM_E_ARG, "grid is NULL");
  for (int d = 0; d < 3; ++d) {
    if (grid->hi[d] < grid->lo[d]) return set_error(NRG_CHEM_E_ARG, "grid hi < lo in dim %d", d);
    if (grid->inner_lo[d] < grid->lo[d] || grid->inner_hi[d] > grid->hi[d])
      return set_error(NRG_CHEM_E_ARG, "inner bounds outside the field bounds in dim %d", d);
  }
  g.lo0 = grid->lo[0];
  g.lo1 = grid->lo[1];
  g.lo2 = grid->lo[2];
  g.nx = grid->hi[0] - grid->lo[0] + 1;
  g.ny = grid->hi[1] - grid->lo[1] + 1;
  g.ilo0 = grid->inner_lo[0];
  g.ilo1 = grid->inner_lo[1];
  g.ilo2 = grid->inner_lo[2];
  g.ix = std::max(0, grid->inner_hi[0] - grid->inner_lo[0] + 1);
  g.iy = std::max(0, grid->inner_hi[1] - grid->inner_lo[1] + 1);
  g.iz = std::max(0, grid->inner_hi[2] - grid->inner_lo[2] + 1);
  g.ninner = (long long)g.ix * g.iy * g.iz;
  g.pad0 = g.pad1 = 0;
  if (g.ninner > 0) {
    auto off = [&](int i, int j, int k) {
      return (long long)(i - g.lo0) + (long long)g.nx * ((j - g.lo1) + (long long)g.ny * (k - g.lo2));
    };
    g.pad0 = off(grid->inner_lo[0], grid->inner_lo[1], grid->inner_lo[2]) & ~63ll;
    g.pad1 = off(grid->inner_hi[0], grid->inner_hi[1], grid->inner_hi[2]) + 1;
  }
  g.idx32 = g.ninner < (1ll << 31) && g.pad1 < (1ll << 31);
  return NRG_CHEM_OK;
}

long long field_cells(const nrg_grid *grid)
{
  long long n = 1;
  for (int d = 0; d < 3; ++d) n *= (long long)(grid->hi[d] - grid->lo[d] + 1);
  return n;
}

int check_device(int dev)
{
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess || n <= 0)
    return set_error(NRG_CHEM_E_NO_DEVICE, "no HIP device");
  if (dev < 0 || dev >= n) return set_error(NRG_CHEM_E_NO_DEVICE, "device %d out of range", dev);
  hipDeviceProp_t p;
  HIP_TRY(hipGetDeviceProperties(&p, dev));
  if (std::strncmp(p.gcnArchName, "gfx950", 6) != 0)
    return set_error(NRG_CHEM_E_NO_DEVICE, "device %d is %s, kernels are built for gfx950", dev,
                     p.gcnArchName);
  return NRG_CHEM_OK;
}

}  // namespace

// Device address of `scratch` on each device, taken once per device (with that
// device current) when the first handle on it is created.
constexpr int NOALLOC_MAX_DEVICES = 64;
static void *g_noalloc_scratch[NOALLOC_MAX_DEVICES];
static std::mutex g_noalloc_mu;

static int noalloc_setup(int dev)
{
#if !NRG_TOPO_PRIMARY
  (void)dev;
  return NRG_CHEM_OK;
#else
  if (dev < 0 || dev >= NOALLOC_MAX_DEVICES)
    return set_error(NRG_CHEM_E_NO_DEVICE, "device %d beyond the %d the library serves", dev,
                     NOALLOC_MAX_DEVICES);
  std::lock_guard<std::mutex> lock(g_noalloc_mu);
  if (g_noalloc_scratch[dev]) return NRG_CHEM_OK;
  void *ptr = nullptr;
  const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
  if (e != hipSuccess || !ptr)
    return set_error(NRG_CHEM_E_HIP, "hipGetSymbolAddress(scratch) on device %d: %s", dev,
                     hipGetErrorString(e));
  g_noalloc_scratch[dev] = ptr;
  return NRG_CHEM_OK;
#endif
}

// The first n counters, once the stream is done (through pinned memory where there
// is some: a copy into a stack variable adds ~10 us to a call).
static hipError_t read_counters(nrg_chem_handle *h, unsigned long long *out, const unsigned long long *dev, int n)
{
  unsigned long long *to = h->acc_host ? h->acc_host : out;
  hipError_t e = hipMemcpyAsync(to, dev, n * sizeof(*out), hipMemcpyDeviceToHost, h->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(h->stream);
  if (e == hipSuccess && to != out) std::memcpy(out, to, n * sizeof(*out));
  return e;
}

// Blocks of 256 threads covering the aligned walk, one offset per thread.
static long long walk_blocks(const GridIdx &g) { return std::max<long long>(1, (g.pad1 - g.pad0 + 255) / 256); }

// Whether a pass over `fields` FP64 fields stores past the caches: where it touches
// more than the 256 MB memory-side cache keeps for whoever reads its outputs next.
// Calls, plain / past the caches: table step (29 fields) 427,050 cells 76 / 79 us, 1.0M
// 98 / 103, 2.0M 178 / 145, 4.1M 302 / 278; closure (37) 427,050 64.7 / 65.9, 1.0M 94 /
// 94, 2.0M 136 / 134; the low-Mach passes (23 to 29, three in turn) 427,050 133 /
// 133, 1.0M 218 / 198, 2.0M 356 / 316.  (Loads that pass the caches lose: the table
// step's kernel 119 us, 140 with both.)
static bool streams(const GridIdx &g, int fields, long long mib)
{
  return (g.pad1 - g.pad0) * 8 * fields > (mib << 20);
}

// Blocks for a kernel that strides over the aligned walk itself: its resident
// blocks per CU times the CUs at most (a block more than fits would run as a
// tail after the others), and as many fewer as leave every block the same number
// of the walk's 256-cell slices (table step of 427,050 cells 78 -> 75 us).
template <class K>
static long long resident_blocks(const nrg_chem_handle *h, K kernel, size_t dyn_lds, const GridIdx &g)
{
  int per_cu = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, 256, dyn_lds) != hipSuccess ||
      per_cu < 1)
    per_cu = 1;
  const long long nb = walk_blocks(g), resident = (long long)per_cu * h->num_cu;
  const long long rounds = (nb + resident - 1) / resident;
  return (nb + rounds - 1) / rounds;
}

// ---- entry points of this topology (forwarded from nrg_api.cpp) ----------

int nrg_chem_create(const nrg_chem_mech *mech, const nrg_chem_opts *opts, nrg_chem_t **out)
{
  if (!out) return set_error(NRG_CHEM_E_ARG, "out is NULL");
  *out = nullptr;
  nrg_chem_opts o;
  if (opts)
    o = *opts;
  else
    nrg_chem_default_opts(&o);
  if (!(o.eps > 0.0) || !(o.ewt > 0.0) || !(o.hmax > 0.0) || o.mxstep <= 0 || o.mxord <= 0)
    return set_error(NRG_CHEM_E_ARG, "invalid integrator options");
  if (o.errtest_gather_pct < 0 || o.errtest_gather_pct > 100)
    return set_error(NRG_CHEM_E_ARG, "errtest_gather_pct must be in 0..100");
  if (o.refill_min_idle < 0 || o.refill_min_idle > WAVE)
    return set_error(NRG_CHEM_E_ARG, "refill_min_idle must be in 0..64");
  if (o.jacobian != NRG_JAC_FD_SLATEC && o.jacobian != NRG_JAC_ANALYTIC)
    return set_error(NRG_CHEM_E_ARG, "jacobian mode %d not available", o.jacobian);
  if (o.form != NRG_FORM_PLAIN && o.form != NRG_FORM_PERSISTENT)
    return set_error(NRG_CHEM_E_ARG, "unknown form %d", o.form);
  if (o.jac_batch_pct < 0 || o.jac_batch_pct > 100)
    return set_error(NRG_CHEM_E_ARG, "jac_batch_pct must be in 0..100");
  if (o.waves_per_cu < 0 || o.waves_per_cu > 32)
    return set_error(NRG_CHEM_E_ARG, "waves_per_cu must be in 0..32");
  if (o.cell_order != NRG_ORDER_NATURAL && o.cell_order != NRG_ORDER_STIFFNESS)
    return set_error(NRG_CHEM_E_ARG, "unknown cell_order %d", o.cell_order);
  if (o.chunk_log2 != 0 && (o.chunk_log2 < 16 || o.chunk_log2 > 26))
    return set_error(NRG_CHEM_E_ARG, "chunk_log2 must be 0 or in 16..26");
  auto *h = new (std::nothrow) nrg_chem_handle();
  if (!h) return set_error(NRG_CHEM_E_ARG, "out of host memory");
  int st = build_mech(mech, h->host_mech);
  if (!st) st = check_device(o.device);
  if (st) {
    delete h;
    return st;
  }
  h->opts = o;
  h->device = o.device;
  h->k = make_const(o);
  h->refill_auto = o.refill_min_idle == 0;
  h->form = o.form;
  h->order = o.cell_order;
  h->use_graph = o.use_graph != 0;
  if (o.chunk_log2) h->chunk_max = 1ll << o.chunk_log2;
  h->jac_pct = o.jac_batch_pct ? o.jac_batch_pct : 50;
  auto fail = [&](int s) {
    nrg_chem_destroy(h);
    return s;
  };
  if (hipSetDevice(h->device) != hipSuccess) return fail(set_error(NRG_CHEM_E_HIP, "hipSetDevice"));
  if (hipStreamCreate(&h->stream) != hipSuccess) return fail(set_error(NRG_CHEM_E_HIP, "hipStreamCreate"));
  if ((st = noalloc_setup(h->device))) return fail(st);
  if (hipMalloc(&h->dev_mech, sizeof(MechCoef)) != hipSuccess)
    return fail(set_error(NRG_CHEM_E_HIP, "hipMalloc mech"));
  if (hipMalloc(&h->dev_acc, ACC_SLOTS * sizeof(unsigned long long)) != hipSuccess)
    return fail(set_error(NRG_CHEM_E_HIP, "hipMalloc acc"));
  if (hipHostMalloc(&h->acc_host, 16 * sizeof(unsigned long long), hipHostMallocDefault) != hipSuccess) {
    (void)hipGetLastError();   // no pinned memory to be had: the counters come without it
    h->acc_host = nullptr;
  }
  {
    hipDeviceProp_t prop;
    int per_cu = 0;
    if (hipGetDeviceProperties(&prop, h->device) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, chem_bdf_kernel<false>, WAVE, 0) !=
            hipSuccess)
      return fail(set_error(NRG_CHEM_E_HIP, "occupancy query"));
    if (o.waves_per_cu > 0) per_cu = o.waves_per_cu;
    if (per_cu < 1) per_cu = 1;
    h->persistent_blocks = per_cu * prop.multiProcessorCount;
    h->lane_blocks = (o.waves_per_cu > 0 ? o.waves_per_cu : LANE_WAVES_PER_CU) * prop.multiProcessorCount;
    h->num_cu = std::max(prop.multiProcessorCount, 1);
  }
  if (hipMemcpy(h->dev_mech, &h->host_mech, sizeof(MechCoef), hipMemcpyHostToDevice) != hipSuccess)
    return fail(set_error(NRG_CHEM_E_HIP, "hipMemcpy mech"));
  if (hipEventCreate(&h->ev0) != hipSuccess || hipEventCreate(&h->ev1) != hipSuccess ||
      hipEventCreate(&h->ev2) != hipSuccess || hipEventCreate(&h->ev3) != hipSuccess)
    return fail(set_error(NRG_CHEM_E_HIP, "hipEventCreate"));
  *out = h;
  return NRG_CHEM_OK;
}

void nrg_chem_destroy(nrg_chem_t *h)
{
  if (!h) return;
  // teardown has no caller to report to: failures here are ignored
  (void)hipSetDevice(h->device);
  if (h->stream) (void)hipStreamSynchronize(h->stream);
  if (h->stage) (void)hipFree(h->stage);
  if (h->pinned) (void)hipHostFree(h->pinned);
  if (h->acc_host) (void)hipHostFree(h->acc_host);
  if (h->dev_mech) (void)hipFree(h->dev_mech);
  if (h->dev_acc) (void)hipFree(h->dev_acc);
  if (h->rates) (void)hipFree(h->rates);
  if (h->graph_exec) (void)hipGraphExecDestroy(h->graph_exec);
  for (hipEvent_t e : {h->ev0, h->ev1, h->ev2, h->ev3})
    if (e) (void)hipEventDestroy(e);
  for (void *p : {(void *)h->sur_X, (void *)h->sur_Y, (void *)h->sur_list, (void *)h->sur_rate_bad,
                  (void *)h->sur_cand, (void *)h->sur_recheck, (void *)h->sur_acc,
                  (void *)h->order_list, (void *)h->hist, (void *)h->bins, (void *)h->table})
    if (p) (void)hipFree(p);
  if (h->stream) (void)hipStreamDestroy(h->stream);
  delete h;
}

void *nrg_chem_stream(nrg_chem_t *h) { return h ? (void *)h->stream : nullptr; }

// Build the stiffness-ordered cell list of this call into h->order_list and
// point a.list / a.hist at it (device work only, so it can be captured).
static int prepare_order(nrg_chem_t *h, long long n)
{
  if (n >= (1ll << 31)) return set_error(NRG_CHEM_E_ARG, "more than 2^31 inner cells");
  if (n > h->order_cells) {
    if (h->order_list) HIP_TRY(hipFree(h->order_list));
    if (h->hist) HIP_TRY(hipFree(h->hist));
    h->order_list = nullptr;
    h->hist = nullptr;
    h->order_cells = 0;
    h->hist_valid = false;
    HIP_TRY(hipMalloc(&h->order_list, (size_t)n * sizeof(int32_t)));
    HIP_TRY(hipMalloc(&h->hist, (size_t)n * sizeof(int32_t)));
    // no step counts yet (never inside a capture: callers prepare before it)
    HIP_TRY(hipMemsetAsync(h->hist, 0, (size_t)n * sizeof(int32_t), h->stream));
    h->order_cells = n;
  }
  if (!h->bins) HIP_TRY(hipMalloc(&h->bins, 2 * NBIN * sizeof(unsigned long long)));
  return NRG_CHEM_OK;
}

// Order the cells in_list[0..n) (all inner cells when in_list is NULL) into
// h->order_list, most expensive bin first.
static void enqueue_order(nrg_chem_t *h, StepArgs &a, bool use_hist, const int32_t *in_list = nullptr,
                          long long n = -1)
{
  if (n < 0) n = a.g.ninner;
  BinArgs b{};
  b.g = a.g;
  b.T = a.T;
  b.bc = a.bc;
  b.t_gate = a.k.t_gate;
  b.hist = use_hist ? h->hist : nullptr;
  b.count = h->bins;
  b.cursor = h->bins + NBIN;
  b.list = h->order_list;
  b.in_list = in_list;
  b.npos = n;
  // runs as long as still give every CU four blocks (84,000 listed cells: 9 + 12 us with
  // one cell a thread; with 32, in an earlier form of both kernels, 55 + 50)
  b.run = (int)std::min<long long>(BIN_RUN_MAX, std::max<long long>(1, n / (4ll * h->num_cu * BIN_THREADS)));
  const unsigned nb = (unsigned)((n + b.run * BIN_THREADS - 1) / (b.run * BIN_THREADS));
  hipLaunchKernelGGL(reset_kernel, dim3(2 * NBIN / 256), dim3(256), 0, h->stream, h->bins, 2 * NBIN);
  hipLaunchKernelGGL(bin_count_kernel, dim3(nb), dim3(BIN_THREADS), 0, h->stream, b);
  hipLaunchKernelGGL(bin_scatter_kernel, dim3(nb), dim3(BIN_THREADS), 0, h->stream, b);
}

// Positions to a chunk: at most chunk_max, each chunk with its own queue head.
static long long chunk_for(const nrg_chem_t *h, long long npos)
{
  long long chunk = std::min<long long>(npos, h->chunk_max);
  const long long min_chunk = (npos + MAX_CHUNKS - 1) / MAX_CHUNKS;
  return std::max<long long>(std::max<long long>(chunk, min_chunk), 1);
}

static int prepare_rates(nrg_chem_t *h, long long npos)
{
  const long long chunk = chunk_for(h, npos);
  if (npos > 0 && h->rates_cells < chunk) {
    if (h->rates) HIP_TRY(hipFree(h->rates));
    h->rates = nullptr;
    h->rates_cells = 0;
    HIP_TRY(hipMalloc(&h->rates, (size_t)chunk * REC_PAIRS * 2 * sizeof(double)));
    h->rates_cells = chunk;
  }
  return NRG_CHEM_OK;
}

static bool same_grid(const GridIdx &x, const GridIdx &y)
{
  return std::memcmp(&x, &y, sizeof(GridIdx)) == 0;
}

// A lane or a lane group to a cell?  A lane's way through a right-hand side and an
// iteration matrix costs the chip less (0.6 to 0.8 of a group's time where the chip is
// full of cells that cost alike), but it is three times as long, and a wave waits
// for the longest of its 64 cells.  So it depends on what a launch holds, which the
// counters of the handle's previous call on the grid tell: right-hand sides in
// all over those of the longest cell are the cells' worth of work (`full`), and that
// over the cells is how alike they are (`alike`: 0.7 a flame, 0.04 a grid of cold gas
// with hot kernels).  Below, time of a lane over that of a group, KEROMNES unless
// said otherwise; 65,536 lanes fill the chip.
//  Stiffness order with a history (a wave's cells cost alike):
//   finite differences, `full` in thousands: hot kernels 13: 2.35, 36: 1.31, 82: 0.67;
//    flame 64: 1.09, 112: 0.92, 434: 0.80; igniting 18: 2.1, 35: 1.5, 70: 0.88, 279: 0.82;
//    one composition at 900 K 23: 1.5, 46: 0.97, 91: 0.85.  In 1 us, where a cell takes
//    many steps to a Jacobian (2.2 right-hand sides a step; 2.6 and up elsewhere), 92:
//    1.09, 192: 1.04: what a lane does better is right-hand sides.  With 16 lanes to a
//    group a lane's state spills (TEREZA flame 90: 1.01, 155: 0.96, igniting 139: 1.03).
//   analytic Jacobian: hot kernels 13: 1.7, 36: 0.79; flame 26: 1.23, 57: 0.82, 392: 0.67;
//    igniting 18: 1.7, 38: 1.06, 75: 0.74; 1100 K 35: 1.24, 71: 0.69; a learned step's
//    fallback list 24: 1.3, 44: 0.9, 89: 0.79.
//   (Under 0.5 of the lanes the longest cell decides; where there are three times as
//   many cells as lanes, the others run beside it.)
//  Without a history there is nothing to tell, and stiffness order has only 50 K
//   temperature bins: finite differences, hot kernels 1.4 to 1.8 (TEREZA 2.6 to 3.1),
//   flame 0.9, one composition 0.8: a group loses less.  Analytic, hot kernels 1.0 to
//   1.4, flame and igniting 0.77, one composition 0.63 (TEREZA 0.4): a lane does, from
//   where it fills the chip a few times (natural order 1.0 to 1.26 and 0.62 to 0.95).
//  Natural order, both with the refill that fits: `alike` 0.82: 0.8 to 0.9, 0.69: 0.85 to
//   1.0, flame (0.67) 112: 1.2, 434: 1.06, 0.58: 1.1 to 0.9, igniting (0.27) 1.2, hot kernels
//   1.4; analytic 0.61: 0.8 to 1.07, 0.54: 0.7 to 0.9, 0.29: 1.05 to 1.2 (TEREZA 0.9), hot kernels
//   1.1 (TEREZA 1.03 at 39, 0.8 above).
// The choice keeps to what it was until the numbers are a fifth past the line, so that
// a captured graph does not change with every call.
static bool alike(const Seen &s)
{
  return s.valid && s.nfe * (s.alike ? 2.5 : 2.0) >= (double)s.cells * s.nfe_max;
}
static bool lane_launch(const nrg_chem_t *h, const Seen &s, bool ordered, bool use_hist, bool fallback,
                        long long npos, long long nchunk, bool before)
{
  if (!LANE_KERNEL) return false;
  const bool analytic = h->opts.jacobian == NRG_JAC_ANALYTIC;
  const double lanes = (double)WAVE * LANE_WAVES_PER_CU * h->num_cu, slack = before ? 0.8 : 1.0;
  if (!s.valid || s.nfe_max <= 0 || (ordered && !use_hist))
    return analytic && nchunk >= (fallback ? 1 : ordered ? 3 : 8) * lanes;
  const double part = (double)nchunk / (fallback ? s.cells : npos);
  const double full = part * s.nfe / s.nfe_max;
  const double fills = analytic ? (!ordered ? 1.0 : part * s.cells >= 3 * lanes ? 0.4 : 0.5625)
                                : (ordered && G == 8 ? 1.0 : 2.0);
  if (full < slack * fills * lanes) return false;
  if (ordered) return analytic || s.nfe >= slack * 2.5 * s.nstep || alike(s);
  return alike(s) || (analytic && G == 16);
}

// The chunks of a call that go one cell to a lane (a bit each), and the refill threshold
// of natural order where the caller has set none.
static unsigned long long plan(nrg_chem_t *h, Seen &s, StepArgs &a, long long npos, long long chunk, bool ordered,
                               bool use_hist, bool fallback)
{
  if (s.valid && !same_grid(s.g, a.g)) s = Seen();
  unsigned long long lanes = 0;
  for (long long ci = 0; ci * chunk < npos; ++ci)
    if (lane_launch(h, s, ordered, use_hist, fallback, npos, std::min(chunk, npos - ci * chunk), s.lanes >> ci & 1))
      lanes |= 1ull << ci;
  s.lanes = lanes;
  s.alike = alike(s);
  if (h->refill_auto)
    a.k.refill_idle = ordered || s.alike ? REFILL_IDLE_ORDERED : REFILL_IDLE_NATURAL;
  return lanes;
}

// Keep what a call has counted for the next one's plan.
static void note(Seen &s, const GridIdx &g, const unsigned long long (&acc)[16])
{
  s.valid = acc[ACC_INTEG] > 0;
  s.g = g;
  s.cells = (long long)acc[ACC_INTEG];
  s.nfe = (double)acc[ACC_NFE];
  s.nstep = (double)acc[ACC_NSTEP];
  s.nfe_max = (long long)acc[ACC_NFE_MAX];
}

// Launch rates_kernel + the integrator kernel per chunk of `chunk` positions, with
// the chunk's rate constants in `rates` and its queue head in acc[ACC_QUEUE0 + ci];
// chunk ci goes to the one-cell-per-lane integrator where bit ci of `lanes` is set.
static void enqueue_chunks(nrg_chem_t *h, StepArgs &a, long long npos, long long chunk,
                           double *rates, unsigned long long *acc, unsigned long long lanes)
{
  const long long nchunks = npos > 0 ? (npos + chunk - 1) / chunk : 0;
  const bool ordered = a.list && a.list == h->order_list;
  a.npos = npos;
  a.gated = ordered ? h->bins : nullptr;   // bin 0 (cost_bin)
  a.rates = rates;
  a.rates_out = rates;
  for (long long ci = 0; ci < nchunks; ++ci) {
    a.base = ci * chunk;
    a.nchunk = std::min<long long>(chunk, npos - a.base);
    a.queue = acc + ACC_QUEUE0 + ci;
    a.live = acc + ACC_LIVE0 + ci;
    hipLaunchKernelGGL(rates_kernel, dim3((unsigned)((a.nchunk + RATES_CELLS - 1) / RATES_CELLS)),
                       dim3(256), 0, h->stream, a);
    // A wave holds fewer cells than it could where the grid gives the SIMDs less
    // than a full wave each: cells that share a wave wait for each other's
    // stages (420 flame cells: one to a wave 0.60 ms, eight 0.75; 16,384: the same).
    a.cpw = (int)std::min<long long>(CPW, std::max<long long>(1, (a.nchunk + 4 * h->num_cu - 1) / (4 * h->num_cu)));
    const bool analytic = h->opts.jacobian == NRG_JAC_ANALYTIC;
    const long long need = (a.nchunk + a.cpw - 1) / a.cpw;
    const dim3 grid((unsigned)std::min<long long>(need, h->persistent_blocks));
    if constexpr (LANE_KERNEL)
      if (lanes >> ci & 1) {
        const dim3 blocks((unsigned)std::min<long long>((a.nchunk + WAVE - 1) / WAVE, h->lane_blocks));
        if (analytic)
          hipLaunchKernelGGL(chem_bdf_lane_kernel<true>, blocks, dim3(WAVE), 0, h->stream, a);
        else
          hipLaunchKernelGGL(chem_bdf_lane_kernel<false>, blocks, dim3(WAVE), 0, h->stream, a);
        continue;
      }
    if (analytic)
      hipLaunchKernelGGL(chem_bdf_kernel<true>, grid, dim3(WAVE), 0, h->stream, a);
    else
      hipLaunchKernelGGL(chem_bdf_kernel<false>, grid, dim3(WAVE), 0, h->stream, a);
  }
}

static int enqueue_integrator(nrg_chem_t *h, StepArgs &a, long long npos, unsigned long long lanes)
{
  int st = prepare_rates(h, npos);
  if (st) return st;
  enqueue_chunks(h, a, npos, chunk_for(h, npos), h->rates, h->dev_acc, lanes);
  HIP_TRY(hipGetLastError());
  return NRG_CHEM_OK;
}

static void fill_stats(const unsigned long long (&acc)[16], long long ninner, float ms,
                       nrg_chem_stats *stats)
{
  std::memset(stats, 0, sizeof(*stats));
  stats->cells_inner = ninner;
  stats->cells_integrated = (int64_t)acc[ACC_INTEG];
  stats->nstep_sum = (int64_t)acc[ACC_NSTEP];
  stats->nfe_sum = (int64_t)acc[ACC_NFE];
  stats->nje_sum = (int64_t)acc[ACC_NJE];
  stats->ncorr_sum = (int64_t)acc[ACC_NCORR];
  stats->natt_sum = (int64_t)acc[ACC_NATT];
  stats->nstep_max = (int32_t)acc[ACC_NSTEP_MAX];
  stats->nfe_max = (int32_t)acc[ACC_NFE_MAX];
  for (int i = 0; i < 6; ++i) stats->status_count[i] = (int64_t)acc[ACC_STATUS0 + i];
  stats->kernel_ms = ms;
}

// The reference STOPs on these (slatec/ddriv3.f90 IERFLG 41, 42); here they are statuses.
static int integrator_status(const unsigned long long (&acc)[16])
{
  if (acc[ACC_STATUS0 + NRG_CELL_STEP_ZERO])
    return set_error(NRG_CHEM_E_STEP_ZERO, "%llu cell(s): step size went to zero",
                     acc[ACC_STATUS0 + NRG_CELL_STEP_ZERO]);
  if (acc[ACC_STATUS0 + NRG_CELL_REPEATED_FAIL] || acc[ACC_STATUS0 + NRG_CELL_SINGULAR])
    return set_error(NRG_CHEM_E_REPEATED_FAIL, "%llu cell(s): repeated integrator failures",
                     acc[ACC_STATUS0 + NRG_CELL_REPEATED_FAIL] + acc[ACC_STATUS0 + NRG_CELL_SINGULAR]);
  return NRG_CHEM_OK;
}

// The device work of one chemistry step: counters reset, optional ordering,
// rate constants and integrator per chunk.  Launches only.
static int enqueue_step(nrg_chem_t *h, StepArgs &a, bool use_hist, unsigned long long lanes)
{
  hipLaunchKernelGGL(reset_kernel, dim3(1), dim3(ACC_SLOTS), 0, h->stream, h->dev_acc, ACC_SLOTS);
  if (a.list) enqueue_order(h, a, use_hist);
  return enqueue_integrator(h, a, a.g.ninner, lanes);
}

// Replay the captured step when the arguments equal the captured ones;
// otherwise capture the step into a new graph first.
static int launch_step_graph(nrg_chem_t *h, StepArgs &a, bool use_hist, unsigned long long lanes)
{
  StepKey key;
  std::memset(&key, 0, sizeof(key));
  std::memcpy(&key.args, &a, sizeof(StepArgs));
  key.rates = h->rates;
  key.use_hist = use_hist;
  key.form = h->form;
  key.chunk_max = h->chunk_max;
  key.persistent_blocks = h->persistent_blocks;
  key.jacobian = h->opts.jacobian;
  key.lanes = lanes;
  if (!h->graph_exec || std::memcmp(&key, &h->graph_key, sizeof(key)) != 0) {
    if (h->graph_exec) HIP_TRY(hipGraphExecDestroy(h->graph_exec));
    h->graph_exec = nullptr;
    hipGraph_t graph = nullptr;
    HIP_TRY(hipStreamBeginCapture(h->stream, hipStreamCaptureModeThreadLocal));
    StepArgs c = a;
    const int st = enqueue_step(h, c, use_hist, lanes);
    const hipError_t e = hipStreamEndCapture(h->stream, &graph);
    if (st) {
      if (graph) (void)hipGraphDestroy(graph);
      return st;
    }
    if (e != hipSuccess) return set_error(NRG_CHEM_E_HIP, "graph capture: %s", hipGetErrorString(e));
    const hipError_t ei = hipGraphInstantiate(&h->graph_exec, graph, nullptr, nullptr, 0);
    (void)hipGraphDestroy(graph);
    if (ei != hipSuccess) {
      h->graph_exec = nullptr;
      return set_error(NRG_CHEM_E_HIP, "graph instantiate: %s", hipGetErrorString(ei));
    }
    h->graph_key = key;
    h->graph_captures++;
  }
  HIP_TRY(hipGraphLaunch(h->graph_exec, h->stream));
  return NRG_CHEM_OK;
}

// Step arguments from an entry point's pointers (checked); the work counters,
// accumulators and queue are left for the caller to set.
static int fill_step_args(nrg_chem_t *h, const nrg_grid *grid, double dt, const double *T,
                          const double *rho, const double *const *Y, const int8_t *bc,
                          double *const *Y_prod, double *const *Y_prod2, double *E_f_prod,
                          int32_t *cell_status, StepArgs &a)
{
  if (!h) return set_error(NRG_CHEM_E_ARG, "handle is NULL");
  if (!(dt > 0.0) || !std::isfinite(dt)) return set_error(NRG_CHEM_E_ARG, "time_step must be > 0");
  if (!T || !rho || !Y || !Y_prod || !Y_prod2 || !E_f_prod)
    return set_error(NRG_CHEM_E_ARG, "required field pointer is NULL");
  int st = make_grid(grid, a.g);
  if (st) return st;
  for (int s = 0; s < S; ++s) {
    if (!Y[s] || !Y_prod[s] || !Y_prod2[s]) return set_error(NRG_CHEM_E_ARG, "species %d field is NULL", s + 1);
    a.Y[s] = Y[s];
    a.Yp[s] = Y_prod[s];
    a.Yp2[s] = Y_prod2[s];
  }
  a.dt = dt;
  a.k = h->k;
  a.mech = h->dev_mech;
  a.T = T;
  a.rho = rho;
  a.bc = bc;
  a.Efp = E_f_prod;
  a.status = cell_status;
  a.jac_pct = h->jac_pct;
  return NRG_CHEM_OK;
}

static int step_dev_impl(nrg_chem_t *h, const nrg_grid *grid, double dt, const double *T,
                         const double *rho, const double *const *Y, const int8_t *bc,
                         double *const *Y_prod, double *const *Y_prod2, double *E_f_prod,
                         int32_t *cell_status, nrg_chem_stats *stats, int32_t *nstep,
                         int32_t *nfe, int32_t *nje)
{
  StepArgs a{};
  int st = fill_step_args(h, grid, dt, T, rho, Y, bc, Y_prod, Y_prod2, E_f_prod, cell_status, a);
  if (st) return st;
  a.nstep = nstep;
  a.nfe = nfe;
  a.nje = nje;
  a.acc = h->dev_acc;
  HIP_TRY(hipSetDevice(h->device));
  unsigned long long acc[16] = {};
  float ms = 0.f;
  if (a.g.ninner <= 0) {
    hipLaunchKernelGGL(reset_kernel, dim3(1), dim3(ACC_SLOTS), 0, h->stream, h->dev_acc, ACC_SLOTS);
    HIP_TRY(hipGetLastError());
  } else {
    // buffers first: nothing below allocates, so the sequence can be captured
    const bool ordered = h->order == NRG_ORDER_STIFFNESS;
    bool use_hist = false;
    if (ordered) {
      if ((st = prepare_order(h, a.g.ninner))) return st;
      use_hist = h->hist_valid && same_grid(h->hist_grid, a.g);
      a.list = h->order_list;
      a.hist = h->hist;
    }
    if ((st = prepare_rates(h, a.g.ninner))) return st;
    const unsigned long long lanes =
        plan(h, h->seen_step, a, a.g.ninner, chunk_for(h, a.g.ninner), ordered, use_hist, false);
    HIP_TRY(hipEventRecord(h->ev0, h->stream));
    if (h->use_graph) {
      if ((st = launch_step_graph(h, a, use_hist, lanes))) return st;
    } else {
      if ((st = enqueue_step(h, a, use_hist, lanes))) return st;
    }
    if (ordered) {
      h->hist_valid = true;
      h->hist_grid = a.g;
    }
    HIP_TRY(hipEventRecord(h->ev1, h->stream));
    HIP_TRY(read_counters(h, acc, h->dev_acc, 16));
    HIP_TRY(hipEventElapsedTime(&ms, h->ev0, h->ev1));
    note(h->seen_step, a.g, acc);
  }
  if (stats) fill_stats(acc, a.g.ninner, ms, stats);
  return integrator_status(acc);
}

int nrg_chem_step_dev(nrg_chem_t *h, const nrg_grid *grid, double dt, const double *T,
                      const double *p, const double *rho, const double *const *Y,
                      const int8_t *bc, double *const *Y_prod, double *const *Y_prod2,
                      double *E_f_prod, int32_t *cell_status, nrg_chem_stats *stats)
{
  (void)p;   // read but unused by the reference step (chemical_kinetics_solver.f90:307)
  return step_dev_impl(h, grid, dt, T, rho, Y, bc, Y_prod, Y_prod2, E_f_prod, cell_status, stats,
                       nullptr, nullptr, nullptr);
}

int nrg_chem_step_dev_diag(nrg_chem_t *h, const nrg_grid *grid, double dt, const double *T,
                           const double *p, const double *rho, const double *const *Y,
                           const int8_t *bc, double *const *Y_prod, double *const *Y_prod2,
                           double *E_f_prod, int32_t *cell_status, nrg_chem_stats *stats,
                           int32_t *nstep, int32_t *nfe, int32_t *nje)
{
  (void)p;
  if ((nstep || nfe || nje) && !(nstep && nfe && nje))
    return set_error(NRG_CHEM_E_ARG, "nstep, nfe and nje must be all NULL or all set");
  return step_dev_impl(h, grid, dt, T, rho, Y, bc, Y_prod, Y_prod2, E_f_prod, cell_status, stats,
                       nstep, nfe, nje);
}

// nrg_chem_step_dev with every device buffer beyond the caller's fields taken
// from `scratch` (through its per-device address): no allocation, no graph,
// natural cell order, chunks of NRG_NOALLOC_CHUNK_CELLS cells.  The kernels and
// their arithmetic are those of nrg_chem_step_dev.
int nrg_chem_step_dev_noalloc(nrg_chem_t *h, const nrg_grid *grid, double dt, const double *T,
                              const double *p, const double *rho, const double *const *Y,
                              const int8_t *bc, double *const *Y_prod, double *const *Y_prod2,
                              double *E_f_prod, int32_t *cell_status, nrg_chem_stats *stats)
{
  (void)p;
#if !NRG_TOPO_PRIMARY
  (void)h; (void)grid; (void)dt; (void)T; (void)rho; (void)Y; (void)bc; (void)Y_prod;
  (void)Y_prod2; (void)E_f_prod; (void)cell_status; (void)stats;
  return set_error(NRG_CHEM_E_MECH, "nrg_chem_step_dev_noalloc serves the KEROMNES kernels only, "
                                    "not " NRG_TOPO_NAME);
#else
  StepArgs a{};
  int st = fill_step_args(h, grid, dt, T, rho, Y, bc, Y_prod, Y_prod2, E_f_prod, cell_status, a);
  if (st) return st;
  if (a.g.ninner > (long long)NRG_NOALLOC_MAX_CELLS)
    return set_error(NRG_CHEM_E_ARG,
                     "%lld inner cells: nrg_chem_step_dev_noalloc serves at most %lld "
                     "(NRG_NOALLOC_MAX_CELLS); use nrg_chem_step_dev",
                     a.g.ninner, (long long)NRG_NOALLOC_MAX_CELLS);
  void *ptr = (h->device >= 0 && h->device < NOALLOC_MAX_DEVICES) ? g_noalloc_scratch[h->device] : nullptr;
  if (!ptr) return set_error(NRG_CHEM_E_HIP, "no scratch address for device %d", h->device);
  auto *acc_dev = (unsigned long long *)ptr;
  auto *rates = (double *)((unsigned char *)ptr + NOALLOC_ACC_BYTES);
  a.acc = acc_dev;
  HIP_TRY(hipSetDevice(h->device));
  unsigned long long acc[16] = {};
  float ms = 0.f;
  HIP_TRY(hipEventRecord(h->ev0, h->stream));
  hipLaunchKernelGGL(reset_kernel, dim3(1), dim3(ACC_SLOTS), 0, h->stream, acc_dev, ACC_SLOTS);
  if (a.g.ninner > 0) {
    const unsigned long long lanes =
        plan(h, h->seen_step, a, a.g.ninner, NRG_NOALLOC_CHUNK_CELLS, false, false, false);
    enqueue_chunks(h, a, a.g.ninner, NRG_NOALLOC_CHUNK_CELLS, rates, acc_dev, lanes);
  }
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipEventRecord(h->ev1, h->stream));
  HIP_TRY(read_counters(h, acc, acc_dev, 16));
  HIP_TRY(hipEventElapsedTime(&ms, h->ev0, h->ev1));
  note(h->seen_step, a.g, acc);
  if (stats) fill_stats(acc, a.g.ninner, ms, stats);
  return integrator_status(acc);
#endif
}

// Host fields: stage them through the handle's device buffers, run the FP64
// step (or the table step) there, copy the outputs back.
static int step_host(nrg_chem_t *h, bool table, const nrg_grid *grid, double dt, const double *T,
                     const double *rho, const double *const *Y, const int8_t *bc,
                     double *const *Y_prod, double *const *Y_prod2, double *E_f_prod,
                     int32_t *cell_status, nrg_chem_stats *stats)
{
  if (!h) return set_error(NRG_CHEM_E_ARG, "handle is NULL");
  if (!grid || !T || !rho || !Y || !Y_prod || !Y_prod2 || !E_f_prod)
    return set_error(NRG_CHEM_E_ARG, "required pointer is NULL");
  const long long n = field_cells(grid);
  if (n <= 0) return set_error(NRG_CHEM_E_ARG, "empty field");
  HIP_TRY(hipSetDevice(h->device));
  for (int q = 0; q < S; ++q)
    if (!Y[q] || !Y_prod[q] || !Y_prod2[q]) return set_error(NRG_CHEM_E_ARG, "species %d field is NULL", q + 1);
  // staging layout: T, rho, Y[S], bc (padded to doubles); then what comes back:
  // Y_prod[S], Y_prod2[S], E_f_prod, status
  auto room = [&](size_t size) { return ((size_t)n * size + 255) / 256 * 256; };
  const size_t in_bytes = (2 + S) * room(8) + room(1), out_bytes = (2 * S + 1) * room(8) + room(4);
  if (h->stage_bytes < in_bytes + out_bytes) {
    void *old = h->stage;
    h->stage = nullptr;   // never freed twice, even when this free fails
    h->stage_bytes = 0;
    if (old) HIP_TRY(hipFree(old));
    HIP_TRY(hipMalloc(&h->stage, in_bytes + out_bytes));
    h->stage_bytes = in_bytes + out_bytes;
  }
  // Small fields go through pinned memory, all in one copy each way: a copy from
  // pageable memory returns only when it is done (~10 us each, 51 of them).  Field by
  // field and in one copy, flame steps, table steps: 10,000 cells 1030 and 605 us, 650 and
  // 220; 30,000 1400 and 1040, 850 and 495; 65,000 2190 and 1960, 1230 and 1030; 100,000
  // 3000 and 2990, 1650 and 1650; 120,000 3430 and 3590, 1870 and 2020: by then the host's
  // own copies are as long as the transfers, which single fields' copies run beside.
  bool pin = in_bytes + out_bytes <= STAGE_PINNED_MAX;
  if (pin && h->pinned_bytes < in_bytes + out_bytes) {
    const size_t grown = std::max(in_bytes + out_bytes, std::min(h->pinned_bytes / 2 * 3, STAGE_PINNED_MAX));
    void *old = h->pinned;
    h->pinned = nullptr;
    h->pinned_bytes = 0;
    if (old) HIP_TRY(hipHostFree(old));
    if (hipHostMalloc(&h->pinned, grown, hipHostMallocDefault) == hipSuccess) {
      h->pinned_bytes = grown;
    } else {
      (void)hipGetLastError();   // no pinned memory to be had: field by field
      h->pinned = nullptr;
      pin = false;
    }
  }
  char *dev = (char *)h->stage, *host = pin ? (char *)h->pinned : nullptr;
  hipStream_t s = h->stream;
  size_t at = 0;
  int rc = NRG_CHEM_OK;
  auto up = [&](const void *src, size_t size) {   // the next field's device address
    char *d = dev + at;
    if (src && pin)
      std::memcpy(host + at, src, n * size);
    else if (src && rc == NRG_CHEM_OK && hipMemcpyAsync(d, src, n * size, hipMemcpyHostToDevice, s) != hipSuccess)
      rc = set_error(NRG_CHEM_E_HIP, "copy of a field to the device");
    at += room(size);
    return src ? d : nullptr;
  };
  const double *Yd[S];
  double *Ypd[S], *Yp2d[S];
  const double *Td = (const double *)up(T, 8), *rhod = (const double *)up(rho, 8);
  for (int q = 0; q < S; ++q) Yd[q] = (const double *)up(Y[q], 8);
  const int8_t *bcd = (const int8_t *)up(bc, 1);
  for (int q = 0; q < S; ++q) Ypd[q] = (double *)up(Y_prod[q], 8);
  for (int q = 0; q < S; ++q) Yp2d[q] = (double *)up(Y_prod2[q], 8);
  double *Efd = (double *)up(E_f_prod, 8);
  int32_t *std_ = (int32_t *)up(cell_status, 4);
  if (rc != NRG_CHEM_OK) return rc;
  if (pin) HIP_TRY(hipMemcpyAsync(dev, host, at, hipMemcpyHostToDevice, s));
  rc = table ? nrg_chem_table_step_dev(h, grid, dt, Td, nullptr, rhod, Yd, bcd, Ypd, Yp2d, Efd, std_, stats)
             : step_dev_impl(h, grid, dt, Td, rhod, Yd, bcd, Ypd, Yp2d, Efd, std_, stats, nullptr, nullptr,
                             nullptr);
  if (rc != NRG_CHEM_OK && rc != NRG_CHEM_E_STEP_ZERO && rc != NRG_CHEM_E_REPEATED_FAIL) return rc;
  if (pin) {
    HIP_TRY(hipMemcpyAsync(host + in_bytes, dev + in_bytes, out_bytes, hipMemcpyDeviceToHost, s));
    HIP_TRY(hipStreamSynchronize(s));
  }
  bool copied = true;
  auto down = [&](void *dst, const void *src, size_t size) {
    if (!dst) return;
    if (pin)
      std::memcpy(dst, host + ((const char *)src - dev), n * size);
    else
      copied = copied && hipMemcpyAsync(dst, src, n * size, hipMemcpyDeviceToHost, s) == hipSuccess;
  };
  for (int q = 0; q < S; ++q) {
    down(Y_prod[q], Ypd[q], 8);
    down(Y_prod2[q], Yp2d[q], 8);
  }
  down(E_f_prod, Efd, 8);
  down(cell_status, std_, 4);
  if (!copied) return set_error(NRG_CHEM_E_HIP, "copy of a field to the host");
  if (!pin) HIP_TRY(hipStreamSynchronize(s));
  return rc;
}

int nrg_chem_step(nrg_chem_t *h, const nrg_grid *grid, double dt, const double *T,
                  const double *p, const double *rho, const double *const *Y, const int8_t *bc,
                  double *const *Y_prod, double *const *Y_prod2, double *E_f_prod,
                  int32_t *cell_status, nrg_chem_stats *stats)
{
  (void)p;
  return step_host(h, false, grid, dt, T, rho, Y, bc, Y_prod, Y_prod2, E_f_prod, cell_status, stats);
}

int nrg_chem_table_step(nrg_chem_t *h, const nrg_grid *grid, double dt, const double *T,
                        const double *p, const double *rho, const double *const *Y, const int8_t *bc,
                        double *const *Y_prod, double *const *Y_prod2, double *E_f_prod,
                        int32_t *cell_status, nrg_chem_stats *stats)
{
  (void)p;
  if (h && !h->table) return set_error(NRG_CHEM_E_ARG, "no table (nrg_chem_set_table)");
  return step_host(h, true, grid, dt, T, rho, Y, bc, Y_prod, Y_prod2, E_f_prod, cell_status, stats);
}

static int closure_impl(nrg_chem_t *h, const nrg_grid *grid, double dt, int apply,
                        const double *rho, const double *const *v, int32_t ndim,
                        const double *E_f_prod, const double *const *Y_prod, const int8_t *bc,
                        double *E_f, double *const *Y, double *T, double *p)
{
  if (!h) return set_error(NRG_CHEM_E_ARG, "handle is NULL");
  if (!rho || !E_f || !Y || !T) return set_error(NRG_CHEM_E_ARG, "required field pointer is NULL");
  if (ndim < 0 || ndim > 3 || (ndim > 0 && !v)) return set_error(NRG_CHEM_E_ARG, "bad velocity");
  if (apply && (!E_f_prod || !Y_prod || !(dt > 0.0)))
    return set_error(NRG_CHEM_E_ARG, "sources and dt > 0 required");
  ClosureArgs a{};
  int st = make_grid(grid, a.g);
  if (st) return st;
  a.dt = dt;
  a.apply_sources = apply;
  a.ndim = ndim;
  a.mech = h->dev_mech;
  a.rho = rho;
  for (int d = 0; d < ndim; ++d) {
    if (!v[d]) return set_error(NRG_CHEM_E_ARG, "velocity component %d is NULL", d);
    a.v[d] = v[d];
  }
  a.Efp = E_f_prod;
  for (int s = 0; s < S; ++s) {
    if (!Y[s] || (apply && !Y_prod[s])) return set_error(NRG_CHEM_E_ARG, "species %d field is NULL", s + 1);
    a.Y[s] = Y[s];
    a.Yp[s] = apply ? Y_prod[s] : nullptr;
  }
  a.bc = bc;
  a.E_f = E_f;
  a.T = T;
  a.p = p;
  HIP_TRY(hipSetDevice(h->device));
  if (a.g.ninner > 0) {
    const long long nb = walk_blocks(a.g);
    const auto kernel = streams(a.g, 4 * S + 1, 320) ? closure_kernel<true> : closure_kernel<false>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)nb), dim3(256), 0, h->stream, a);
    HIP_TRY(hipGetLastError());
  }
  HIP_TRY(hipStreamSynchronize(h->stream));
  return NRG_CHEM_OK;
}

int nrg_chem_closure_dev(nrg_chem_t *h, const nrg_grid *grid, double dt, const double *rho,
                         const double *const *v, int32_t ndim, const double *E_f_prod,
                         const double *const *Y_prod, const int8_t *bc, double *E_f,
                         double *const *Y, double *T, double *p)
{
  return closure_impl(h, grid, dt, 1, rho, v, ndim, E_f_prod, Y_prod, bc, E_f, Y, T, p);
}

int nrg_state_equation_dev(nrg_chem_t *h, const nrg_grid *grid, const double *rho,
                           const double *const *v, int32_t ndim, const double *E_f,
                           const double *const *Y, const int8_t *bc, double *T, double *p)
{
  return closure_impl(h, grid, 0.0, 0, rho, v, ndim, nullptr, nullptr, bc, const_cast<double *>(E_f),
                      const_cast<double *const *>(Y), T, p);
}

int nrg_energy_from_temperature_dev(nrg_chem_t *h, const nrg_grid *grid, const double *T,
                                    const double *const *Y, const double *const *v, int32_t ndim,
                                    double *E_f)
{
  if (!h) return set_error(NRG_CHEM_E_ARG, "handle is NULL");
  if (!T || !Y || !E_f) return set_error(NRG_CHEM_E_ARG, "required field pointer is NULL");
  if (ndim < 0 || ndim > 3 || (ndim > 0 && !v)) return set_error(NRG_CHEM_E_ARG, "bad velocity");
  EnergyArgs a{};
  int st = make_grid(grid, a.g);
  if (st) return st;
  a.ndim = ndim;
  a.mech = h->dev_mech;
  a.T = T;
  for (int s = 0; s < S; ++s) {
    if (!Y[s]) return set_error(NRG_CHEM_E_ARG, "species %d field is NULL", s + 1);
    a.Y[s] = Y[s];
  }
  for (int d = 0; d < ndim; ++d) a.v[d] = v[d];
  a.E_f = E_f;
  HIP_TRY(hipSetDevice(h->device));
  if (a.g.ninner > 0) {
    const long long nb = (a.g.ninner + 255) / 256;
    hipLaunchKernelGGL(energy_kernel, dim3((unsigned)nb), dim3(256), 0, h->stream, a);
    HIP_TRY(hipGetLastError());
  }
  HIP_TRY(hipStreamSynchronize(h->stream));
  return NRG_CHEM_OK;
}

int nrg_chem_set_table(nrg_chem_t *h, int32_t rows, const double *T_t, const double *dC_t)
{
  if (!h) return set_error(NRG_CHEM_E_ARG, "handle is NULL");
  if (rows < 2 || !T_t || !dC_t) return set_error(NRG_CHEM_E_ARG, "a table needs >= 2 rows and both arrays");
  if (rows > (1 << 24)) return set_error(NRG_CHEM_E_ARG, "a table has at most 2^24 rows, got %d", rows);
  HIP_TRY(hipSetDevice(h->device));
  HIP_TRY(hipStreamSynchronize(h->stream));
  if (h->table) HIP_TRY(hipFree(h->table));
  h->table = nullptr;
  h->table_rows = 0;
  std::vector<double> t((size_t)(S + 1) * rows);
  std::memcpy(t.data(), T_t, sizeof(double) * rows);
  std::memcpy(t.data() + rows, dC_t, sizeof(double) * S * rows);
  HIP_TRY(hipMalloc(&h->table, t.size() * sizeof(double)));
  HIP_TRY(hipMemcpy(h->table, t.data(), t.size() * sizeof(double), hipMemcpyHostToDevice));
  h->table_rows = rows;
  h->table_ascending = 1;
  for (int32_t i = 0; i + 1 < rows; ++i)
    if (!(T_t[i] < T_t[i + 1])) h->table_ascending = 0;
  return NRG_CHEM_OK;
}

int nrg_chem_table_step_dev(nrg_chem_t *h, const nrg_grid *grid, double dt, const double *T,
                            const double *p, const double *rho, const double *const *Y,
                            const int8_t *bc, double *const *Y_prod, double *const *Y_prod2,
                            double *E_f_prod, int32_t *cell_status, nrg_chem_stats *stats)
{
  (void)p;
  (void)rho;
  if (!h) return set_error(NRG_CHEM_E_ARG, "handle is NULL");
  if (!h->table) return set_error(NRG_CHEM_E_ARG, "no table (nrg_chem_set_table)");
  if (!(dt > 0.0) || !std::isfinite(dt)) return set_error(NRG_CHEM_E_ARG, "time_step must be > 0");
  if (!T || !Y || !Y_prod || !Y_prod2 || !E_f_prod)
    return set_error(NRG_CHEM_E_ARG, "required field pointer is NULL");
  TableArgs a{};
  int st = make_grid(grid, a.g);
  if (st) return st;
  for (int s = 0; s < S; ++s) {
    if (!Y[s] || !Y_prod[s] || !Y_prod2[s]) return set_error(NRG_CHEM_E_ARG, "species %d field is NULL", s + 1);
    a.Y[s] = Y[s];
    a.Yp[s] = Y_prod[s];
    a.Yp2[s] = Y_prod2[s];
  }
  a.dt = dt;
  a.t_gate = h->k.t_gate;
  a.mech = h->dev_mech;
  a.T = T;
  a.bc = bc;
  a.Efp = E_f_prod;
  a.status = cell_status;
  a.table = h->table;
  a.rows = h->table_rows;
  a.ascending = h->table_ascending;
  a.acc = h->dev_acc;
  HIP_TRY(hipSetDevice(h->device));
  hipLaunchKernelGGL(reset_kernel, dim3(1), dim3(ACC_SLOTS), 0, h->stream, h->dev_acc, ACC_SLOTS);
  unsigned long long acc[16] = {};
  float ms = 0.f;
  HIP_TRY(hipEventRecord(h->ev0, h->stream));
  if (a.g.ninner > 0) {
    const size_t tab_bytes = sizeof(double) * (size_t)(S + 1) * (size_t)a.rows;
    const bool lds = tab_bytes <= (size_t)TABLE_LDS_BYTES, st = streams(a.g, 3 * S + 2, 320);
    const auto kernel = lds ? (st ? table_kernel<true, true> : table_kernel<true, false>)
                            : (st ? table_kernel<false, true> : table_kernel<false, false>);
    const size_t dyn = lds ? tab_bytes : 0;
    hipLaunchKernelGGL(kernel, dim3((unsigned)resident_blocks(h, kernel, dyn, a.g)), dim3(TABLE_THREADS), dyn,
                       h->stream, a);
    HIP_TRY(hipGetLastError());
  }
  HIP_TRY(hipEventRecord(h->ev1, h->stream));
  HIP_TRY(read_counters(h, acc, h->dev_acc, 16));
  HIP_TRY(hipEventElapsedTime(&ms, h->ev0, h->ev1));
  if (stats) fill_stats(acc, a.g.ninner, ms, stats);
  return NRG_CHEM_OK;
}

// ---------------------------------------------------------------------------
// Low-Mach coupling entry points (include/nrg_low_mach.h)
// ---------------------------------------------------------------------------
int nrg_low_mach_state_equation_dev(nrg_chem_t *h, const nrg_grid *grid, double time_step,
                                    int32_t predictor, const double *rho,
                                    const double *const *Y, const double *const *v, int32_t ndim,
                                    const double *dp_stat_dt, const int8_t *bc, double *p_stat,
                                    double *p_stat_old, double *T, double *mix_mol_mass, double *p,
                                    double *mixture_cp, double *gamma, double *h_s, double *v_s,
                                    double *e_i, double *E_f)
{
  if (!h) return set_error(NRG_CHEM_E_ARG, "handle is NULL");
  if (!rho || !Y || !dp_stat_dt || !p_stat || !p_stat_old || !T || !mix_mol_mass)
    return set_error(NRG_CHEM_E_ARG, "required field pointer is NULL");
  if (ndim < 0 || ndim > 3 || (ndim > 0 && !v)) return set_error(NRG_CHEM_E_ARG, "bad velocity");
  if (!std::isfinite(time_step)) return set_error(NRG_CHEM_E_ARG, "time_step is not finite");
  LowMachEosArgs a{};
  int st = make_grid(grid, a.g);
  if (st) return st;
  for (int s = 0; s < S; ++s) {
    if (!Y[s]) return set_error(NRG_CHEM_E_ARG, "species %d field is NULL", s + 1);
    a.Y[s] = Y[s];
  }
  for (int d = 0; d < ndim; ++d) {
    if (!v[d]) return set_error(NRG_CHEM_E_ARG, "velocity %d is NULL", d + 1);
    a.v[d] = v[d];
  }
  a.dt = time_step;
  a.predictor = predictor != 0;
  a.ndim = ndim;
  a.mech = h->dev_mech;
  a.rho = rho;
  a.dp = dp_stat_dt;
  a.bc = bc;
  a.p_stat = p_stat;
  a.p_stat_old = p_stat_old;
  a.T = T;
  a.mmm = mix_mol_mass;
  a.p = p;
  a.cp = mixture_cp;
  a.gamma = gamma;
  a.h_s = h_s;
  a.v_s = v_s;
  a.e_i = e_i;
  a.E_f = E_f;
  HIP_TRY(hipSetDevice(h->device));
  if (a.g.ninner > 0) {
    const auto kernel = streams(a.g, S + 16, 128) ? low_mach_eos_kernel<true> : low_mach_eos_kernel<false>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)walk_blocks(a.g)), dim3(LM_THREADS), 0,
                       h->stream, a);
    HIP_TRY(hipGetLastError());
  }
  HIP_TRY(hipStreamSynchronize(h->stream));
  return NRG_CHEM_OK;
}

int nrg_low_mach_species_dev(nrg_chem_t *h, const nrg_grid *grid, double time_step,
                             int32_t corrector, const double *rho_a, const double *const *Y_a,
                             const double *rho_b, const double *const *Y_b,
                             const double *const *rhs, const double *const *Y_prod_diff,
                             const double *const *Y_prod_chem, const int8_t *bc, double *rho_out,
                             double *const *Y_out)
{
  if (!h) return set_error(NRG_CHEM_E_ARG, "handle is NULL");
  if (!rho_a || !Y_a || !rho_out || !Y_out) return set_error(NRG_CHEM_E_ARG, "required field pointer is NULL");
  if (corrector && (!rho_b || !Y_b)) return set_error(NRG_CHEM_E_ARG, "the corrector needs rho_b and Y_b");
  if (!std::isfinite(time_step)) return set_error(NRG_CHEM_E_ARG, "time_step is not finite");
  LowMachSpeciesArgs a{};
  int st = make_grid(grid, a.g);
  if (st) return st;
  for (int s = 0; s < S; ++s) {
    if (!Y_a[s] || !Y_out[s] || (corrector && !Y_b[s]) || (rhs && !rhs[s]) ||
        (Y_prod_diff && !Y_prod_diff[s]) || (Y_prod_chem && !Y_prod_chem[s]))
      return set_error(NRG_CHEM_E_ARG, "species %d field is NULL", s + 1);
    a.Y_a[s] = Y_a[s];
    a.Y_b[s] = corrector ? Y_b[s] : nullptr;
    a.rhs[s] = rhs ? rhs[s] : nullptr;
    a.Yd[s] = Y_prod_diff ? Y_prod_diff[s] : nullptr;
    a.Yc[s] = Y_prod_chem ? Y_prod_chem[s] : nullptr;
    a.Y_out[s] = Y_out[s];
  }
  a.dt = time_step;
  a.corrector = corrector != 0;
  a.rho_a = rho_a;
  a.rho_b = corrector ? rho_b : nullptr;
  a.bc = bc;
  a.rho_out = rho_out;
  HIP_TRY(hipSetDevice(h->device));
  if (a.g.ninner > 0) {
    const auto kernel = streams(a.g, 3 * S + 2, 128) ? low_mach_species_kernel<true> : low_mach_species_kernel<false>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)walk_blocks(a.g)), dim3(LM_THREADS), 0,
                       h->stream, a);
    HIP_TRY(hipGetLastError());
  }
  HIP_TRY(hipStreamSynchronize(h->stream));
  return NRG_CHEM_OK;
}

int nrg_low_mach_chem_divergence_dev(nrg_chem_t *h, const nrg_grid *grid, const double *rho,
                                     const double *T, const double *const *Y,
                                     const double *mix_mol_mass, const double *E_f_prod_chem,
                                     const double *const *Y_prod_chem, const int8_t *bc,
                                     double *div_v)
{
  if (!h) return set_error(NRG_CHEM_E_ARG, "handle is NULL");
  if (!rho || !T || !Y || !mix_mol_mass || !E_f_prod_chem || !Y_prod_chem || !div_v)
    return set_error(NRG_CHEM_E_ARG, "required field pointer is NULL");
  LowMachDivArgs a{};
  int st = make_grid(grid, a.g);
  if (st) return st;
  for (int s = 0; s < S; ++s) {
    if (!Y[s] || !Y_prod_chem[s]) return set_error(NRG_CHEM_E_ARG, "species %d field is NULL", s + 1);
    a.Y[s] = Y[s];
    a.Yc[s] = Y_prod_chem[s];
  }
  a.mech = h->dev_mech;
  a.rho = rho;
  a.T = T;
  a.mmm = mix_mol_mass;
  a.Efc = E_f_prod_chem;
  a.bc = bc;
  a.div = div_v;
  HIP_TRY(hipSetDevice(h->device));
  if (a.g.ninner > 0) {
    const auto kernel = streams(a.g, 2 * S + 5, 128) ? low_mach_div_kernel<true> : low_mach_div_kernel<false>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)walk_blocks(a.g)), dim3(LM_THREADS), 0,
                       h->stream, a);
    HIP_TRY(hipGetLastError());
  }
  HIP_TRY(hipStreamSynchronize(h->stream));
  return NRG_CHEM_OK;
}

int nrg_chem_autotune_dev(nrg_chem_t *h, const nrg_grid *grid, double dt, const double *T,
                          const double *p, const double *rho, const double *const *Y,
                          const int8_t *bc, double *const *Y_prod, double *const *Y_prod2,
                          double *E_f_prod, nrg_chem_tuning *out)
{
  (void)p;
  if (!h || !out) return set_error(NRG_CHEM_E_ARG, "handle or out is NULL");
  std::memset(out, 0, sizeof(*out));
  hipDeviceProp_t prop;
  HIP_TRY(hipGetDeviceProperties(&prop, h->device));
  int occ = 0;
  HIP_TRY(hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, chem_bdf_kernel<false>, WAVE, 0));
  occ = std::max(occ, 1);
  struct Cfg {
    int form, order, jac, wpc;
    long long chunk;
    int gather, refill;
  };
  auto apply = [&](const Cfg &c) {
    h->k.gather_pct = c.gather;
    h->k.refill_idle = c.refill;
    h->refill_auto = false;
    h->form = c.form;
    h->order = c.order;
    h->jac_pct = c.jac;
    h->persistent_blocks = (c.wpc > 0 ? c.wpc : occ) * prop.multiProcessorCount;
    h->lane_blocks = (c.wpc > 0 ? c.wpc : LANE_WAVES_PER_CU) * prop.multiProcessorCount;
    h->chunk_max = c.chunk;
  };
  auto trial = [&](const Cfg &c, double &ms) -> int {
    apply(c);
    nrg_chem_stats s;
    const int st = step_dev_impl(h, grid, dt, T, rho, Y, bc, Y_prod, Y_prod2, E_f_prod, nullptr,
                                 &s, nullptr, nullptr, nullptr);
    ms = s.kernel_ms;
    if (st == NRG_CHEM_OK && out->n_trials < NRG_TUNE_MAX_TRIALS) {
      nrg_chem_tune_trial &t = out->trials[out->n_trials++];
      t.form = c.form; t.cell_order = c.order; t.jac_batch_pct = c.jac;
      t.waves_per_cu = c.wpc > 0 ? c.wpc : occ; t.chunk_cells = c.chunk; t.kernel_ms = ms;
      t.errtest_gather_pct = c.gather;
      t.refill_min_idle = c.refill;
    }
    return st;
  };
  // trials run eagerly: a capture per trial set-up would add host latency to its time
  const bool graph = h->use_graph;
  h->use_graph = false;
  struct Restore {
    nrg_chem_t *h;
    bool g;
    ~Restore() { h->use_graph = g; }
  } restore{h, graph};
  const int wpc0 = h->persistent_blocks / std::max(prop.multiProcessorCount, 1);
  Cfg best{h->form, h->order, h->jac_pct, wpc0 == occ ? 0 : wpc0, h->chunk_max, h->k.gather_pct,
           h->k.refill_idle};
  double best_ms = 0.0;
  int st;
  // the first run sets up the stiffness history that the ordered trials use
  if ((st = trial(best, best_ms))) return st;
  if ((st = trial(best, best_ms))) return st;
  auto consider = [&](Cfg c) -> int {
    double ms = 0.0;
    int s = NRG_CHEM_OK;
    if (c.order == NRG_ORDER_STIFFNESS && best.order != NRG_ORDER_STIFFNESS && (s = trial(c, ms))) return s;
    if ((s = trial(c, ms))) return s;      // (in stiffness order, with a history)
    if (ms < best_ms) {
      best_ms = ms;
      best = c;
    }
    return NRG_CHEM_OK;
  };
  for (int order : {NRG_ORDER_NATURAL, NRG_ORDER_STIFFNESS})
    if (order != best.order) {
      Cfg c = best;
      c.order = order;
      if ((st = consider(c))) return st;
    }
  for (int gather : {0, 100})
    if (gather != best.gather) {
      Cfg c = best;
      c.gather = gather;
      if ((st = consider(c))) return st;
    }
  for (int jac : {10, 25, 50, 75, 100})
    if (jac != best.jac) {
      Cfg c = best;
      c.jac = jac;
      if ((st = consider(c))) return st;
    }
  for (int refill : {REFILL_IDLE_NATURAL, REFILL_IDLE_ORDERED})
    if (refill != best.refill) {
      Cfg c = best;
      c.refill = refill;
      if ((st = consider(c))) return st;
    }
  for (int w : {2 * occ, 4 * occ}) {
    Cfg c = best;
    c.wpc = w;
    if ((st = consider(c))) return st;
  }
  for (long long ch : {1ll << 21, 1ll << 22, 1ll << 23, 1ll << 24})
    if (ch != best.chunk) {
      Cfg c = best;
      c.chunk = ch;
      if ((st = consider(c))) return st;
    }
  apply(best);
  out->best.form = best.form;
  out->best.cell_order = best.order;
  out->best.jac_batch_pct = best.jac;
  out->best.waves_per_cu = best.wpc > 0 ? best.wpc : occ;
  out->best.chunk_cells = best.chunk;
  out->best.kernel_ms = best_ms;
  out->best.errtest_gather_pct = best.gather;
  out->best.refill_min_idle = best.refill;
  return NRG_CHEM_OK;
}

int nrg_chem_surrogate_step_dev(nrg_chem_t *h, nrg_mlp_t *mlp, const nrg_surrogate_norm *norm,
                                const nrg_surrogate_gate *gate, const nrg_grid *grid, double dt,
                                const double *T, const double *p, const double *rho,
                                const double *const *Y, const int8_t *bc,
                                double *const *Y_prod, double *const *Y_prod2, double *E_f_prod,
                                int32_t *cell_status, nrg_surrogate_stats *stats)
{
  if (!h || !gate) return set_error(NRG_CHEM_E_ARG, "handle or gate is NULL");
  const bool use_net = gate->screen != NRG_SUR_SCREEN_ONLY;
  if (use_net && (!mlp || !norm)) return set_error(NRG_CHEM_E_ARG, "network or norm is NULL");
  if (!(dt > 0.0) || !std::isfinite(dt)) return set_error(NRG_CHEM_E_ARG, "time_step must be > 0");
  if (!T || !rho || !Y || !Y_prod || !Y_prod2 || !E_f_prod || (use_net && !p))
    return set_error(NRG_CHEM_E_ARG, "required field pointer is NULL (the network needs p)");
  if (use_net && (mlp_n_in(mlp) != NIN || mlp_n_out(mlp) != NOUT))
    return set_error(NRG_CHEM_E_ARG, "network maps %d -> %d, the step needs %d -> %d", mlp_n_in(mlp),
                     mlp_n_out(mlp), NIN, NOUT);
  if (gate->n_elements < 0 || gate->n_elements > NRG_SUR_MAX_ELEMENTS)
    return set_error(NRG_CHEM_E_ARG, "n_elements must be in 0..%d", NRG_SUR_MAX_ELEMENTS);
  StepArgs a{};
  int st = make_grid(grid, a.g);
  if (st) return st;
  if (a.g.ninner >= (1ll << 31)) return set_error(NRG_CHEM_E_ARG, "more than 2^31 inner cells");
  SurArgs sa{};
  sa.g = a.g;
  for (int s = 0; s < S; ++s) {
    if (!Y[s] || !Y_prod[s] || !Y_prod2[s]) return set_error(NRG_CHEM_E_ARG, "species %d field is NULL", s + 1);
    a.Y[s] = sa.Y[s] = Y[s];
    a.Yp[s] = sa.Yp[s] = Y_prod[s];
    a.Yp2[s] = sa.Yp2[s] = Y_prod2[s];
  }
  a.dt = sa.dt = dt;
  a.k = h->k;
  a.mech = sa.mech = h->dev_mech;
  a.T = sa.T = T;
  a.rho = sa.rho = rho;
  sa.p = p;
  a.bc = sa.bc = bc;
  a.Efp = sa.Efp = E_f_prod;
  a.status = sa.status = cell_status;
  a.acc = h->dev_acc;
  a.jac_pct = h->jac_pct;
  sa.t_gate = h->k.t_gate;
  if (norm) {
    for (int i = 0; i < NIN; ++i) {
      sa.in_shift[i] = norm->in_shift[i];
      sa.in_scale[i] = norm->in_scale[i];
    }
    for (int i = 0; i < NOUT; ++i) {
      sa.out_shift[i] = norm->out_shift[i];
      sa.out_scale[i] = norm->out_scale[i];
    }
    sa.y_floor = norm->y_floor;
  }
  sa.t_min = gate->t_min; sa.t_max = gate->t_max;
  sa.p_min = gate->p_min; sa.p_max = gate->p_max;
  sa.dt_ok = dt >= gate->dt_min && dt <= gate->dt_max;
  sa.elem_tol = gate->elem_tol; sa.elem_floor = gate->elem_floor;
  sa.y_neg_tol = gate->y_neg_tol; sa.energy_tol = gate->energy_tol; sa.dT_max = gate->dT_max;
  sa.dT_freeze = gate->dT_freeze; sa.dY_freeze = gate->dY_freeze;
  if (!(gate->rate_tol >= 0.0)) return set_error(NRG_CHEM_E_ARG, "gate rate_tol must be >= 0");
  sa.rate_tol = gate->rate_tol;
  const int screen = gate->screen;
  if (screen != NRG_SUR_SCREEN_NONE && screen != NRG_SUR_SCREEN_RATES && screen != NRG_SUR_SCREEN_ONLY)
    return set_error(NRG_CHEM_E_ARG, "unknown gate screen %d", screen);
  if (screen != NRG_SUR_SCREEN_NONE && !(gate->dT_freeze > 0.0))
    return set_error(NRG_CHEM_E_ARG, "the explicit-rate screen needs dT_freeze > 0");
  sa.ne = gate->n_elements;
  for (int e = 0; e < sa.ne; ++e)
    for (int s = 0; s < S; ++s) sa.E[e][s] = gate->elements[e][s];

  HIP_TRY(hipSetDevice(h->device));
  const long long n = a.g.ninner;
  if (n > h->sur_cells) {
    for (void *q : {(void *)h->sur_X, (void *)h->sur_Y, (void *)h->sur_list, (void *)h->sur_rate_bad,
                    (void *)h->sur_cand, (void *)h->sur_recheck})
      if (q) HIP_TRY(hipFree(q));
    h->sur_X = nullptr; h->sur_Y = nullptr; h->sur_list = nullptr; h->sur_rate_bad = nullptr;
    h->sur_cand = nullptr; h->sur_recheck = nullptr;
    h->sur_cells = 0;
    HIP_TRY(hipMalloc(&h->sur_X, (size_t)n * MLP_IN_PAD * sizeof(bf16)));
    HIP_TRY(hipMalloc(&h->sur_Y, (size_t)n * NOUT * sizeof(float)));
    HIP_TRY(hipMalloc(&h->sur_list, (size_t)n * sizeof(int32_t)));
    HIP_TRY(hipMalloc(&h->sur_rate_bad, (size_t)n * sizeof(int8_t)));
    HIP_TRY(hipMalloc(&h->sur_cand, (size_t)n * sizeof(int32_t)));
    HIP_TRY(hipMalloc(&h->sur_recheck, (size_t)n * sizeof(int32_t)));
    h->sur_cells = n;
  }
  if (!h->sur_acc) HIP_TRY(hipMalloc(&h->sur_acc, SUR_SLOTS * sizeof(unsigned long long)));
  sa.X = h->sur_X;
  sa.Ypred = h->sur_Y;
  sa.list = h->sur_list;
  sa.rate_bad = h->sur_rate_bad;
  sa.acc = h->sur_acc;
  sa.cand = nullptr;
  sa.npos = n;

  hipLaunchKernelGGL(reset_kernel, dim3(1), dim3(ACC_SLOTS), 0, h->stream, h->dev_acc, ACC_SLOTS);
  hipLaunchKernelGGL(reset_kernel, dim3(1), dim3(SUR_SLOTS), 0, h->stream, h->sur_acc, SUR_SLOTS);
  HIP_TRY(hipGetLastError());
  unsigned long long sur[SUR_SLOTS] = {}, acc[16] = {};
  float ms_scr = 0.f, ms_inf = 0.f, ms_gate = 0.f, ms_fb = 0.f;
  long long ncand = n;
  if (n > 0) {
    HIP_TRY(hipEventRecord(h->ev0, h->stream));
    if (screen != NRG_SUR_SCREEN_NONE) {
      // the explicit-rate screen freezes the inert cells; the others go to the
      // network (SCREEN_RATES) or straight to the FP64 integrator (SCREEN_ONLY)
      sa.screen_out = screen == NRG_SUR_SCREEN_RATES ? h->sur_cand : h->sur_list;
      sa.screen_slot = screen == NRG_SUR_SCREEN_RATES ? SUR_CAND : SUR_FALLBACK;
      sa.screen_fp64 = gate->screen_fp64 != 0;
      sa.recheck = h->sur_recheck;
      sa.recheck_n = h->sur_acc + SUR_RECHECK;
      if (!h->recheck_blocks) {
        // resident blocks of the FP64 pass, which strides over its list
        int per_cu = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, rate_screen_kernel, 256, 0) != hipSuccess ||
            per_cu < 1)
          per_cu = 1;
        h->recheck_blocks = (long long)per_cu * h->num_cu;
      }
      // the FP32 pass over every cell, then the FP64 estimate on the cells it
      // lists (a grid that reads their number on the device)
      hipLaunchKernelGGL(screen_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, h->stream, sa);
      hipLaunchKernelGGL(rate_screen_kernel,
                         dim3((unsigned)std::min<long long>(h->recheck_blocks, (n + RCHECK_CELLS - 1) / RCHECK_CELLS)),
                         dim3(256), 0, h->stream, sa);
      HIP_TRY(hipGetLastError());
      HIP_TRY(read_counters(h, sur, h->sur_acc, SUR_SLOTS));
      ncand = screen == NRG_SUR_SCREEN_RATES ? (long long)sur[SUR_CAND] : 0;
      if (ncand > n || (long long)sur[SUR_FALLBACK] > n || (long long)sur[SUR_RECHECK] > n)
        return set_error(NRG_CHEM_E_HIP, "screen counts exceed %lld cells", n);
      sa.cand = h->sur_cand;
      sa.npos = ncand;
    }
    HIP_TRY(hipEventRecord(h->ev2, h->stream));
    if (ncand > 0) {
      const unsigned nb = (unsigned)((ncand + 255) / 256);
      hipLaunchKernelGGL(featurize_kernel, dim3(nb), dim3(256), 0, h->stream, sa);
      HIP_TRY(hipGetLastError());
      if ((st = mlp_infer_bf16(mlp, ncand, h->sur_X, h->sur_Y, h->stream))) return st;
    }
    HIP_TRY(hipEventRecord(h->ev3, h->stream));
    HIP_TRY(hipEventSynchronize(h->ev3));
    HIP_TRY(hipEventElapsedTime(&ms_scr, h->ev0, h->ev2));
    HIP_TRY(hipEventElapsedTime(&ms_inf, h->ev2, h->ev3));
    if (ncand > 0) {
      const unsigned nb = (unsigned)((ncand + 255) / 256);
      if (sa.rate_tol > 0.0) {
        hipLaunchKernelGGL(rate_check_kernel, dim3((unsigned)((ncand + RCHECK_CELLS - 1) / RCHECK_CELLS)),
                           dim3(256), 0, h->stream, sa);
        hipLaunchKernelGGL(gate_kernel<true>, dim3(nb), dim3(256), 0, h->stream, sa);
      } else
        hipLaunchKernelGGL(gate_kernel<false>, dim3(nb), dim3(256), 0, h->stream, sa);
      HIP_TRY(hipGetLastError());
    }
    HIP_TRY(hipEventRecord(h->ev2, h->stream));
    HIP_TRY(read_counters(h, sur, h->sur_acc, SUR_SLOTS));
    HIP_TRY(hipEventElapsedTime(&ms_gate, h->ev3, h->ev2));
    HIP_TRY(hipEventRecord(h->ev3, h->stream));
    const long long nfb = (long long)sur[SUR_FALLBACK];
    if (nfb > n) return set_error(NRG_CHEM_E_HIP, "fallback count %lld exceeds %lld cells", nfb, n);
    if (nfb > 0) {
      a.list = h->sur_list;
      // the fallback cells are the stiffest of the field: hand them out most
      // expensive first, by the step counts this handle recorded for them
      // (an FP64 step or an earlier fallback; temperature bins when it has
      // none for this grid), and record their step counts for the next call
      const bool ordered = h->order == NRG_ORDER_STIFFNESS;
      bool use_hist = false;
      if (ordered) {
        if ((st = prepare_order(h, n))) return st;
        use_hist = h->hist_valid && same_grid(h->hist_grid, a.g);
        enqueue_order(h, a, use_hist, h->sur_list, nfb);
        a.list = h->order_list;
        a.hist = h->hist;
        h->hist_valid = true;
        h->hist_grid = a.g;
      }
      const unsigned long long lanes =
          plan(h, h->seen_fallback, a, nfb, chunk_for(h, nfb), ordered, use_hist, true);
      if ((st = enqueue_integrator(h, a, nfb, lanes))) return st;
    }
    HIP_TRY(hipEventRecord(h->ev1, h->stream));
    HIP_TRY(read_counters(h, acc, h->dev_acc, 16));
    HIP_TRY(hipEventElapsedTime(&ms_fb, h->ev3, h->ev1));
    if (nfb > 0) note(h->seen_fallback, a.g, acc);
  }
  if (stats) {
    std::memset(stats, 0, sizeof(*stats));
    stats->cells_inner = n;
    stats->cells_gated = (int64_t)sur[SUR_GATED];
    stats->cells_accepted = (int64_t)sur[SUR_ACCEPT];
    stats->cells_fallback = (int64_t)sur[SUR_FALLBACK];
    stats->reject_domain = (int64_t)sur[SUR_R_DOMAIN];
    stats->reject_elements = (int64_t)sur[SUR_R_ELEM];
    stats->reject_negative = (int64_t)sur[SUR_R_NEG];
    stats->reject_energy = (int64_t)sur[SUR_R_ENERGY];
    stats->reject_confidence = (int64_t)sur[SUR_R_CONF];
    stats->reject_rate = (int64_t)sur[SUR_R_RATE];
    stats->cells_frozen = (int64_t)sur[SUR_FROZEN];
    stats->cells_network = ncand;
    stats->screen_ms = ms_scr;
    stats->cells_screen_fp64 = (int64_t)sur[SUR_RECHECK];
    stats->infer_ms = ms_inf;
    stats->gate_ms = ms_gate;
    stats->fallback_ms = ms_fb;
    fill_stats(acc, (long long)sur[SUR_FALLBACK], ms_fb, &stats->fallback);
  }
  return integrator_status(acc);
}

// ---- this topology's table for the C-ABI -------------------------------------
#define H(h) reinterpret_cast<nrg_chem_t *>(h)
#define NRG_TOPO_ADAPTER(name, params, args) static int op_##name params { return name args; }
NRG_TOPO_ENTRY_POINTS(NRG_TOPO_ADAPTER)
#undef NRG_TOPO_ADAPTER

static int op_check(const nrg_chem_mech *mech)
{
  MechCoef tmp;
  return build_mech(mech, tmp);
}
static int op_create(const nrg_chem_mech *mech, const nrg_chem_opts *opts, ::nrg_chem_t **out)
{
  nrg_chem_t *h = nullptr;
  const int st = nrg_chem_create(mech, opts, &h);
  *out = reinterpret_cast<::nrg_chem_t *>(h);
  return st;
}
static void op_destroy(::nrg_chem_t *h) { nrg_chem_destroy(H(h)); }
static void *op_stream(::nrg_chem_t *h) { return nrg_chem_stream(H(h)); }
#undef H

}  // namespace NRG_TOPO_NS
#pragma GCC visibility pop

__attribute__((visibility("hidden"))) const nrg_topo_ops *NRG_TOPO_OPS_FN()
{
  using namespace NRG_TOPO_NS;
#define NRG_TOPO_OP_INIT(name, params, args) t.name = op_##name;
  static const nrg_topo_ops table = [] {
    nrg_topo_ops t{};
    t.name = NRG_TOPO_NAME;
    t.check = op_check;
    t.create = op_create;
    t.destroy = op_destroy;
    t.stream = op_stream;
    NRG_TOPO_ENTRY_POINTS(NRG_TOPO_OP_INIT)
    return t;
  }();
#undef NRG_TOPO_OP_INIT
  return &table;
}
#endif  // NRG_PART < 2
