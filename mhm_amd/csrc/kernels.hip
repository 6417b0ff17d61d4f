// kernels.hip -- HIP kernels for gfx950: the per-cell chain and the routing.
//
// Cell kernels run one lane per (cell, parameter set).  Every row of P, S, X
// and F is a structure-of-arrays slab, so each of the ~70 loads and stores a
// lane makes per step is a fully coalesced 512-byte wavefront access.  Rows
// are addressed as a wave-uniform base (SGPRs) plus one 32-bit byte offset
// per lane shared by all rows, which maps onto global_load/store with
// saddr + voffset and keeps per-row 64-bit addresses out of the VGPRs.
//
// Routing is pipelined over (depth, time) diagonals: node p at depth delta
// (distance to its outlet) handles step t on diagonal d = t + dmax - delta.
// Its upstream nodes sit one level deeper, so they produced step t on
// diagonal d-1; a two-slot parity buffer of routed outflow (qTR) keeps step t
// readable while those nodes already write step t+1.  A whole run of T steps
// takes T + dmax diagonals instead of T * dmax level sweeps.  The default
// schedules run the same diagonals inside tiles of the tree, one workgroup per
// bin of tiles: route_stream_kernel all steps of the ring in one launch, tiles
// handing steps on while it runs, route_tile_kernel a window of steps per
// launch, handed from tile to tile between launches (one_launch_pays in api.hip
// chooses), route_step_kernel a single step; route_diag_kernel and
// route_wg_kernel run them over the whole grid or inside one workgroup.
#include <hip/hip_runtime.h>

#include "chain.h"
#include "internal.h"
#include "launch.h"

namespace mhmhip {

// row[boff / 8] with a uniform row base and a 32-bit per-lane byte offset
__device__ __forceinline__ double ldr(const double *row, uint32_t boff) {
  return *reinterpret_cast<const double *>(reinterpret_cast<const char *>(row) + boff);
}
__device__ __forceinline__ void str(double *row, uint32_t boff, double x) {
  *reinterpret_cast<double *>(reinterpret_cast<char *>(row) + boff) = x;
}
// Waits for v's load here and makes v count as defined by this (empty)
// statement.  A value loaded in a block that runs once per day or month and
// used every step otherwise leaves the compiler's memory-counter tracking
// unsure whether its load is still in flight where the paths merge, and the
// wait it puts there (every step) also waits for the step before's ring
// store.
__device__ __forceinline__ void settle(double &v) { asm volatile("" : "+v"(v)); }
// The lane's byte offset, made opaque where it is used: an address formed
// from it inside a loop cannot be hoisted out of the loop.  Rows stored in a
// block that runs once per launch (the last step's fluxes) then keep no
// 64-bit per-lane address in VGPRs across the whole time loop.
__device__ __forceinline__ uint32_t opaque(uint32_t v) {
  asm volatile("" : "+v"(v));
  return v;
}
// streaming store for outputs no kernel of the step reads back
#ifndef MHMHIP_NT_STORE
#define MHMHIP_NT_STORE 1
#endif
__device__ __forceinline__ void stn(double *row, uint32_t boff, double x) {
#if MHMHIP_NT_STORE
  __builtin_nontemporal_store(x, reinterpret_cast<double *>(reinterpret_cast<char *>(row) + boff));
#else
  str(row, boff, x);
#endif
}

// The kernel's arguments read through the constant address space: CellArgs is
// the first argument of every cell kernel, so its copy is at the start of the
// argument segment.  Members that are indexed at run time (OutAcc's) and
// out-of-line functions read it there with scalar loads; a by-value copy of
// them would live in scratch memory.
typedef const __attribute__((address_space(4))) CellArgs ConstArgs;
__device__ __forceinline__ ConstArgs *kernel_args() {
  return (ConstArgs *)__builtin_amdgcn_kernarg_segment_ptr();
}
// A pointer that is the same in every lane, as one the compiler knows to be
__device__ __forceinline__ ConstArgs *uniform(ConstArgs *p) {
  const uint64_t v = (uint64_t)p;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return (ConstArgs *)(((uint64_t)hi << 32) | lo);
}
// For a block that a time loop runs now and then: the arguments read there
// instead of being held in scalar registers across the loop.
__device__ __forceinline__ ConstArgs *rare(ConstArgs *p) {
  asm volatile("" : "+s"(p));
  return p;
}
// every argument but the output sums
__device__ __forceinline__ CellArgs read_args(ConstArgs *p) {
  CellArgs a;
  a.P = p->P, a.S = p->S, a.X = p->X, a.F = p->F, a.ring = p->ring, a.area = p->area;
  a.lag = p->lag, a.tst = p->tst, a.steps = p->steps;
  a.n_cells = p->n_cells, a.sstride = p->sstride, a.ld = p->ld;
  a.forcing_days = p->forcing_days, a.ring_len = p->ring_len, a.pet_case = p->pet_case;
  a.jarvis = p->jarvis, a.hourly = p->hourly, a.ring_rep = p->ring_rep;
  a.raw_total = p->raw_total, a.nT = p->nT, a.rnT = p->rnT, a.W = p->W;
  a.sun = p->sun, a.sun_step0 = p->sun_step0, a.skip_fluxes = p->skip_fluxes;
  return a;
}

template <int NH>
struct CellRegs {
  double fS, thrS, c1, k0s, k1s, k2s, kps, alpha, karst, thrU, dmaxs, dnps, incr, tth;
  double sat[NH], fr[NH], fc[NH], wp[NH], bexp[NH];
  // correctly rounded reciprocals of the per-cell divisors (div_rcp)
  double rthrS, rsat[NH];
  double inter, pack, seal, unsat, satS;
  double sm[NH];
};

// Waits for every load of a cell's parameters and states.
template <int NH>
__device__ __forceinline__ void settle_all(CellRegs<NH> &c) {
  settle(c.fS), settle(c.thrS), settle(c.c1), settle(c.k0s), settle(c.k1s), settle(c.k2s);
  settle(c.kps), settle(c.alpha), settle(c.karst), settle(c.thrU), settle(c.dmaxs);
  settle(c.dnps), settle(c.incr), settle(c.tth), settle(c.inter), settle(c.pack);
  settle(c.seal), settle(c.unsat), settle(c.satS);
#pragma unroll
  for (int h = 0; h < NH; ++h) {
    settle(c.sat[h]), settle(c.bexp[h]), settle(c.sm[h]);
    settle(c.fr[h]), settle(c.fc[h]), settle(c.wp[h]);
  }
}

template <int NH>
struct FluxRegs {
  double pet, temp, prec, thr, ecan, ddf, melt, peff, rain, snow, rseal, aseal, fast, slow, perc,
      bflow, total;
  double infil[NH], aet[NH];
};

template <int NH, bool JV>
__device__ __forceinline__ void load_params(const CellArgs &a, uint32_t bv, CellRegs<NH> &c) {
  auto P = [&](int r) { return ldr(a.P + (int64_t)r * a.ld, bv); };
  c.fS = P(PR_FS);
  c.thrS = P(PR_SEALTHR);
  c.c1 = JV ? P(PR_JARVIS) : 0.0;
  c.k0s = P(PR_K0S);
  c.k1s = P(PR_K1S);
  c.k2s = P(PR_K2S);
  c.kps = P(PR_KPS);
  c.alpha = P(PR_ALPHA);
  c.karst = P(PR_KARST);
  c.thrU = P(PR_UNSATTHR);
  c.dmaxs = P(PR_DMAXS);
  c.dnps = P(PR_DNPS);
  c.incr = P(PR_INCR);
  c.tth = P(PR_TTH);
#pragma unroll
  for (int h = 0; h < NH; ++h) {
    c.sat[h] = P(pr_sat(NH) + h);
    c.fr[h] = P(pr_froots(NH) + h);
    c.fc[h] = P(pr_fc(NH) + h);
    c.wp[h] = P(pr_wp(NH) + h);
    c.bexp[h] = P(pr_exp(NH) + h);
  }
  c.rthrS = 1.0 / c.thrS;
#pragma unroll
  for (int h = 0; h < NH; ++h) c.rsat[h] = 1.0 / c.sat[h];
}

template <int NH>
__device__ __forceinline__ void load_states(const CellArgs &a, uint32_t bv, CellRegs<NH> &c) {
  auto S = [&](int r) { return ldr(a.S + (int64_t)r * a.ld, bv); };
  c.inter = S(SR_INTER);
  c.pack = S(SR_SNOW);
  c.seal = S(SR_SEAL);
  c.unsat = S(SR_UNSAT);
  c.satS = S(SR_SAT);
#pragma unroll
  for (int h = 0; h < NH; ++h) c.sm[h] = S(SR_NSCALAR + h);
}

template <int NH>
__device__ __forceinline__ void store_states(const CellArgs &a, uint32_t bv0,
                                             const CellRegs<NH> &c) {
  const uint32_t bv = opaque(bv0);
  auto S = [&](int r, double x) { str(a.S + (int64_t)r * a.ld, bv, x); };
  S(SR_INTER, c.inter);
  S(SR_SNOW, c.pack);
  S(SR_SEAL, c.seal);
  S(SR_UNSAT, c.unsat);
  S(SR_SAT, c.satS);
#pragma unroll
  for (int h = 0; h < NH; ++h) S(SR_NSCALAR + h, c.sm[h]);
}

// the step's meteo values and the fluxes of the canopy and the snow
template <int NH>
__device__ __forceinline__ void store_fluxes_canopy(const CellArgs &a, uint32_t bv0,
                                                    const FluxRegs<NH> &x) {
  const uint32_t bv = opaque(bv0);
  auto X = [&](int r, double y) { stn(a.X + (int64_t)r * a.ld, bv, y); };
  X(XR_PET, x.pet);
  X(XR_TEMP, x.temp);
  X(XR_PREC, x.prec);
  X(XR_THROUGHFALL, x.thr);
  X(XR_AETCAN, x.ecan);
  X(XR_DEGDAY, x.ddf);
  X(XR_MELT, x.melt);
  X(XR_PEFF, x.peff);
  X(XR_RAIN, x.rain);
  X(XR_SNOW, x.snow);
}

// those of the sealed area, the soil and the fast interflow
template <int NH>
__device__ __forceinline__ void store_fluxes_soil(const CellArgs &a, uint32_t bv0,
                                                  const FluxRegs<NH> &x) {
  const uint32_t bv = opaque(bv0);
  auto X = [&](int r, double y) { stn(a.X + (int64_t)r * a.ld, bv, y); };
  X(XR_RUNOFFSEAL, x.rseal);
  X(XR_AETSEAL, x.aseal);
  X(XR_FAST, x.fast);
#pragma unroll
  for (int h = 0; h < NH; ++h) {
    X(xr_infil(NH) + h, x.infil[h]);
    X(xr_aet(NH) + h, x.aet[h]);
  }
}

// those of the slow interflow and the groundwater
template <int NH>
__device__ __forceinline__ void store_fluxes_post(const CellArgs &a, uint32_t bv0,
                                                  const FluxRegs<NH> &x) {
  const uint32_t bv = opaque(bv0);
  auto X = [&](int r, double y) { stn(a.X + (int64_t)r * a.ld, bv, y); };
  X(XR_SLOW, x.slow);
  X(XR_PERC, x.perc);
  X(XR_BASEFLOW, x.bflow);
  X(XR_TOTAL, x.total);
}

template <int NH>
__device__ __forceinline__ void store_fluxes(const CellArgs &a, uint32_t bv, const FluxRegs<NH> &x) {
  store_fluxes_canopy<NH>(a, bv, x);
  store_fluxes_soil<NH>(a, bv, x);
  store_fluxes_post<NH>(a, bv, x);
}

// One step's contribution to the output sums (mHM_updateDataset,
// src/mHM/mo_write_fluxes_states.f90:283-438, updateVariable): each selected
// output's value of the step -- states after it, its fluxes -- in the
// reference's expression and operation order, added to its sum.  Horizon
// sums run from 0 over the horizons in order (sum(..., dim = 2)); the
// unsealed fraction is 1 - fSealed (mo_mhm_interface_run.f90:239).  In three
// parts, each as soon as its values are known; put(bit, value) is called
// for the outputs in the order of their bits.
template <int NH, typename Put>
__device__ __forceinline__ void outputs_canopy(const CellRegs<NH> &c, const FluxRegs<NH> &x,
                                               Put put) {
  put(out_bit(1, 0, NH), [&] { return c.inter; });
  put(out_bit(2, 0, NH), [&] { return c.pack; });
  put(out_bit(9, 0, NH), [&] { return x.pet; });
  put(out_bit(20, 0, NH), [&] { return x.peff; });
  put(out_bit(21, 0, NH), [&] { return x.melt; });
}

template <int NH, typename Put>
__device__ __forceinline__ void outputs_soil(const CellRegs<NH> &c, const FluxRegs<NH> &x,
                                             double ecan, Put put) {
  const double fs = c.fS, fns = 1.0 - c.fS;
  auto hsum = [](const double (&v)[NH]) {
    double s = 0.0;
#pragma unroll
    for (int h = 0; h < NH; ++h) s = s + v[h];
    return s;
  };
#pragma unroll
  for (int h = 0; h < NH; ++h) put(out_bit(3, h, NH), [&] { return c.sm[h]; });
#pragma unroll
  for (int h = 0; h < NH; ++h) put(out_bit(4, h, NH), [&] { return c.sm[h] / c.sat[h]; });
  put(out_bit(5, 0, NH), [&] { return hsum(c.sm) / hsum(c.sat); });
  put(out_bit(6, 0, NH), [&] { return c.seal; });
  put(out_bit(10, 0, NH), [&] { return hsum(x.aet) * fns + ecan + x.aseal * fs; });
  put(out_bit(12, 0, NH), [&] { return x.rseal * fs; });
  put(out_bit(13, 0, NH), [&] { return x.fast * fns; });
#pragma unroll
  for (int h = 0; h < NH; ++h) put(out_bit(17, h, NH), [&] { return x.infil[h] * fns; });
#pragma unroll
  for (int h = 0; h < NH; ++h) put(out_bit(19, h, NH), [&] { return x.aet[h] * fns; });
}

template <int NH, typename Put>
__device__ __forceinline__ void outputs_post(const CellRegs<NH> &c, const FluxRegs<NH> &x,
                                             Put put) {
  const double fns = 1.0 - c.fS;
  put(out_bit(7, 0, NH), [&] { return c.unsat; });
  put(out_bit(8, 0, NH), [&] { return c.satS; });
  put(out_bit(11, 0, NH), [&] { return x.total; });
  put(out_bit(14, 0, NH), [&] { return x.slow * fns; });
  put(out_bit(15, 0, NH), [&] { return x.bflow * fns; });
  put(out_bit(16, 0, NH), [&] { return x.perc * fns; });
}

// The plain kernel's: straight to the sums.
template <int NH>
__device__ __forceinline__ void add_outputs(ConstArgs *k, int64_t ld, uint32_t bv,
                                            const CellRegs<NH> &c, const FluxRegs<NH> &x) {
  const uint64_t mask = k->out.mask;
  double *row = k->out.sum;
  auto put = [&](int bit, auto value) {
    if (!(mask >> bit & 1)) return;
    str(row, bv, ldr(row, bv) + value());
    row += ld;
  };
  outputs_canopy<NH>(c, x, put);
  outputs_soil<NH>(c, x, x.ecan, put);
  outputs_post<NH>(c, x, put);
}

// Daily PET before disaggregation (get_corrected_pet, mo_meteo_handler.f90:1050-1097).
// Its per-cell parameters are read here, when a new forcing day starts, rather
// than held in registers across steps.  bc: byte offset of the cell in a
// forcing row; bv: byte offset of (cell, set) in a parameter row.
__device__ __forceinline__ const double *frow_ptr(const CellArgs &a, int v, int32_t day) {
  return a.F + ((int64_t)forcing_row(v, a.pet_case) * a.forcing_days + day) * a.sstride;
}

template <int NH>
__device__ __forceinline__ double pet_day(const CellArgs &a, const StepDev &st, uint32_t bv,
                                          uint32_t bc, double tavg, double tmax, double tmin) {
  auto P = [&](int r) { return ldr(a.P + (int64_t)r * a.ld, bv); };
  if (a.pet_case == 1)
    return P(PR_FASP) * pet_hargreaves(P(PR_HARSAM), tavg, tmax, tmin, P(PR_TANLAT),
                                       P(PR_SINLAT), P(PR_COSLAT), st.dr, st.tand, st.sind,
                                       st.cosd);
  if (a.pet_case >= 2) {
    // Priestley-Taylor and Penman-Monteith are not defined for netrad < 0
    const double rn = vmax0(ldr(frow_ptr(a, MHMHIP_F_NETRAD, st.day), bc));
    if (a.pet_case == 2) return pet_priestly(P(pr_prietay(NH) + st.month0), rn, tavg);
    const double avp = ldr(frow_ptr(a, MHMHIP_F_ABSVAPPRESS, st.day), bc) / 1000.0;
    const double ws = ldr(frow_ptr(a, MHMHIP_F_WINDSPEED, st.day), bc);
    return pet_penman(rn, tavg, avp, P(pr_aero(NH) + st.month0) / ws,
                      P(pr_surf(NH) + st.month0));
  }
  const double petin = ldr(frow_ptr(a, MHMHIP_F_PET, st.day), bc);
  if (a.pet_case == 0) return P(PR_FASP) * petin;
  return P(pr_petlai(NH) + st.month0) * petin;
}

// The step's pet, temp and prec from the daily values: the meteo weights of
// the step's month and hour when given, else the day/night factors
// (get_corrected_pet 1099-1118, get_temp 1183-1200, get_prec 1265-1282).
template <int NH>
__device__ __forceinline__ void disagg_step(const CellArgs &a, const StepDev &st, uint32_t bc,
                                            double pd, double tavg, double pre, double &pet,
                                            double &temp, double &prec) {
  if (a.hourly) {
    pet = pd;
    temp = tavg;
    prec = pre;
  } else if (a.W) {
    const int64_t wv = (int64_t)12 * 24 * a.sstride;
    const double *w = a.W + (int64_t)st.wrow * a.sstride;
    pet = disagg_weights(pd, ldr(w + 2 * wv, bc), 0.0);
    temp = disagg_weights(tavg, ldr(w + wv, bc), kT0);
    prec = disagg_weights(pre, ldr(w, bc), 0.0);
  } else {
    pet = disagg_flux(a.nT, a.rnT, pd, st.f_pet);
    temp = disagg_state_add(a.nT, tavg, st.f_temp);
    prec = disagg_flux(a.nT, a.rnT, pre, st.f_prec);
  }
}

// The step table is read-only during a launch and the same for every lane:
// read through the constant address space, it comes in with scalar loads
// into SGPRs instead of vector loads into VGPRs.
typedef const __attribute__((address_space(4))) StepDev ConstStep;
// read_step copies every field: a field added to StepDev is added there too
static_assert(sizeof(StepDev) == 9 * sizeof(double) + 7 * sizeof(int32_t) + 4,
              "StepDev changed: update read_step");
__device__ __forceinline__ StepDev read_step(const ConstStep *p) {
  StepDev st;
  st.dr = p->dr;
  st.tand = p->tand;
  st.sind = p->sind;
  st.cosd = p->cosd;
  st.f_pet = p->f_pet;
  st.f_prec = p->f_prec;
  st.f_temp = p->f_temp;
  st.evap = p->evap;
  st.revap = p->revap;
  st.day = p->day;
  st.month0 = p->month0;
  st.isday = p->isday;
  st.init_sm = p->init_sm;
  st.doy = p->doy;
  st.change = p->change;
  st.wrow = p->wrow;
  return st;
}

// L11_runoff_acc for L1 = L11 with map_flag (mo_mrm_pre_routing.f90:110-126):
// qAcc = 0; qAcc = qAcc + q * area; qAcc = qAcc * 1000 / TST   [m3 s-1], as q
// times the cell's area * 1000 / TST (one product a step instead of two and a
// division; as many roundings).  raw_total: the total itself.
__device__ __forceinline__ double runoff_scale(const CellArgs &a, uint32_t bc) {
  return a.raw_total ? 1.0 : ldr(a.area, bc) * 1000.0 / a.tst;
}

// Every horizon's (sm / sat)**beta depends only on the soil moisture at the
// start of the step: the bases and exponents of these NH powers, into
// slots off .. off + NH - 1.  Bases the reference never raises to a power
// are replaced by 1 and their results left unused.
template <int NH, int N>
__device__ __forceinline__ void horizon_pow_args(const CellRegs<NH> &c, DV<N> &py, DV<N> &px,
                                                 int off) {
#pragma unroll
  for (int h = 0; h < NH; ++h) {
    const double q = div_rcp(c.sm[h], c.sat[h], c.rsat[h]);
    py.v[off + h] = c.bexp[h];
    px.v[off + h] = q > 0.0 ? q : 1.0;
  }
}

template <int NH>
__device__ __forceinline__ DV<NH> horizon_pows(const CellRegs<NH> &c) {
  DV<NH> py, px;
  horizon_pow_args<NH, NH>(c, py, px, 0);
  return exp_ylogx_v<NH>(py, px);
}

// One step of mHM() for one cell after the meteo getters (mo_mhm.f90:455-519),
// in two parts around the slow interflow's power: chain_pre (canopy, snow,
// soil moisture with the horizon powers pwh of the step's starting soil
// moisture, fast interflow) and chain_post (slow interflow with pw_slow =
// unsat**(1 + alpha), percolation, baseflow, total runoff).  The canopy's
// (interc / interc_max)**(2/3) is pow23.
// JV: Jarvis soil-moisture stress (processCase(3) = 2, 3) instead of Feddes
// The soil-moisture stress parameters of a cell, passed on their own: the
// fused kernel keeps them in LDS between steps.  For the general functions
// fw is the field capacity and slope RN(1 / (fc - wp)); for the ordinary ones
// see stress_ordinary (Feddes does not read fw).
template <int NH>
struct Stress {
  double fr[NH], wp[NH], slope[NH], fw[NH];
};

template <int NH, bool JV>
__device__ __forceinline__ Stress<NH> stress_of(const CellRegs<NH> &c, bool ordinary) {
  Stress<NH> t;
#pragma unroll
  for (int h = 0; h < NH; ++h) {
    const double range = (JV && ordinary ? c.sat[h] : c.fc[h]) - c.wp[h];
    t.fr[h] = c.fr[h];
    t.wp[h] = c.wp[h];
    t.slope[h] = (!JV && ordinary ? c.fr[h] : 1.0) / range;
    t.fw[h] = ordinary ? range : c.fc[h];
  }
  return t;
}

// odd: the cell's weather mark (CellArgs::odd_weather)
template <int NH, bool JV>
__device__ __forceinline__ bool ordinary_cell(const CellRegs<NH> &c, bool init_sm, uint32_t odd) {
  // no branch on odd: the loads it would hold back are as far away as its own
  const bool ok = (odd == 0) & ordinary_params<NH, JV>(
                                   c.fS, c.thrS, c.incr, c.dmaxs, c.dnps, c.tth, c.k0s, c.k1s,
                                   c.k2s, c.kps, c.karst, c.alpha, c.thrU, c.sat, c.fr, c.fc,
                                   c.wp, c.bexp, c.c1);
  // a step that resets the soil moisture starts from half the field capacity
  double sm[NH];
#pragma unroll
  for (int h = 0; h < NH; ++h) sm[h] = init_sm ? 0.5 * c.fc[h] : c.sm[h];
  return ok && ordinary_states<NH>(c.inter, c.pack, c.seal, c.unsat, c.satS, sm, c.sat);
}

template <int NH, bool JV>
__device__ __forceinline__ void chain_pre(CellRegs<NH> &c, FluxRegs<NH> &x, double maxinter,
                                          double rmaxinter, double evap, double revap,
                                          const double *pwh, const Stress<NH> &t) {
  const double ratio = canopy_fill(maxinter, rmaxinter, x.prec, c.inter, x.thr);
  canopy_evap(x.pet, maxinter, ratio, ratio > 0.0 ? pow23(ratio) : 0.0, c.inter, x.ecan);
  // snow_accum_melt's branch threshold (mo_snow_accum_melt.f90:127)
  const double ddthr = (c.dmaxs - c.dnps) / c.incr;
  snow_accum_melt(c.incr, c.dmaxs, c.dnps, ddthr, x.prec, x.temp, c.tth, x.thr, c.pack, x.ddf,
                  x.melt, x.peff, x.rain, x.snow);
  soil_moisture<NH, JV>(c.fS, c.thrS, c.rthrS, x.pet, evap, revap, c.sat, t.fr, t.fw, t.wp, t.slope,
                        c.c1, x.ecan, x.peff, pwh, x.rseal, c.seal, x.infil, c.sm, x.aet, x.aseal);
  runoff_fast(c.k0s, x.infil[NH - 1], c.thrU, c.unsat, x.fast);
}

template <int NH>
__device__ __forceinline__ void chain_post(CellRegs<NH> &c, FluxRegs<NH> &x, double pw_slow) {
  runoff_slow_perc(c.k1s, c.kps, c.karst, pw_slow, c.satS, c.unsat, x.slow, x.perc);
  runoff_sat_zone(c.k2s, c.satS, x.bflow);
  x.total = total_runoff(c.fS, x.fast, x.slow, x.bflow, x.rseal);
}

template <int NH, bool JV>
__device__ __forceinline__ void chain_step(CellRegs<NH> &c, FluxRegs<NH> &x, double maxinter,
                                           double rmaxinter, double evap, double revap,
                                           const Stress<NH> &t) {
  const DV<NH> pwh = horizon_pows<NH>(c);
  chain_pre<NH, JV>(c, x, maxinter, rmaxinter, evap, revap, pwh.v, t);
  chain_post<NH>(c, x, c.unsat > 0.0 ? exp_ylogx(1.0 + c.alpha, c.unsat) : 0.0);
}

// The same step for an ordinary cell, in the parts the fused kernel
// interleaves: canopy and snow; the soil with the horizon powers of the
// step's starting soil moisture (wet: some lane of the wave has water to
// infiltrate; a dry wave's powers are not needed) and the fast interflow; the
// slow interflow (pw_slow: its power), groundwater and total runoff.
template <int NH>
__device__ __forceinline__ void ordinary_canopy(CellRegs<NH> &c, FluxRegs<NH> &x, double melt_meteo,
                                                double cold, double maxinter, double rmaxinter) {
  canopy_ordinary(x.pet, maxinter, rmaxinter, x.prec, c.inter, x.thr, x.ecan);
  snow_ordinary(melt_meteo, cold, x.thr, c.pack, x.melt, x.peff, x.rain, x.snow);
}

template <int NH, bool JV>
__device__ __forceinline__ void ordinary_soil(CellRegs<NH> &c, FluxRegs<NH> &x, double demand,
                                              double pe, double ecan, double peff, bool wet,
                                              const double *pwh, double rc1,
                                              const Stress<NH> &t) {
  sealed_ordinary(c.fS > 0.0, c.thrS, c.rthrS, pe, ecan, peff, x.rseal, c.seal, x.aseal);
#pragma unroll
  for (int h = 0; h < NH; ++h) x.infil[h] = 0.0;
  if (wet) {
#pragma unroll
    for (int h = 0; h < NH; ++h)
      x.infil[h] = infiltrate_ordinary(h ? x.infil[h ? h - 1 : 0] : peff, pwh[h], c.sat[h], c.sm[h]);
  }
  double used = 0.0;
#pragma unroll
  for (int h = 0; h < NH; ++h) {
    const double f = stress_ordinary<JV>(c.sm[h], t.wp[h], t.fr[h], t.slope[h], t.fw[h], c.c1, rc1);
    x.aet[h] = evaporate_ordinary(h ? demand - used : demand, f, c.sm[h]);
    used = h ? used + x.aet[h] : x.aet[h];
  }
  runoff_fast_ordinary(c.k0s, x.infil[NH - 1], c.thrU, c.unsat, x.fast);
}

// what a cell without sealed area reports for it
template <int NH>
__device__ __forceinline__ void report_sealed(const CellRegs<NH> &c, FluxRegs<NH> &x) {
  x.rseal = c.fS > 0.0 ? x.rseal : 0.0;
  x.aseal = c.fS > 0.0 ? x.aseal : 0.0;
}

template <int NH>
__device__ __forceinline__ void ordinary_post(CellRegs<NH> &c, FluxRegs<NH> &x, double pw_slow,
                                              double rseal) {
  runoff_slow_perc_ordinary(c.k1s, c.kps, c.karst, pw_slow, c.satS, c.unsat, x.slow, x.perc);
  x.bflow = c.k2s * c.satS;
  c.satS = c.satS - x.bflow;
  x.total = total_runoff(c.fS, x.fast, x.slow, x.bflow, rseal);
}

// base of the slow interflow's power (an empty store: a power next to 0)
__device__ __forceinline__ double slow_base(double unsat) { return vmax_k(unsat, DBL_MIN); }

// The plain kernel's: each flux leaves as soon as it is known, so that the
// registers do not hold them across the powers.
template <int NH, bool JV>
__device__ __forceinline__ void ordinary_step(const CellArgs &a, uint32_t bv, CellRegs<NH> &c,
                                              FluxRegs<NH> &x, double maxinter, double rmaxinter,
                                              double pe, const Stress<NH> &t) {
  const SnowMeteo m = snow_meteo(c.incr, c.dmaxs, c.dnps, c.tth, x.prec, x.temp);
  x.ddf = m.ddf;
  ordinary_canopy<NH>(c, x, m.melt, m.cold, maxinter, rmaxinter);
  store_fluxes_canopy<NH>(a, bv, x);
  const bool wet = __any(x.peff != 0.0);
  DV<NH> py, px;
  if (wet) {
#pragma unroll
    for (int h = 0; h < NH; ++h) {
      py.v[h] = 256.0 * c.bexp[h];
      px.v[h] = div_rcp(c.sm[h], c.sat[h], c.rsat[h]);
    }
    px = pow_v<NH>(py, px);
  }
  ordinary_soil<NH, JV>(c, x, x.pet - x.ecan, pe, x.ecan, x.peff, wet, px.v, JV ? 1.0 / c.c1 : 0.0,
                        t);
  const double rseal = x.rseal;  // finite, of weight 0 without sealed area
  report_sealed<NH>(c, x);
  store_fluxes_soil<NH>(a, bv, x);
  const DV<1> pw = pow_v<1>(DV<1>{{256.0 * (1.0 + c.alpha)}}, DV<1>{{slow_base(c.unsat)}});
  ordinary_post<NH>(c, x, pw.v[0], rseal);
  store_fluxes_post<NH>(a, bv, x);
}

// ---------------------------------------------------------------------------
// Plain path: one launch per model step; every state and flux is written.
// The cell's loads are issued before the log / exp tables are filled, so the
// fill's reads and barrier wait behind them rather than in front.
//
// Bound by the memory it reads and writes (700x900 cells, 3 horizons: 55 us at
// 5.6 TB/s).  A cell outside the ordinary ranges takes the branches in the
// same kernel, from the same loads; the end of the step stands in both ways,
// so that nothing but the step's start is live where they part (four waves
// per SIMD, no spilled registers at up to 3 horizons).  With the branches in a
// function of their own, which saves the caller's registers and loads the cell
// again, 512x512 cells took 91 us a step where all are such cells, 57 with one
// in 64 and 34 with none; now 31, 34 and 31.
struct StepArgs {
  StepDev st;
  int64_t t;
};

template <int NH, bool JV, bool OUT>
__device__ __forceinline__ void step_end(ConstArgs *k, const CellArgs &a, uint32_t c, uint32_t bv,
                                         int64_t t, double scale, int32_t g,
                                         const CellRegs<NH> &r, const FluxRegs<NH> &x) {
  store_states<NH>(a, bv, r);
  if (OUT) add_outputs<NH>(k, a.ld, bv, r, x);
  if (a.ring) {
    const double q = x.total * scale;
    for (int32_t i = 0; i < a.ring_rep; ++i)
      a.ring[ring_row(t * a.ring_rep + i, g, a.ring_len) * a.ld + bv / 8u] = q;
  }
}

template <int NH>
__device__ __forceinline__ void step_start(const CellArgs &a, const StepDev &st, uint32_t bc,
                                           uint32_t bv, double pre, double tavg, double tmax,
                                           double tmin, CellRegs<NH> &r, FluxRegs<NH> &x) {
  const double pd = pet_day<NH>(a, st, bv, bc, tavg, tmax, tmin);
  disagg_step<NH>(a, st, bc, pd, tavg, pre, x.pet, x.temp, x.prec);
  if (st.init_sm) {
#pragma unroll
    for (int h = 0; h < NH; ++h) r.sm[h] = 0.5 * r.fc[h];
  }
}

template <int NH, bool JV, bool OUT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(NH > 3 ? 2 : OUT ? 3 : 4)))
void cell_step_kernel(CellArgs a, StepArgs sa) {
  static_assert(sizeof(CellArgs) % alignof(StepArgs) == 0, "StepArgs follows CellArgs");
  const StepDev &st = sa.st;
  const uint32_t c0 = blockIdx.x * blockDim.x + threadIdx.x;
  const bool act = c0 < a.n_cells;
  const uint32_t c = act ? c0 : 0u;  // an idle lane loads cell 0 and leaves after the fill
  const uint32_t bc = c * 8u;
  const uint32_t bv = (uint32_t)(blockIdx.y * a.sstride + c) * 8u;
  CellRegs<NH> r;
  FluxRegs<NH> x;
  load_params<NH, JV>(a, bv, r);
  load_states<NH>(a, bv, r);
  const double pre = ldr(frow_ptr(a, MHMHIP_F_PRE, st.day), bc);
  const double tavg = ldr(frow_ptr(a, MHMHIP_F_TAVG, st.day), bc);
  const double tmax = a.pet_case == 1 ? ldr(frow_ptr(a, MHMHIP_F_TMAX, st.day), bc) : 0.0;
  const double tmin = a.pet_case == 1 ? ldr(frow_ptr(a, MHMHIP_F_TMIN, st.day), bc) : 0.0;
  const uint32_t odd = a.odd_weather[c];
  mathtab_fill();  // the chain's powers read it (every thread, before any returns)
  if (!act) return;
  const bool ordinary = ordinary_cell<NH, JV>(r, st.init_sm != 0, odd);
  step_start<NH>(a, st, bc, bv, pre, tavg, tmax, tmin, r, x);
  // after the daily PET's call, which they would have to be kept across
  double maxinter = ldr(a.P + (int64_t)(pr_maxinter(NH) + st.month0) * a.ld, bv);
  double scale = a.ring ? runoff_scale(a, bc) : 0.0;
  int32_t g = a.ring && a.lag ? a.lag[c] : 0;
  // no load is waited for once the stores start: they share a counter
  settle(maxinter);
  settle(scale);
  asm volatile("" : "+v"(g));
  settle_all<NH>(r);
  if (ordinary) {
    ordinary_step<NH, JV>(a, bv, r, x, maxinter, maxinter > kEps ? 1.0 / maxinter : 0.0,
                          div_rcp(x.pet, st.evap, st.revap), stress_of<NH, JV>(r, true));
    step_end<NH, JV, OUT>(kernel_args(), a, c, bv, sa.t, scale, g, r, x);
  } else {
    chain_step<NH, JV>(r, x, maxinter, 1.0 / maxinter, st.evap, st.revap,
                       stress_of<NH, JV>(r, false));
    store_fluxes<NH>(a, bv, x);
    step_end<NH, JV, OUT>(kernel_args(), a, c, bv, sa.t, scale, g, r, x);
  }
}

// Per-lane LDS slots of the fused kernel (dynamic shared memory,
// lane_slots doubles per thread, laid out lane after lane; an odd count
// puts the 64-bit accesses of a wave's lanes on distinct bank pairs): the
// values that change once per forcing day, month or day/night switch, the
// soil-moisture stress parameters read once per step and the launch's output
// sums -- in LDS rather than in registers across the whole time loop.  The
// sums take the steps' values in step order as they would in memory, and cost
// a launch one read and one write of a row instead of one per step.
enum LaneSlot {
  LS_PD = 0, LS_MAXI, LS_RMAXI, LS_XPET, LS_XPE, LS_XPREC, LS_XMELT, LS_XCOLD, LS_STRESS
};
// Jarvis and the general functions read a fourth stress parameter; a general
// lane of the Feddes kernel takes it from memory
__host__ __device__ constexpr int stress_slots(int nh, bool jv) { return (jv ? 4 : 3) * nh; }
__host__ __device__ constexpr int lane_slots(int nh, bool jv, int n_out) {
  return (LS_STRESS + stress_slots(nh, jv) + n_out) | 1;
}
extern __shared__ double s_lane[];

// The lane's place in a fused launch.
struct FusedLane {
  uint32_t bc, bv;     // byte offsets of the cell in a forcing row, of (cell, set) in a row
  uint32_t slot;       // first LDS slot
  double scale;        // runoff_scale
  double *ring;        // ring row 0 of the node (its lag folded in), null: no routing
  int64_t roff;        // element offset of the step's first ring row
  int32_t sun;         // 1: the wave reads its days' sun terms (sun_kernel)
};

// The step's qOUT to its rep ring rows.
__device__ __forceinline__ void put_ring(const CellArgs &a, FusedLane &u, int64_t wrap, int rep,
                                         double total) {
  if (!a.ring) return;
  const double q = total * u.scale;
  int i = rep;
  do {
    u.ring[u.roff] = q;
    u.roff += a.ld;
    if (u.roff == wrap) u.roff = 0;
  } while (--i > 0);
}

// disagg_step with the forcing day's values read here
template <int NH>
__device__ __forceinline__ void disagg_at(const CellArgs &a, const StepDev &st, uint32_t bc,
                                          double pd, double &pet, double &temp, double &prec) {
  const double pre = ldr(frow_ptr(a, MHMHIP_F_PRE, st.day), bc);
  const double tavg = ldr(frow_ptr(a, MHMHIP_F_TAVG, st.day), bc);
  disagg_step<NH>(a, st, bc, pd, tavg, pre, pet, temp, prec);
}

// The daily PET into its slot, out of line and from its own loads: the time
// loop around it holds no register for it.  shared: the sun terms are there.
template <int NH>
__device__ __attribute__((noinline)) void day_pet(ConstArgs *args, uint32_t bc, uint32_t bv,
                                                  uint32_t slot, const ConstStep *step,
                                                  int32_t shared) {
  const CellArgs a = read_args(uniform(args));
  const ConstStep *p = (const ConstStep *)uniform((ConstArgs *)step);
  const StepDev st = read_step(p);
  const double tavg = ldr(frow_ptr(a, MHMHIP_F_TAVG, st.day), bc);
  if (__builtin_amdgcn_readfirstlane(shared)) {
    auto P = [&](int r) { return ldr(a.P + (int64_t)r * a.ld, bv); };
    const int32_t i = (int32_t)(p - (const ConstStep *)a.steps) - a.sun_step0;
    const double *row = a.sun + (int64_t)(2 * i) * a.sstride;
    const SunTerms t{ldr(row, bc), ldr(row + a.sstride, bc)};
    s_lane[slot + LS_PD] = P(PR_FASP) * pet_of_sun(P(PR_HARSAM), tavg, t);
    return;
  }
  const double tmax = a.pet_case == 1 ? ldr(frow_ptr(a, MHMHIP_F_TMAX, st.day), bc) : 0.0;
  const double tmin = a.pet_case == 1 ? ldr(frow_ptr(a, MHMHIP_F_TMIN, st.day), bc) : 0.0;
  s_lane[slot + LS_PD] = pet_day<NH>(a, st, bv, bc, tavg, tmax, tmin);
}

// The daily PET, the month's interception capacity and the step's
// disaggregated meteo values, with what follows from them alone, into the
// lane's slots, as far as the step changes them.
// DY: h holds the lane's parameters for it, and f the step's forcing and sun
// terms, fetched before the soil of the step before.
struct DayParams {
  double incr, dmaxs, dnps, tth, fasp, harsam;
};
struct DayFetch {
  double ra, sq, tavg, pre;
};
__device__ __forceinline__ DayFetch day_fetch(ConstArgs *k, const FusedLane &u, const ConstStep *p) {
  const CellArgs a = read_args(rare(k));
  const uint32_t oc = opaque(u.bc);
  const double *row =
      a.sun + (int64_t)(2 * ((int32_t)(p - (const ConstStep *)a.steps) - a.sun_step0)) * a.sstride;
  return {ldr(row, oc), ldr(row + a.sstride, oc), ldr(frow_ptr(a, MHMHIP_F_TAVG, p->day), oc),
          ldr(frow_ptr(a, MHMHIP_F_PRE, p->day), oc)};
}
template <int NH, bool DY = false>
__device__ __forceinline__ void look_up(ConstArgs *k, const FusedLane &u, const ConstStep *p,
                                        int change, bool ordinary, const DayParams *h = nullptr,
                                        const DayFetch *f = nullptr) {
  if (change & SC_DAY) {
    if (DY && u.sun)
      s_lane[opaque(u.slot) + LS_PD] =
          h->fasp * pet_of_sun(h->harsam, f->tavg, SunTerms{f->ra, f->sq});
    else
      day_pet<NH>(k, u.bc, u.bv, u.slot, p, u.sun);
  }
  const CellArgs a = read_args(rare(k));
  const StepDev st = read_step(p);
  // offsets opaque here: no per-lane address of these rows is held across
  // the time loop
  const uint32_t li = opaque(u.slot), oc = opaque(u.bc), ov = opaque(u.bv);
  auto P = [&](int r) { return ldr(a.P + (int64_t)r * a.ld, ov); };
  if (change & SC_MONTH) {
    const double maxinter = P(pr_maxinter(NH) + st.month0);
    s_lane[li + LS_MAXI] = maxinter;
    s_lane[li + LS_RMAXI] = maxinter > kEps || !ordinary ? 1.0 / maxinter : 0.0;
  }
  double pet, temp, prec;
  if (DY)
    disagg_step<NH>(a, st, oc, s_lane[li + LS_PD], f->tavg, f->pre, pet, temp, prec);
  else
    disagg_at<NH>(a, st, oc, s_lane[li + LS_PD], pet, temp, prec);
  s_lane[li + LS_XPET] = pet;
  s_lane[li + LS_XPREC] = prec;
  if (ordinary) {
    const SnowMeteo m =
        DY ? snow_meteo(h->incr, h->dmaxs, h->dnps, h->tth, prec, temp)
           : snow_meteo(P(PR_INCR), P(PR_DMAXS), P(PR_DNPS), P(PR_TTH), prec, temp);
    s_lane[li + LS_XPE] = div_rcp(pet, st.evap, st.revap);
    s_lane[li + LS_XMELT] = m.melt;
    s_lane[li + LS_XCOLD] = m.cold;
  } else {
    s_lane[li + LS_XMELT] = temp;  // a general lane keeps the temperature there
  }
}

// The temperature and the degree-day factor of a launch's last step, for its
// fluxes: looked up again (the loop keeps what follows from them).
template <int NH>
__device__ __forceinline__ void last_meteo(ConstArgs *k, const FusedLane &u, const ConstStep *p,
                                           FluxRegs<NH> &x) {
  const CellArgs a = read_args(rare(k));
  const StepDev st = read_step(p);
  const uint32_t ov = opaque(u.bv);
  auto P = [&](int r) { return ldr(a.P + (int64_t)r * a.ld, ov); };
  double pet, prec;
  disagg_at<NH>(a, st, opaque(u.bc), 0.0, pet, x.temp, prec);
  x.ddf = snow_meteo(P(PR_INCR), P(PR_DMAXS), P(PR_DNPS), P(PR_TTH), prec, x.temp).ddf;
}

// Adds an output's value to the lane's sum slots, which follow one another in
// the order of the selected bits (o: the next one's slot).
__device__ __forceinline__ auto out_slots(uint64_t mask, uint32_t &o) {
  return [mask, &o](int bit, auto value) {
    if (!(mask >> bit & 1)) return;
    s_lane[o] = s_lane[o] + value();
    ++o;
  };
}
__device__ __forceinline__ void load_sums(ConstArgs *k, int64_t ld, uint32_t bv, uint32_t o) {
  for (int r = 0; r < k->out.n; ++r) s_lane[o + r] = ldr(k->out.sum + r * ld, bv);
}
__device__ __forceinline__ void store_sums(ConstArgs *k, int64_t ld, uint32_t bv, uint32_t o) {
  for (int r = 0; r < k->out.n; ++r) str(k->out.sum + r * ld, bv, s_lane[o + r]);
}

template <int NH, bool JV>
__device__ __forceinline__ Stress<NH> read_stress(uint32_t li) {
  Stress<NH> t;
#pragma unroll
  for (int h = 0; h < NH; ++h) {
    t.fr[h] = s_lane[li + LS_STRESS + h];
    t.wp[h] = s_lane[li + LS_STRESS + NH + h];
    t.slope[h] = s_lane[li + LS_STRESS + 2 * NH + h];
    t.fw[h] = JV ? s_lane[li + LS_STRESS + (JV ? 3 : 0) * NH + h] : 0.0;
  }
  return t;
}

// Sun terms of the steps step0 .. of a launch that begin a day (and of its
// first), per cell: rows 2 i and 2 i + 1 of sun hold ra and sq of step
// step0 + i.  With daily steps each lane's own were a third of a step's
// instructions, the same for every set of a cell: 256 sets of 4096 cells, 1095
// days, 23.7 -> 19.9 ms with every set's lanes reading them (they come from L2:
// a step's rows are 64 KB).
__global__ __launch_bounds__(256) void sun_kernel(CellArgs a, int32_t step0, double *sun) {
  const uint32_t c = blockIdx.x * blockDim.x + threadIdx.x, i = blockIdx.y;
  const StepDev st = a.steps[step0 + i];
  if (c >= a.n_cells || !(i == 0 || (st.change & SC_DAY))) return;
  const uint32_t bc = c * 8u;
  auto P = [&](int r) { return ldr(a.P + (int64_t)r * a.ld, bc); };
  const SunTerms t = sun_terms(ldr(frow_ptr(a, MHMHIP_F_TAVG, st.day), bc),
                               ldr(frow_ptr(a, MHMHIP_F_TMAX, st.day), bc),
                               ldr(frow_ptr(a, MHMHIP_F_TMIN, st.day), bc), P(PR_TANLAT),
                               P(PR_SINLAT), P(PR_COSLAT), st.dr, st.tand, st.sind, st.cosd);
  double *row = sun + (int64_t)(2 * i) * a.sstride;
  str(row, bc, t.ra);
  str(row + a.sstride, bc, t.sq);
}

// Whether the wave's cells have set 0's latitude, whose sun terms sun holds.
__device__ __forceinline__ bool shares_sun(const CellArgs &a, uint32_t bc, uint32_t bv) {
  if (!a.sun) return false;
  bool same = true;
  for (int r : {PR_TANLAT, PR_SINLAT, PR_COSLAT}) {
    const double *row = a.P + (int64_t)r * a.ld;
    same = same & (__double_as_longlong(ldr(row, bc)) == __double_as_longlong(ldr(row, bv)));
  }
  return __all(same);
}

// The lane's slots and its place in the ring: the lane's row offset (its lag)
// is fixed, the step's row uniform.
template <int NH, bool JV>
__device__ __forceinline__ void fused_lane(const CellArgs &a, uint32_t c, uint32_t bv,
                                           uint32_t slot, int64_t t0, const Stress<NH> &t,
                                           FusedLane &u) {
  u.bc = c * 8u;
  u.bv = bv;
  u.slot = slot;
  u.sun = shares_sun(a, u.bc, bv);
#pragma unroll
  for (int h = 0; h < NH; ++h) {
    s_lane[slot + LS_STRESS + h] = t.fr[h];
    s_lane[slot + LS_STRESS + NH + h] = t.wp[h];
    s_lane[slot + LS_STRESS + 2 * NH + h] = t.slope[h];
    if (JV) s_lane[slot + LS_STRESS + (JV ? 3 : 0) * NH + h] = t.fw[h];
  }
  u.scale = 0.0;
  u.ring = nullptr;
  u.roff = 0;
  if (a.ring) {
    u.scale = runoff_scale(a, u.bc);
    u.ring = a.ring + (int64_t)(a.lag ? a.lag[c] : 0) * a.ld + bv / 8u;
    u.roff = t0 * a.ring_rep % a.ring_len * a.ld;
  }
}

// what the first step of a launch looks up
constexpr int kAllChanged = SC_METEO | SC_DAY | SC_MONTH;

// The time loop of an ordinary cell.  Turn s of the loop finishes step s and
// starts step s + 1: the canopy and snow of step s + 1 need nothing of the
// soil and its horizon powers nothing but the soil moisture step s leaves, so
// these powers and step s's slow-interflow power run as one batch of
// independent chains, and a wave in which no lane has water to infiltrate at
// step s + 1 leaves the horizon powers out.  The first turn only starts.
template <int NH, bool JV, bool OUT, bool DY>
__device__ __forceinline__ void fused_ordinary(const CellArgs &a, FusedLane &u, CellRegs<NH> &r,
                                               const ConstStep *steps, int32_t nsteps,
                                               const DayParams &day) {
  ConstArgs *k = kernel_args();
  const uint64_t mask = OUT ? k->out.mask : 0;
  const int n_canopy = __builtin_popcountll(mask & 0x1F);  // outputs_canopy's bits
  if (OUT) load_sums(k, a.ld, u.bv, u.slot + LS_STRESS + stress_slots(NH, JV));
  const int rep = a.ring_rep;
  const int64_t wrap = a.ring_len * a.ld;
  const int32_t flux_at = a.skip_fluxes ? -2 : nsteps - 1;  // step whose fluxes are stored
  // exponents in units of 1/256 (pow_v)
  const double alpha256 = 256.0 * (1.0 + r.alpha), rc1 = JV ? 1.0 / r.c1 : 0.0;
#pragma unroll
  for (int h = 0; h < NH; ++h) r.bexp[h] = 256.0 * r.bexp[h];
  FluxRegs<NH> x;
  // step s + 1's canopy evaporation, demand left (pet - ecan), effective
  // precipitation and horizon powers, carried into the next turn
  double ecan = 0.0, demand = 0.0, peff = 0.0;
  DV<NH> pwh;
#pragma unroll
  for (int h = 0; h < NH; ++h) pwh.v[h] = 0.0;
  bool wet = false;
#pragma nounroll
  for (int32_t s = -1; s < nsteps; ++s) {
    const bool last = s == nsteps - 1;
    uint32_t o = opaque(u.slot) + LS_STRESS + stress_slots(NH, JV);  // output sum slots
    DayFetch fetched{};
    if (DY && !last) fetched = day_fetch(k, u, steps + (s + 1));
    if (s >= 0) {
      const uint32_t li = opaque(u.slot);
      ordinary_soil<NH, JV>(r, x, demand, s_lane[li + LS_XPE], ecan, peff, wet, pwh.v, rc1,
                            read_stress<NH, JV>(li));
      if (s == flux_at || OUT) {
        FluxRegs<NH> y = x;
        report_sealed<NH>(r, y);
        if (s == flux_at) store_fluxes_soil<NH>(read_args(rare(k)), u.bv, y);
        if (OUT) {
          o = opaque(u.slot) + LS_STRESS + stress_slots(NH, JV) + n_canopy;
          outputs_soil<NH>(r, y, ecan, out_slots(mask, o));
        }
      }
    }
    // waited for here whatever the step reads: no load is in flight where the
    // loop's turns meet
    if (DY) settle(fetched.ra), settle(fetched.sq), settle(fetched.tavg), settle(fetched.pre);
    if (!last) {
      const ConstStep *next = steps + (s + 1);
      const int change = next->change | (s < 0 ? kAllChanged : 0);
      if (change) {
        if (change & kAllChanged) look_up<NH, DY>(k, u, next, change, true, &day, &fetched);
        if (change & SC_INIT) {
          ConstArgs *q = rare(k);
          const uint32_t ov = opaque(u.bv);
#pragma unroll
          for (int h = 0; h < NH; ++h) {
            r.sm[h] = 0.5 * ldr(q->P + (int64_t)(pr_fc(NH) + h) * q->ld, ov);
            settle(r.sm[h]);
          }
        }
      }
      const uint32_t li = opaque(u.slot);
      x.pet = s_lane[li + LS_XPET];
      x.prec = s_lane[li + LS_XPREC];
      ordinary_canopy<NH>(r, x, s_lane[li + LS_XMELT], s_lane[li + LS_XCOLD],
                          s_lane[li + LS_MAXI], s_lane[li + LS_RMAXI]);
      if (s + 1 == flux_at) {
        last_meteo<NH>(k, u, next, x);
        store_fluxes_canopy<NH>(read_args(rare(k)), u.bv, x);
      }
      if (OUT) {
        uint32_t oc = opaque(u.slot) + LS_STRESS + stress_slots(NH, JV);
        outputs_canopy<NH>(r, x, out_slots(mask, oc));
      }
      ecan = x.ecan;
      demand = x.pet - x.ecan;
      peff = x.peff;
      wet = __any(peff != 0.0);
    }
    double pw_slow;
    if (wet && !last) {
      DV<NH + 1> py, px;
      py.v[0] = alpha256;
      px.v[0] = slow_base(r.unsat);
#pragma unroll
      for (int h = 0; h < NH; ++h) {
        py.v[h + 1] = r.bexp[h];
        px.v[h + 1] = div_rcp(r.sm[h], r.sat[h], r.rsat[h]);
      }
      px = pow_v<NH + 1>(py, px);
      pw_slow = px.v[0];
#pragma unroll
      for (int h = 0; h < NH; ++h) pwh.v[h] = px.v[h + 1];
    } else {
      pw_slow = pow_v<1>(DV<1>{{alpha256}}, DV<1>{{slow_base(r.unsat)}}).v[0];
    }
    if (s >= 0) {
      ordinary_post<NH>(r, x, pw_slow, x.rseal);
      put_ring(a, u, wrap, rep, x.total);
      if (s == flux_at) store_fluxes_post<NH>(read_args(rare(k)), u.bv, x);
      if (OUT) outputs_post<NH>(r, x, out_slots(mask, o));
    }
  }
  if (OUT) store_sums(k, a.ld, u.bv, u.slot + LS_STRESS + stress_slots(NH, JV));
}

// The time loop of any other cell, out of line and from its own loads: the
// registers of the kernel are those of the ordinary loop (in one kernel the two
// loops need 156, three waves per SIMD, and 1024x1024 ordinary cells take 1301
// instead of 1142 us per 144 steps).  A wave with such cells runs both loops:
// 512x512 cells, 24 steps 85 us without them, 180 with one in 64, 200 where all
// are.
struct FusedArgs {
  int64_t t0;
  int32_t nsteps, step0;
};

template <int NH, bool JV, bool OUT>
__device__ __attribute__((noinline)) void fused_general(ConstArgs *args, uint32_t c, uint32_t bv,
                                                        uint32_t slot) {
  ConstArgs *k = uniform(args);
  const CellArgs a = read_args(k);
  const __attribute__((address_space(4))) FusedArgs *fa =
      (const __attribute__((address_space(4))) FusedArgs *)(k + 1);
  const int32_t nsteps = fa->nsteps;
  const ConstStep *steps = (const ConstStep *)(a.steps + fa->step0);
  CellRegs<NH> r;
  load_params<NH, JV>(a, bv, r);
  load_states<NH>(a, bv, r);
  FusedLane u;
  fused_lane<NH, JV>(a, c, bv, slot, fa->t0, stress_of<NH, JV>(r, false), u);
  const int rep = a.ring_rep;
  const int64_t wrap = a.ring_len * a.ld;
#pragma nounroll
  for (int32_t s = 0; s < nsteps; ++s) {
    const ConstStep *p = steps + s;
    const int change = p->change | (s == 0 ? kAllChanged : 0);
    if (change & kAllChanged) look_up<NH>(k, u, p, change, false);
    const uint32_t li = opaque(u.slot);
    Stress<NH> t = read_stress<NH, JV>(li);
#pragma unroll
    for (int h = 0; h < NH; ++h)
      t.fw[h] = ldr(a.P + (int64_t)(pr_fc(NH) + h) * a.ld, opaque(bv));
    if (change & SC_INIT) {
#pragma unroll
      for (int h = 0; h < NH; ++h) r.sm[h] = 0.5 * t.fw[h];
    }
    FluxRegs<NH> x;
    x.pet = s_lane[li + LS_XPET];
    x.temp = s_lane[li + LS_XMELT];
    x.prec = s_lane[li + LS_XPREC];
    chain_step<NH, JV>(r, x, s_lane[li + LS_MAXI], s_lane[li + LS_RMAXI], p->evap, p->revap, t);
    put_ring(a, u, wrap, rep, x.total);
    if (s == nsteps - 1 && !a.skip_fluxes) store_fluxes<NH>(a, u.bv, x);
    if (OUT) add_outputs<NH>(k, a.ld, u.bv, r, x);
  }
  store_states<NH>(a, bv, r);
}

// ---------------------------------------------------------------------------
// Fused path: nsteps model steps per launch with parameters and states held
// in registers.  Forcing and daily PET are read/evaluated once per forcing day
// (the reference recomputes the same value every hour), maximum interception
// once per month.  Only the routing input leaves the lane each step; states
// are written at the end and the last step's fluxes as soon as each is known.
// A cell takes the ordinary or the general loop by its own parameters, states
// and weather, whatever the wave's other lanes take.
// DY: a launch of daily steps with shared sun terms.  Its lookups run every
// step, and reading their six parameters again each time (48 bytes per cell
// and step, more than its states) cost more than the fourth wave per SIMD
// brings: they stay in registers, at three waves, and the next step's forcing
// and sun terms are fetched before this step's soil.  256 sets of 4096 cells,
// 1095 days: 19.9 -> 18.1 -> 17.0 ms.
template <int NH, bool JV, bool OUT, bool DY>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(NH > 3 ? 2 : JV || OUT || DY ? 3 : 4)))
void cell_fused_kernel(CellArgs a, FusedArgs fa) {
  static_assert(sizeof(CellArgs) % alignof(FusedArgs) == 0, "FusedArgs follows CellArgs");
  mathtab_fill();  // the chain's powers read it (before any thread returns)
  const uint32_t c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= a.n_cells) return;
  const uint32_t bv = (uint32_t)(blockIdx.y * a.sstride + c) * 8u;
  // this lane's LDS slots (lane_slots doubles, laid out lane by lane)
  const uint32_t slot = threadIdx.x * (uint32_t)lane_slots(NH, JV, OUT ? a.out.n : 0);
  const ConstStep *steps = (const ConstStep *)(a.steps + fa.step0);
  CellRegs<NH> r;
  load_params<NH, JV>(a, bv, r);
  load_states<NH>(a, bv, r);
  const bool ordinary = ordinary_cell<NH, JV>(r, steps->init_sm != 0, a.odd_weather[c]);
  if (ordinary) {
    FusedLane u;
    fused_lane<NH, JV>(a, c, bv, slot, fa.t0, stress_of<NH, JV>(r, true), u);
    settle(u.scale);
    settle_all<NH>(r);
    DayParams day{};
    if (DY) {
      auto P = [&](int row) { return ldr(a.P + (int64_t)row * a.ld, bv); };
      day = {r.incr, r.dmaxs, r.dnps, r.tth, P(PR_FASP), P(PR_HARSAM)};
      settle(day.fasp), settle(day.harsam);
    }
    fused_ordinary<NH, JV, OUT, DY>(a, u, r, steps, fa.nsteps, day);
    store_states<NH>(a, bv, r);
  }
  // last, where the call finds no other value in use
  if (!ordinary) fused_general<NH, JV, OUT>(kernel_args(), c, bv, slot);
}

// ---------------------------------------------------------------------------
// One node, one step of L11_runoff_acc + add_inflow + L11_routing
// (mo_mrm_pre_routing.f90:77-143,179-214; mo_mrm_routing.f90:425-472).
__device__ __forceinline__ void route_node(const RouteArgs &r, uint32_t p, int32_t set, int64_t t,
                                           NodeMeta m) {
  const int64_t ld = (int64_t)r.n_sets * r.sstride;
  const uint32_t bv = (uint32_t)(set * r.sstride + p) * 8u;
  const int32_t y = m.packed;
  // qOUT of this node and step (L11_runoff_acc, done by the cell kernel)
  double qout = ldr(r.ring + (t % r.ring_len) * ld, bv);
  if (y & NF_INFLOW) {
    for (int32_t g = 0; g < r.n_inflow; ++g) {
      if (r.inflow_node[g] == (int32_t)p) {
        const double qi = r.inflow_q[(t - r.t_base) / r.rep * r.n_inflow + g];
        qout = r.inflow_hw[g] ? qout + qi : qi;
      }
    }
  }
  if (r.qOUT && t == r.t_hi - 1) str(r.qOUT, bv, qout);
  // qTIN(iNode,IT): upstream qTR in routing rank, then own qOUT
  const double *pub_t = r.pub + (t & 1) * ld + (int64_t)set * r.sstride;
  const int32_t *up = r.child_list + m.child;
  double s = 0.0;
  const int nc = nm_nchild(y);
  for (int c = 0; c < nc; ++c) s = s + pub_t[up[c]];
  if (y & NF_QOUT) s = s + qout;
  if (y & NF_LINK) {
    const double qtin1 = ldr(r.qTIN, bv);
    const double qtr1 = ldr(r.pub + ((t - 1) & 1) * ld, bv);
    double qtr = qtr1 + ldr(r.C1, bv) * (qtin1 - qtr1) + ldr(r.C2, bv) * (s - qtin1);
    if (y & NF_CUT) qtr = 0.0;
    str(r.pub + (t & 1) * ld, bv, qtr);
  }
  str(r.qTIN, bv, s);
  if (r.qacc && t >= r.acc_from) str(r.qacc, bv, ldr(r.qacc, bv) + s);
  if (y & NF_GAUGE) {
    for (int32_t g = 0; g < r.n_gauges; ++g)
      if (r.gauge_node[g] == (int32_t)p)
        r.gauge_out[((t - r.t_base) * r.n_sets + set) * r.n_gauges + g] = s;
  }
}

__global__ __launch_bounds__(256) void route_diag_kernel(RouteArgs r, int64_t d, uint32_t p_lo,
                                                         uint32_t p_hi) {
  const uint32_t p = p_lo + blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= p_hi) return;
  const NodeMeta m = r.meta[p];
  const int64_t t = d - (int64_t)(r.dmax - nm_depth(m.packed));
  if (t < r.t_lo || t >= r.t_hi) return;
  route_node(r, p, (int32_t)blockIdx.y, t, m);
}

// Workgroup-resident routing: one workgroup owns one (domain, parameter set)
// tree and walks that domain's own diagonals d in [d_lo, d_end) -- node at
// depth delta handles step t = d - (dmax_dom - delta) -- with a workgroup
// barrier between diagonals instead of a kernel boundary.  drain != 0 walks
// the dmax_dom diagonals that finish the last steps of a run.
__global__ __launch_bounds__(1024) void route_wg_kernel(RouteArgs r, const int64_t *dom_start,
                                                        const int32_t *dom_dmax, int64_t d_lo,
                                                        int64_t d_hi, int32_t drain) {
  const int32_t dom = blockIdx.x;
  const int32_t set = blockIdx.y;
  const uint32_t lo = (uint32_t)dom_start[dom], hi = (uint32_t)dom_start[dom + 1];
  const int32_t dm = dom_dmax[dom];
  const int64_t d_end = drain ? d_lo + dm : d_hi;
  for (int64_t d = d_lo; d < d_end; ++d) {
    for (uint32_t p = lo + threadIdx.x; p < hi; p += blockDim.x) {
      const NodeMeta m = r.meta[p];
      const int64_t t = d - (int64_t)(dm - nm_depth(m.packed));
      if (t >= r.t_lo && t < r.t_hi) route_node(r, p, set, t, m);
    }
    __syncthreads();
  }
}

// Workgroup barrier that orders LDS only: waits for this wave's LDS
// operations, not for its global stores (no other lane of the workgroup
// reads those before the kernel ends).
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Diagonals that a tiled kernel fetches ahead of use.
constexpr int kTileAhead = 4;
// LDS parity buffers, in doubles: a value per slot and for the zero slot W,
// whose +0.0 stands for a node's missing upstream slots (adding it leaves the
// running sum's value unchanged).
constexpr int kTileBuf = kTileSlots + 1;

// ---------------------------------------------------------------------------
// Tiled routing: launch L handles, for every tile of depth tau, the window
// k = L - (tau_max - tau) of B steps.  Tile-root outflow of window k is
// written to the boundary buffer (parity k & 1) in launch L and read by the
// downstream tile's proxy slot in launch L + 1.  Inside the window the
// workgroup walks its own (depth, step) diagonals: slot with lag g handles
// window step j on diagonal j + g, upstream slots (lag g - 1) produced step j
// on the diagonal before, and a two-entry LDS parity buffer keeps it
// readable while they write step j + 1.  Each slot streams its own series --
// qOUT rows of the ring (real slots, inflow gauges already applied by
// inflow_patch_kernel) or the upstream tile root's boundary series (proxies)
// -- from memory, kTileAhead diagonals ahead of use, so LDS holds only the
// parity buffers and the window length is not bounded by it.
// The host keeps a window's ring rows contiguous (ring length and window
// starts are multiples of B).
// Same per-node arithmetic as route_node (mo_mrm_routing.f90:425-472).
//
// What bounds it: where a launch has many bins due, the ring's reads (1,800
// bins x 64 steps: 236 MB in 56 us, the rate of a large copy); at the ends of
// a run's tile pipeline and on small basins a diagonal's latency: LDS write,
// barrier and read (146 cycles), eight dependent FP64 operations and whatever
// else a wave issues (a lone wave issues an FP64 instruction every 8 cycles,
// others every 4).  So a wave runs a loop with only what its slots need
// (ROOTS, RARE below), masked instead of selected, between the first and the
// last diagonal that one of its slots handles (slots are laid out by lag), and
// outside those keeps the barriers only: some 32 instructions per diagonal for
// most waves.  Against one loop for all slots, with selects and an index per
// fetch: the average launch of 1024x1024 nodes over 1440 steps 44.4 -> 38.8 us,
// 1,800 bins 63 -> 56 us, eleven bins (latency alone, 0.2 us a diagonal) 21.0 ->
// 19.4 us; 8 fetches ahead instead of 4 gave the same.  Four steps per diagonal
// (one LDS round trip for four steps) were slower where many bins are due (68
// us: a window fills and drains over four times the steps), 17.7 us for eleven.
struct TileLane {
  const double *p;      // series element of window step 0
  uint64_t stride;      // bytes between consecutive elements of the series (0: idle)
  double *bout;         // tile root: boundary series of this window, else null
  int64_t t0;           // global step of window step 0
  int32_t lag, nb, nc, c0;  // nb: steps of this window, 0: idle
  uint32_t bv;          // byte offset of (set, node) in a row
  int32_t a, set;
  int32_t gauge;        // first gauge at the node, -1: none
  int32_t orow_t, orow_g;  // LDS output rows of the tile-root series / gauge sums, -1: none
  bool real, proxy;
  double qtin1, qtr1, c1, c2;
  double qacc;          // Qmod summed over the steps (ACC)
};

// Output row of the tiled kernel's LDS staging: where its B values go.
struct TileOutRow {
  double *base;
  int32_t stride;  // elements between consecutive steps
  int32_t nb;      // steps to write
};

// The diagonals [lo, hi) of the bin's nd (a multiple of kTileAhead) that a
// wave's slots handle, lo a multiple of kTileAhead.
struct TileSpan {
  int lo, hi, nd;
};

// One sweep over the bin's diagonals; NCW bounds the upstream slots read
// together.  ROOTS: a slot of the wave hands a series on (a tile root's, a
// gauge's); RARE: a slot has more than NCW upstream slots, does not add its
// own qOUT or is cut by an inflow gauge.  STAGE: the tile-root series and
// gauge sums go to LDS rows (out, B + 1 values apart: the lanes of a wave
// write different banks) and leave after the sweep, so that the loop holds no
// global store: stores count in the same counter as the loads in flight, and
// each one would shorten the wait for a fetched value.  Every lane then writes,
// without a branch: a lane without a row its scratch entry after them.
template <int NCW, bool ROOTS, bool RARE, bool STAGE, bool ACC>
__device__ __forceinline__ void tile_sweep(const RouteArgs &r, TileLane &u, double *qtr,
                                           TileSpan w, double *out, int out_rows, int B) {
  constexpr int W = kTileSlots, A = kTileAhead;
  const int s = threadIdx.x;
  const double *up[NCW];  // the upstream slots in buffer 0
#pragma unroll
  for (int c = 0; c < NCW; ++c) up[c] = qtr + (c < u.nc ? u.c0 + c : W);
  const bool noq = u.real && !(u.a & NF_QOUT), cut = u.real && (u.a & NF_CUT);
  const int scratch = out_rows * (B + 1) + s;
  double *ot = out + (u.orow_t >= 0 ? u.orow_t * (B + 1) : scratch);
  double *og = out + (u.orow_g >= 0 ? u.orow_g * (B + 1) : scratch);
  const int tstep = u.orow_t >= 0 ? 1 : 0, gstep = u.orow_g >= 0 ? 1 : 0;
  const bool gauges = ROOTS && __any(u.gauge >= 0);
  // value for diagonal d: the slot's step d - lag, its first or last one
  // outside its diagonals
  const char *p = reinterpret_cast<const char *>(u.p);
  const uint32_t moves = u.nb > 0 ? u.nb - 1 : 0;
  double qq[A];
  auto fetch = [&](int d, double &q) {
    if ((uint32_t)(d - u.lag - 1) < moves) p += u.stride;
    q = *reinterpret_cast<const double *>(p);
  };
  double musk = u.qtr1 + u.c1 * (u.qtin1 - u.qtr1);  // qTR(IT1) + C1 (qTIN(IT1) - qTR(IT1))
  // Diagonal d reads parity buffer (d + 1) & 1, written on diagonal d - 1 by
  // the upstream slots (one level deeper, one diagonal earlier, same step),
  // and writes buffer d & 1 (wb).
  auto diagonal = [&](int d, int wb, double qo) {
    const int j = d - u.lag;
    if ((uint32_t)j >= (uint32_t)u.nb) return;
    double v[NCW];
#pragma unroll
    for (int c = 0; c < NCW; ++c) v[c] = up[c][(wb ^ 1) * kTileBuf];
    // upstream qTR in routing rank, then the node's own qOUT
    double sum = v[0];
#pragma unroll
    for (int c = 1; c < NCW; ++c) sum = sum + v[c];
    if (RARE) {
#pragma nounroll
      for (int c = NCW; c < u.nc; ++c) sum = sum + qtr[(wb ^ 1) * kTileBuf + u.c0 + c];
    }
    sum = sum + (RARE && noq ? 0.0 : qo);
    // musk = qTR(IT1) + C1 (qTIN(IT1) - qTR(IT1)), formed on the diagonal before
    double q = musk + u.c2 * (sum - u.qtin1);
    if (RARE && cut) q = 0.0;
    qtr[wb * kTileBuf + s] = u.proxy ? qo : q;
    u.qtr1 = q;
    u.qtin1 = sum;
    musk = q + u.c1 * (sum - q);
    // Qmod of step j, added in step order
    if (ACC && u.t0 + j >= r.acc_from) u.qacc = u.qacc + sum;
    if (STAGE && ROOTS) {
      *ot = q;
      ot += tstep;
      if (gauges) {
        *og = sum;
        og += gstep;
      }
    } else if (ROOTS) {
      if (u.bout) u.bout[j] = q;
      if (u.gauge >= 0)
        r.gauge_out[((u.t0 + j - r.t_base) * r.n_sets + u.set) * r.n_gauges + u.gauge] = sum;
    }
  };
#pragma unroll
  for (int i = 0; i < A; ++i) fetch(w.lo + i, qq[i]);
#pragma nounroll
  for (int d = 0; d < w.lo; ++d) lds_barrier();
  int d0 = w.lo;
#pragma nounroll
  for (; d0 < w.hi; d0 += A) {
#pragma unroll
    for (int i = 0; i < A; ++i) {
      // every lane waits for this diagonal's value here, whether it uses it
      // or not: the register is free for the next fetch
      settle(qq[i]);
      diagonal(d0 + i, i & 1, qq[i]);
      lds_barrier();
      fetch(d0 + i + A, qq[i]);
    }
  }
#pragma nounroll
  for (; d0 < w.nd; ++d0) lds_barrier();
}

// LDS: the parity buffers, then (STAGE) the bin's output rows: v.out_rows
// TileOutRow, then v.out_rows x (B + 1) values and a scratch value per slot.
// ACC: Qmod summed per node (r.qacc).
template <bool STAGE, bool ACC>
__global__ __launch_bounds__(kTileSlots) void route_tile_kernel(RouteArgs r, TileArgs g,
                                                                WindowArgs v, int32_t L,
                                                                int32_t bin0) {
  extern __shared__ double lds[];
  __shared__ int32_t n_rows;  // output rows given out
  constexpr int W = kTileSlots;
  const int bin = bin0 + blockIdx.x, set = blockIdx.y, s = threadIdx.x;
  const BinInfo bi = g.bin[bin];
  // whole bin idle in this launch: every thread leaves before any barrier
  if (L - (v.tau_max - bi.tau_hi) < 0 || L - (v.tau_max - bi.tau_lo) >= v.nwin) return;
  const SlotMeta m = g.slot[(int64_t)bin * W + s];
  TileLane u;
  const int32_t k = L - (v.tau_max - (m.b >> 16));
  u.a = m.a;
  u.set = set;
  u.real = (m.a & SF_REAL) != 0;
  u.proxy = (m.a & SF_PROXY) != 0;
  const bool act = (u.real || u.proxy) && k >= 0 && k < v.nwin;
  u.t0 = r.t_lo + (int64_t)k * v.B;
  u.nb = act ? (int)min((int64_t)v.B, r.t_hi - u.t0) : 0;
  u.lag = m.a & 0xFFF;
  u.nc = (m.a >> 12) & 0xF;
  u.c0 = m.b & 0xFFFF;
  const int64_t ld = (int64_t)r.n_sets * r.sstride;
  u.bv = u.real ? (uint32_t)(set * r.sstride + m.pos) * 8u : 0u;
  u.qtin1 = u.qtr1 = u.c1 = u.c2 = 0.0;
  // series of the slot: ring rows t0 mod R + lag + j (t0 and R are multiples
  // of B, and the ring has the tiles' height in rows past R) or the boundary
  // series of the proxy's tile root; idle slots re-read one valid element
  const int64_t bseries = ((int64_t)(k & 1) * r.n_sets + set) * g.n_bnd;
  if (act && u.real) {
    u.p = r.ring + ring_row(u.t0, u.lag, r.ring_len) * ld + (int64_t)set * r.sstride + m.pos;
    u.stride = (uint64_t)ld * 8u;
    u.qtin1 = ldr(r.qTIN, u.bv);
    if (m.a & NF_LINK) {
      u.qtr1 = ldr(r.pub + ((u.t0 - 1) & 1) * ld, u.bv);
      u.c1 = ldr(r.C1, u.bv);
      u.c2 = ldr(r.C2, u.bv);
    }
  } else if (act) {
    u.p = v.bnd + (bseries + m.bnd) * v.bstride;
    u.stride = 8;
  } else {
    u.p = v.bnd;
    u.stride = 0;
  }
  u.bout = (act && (m.a & SF_TROOT)) ? v.bnd + (bseries + m.bnd) * v.bstride : nullptr;
  // gauges: the node's first gauge only (the host copies it to the others)
  u.gauge = (act && u.real && (m.a & NF_GAUGE)) ? g.node_gauge[m.pos] : -1;
  u.orow_t = u.orow_g = -1;
  u.qacc = ACC && act && u.real ? ldr(r.qacc, u.bv) : 0.0;
  double *qtr = lds;
  TileOutRow *rows = reinterpret_cast<TileOutRow *>(lds + 2 * kTileBuf);
  double *out = reinterpret_cast<double *>(rows + v.out_rows);
  if (STAGE) {
    // a row for each tile-root series and gauge, in any order
    if (s == 0) n_rows = 0;
    lds_barrier();
    if (u.bout) {
      u.orow_t = atomicAdd(&n_rows, 1);
      rows[u.orow_t] = TileOutRow{u.bout, 1, u.nb};
    }
    if (u.gauge >= 0) {
      const int64_t gi = ((u.t0 - r.t_base) * r.n_sets + set) * r.n_gauges + u.gauge;
      u.orow_g = atomicAdd(&n_rows, 1);
      rows[u.orow_g] = TileOutRow{r.gauge_out + gi, r.n_sets * r.n_gauges, u.nb};
    }
  }
  if (s < 2) qtr[s * kTileBuf + W] = 0.0;
  lds_barrier();
  TileSpan w;
  w.nd = (bi.height + v.B - 1 + kTileAhead - 1) / kTileAhead * kTileAhead;
  int lo = u.nb > 0 ? u.lag : 0x7FFFFFFF, hi = u.nb > 0 ? u.lag + u.nb : 0;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    lo = min(lo, __shfl_xor(lo, o));
    hi = max(hi, __shfl_xor(hi, o));
  }
  w.hi = __builtin_amdgcn_readfirstlane(hi);
  w.lo = min(__builtin_amdgcn_readfirstlane(lo), w.hi) & ~(kTileAhead - 1);
  const bool rare = u.nc > 5 || (u.real && (!(u.a & NF_QOUT) || (u.a & NF_CUT)));
  if (__any(rare))
    tile_sweep<5, true, true, STAGE, ACC>(r, u, qtr, w, out, v.out_rows, v.B);
  else if (__any(u.bout != nullptr || u.gauge >= 0))
    tile_sweep<5, true, false, STAGE, ACC>(r, u, qtr, w, out, v.out_rows, v.B);
  else if (__any(u.nc > 3))
    tile_sweep<5, false, false, STAGE, ACC>(r, u, qtr, w, out, v.out_rows, v.B);
  else
    tile_sweep<3, false, false, STAGE, ACC>(r, u, qtr, w, out, v.out_rows, v.B);
  if (STAGE) {
    // the sweep's last barrier follows its last rows
    for (int idx = s; idx < n_rows * v.B; idx += W) {
      const int rr = idx / v.B, j = idx - rr * v.B;
      const TileOutRow o = rows[rr];
      if (j < o.nb) o.base[(int64_t)j * o.stride] = out[rr * (v.B + 1) + j];
    }
  }
  if (act && u.real) {
    str(r.qTIN, u.bv, u.qtin1);
    if (m.a & NF_LINK) str(r.pub + ((u.t0 + u.nb - 1) & 1) * ld, u.bv, u.qtr1);
    // qOUT of the run's last step, from its ring row
    if (r.qOUT && r.t_hi - 1 - u.t0 < u.nb) str(r.qOUT, u.bv, u.p[(r.t_hi - 1 - u.t0) * ld]);
    if (ACC) str(r.qacc, u.bv, u.qacc);
  }
}

// ---------------------------------------------------------------------------
// One routed step in one launch (mhmhip_mrm_step): every workgroup routes one
// bin of one set as soon as the tiles upstream of it are done, instead of one
// launch per tile depth.
//
// What bounds it: the chain of levels from the deepest node to the outlet.
// With a launch per tile depth that was 8.9 us per 32 levels (launch, loads of
// the slots' states, 33 barriers).  Here the loads come before the wait for
// the upstream tiles, a tile root's outflow reaches the waiting workgroup in
// 0.6 us (measured over a chain of 512), and inside a tile a wave walks its
// own levels without barriers (slots are laid out by lag: waves in turn, the
// last, which holds the lowest lags, first) at 85 ns a level: an LDS write and
// read and six to eight dependent FP64 operations.  A step of 1024x1024 nodes
// in tiles of 32 levels, 53 deep: 473 -> 183 us; of 24x30 nodes: 27 -> 11 us.
// Many bins do not change that (a ticket each, one counter per set), with eight
// coupled steps in place of a launch per depth: 600 basins of 400 nodes 749 ->
// 490 us, 2000 of 42 nodes 480 -> 255, 256 sets of 2000 nodes 1199 -> 690.
// Levels with only their own slots unmasked took 220 us.
//
// Order: a workgroup's bin is its ticket, not its block index, and tickets
// count bins from the last (deepest) to the first.  A tile's upstream tiles
// are in a bin of a lower ticket or in its own bin at a larger depth, which
// the workgroup handles before: a workgroup only waits for workgroups that
// are already running, so the waits end whatever else is on the device.  A
// ticket costs 12 ns (one counter per set).
//
// Hand-over: a tile root's value as two 64-bit words, each a 32-bit half and
// the launch's 32-bit tag, so that each word says by itself whether it is
// this launch's; relaxed device-scope accesses suffice.  The counter holds
// the launch number and the tickets taken; who takes the last ticket sets it
// for the next launch.
constexpr int kFlowHead = 16;
// polls (0.6 us each) after which a wait gives up: the kernel ends, with an error
constexpr int kFlowPolls = 1 << 22;

__device__ __forceinline__ uint64_t flow_load(const uint64_t *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void flow_store(uint64_t *p, uint64_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Workgroup's ticket (32 bits) under the launch number; without tile
// boundaries nobody waits, and the block index serves.
__device__ __forceinline__ uint64_t flow_ticket(const FlowArgs &f, uint64_t *area) {
  if (!f.tickets) return blockIdx.x;
  const uint64_t t = __hip_atomic_fetch_add(area, (uint64_t)1, __ATOMIC_RELAXED,
                                            __HIP_MEMORY_SCOPE_AGENT);
  if ((uint32_t)t == (uint32_t)f.n_bins - 1) flow_store(area, ((t >> 32) + 1) << 32);
  return t;
}

// A wait that took too long: all waits give up, and the host is told.
__device__ __forceinline__ bool flow_gives_up(const FlowArgs &f, uint64_t *area, int polls) {
  if ((polls & 1023) != 1023 || (polls < kFlowPolls && flow_load(area + 1) == 0)) return false;
  flow_store(area + 1, 1);
  __hip_atomic_store(f.fail, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  return true;
}

__device__ __forceinline__ void flow_put(uint64_t *w, uint32_t tag, double v) {
  const uint64_t b = (uint64_t)__double_as_longlong(v), t = (uint64_t)tag << 32;
  flow_store(w, t | (b & 0xFFFFFFFFu));
  flow_store(w + 1, t | (b >> 32));
}

__device__ __forceinline__ double flow_get(const FlowArgs &f, uint64_t *area, const uint64_t *w,
                                           uint32_t tag) {
  uint64_t lo, hi;
  for (int i = 0;; ++i) {
    lo = flow_load(w);
    hi = flow_load(w + 1);
    if ((uint32_t)(lo >> 32) == tag && (uint32_t)(hi >> 32) == tag) break;
    if (flow_gives_up(f, area, i)) break;
    __builtin_amdgcn_s_sleep(1);
  }
  return __longlong_as_double((long long)((hi << 32) | (lo & 0xFFFFFFFFu)));
}

// One slot's update in route_step_kernel.
struct StepLane {
  int32_t lag, nc, c0;
  bool link, cut;
  double qo, qtin, c2, musk;
  double q;       // qTR of the step (a proxy's: the upstream tile root's)
  double sum;     // qTIN of the step
};

// The levels of one wave's slots that are due, lowest lag first.  Every slot
// is computed on every level, from what its upstream slots hold by then: once
// those are final (after as many levels as the slot lies above the wave's
// lowest) so is it, and computing it again gives the same value.  That leaves
// the loop without masks or comparisons, and levels too many do no harm.
// LDS accesses of a wave happen in order.
template <int NCW, bool RARE>
__device__ __forceinline__ void step_levels(StepLane &u, double *qtr, const double *const *up,
                                            int levels) {
  const int s = threadIdx.x;
  auto level = [&]() {
    double v[NCW];
#pragma unroll
    for (int c = 0; c < NCW; ++c) v[c] = *up[c];
    // upstream qTR in routing rank, then the node's own qOUT
    double sum = v[0];
#pragma unroll
    for (int c = 1; c < NCW; ++c) sum = sum + v[c];
    if (RARE) {
#pragma nounroll
      for (int c = NCW; c < u.nc; ++c) sum = sum + qtr[u.c0 + c];
    }
    sum = sum + u.qo;
    double q = u.musk + u.c2 * (sum - u.qtin);
    if (RARE && u.cut) q = 0.0;
    qtr[s] = q;
    u.q = q;
    u.sum = sum;
    // the next level's reads stay behind this level's writes
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  };
#pragma nounroll
  for (int i = 0; i < levels; i += 2) {
    level();
    level();
  }
}

// r.pub: the qTR row in use, updated in place.  r.t_lo = 0, r.t_hi = 1, a ring
// of one step (rows by lag).
template <bool ACC>
__global__ __launch_bounds__(kTileSlots) void route_step_kernel(RouteArgs r, TileArgs g, FlowArgs f) {
  constexpr int W = kTileSlots;
  __shared__ double qtr[W + 1];
  __shared__ uint64_t ticket;
  const int s = threadIdx.x, set = blockIdx.y;
  uint64_t *area = f.area + (int64_t)set * f.astride;
  if (s == 0) {
    ticket = flow_ticket(f, area);
    qtr[W] = 0.0;
  }
  lds_barrier();
  const uint64_t t = ticket;
  const uint32_t tag = __builtin_amdgcn_readfirstlane((uint32_t)(t >> 32) + 1);
  const int bin = __builtin_amdgcn_readfirstlane(f.n_bins - 1 - (int32_t)(uint32_t)t);
  const BinInfo bi = g.bin[bin];
  const SlotMeta m = g.slot[(int64_t)bin * W + s];
  const bool real = (m.a & SF_REAL) != 0, proxy = (m.a & SF_PROXY) != 0;
  const int32_t tau = m.b >> 16;
  const int64_t ld = (int64_t)r.n_sets * r.sstride;
  const uint32_t bv = real ? (uint32_t)(set * r.sstride + m.pos) * 8u : 0u;
  uint64_t *word = area + kFlowHead + 2 * (int64_t)(m.bnd >= 0 ? m.bnd : 0);
  StepLane u{};
  u.lag = m.a & 0xFFF;
  u.nc = (m.a >> 12) & 0xF;
  u.c0 = m.b & 0xFFFF;
  u.link = (m.a & NF_LINK) != 0;
  u.cut = real && (m.a & NF_CUT);
  const bool troot = real && (m.a & SF_TROOT);
  double qo = 0.0;
  int32_t gauge = -1;
  if (real) {
    qo = ldr(r.ring + (int64_t)u.lag * ld, bv);
    u.qtin = ldr(r.qTIN, bv);
    if (m.a & NF_GAUGE) gauge = g.node_gauge[m.pos];
    if (u.link) {
      const double qtr1 = ldr(r.pub, bv), c1 = ldr(r.C1, bv);
      u.c2 = ldr(r.C2, bv);
      // qTR(IT1) + C1 (qTIN(IT1) - qTR(IT1))
      u.musk = qtr1 + c1 * (u.qtin - qtr1);
    }
    u.qo = (m.a & NF_QOUT) ? qo : 0.0;
  }
  const int wave = __builtin_amdgcn_readfirstlane(s / 64);
  // everything that needs no upstream value comes before the wait for one
  const double *up[5];  // the upstream slots; the zero slot W for missing ones
#pragma unroll
  for (int c = 0; c < 5; ++c) up[c] = qtr + (c < u.nc ? u.c0 + c : W);
  const int form = __any(u.nc > 5 || u.cut) ? 2 : __any(u.nc > 3) ? 1 : 0;
  for (int32_t k = bi.tau_hi; k >= bi.tau_lo; --k) {
    const bool due = real && tau == k;
    const uint64_t mask = __ballot(due);
    int levels = 0;  // of the wave's slots that are due
    if (mask != 0)
      levels = 1 + __builtin_amdgcn_readlane(u.lag, __builtin_ctzll(mask)) -
               __builtin_amdgcn_readlane(u.lag, 63 - __builtin_clzll(mask));
    if (proxy && tau == k) qtr[s] = flow_get(f, area, word, tag);
#pragma nounroll
    for (int turn = W / 64 - 1; turn >= 0; --turn) {
      if (turn == wave && due) {
        if (form == 2) step_levels<5, true>(u, qtr, up, levels);
        else if (form == 1) step_levels<5, false>(u, qtr, up, levels);
        else step_levels<3, false>(u, qtr, up, levels);
        if (troot) flow_put(word, tag, u.q);
      }
      if (turn > 0) lds_barrier();
    }
  }
  if (real) {
    str(r.qTIN, bv, u.sum);
    if (u.link) str(r.pub, bv, u.q);
    if (r.qOUT) str(r.qOUT, bv, qo);
    // gauges: the node's first gauge only (the host copies it to the others)
    if (gauge >= 0) r.gauge_out[(int64_t)set * r.n_gauges + gauge] = u.sum;
    if (ACC) str(r.qacc, bv, ldr(r.qacc, bv) + u.sum);
  }
}

// ---------------------------------------------------------------------------
// Routing of the steps [t_lo, t_hi) of the ring in one launch: every workgroup
// routes one bin of one set, all steps, as soon as the tiles upstream of it
// hand their steps on.  The workgroup walks its own (depth, step) diagonals:
// the slot with lag g handles step j on diagonal j + g, its upstream slots
// (lag g - 1) produced step j on the diagonal before, and a two-entry LDS
// parity buffer keeps it readable while they write step j + 1.  The tiles of a
// bin that lie s levels of tile depth below its deepest ones run s (height +
// kStreamSkew) diagonals late: by then the tiles they may wait for in the same
// bin have handed the step on.
// Same per-node arithmetic as route_node (mo_mrm_routing.f90:425-472).
//
// Waves by role.  0..3, a slot per lane: each real slot streams its qOUT from
// the ring (inflow gauges already applied by inflow_patch_kernel), kTileAhead
// diagonals ahead of use.  Then f.proxy_waves: each lane takes a proxy's steps
// from the upstream tile.  Then f.out_waves: each lane hands a tile root's
// steps on or stores a gauge's.  Loads, waits for other workgroups and stores
// would hold up the slots' diagonals in one wave (stores and loads share a
// counter, so a wait for a fetched value would wait for later stores).
//
// Hand-over: a root's step as two words in the ring, in the entries of that
// step of the root itself and of its first upstream node, which nobody reads
// any more: both hold 32 bits of the value under a tag.  The tags are
// signalling NaNs, which no arithmetic yields, so that an entry's qOUT is
// never taken for a word; an entry gets its next qOUT from a cell kernel after
// this launch.  Tickets as in route_step_kernel.
//
// What bounds it: where the bins fill the chip, the ring's reads; else the
// chain of diagonals, steps + levels of them (0.2 us each: LDS write, barrier
// and read, 146 cycles, eight dependent FP64 operations, and whatever else a
// wave issues).  Against the windowed launches: 150x220 nodes, 960 routing
// steps through a ring of 192 rows 1504 -> 936 us; 215x301 nodes, 720 steps
// 979 -> 579 us; 64x64 nodes, a year 2636 -> 2034 us; with the chip full no
// gain (one_launch_pays in api.hip).
constexpr int kStreamSkew = 8;
constexpr uint32_t kTagLo = 0x7FF5A5A1u, kTagHi = 0x7FF5A5A2u;

struct StreamLane {
  const char *p;    // series element of step 0
  uint64_t stride;  // bytes between consecutive elements
  int32_t lag, n;   // n: steps, 0: idle
  int32_t nc, c0;
  bool noq, cut;
  double qtin1, qtr1, c1, c2;
  double qlast;     // qOUT of the last step
  double qacc;      // Qmod summed over the steps (ACC)
};

// What a proxy or output lane does (LDS lists).
struct StreamItem {
  int32_t slot, lag;
  int32_t a, b;  // nodes whose ring entries hold the words; output: b = -1: gauge a
};

// A wave's slots over the nd diagonals (a multiple of kTileAhead); NCW bounds
// the upstream slots read together.  RARE: a slot has more than NCW upstream
// slots, does not add its own qOUT or is cut by an inflow gauge.  Slots outside
// their steps are masked; before the first and after the last diagonal that
// one of its slots handles [lo, hi) the wave only keeps the barriers.
template <int NCW, bool RARE, bool ACC>
__device__ __forceinline__ void stream_slots(const RouteArgs &r, StreamLane &u, double *qtr,
                                             double *gsum, bool gauges, int nd) {
  constexpr int W = kTileSlots, A = kTileAhead;
  const int s = threadIdx.x;
  int lo = u.n > 0 ? u.lag : 0x7FFFFFFF, hi = u.n > 0 ? u.lag + u.n : 0;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    lo = min(lo, __shfl_xor(lo, o));
    hi = max(hi, __shfl_xor(hi, o));
  }
  hi = __builtin_amdgcn_readfirstlane(hi);
  lo = min(__builtin_amdgcn_readfirstlane(lo), hi) & ~(A - 1);
  const double *up[NCW];  // the upstream slots in buffer 0
#pragma unroll
  for (int c = 0; c < NCW; ++c) up[c] = qtr + (c < u.nc ? u.c0 + c : W);
  // value for diagonal d: the slot's step d - lag, its first or last one
  // outside its diagonals
  const char *p = u.p;
  const uint32_t moves = u.n > 0 ? u.n - 1 : 0;
  double qq[A];
  auto fetch = [&](int d, double &q) {
    if ((uint32_t)(d - u.lag - 1) < moves) p += u.stride;
    q = *reinterpret_cast<const double *>(p);
  };
  double musk = u.qtr1 + u.c1 * (u.qtin1 - u.qtr1);  // qTR(IT1) + C1 (qTIN(IT1) - qTR(IT1))
  // Diagonal d reads parity buffer (d + 1) & 1, written on diagonal d - 1, and
  // writes buffer d & 1 (wb).
  auto diagonal = [&](int d, int wb, double qo) {
    const int j = d - u.lag;
    if ((uint32_t)j >= (uint32_t)u.n) return;
    double v[NCW];
#pragma unroll
    for (int c = 0; c < NCW; ++c) v[c] = up[c][(wb ^ 1) * kTileBuf];
    // upstream qTR in routing rank, then the node's own qOUT
    double sum = v[0];
#pragma unroll
    for (int c = 1; c < NCW; ++c) sum = sum + v[c];
    if (RARE) {
#pragma nounroll
      for (int c = NCW; c < u.nc; ++c) sum = sum + qtr[(wb ^ 1) * kTileBuf + u.c0 + c];
    }
    sum = sum + (RARE && u.noq ? 0.0 : qo);
    // musk = qTR(IT1) + C1 (qTIN(IT1) - qTR(IT1)), formed on the diagonal before
    double q = musk + u.c2 * (sum - u.qtin1);
    if (RARE && u.cut) q = 0.0;
    qtr[wb * kTileBuf + s] = q;
    if (gauges) gsum[wb * W + s] = sum;
    u.qtr1 = q;
    u.qtin1 = sum;
    u.qlast = qo;
    musk = q + u.c1 * (sum - q);
    // Qmod of step j, added in step order
    if (ACC && r.t_lo + j >= r.acc_from) u.qacc = u.qacc + sum;
  };
#pragma unroll
  for (int i = 0; i < A; ++i) fetch(lo + i, qq[i]);
#pragma nounroll
  for (int d = 0; d < lo; ++d) lds_barrier();
  int d0 = lo;
#pragma nounroll
  for (; d0 < hi; d0 += A) {
#pragma unroll
    for (int i = 0; i < A; ++i) {
      // every lane waits for this diagonal's value here, whether it uses it
      // or not: the register is free for the next fetch
      settle(qq[i]);
      diagonal(d0 + i, i & 1, qq[i]);
      lds_barrier();
      fetch(d0 + i + A, qq[i]);
    }
  }
#pragma nounroll
  for (; d0 < nd; ++d0) lds_barrier();
}

// A proxy wave: each lane brings an upstream tile root's steps into its
// proxy's slot, kTileAhead diagonals ahead of use, and waits for a step that
// was not there yet.
__device__ __forceinline__ void stream_proxies(const RouteArgs &r, const FlowArgs &f, uint64_t *area,
                                               const StreamItem &m, bool have, int n,
                                               const char *pa, const char *pb, uint64_t stride,
                                               double *qtr, int nd) {
  constexpr int A = kTileAhead;
  const char *p = pa, *p2 = pb;
  const uint32_t moves = have ? n - 1 : 0;
  uint64_t wa[A], wb[A];
  bool dead = false;  // a wait gave up
  auto fetch = [&](int d, uint64_t &a, uint64_t &b) {
    if ((uint32_t)(d - m.lag - 1) < moves) {
      p += stride;
      p2 += stride;
    }
    a = flow_load(reinterpret_cast<const uint64_t *>(p));
    b = flow_load(reinterpret_cast<const uint64_t *>(p2));
  };
  auto ready = [](uint64_t a, uint64_t b) {
    return (uint32_t)(a >> 32) == kTagLo && (uint32_t)(b >> 32) == kTagHi;
  };
#pragma unroll
  for (int i = 0; i < A; ++i) fetch(i, wa[i], wb[i]);
#pragma nounroll
  for (int d0 = 0; d0 < nd; d0 += A) {
#pragma unroll
    for (int i = 0; i < A; ++i) {
      const int j = d0 + i - m.lag;
      if (have && (uint32_t)j < (uint32_t)n) {
        uint64_t a = wa[i], b = wb[i];
        if (!ready(a, b) && !dead) {
          const uint64_t *qa = reinterpret_cast<const uint64_t *>(pa + (uint64_t)j * stride);
          const uint64_t *qb = reinterpret_cast<const uint64_t *>(pb + (uint64_t)j * stride);
          for (int k = 0;; ++k) {
            a = flow_load(qa);
            b = flow_load(qb);
            if (ready(a, b)) break;
            if (flow_gives_up(f, area, k)) {
              dead = true;
              break;
            }
            __builtin_amdgcn_s_sleep(1);
          }
        }
        qtr[(i & 1) * kTileBuf + m.slot] =
            __longlong_as_double((long long)((b << 32) | (a & 0xFFFFFFFFu)));
      }
      lds_barrier();
      fetch(d0 + i + A, wa[i], wb[i]);
    }
  }
}

// An output wave: on the diagonal after a slot's, each lane hands its tile
// root's step on or stores its gauge's.
__device__ __forceinline__ void stream_outputs(const StreamItem &m, bool have, int n, char *pa,
                                               char *pb, uint64_t stride, const double *qtr,
                                               const double *gsum, int nd) {
  const bool gauge = m.b < 0;
  auto put = [&](int d, int rb) {  // diagonal d's values, in parity buffer rb
    if (!have || (uint32_t)(d - m.lag) >= (uint32_t)n) return;
    if (gauge) {
      *reinterpret_cast<double *>(pa) = gsum[rb * kTileSlots + m.slot];
    } else {
      const uint64_t v = (uint64_t)__double_as_longlong(qtr[rb * kTileBuf + m.slot]);
      flow_store(reinterpret_cast<uint64_t *>(pa), (uint64_t)kTagLo << 32 | (v & 0xFFFFFFFFu));
      flow_store(reinterpret_cast<uint64_t *>(pb), (uint64_t)kTagHi << 32 | (v >> 32));
      pb += stride;
    }
    pa += stride;
  };
  lds_barrier();  // diagonal 0
#pragma nounroll
  for (int d = 1; d < nd; d += 2) {
    put(d - 1, 0);
    lds_barrier();
    put(d, 1);
    if (d + 1 < nd) lds_barrier();
  }
}

// ACC: Qmod summed per node (r.qacc).  last: t_hi ends the run (r.qOUT).
template <bool ACC>
__global__ __launch_bounds__(1024) void route_stream_kernel(RouteArgs r, TileArgs g, FlowArgs f) {
  constexpr int W = kTileSlots;
  __shared__ double qtr[2 * kTileBuf];
  __shared__ double gsum[2 * W];
  __shared__ StreamItem proxy[W], output[2 * W];
  __shared__ uint64_t ticket;
  __shared__ int32_t n_proxy, n_output;
  const int s = threadIdx.x, set = blockIdx.y;
  uint64_t *area = f.area + (int64_t)set * f.astride;
  if (s == 0) {
    ticket = flow_ticket(f, area);
    n_proxy = n_output = 0;
    qtr[W] = qtr[kTileBuf + W] = 0.0;
  }
  lds_barrier();
  const int bin = __builtin_amdgcn_readfirstlane(f.n_bins - 1 - (int32_t)(uint32_t)ticket);
  const BinInfo bi = g.bin[bin];
  const int n = (int)(r.t_hi - r.t_lo);
  const int skew = bi.height + kStreamSkew;
  const int64_t ld = (int64_t)r.n_sets * r.sstride;
  const int64_t row0 = ring_row(r.t_lo, 0, r.ring_len);
  char *ring = reinterpret_cast<char *>(const_cast<double *>(r.ring) + row0 * ld +
                                        (int64_t)set * r.sstride);
  const int wave = __builtin_amdgcn_readfirstlane(s / 64);
  StreamLane u{};
  uint32_t bv = 0;
  bool real = false, link = false, gauges = false;
  if (wave < W / 64) {
    const SlotMeta m = g.slot[(int64_t)bin * W + s];
    const int32_t spare = g.spare[(int64_t)bin * W + s];
    real = (m.a & SF_REAL) != 0;
    link = (m.a & NF_LINK) != 0;
    const int32_t lag = m.a & 0xFFF;
    u.lag = lag + (bi.tau_hi - (m.b >> 16)) * skew;
    u.nc = (m.a >> 12) & 0xF;
    u.c0 = m.b & 0xFFFF;
    u.noq = real && !(m.a & NF_QOUT);
    u.cut = real && (m.a & NF_CUT);
    u.p = ring;
    if (m.a & SF_PROXY) proxy[atomicAdd(&n_proxy, 1)] = StreamItem{s, u.lag, m.pos, spare};
    if (real) {
      u.n = n;
      u.p = ring + ((int64_t)lag * ld + m.pos) * 8;
      u.stride = (uint64_t)ld * 8u;
      bv = (uint32_t)(set * r.sstride + m.pos) * 8u;
      u.qtin1 = ldr(r.qTIN, bv);
      if (link) {
        u.qtr1 = ldr(r.pub + ((r.t_lo - 1) & 1) * ld, bv);
        u.c1 = ldr(r.C1, bv);
        u.c2 = ldr(r.C2, bv);
      }
      if (ACC) u.qacc = ldr(r.qacc, bv);
      if (m.a & SF_TROOT) output[atomicAdd(&n_output, 1)] = StreamItem{s, u.lag, m.pos, spare};
      // gauges: the node's first gauge only (the host copies it to the others)
      if (m.a & NF_GAUGE)
        output[atomicAdd(&n_output, 1)] = StreamItem{s, u.lag, g.node_gauge[m.pos], -1};
    }
    gauges = __any(real && (m.a & NF_GAUGE));
  }
  lds_barrier();
  const int nd = (n + bi.height - 1 + (bi.tau_hi - bi.tau_lo) * skew + kTileAhead - 1) /
                 kTileAhead * kTileAhead;
  if (wave < W / 64) {
    if (__any(u.nc > 5 || u.noq || u.cut)) stream_slots<5, true, ACC>(r, u, qtr, gsum, gauges, nd);
    else if (__any(u.nc > 3)) stream_slots<5, false, ACC>(r, u, qtr, gsum, gauges, nd);
    else stream_slots<3, false, ACC>(r, u, qtr, gsum, gauges, nd);
    if (real) {
      str(r.qTIN, bv, u.qtin1);
      if (link) str(r.pub + ((r.t_hi - 1) & 1) * ld, bv, u.qtr1);
      if (f.last && r.qOUT) str(r.qOUT, bv, u.qlast);
      if (ACC) str(r.qacc, bv, u.qacc);
    }
  } else if (wave < W / 64 + f.proxy_waves) {
    const int i = s - W;
    const bool have = i < n_proxy;
    const StreamItem m = have ? proxy[i] : StreamItem{0, 0, 0, 0};
    if (__any(have))
      stream_proxies(r, f, area, m, have, n, ring + ((int64_t)f.lag[m.a] * ld + m.a) * 8,
                     ring + ((int64_t)f.lag[m.b] * ld + m.b) * 8, have ? (uint64_t)ld * 8u : 0,
                     qtr, nd);
    else
      for (int d = 0; d < nd; ++d) lds_barrier();
  } else {
    const int i = s - W - 64 * f.proxy_waves;
    const bool have = i < n_output;
    const StreamItem m = have ? output[i] : StreamItem{0, 0, 0, 0};
    const bool gauge = m.b < 0;
    char *pa = ring + ((int64_t)f.lag[gauge ? 0 : m.a] * ld + m.a) * 8;
    char *pb = ring + ((int64_t)f.lag[gauge ? 0 : m.b] * ld + m.b) * 8;
    uint64_t stride = (uint64_t)ld * 8u;
    if (gauge) {
      pa = reinterpret_cast<char *>(
          r.gauge_out + ((r.t_lo - r.t_base) * r.n_sets + set) * r.n_gauges + m.a);
      stride = (uint64_t)r.n_sets * r.n_gauges * 8u;
    }
    if (__any(have))
      stream_outputs(m, have, n, pa, pb, stride, qtr, gsum, nd);
    else
      for (int d = 0; d < nd; ++d) lds_barrier();
  }
}

// Forcing on the meteo grid (L2) to the L1 cells of one domain, as
// meteo_forcings_wrapper maps it (mo_meteo_helper.f90:119-143).  One thread
// per (L1 cell, day).  Aggregation (L1 coarser, mo_meteo_spatial_tools.f90:
// 94-200): the valid L2 cells of the cell's block added column by column (j
// outer, i inner, the reference's order, from 0.0) and divided by their
// count (0/0 gives NaN, as there).  Disaggregation (313-377) and equal grids
// (mo_meteo_helper.f90:129-131): the source L2 cell, or nodata (-9999).
__global__ __launch_bounds__(256) void meteo_l2_kernel(const double *data2, const uint8_t *mask2,
                                                       int32_t nr2, int64_t n2,
                                                       const MeteoL2Cell *cells, int64_t ncells,
                                                       int32_t ndays, double *F,
                                                       int64_t day_stride, int32_t aggregate) {
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= ncells) return;
  const MeteoL2Cell m = cells[c];
  for (int32_t t = blockIdx.y; t < ndays; t += gridDim.y) {
    const double *d2 = data2 + (int64_t)t * n2;
    double v;
    if (aggregate) {
      double sum = 0.0;
      for (int32_t j = m.c0; j <= m.c1; ++j)
        for (int32_t i = m.r0; i <= m.r1; ++i) {
          const int64_t k = (int64_t)j * nr2 + i;
          if (mask2[k]) sum = sum + d2[k];
        }
      v = sum / (double)m.n;
    } else {
      v = m.src >= 0 ? d2[m.src] : -9999.0;
    }
    F[(int64_t)t * day_stride + m.dst] = v;
  }
}

hipError_t launch_meteo_l2(const double *data2, const uint8_t *mask2, int32_t nr2, int64_t n2,
                           const MeteoL2Cell *cells, int64_t ncells, int32_t ndays, double *F,
                           int64_t day_stride, bool aggregate, hipStream_t s) {
  if (ncells <= 0 || ndays <= 0) return hipSuccess;
  const dim3 grid((unsigned)((ncells + 255) / 256), (unsigned)(ndays < 65535 ? ndays : 65535));
  hipLaunchKernelGGL(meteo_l2_kernel, grid, dim3(256), 0, s, data2, mask2, nr2, n2, cells, ncells,
                     ndays, F, day_stride, aggregate ? 1 : 0);
  return hipGetLastError();
}

// reg_rout (mo_mrm_mpr.f90:61-119) over the links [l0, l1), into their source
// nodes' C1, C2; TS = real(timestep) [h].  in: length [m], slope, sealed flood
// plain fraction and the domain's largest slope of every link, rows n apart;
// in and pos (device index of a link's source node) are pinned host memory,
// read once per call at the link's rate: 20k links in 25 us, without the host
// waiting, against 136 us for the coefficients evaluated on the host between
// two downloads and two uploads.
__global__ __launch_bounds__(256) void reg_rout_kernel(const double *in, int64_t n,
                                                       const int32_t *pos, int64_t l0, int64_t l1,
                                                       RegRout g, double *C1, double *C2) {
  const int64_t i = l0 + (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= l1) return;
  const double length = in[i], slope = in[n + i], sealed = in[2 * n + i], ss_max = in[3 * n + i];
  const double TS = g.ts;
  double K = g.p[0] + g.p[1] * (length * 0.001) + g.p[2] * slope + g.p[3] * sealed;
  double xi = g.p[4] * (1.0 + slope / ss_max);
  if (xi > 0.5) xi = 0.5;
  if (xi < 0.005) xi = 0.005;
  if (K > 0.5 * TS / xi) K = 0.5 * TS / xi;
  if (K < 0.5 * TS / (1.0 - xi)) K = 0.5 * TS / (1.0 - xi);
  const double c1 = TS / (K * (1.0 - xi) + 0.5 * TS);
  const int64_t q = pos[i];
  C1[q] = c1;
  C2[q] = 1.0 - c1 * K / TS;
}

hipError_t launch_reg_rout(const double *in, int64_t n, const int32_t *pos, int64_t l0, int64_t l1,
                           const RegRout &g, double *C1, double *C2, hipStream_t s) {
  if (l0 < 0 || l1 > n || l1 <= l0) return hipErrorInvalidValue;
  hipLaunchKernelGGL(reg_rout_kernel, dim3((unsigned)((l1 - l0 + 255) / 256)), dim3(256), 0, s, in,
                     n, pos, l0, l1, g, C1, C2);
  return hipGetLastError();
}

// State rows at one value each, of every set; the padding past the cells is 0.
// 24 sets of 20k cells with their zeroed fluxes: 12.5 ms -> 0.1 ms against a
// row at a time through the host (bound by writing 0.1 GB).
__global__ __launch_bounds__(256) void state_rows_kernel(double *S, StateValues v, int64_t n_cells,
                                                         int64_t sstride, int64_t ld) {
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= sstride) return;
  S[(int64_t)blockIdx.z * ld + (int64_t)blockIdx.y * sstride + c] =
      c < n_cells ? v.row[blockIdx.z] : 0.0;
}

hipError_t launch_state_rows(double *S, const StateValues &v, int32_t n_rows, int64_t n_cells,
                             int64_t sstride, int64_t ld, int32_t n_sets, hipStream_t s) {
  if (n_rows < 1 || n_rows > (int32_t)(sizeof(v.row) / sizeof(v.row[0])) || n_sets < 1 ||
      n_cells < 1 || n_cells > sstride || ld != sstride * n_sets)
    return hipErrorInvalidValue;
  for (int32_t s0 = 0; s0 < n_sets; s0 += 32768) {
    const dim3 grid((unsigned)((sstride + 255) / 256), (unsigned)(n_sets - s0 < 32768 ? n_sets - s0 : 32768),
                    (unsigned)n_rows);
    hipLaunchKernelGGL(state_rows_kernel, grid, dim3(256), 0, s, S + (int64_t)s0 * sstride, v,
                       n_cells, sstride, ld);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

// A row for the host: out[k] = row[pos[k]] for k in [lo, hi).  pos and out are
// pinned host memory, so the values cross the link once and in the host's
// order: 1M cells in 207 us, bound by the link (the plain copy 150 us, which a
// host loop then had to put in order, every read a cache miss).  The download
// of a row of 1M cells as a whole: 1.8 -> 0.40 ms, of 65k cells 97 -> 38 us.
__global__ __launch_bounds__(256) void row_gather_kernel(const double *row, const int32_t *pos,
                                                         double *out, int64_t lo, int64_t hi) {
  const int64_t k = lo + (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < hi) out[k] = row[pos[k]];
}

hipError_t launch_row_gather(const double *row, const int32_t *pos, double *out, int64_t lo,
                             int64_t hi, hipStream_t s) {
  if (lo < 0 || hi <= lo) return hipErrorInvalidValue;
  hipLaunchKernelGGL(row_gather_kernel, dim3((unsigned)((hi - lo + 255) / 256)), dim3(256), 0, s,
                     row, pos, out, lo, hi);
  return hipGetLastError();
}

// Marks the cells whose n_rows rows of precipitation (pre) hold a value outside
// [0, kBig) with bit, those whose rows of temperature (temp) hold one outside
// (-kBig, kBig) with 2 bit (CellArgs::odd_weather); either may be null.  For the
// other cells the degree-day factor is not below zero at any step.
__global__ __launch_bounds__(256) void forcing_scan_kernel(const double *pre, const double *temp,
                                                           int64_t stride, int32_t n_rows,
                                                           int64_t n_cells, int32_t bit,
                                                           uint8_t *odd) {
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n_cells) return;
  bool odd_pre = false, odd_temp = false;
  for (int32_t t = blockIdx.y; t < n_rows; t += gridDim.y) {
    if (pre) {
      const double v = pre[(int64_t)t * stride + c];
      odd_pre = odd_pre | !(v >= 0.0) | !(v < kBig);
    }
    if (temp) odd_temp = odd_temp | !(fabs(temp[(int64_t)t * stride + c]) < kBig);
  }
  const uint32_t bits = (odd_pre ? bit : 0) | (odd_temp ? 2 * bit : 0);
  if (bits) atomicOr(reinterpret_cast<uint32_t *>(odd) + c / 4, bits << 8 * (c % 4));
}

// Takes bits out of the marks (n: a multiple of 4).
__global__ __launch_bounds__(256) void odd_clear_kernel(int64_t n, int32_t bits, uint8_t *odd) {
  const int64_t w = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (w < n / 4) atomicAnd(reinterpret_cast<uint32_t *>(odd) + w, ~((uint32_t)bits * 0x01010101u));
}

hipError_t launch_forcing_scan(const double *pre, const double *temp, int64_t stride,
                               int32_t n_rows, int64_t n_cells, int32_t bit, uint8_t *odd,
                               hipStream_t s) {
  if (n_rows < 1 || n_cells < 1 || (!pre && !temp) || !odd) return hipErrorInvalidValue;
  const dim3 grid((unsigned)((n_cells + 255) / 256), (unsigned)(n_rows < 64 ? n_rows : 64));
  hipLaunchKernelGGL(forcing_scan_kernel, grid, dim3(256), 0, s, pre, temp, stride, n_rows,
                     n_cells, bit, odd);
  return hipGetLastError();
}

hipError_t launch_odd_clear(int64_t n, int32_t bits, uint8_t *odd, hipStream_t s) {
  if (n < 4 || n % 4 != 0 || !odd) return hipErrorInvalidValue;
  hipLaunchKernelGGL(odd_clear_kernel, dim3((unsigned)((n / 4 + 255) / 256)), dim3(256), 0, s, n,
                     bits, odd);
  return hipGetLastError();
}

// Streamed forcing: a chunk of days of the variables in var_mask (bit v:
// forcing variable v), uploaded in reference cell order (raw[k][j][cell],
// k counting the variables given), scattered into the forcing columns in
// device order: F[v][col(j)][pos[cell]], col(j) = (day0 + j) mod n_cols.  One
// thread per (cell, day of the chunk): the reads are coalesced, the writes
// follow the tile layout (cells of a tile close together).
__global__ __launch_bounds__(256) void forcing_gather_kernel(const double *raw, FRowMap m,
                                                             int32_t ndays, int64_t n_cells,
                                                             const int32_t *pos, double *F,
                                                             int32_t n_cols, int32_t day0,
                                                             int64_t sstride) {
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int32_t j = blockIdx.y;
  if (c >= n_cells || j >= ndays) return;
  const int64_t p = pos[c];
  const int64_t col = (int64_t)((day0 + j) % n_cols);
  for (int32_t k = 0; k < m.n; ++k)
    F[((int64_t)m.row[k] * n_cols + col) * sstride + p] = raw[((int64_t)k * ndays + j) * n_cells + c];
}

hipError_t launch_forcing_gather(const double *raw, const FRowMap &m, int32_t ndays,
                                 int64_t n_cells, const int32_t *pos, double *F, int32_t n_cols,
                                 int32_t day0, int64_t sstride, hipStream_t s) {
  if (m.n < 1 || m.n > MHMHIP_F_COUNT || ndays < 1 || ndays > 65535 || n_cells < 1 ||
      n_cols < 1 || day0 < 0)
    return hipErrorInvalidValue;
  for (int32_t k = 0; k < m.n; ++k)
    if (m.row[k] < 0 || m.row[k] >= MHMHIP_F_COUNT) return hipErrorInvalidValue;
  const dim3 grid((unsigned)((n_cells + 255) / 256), (unsigned)ndays);
  hipLaunchKernelGGL(forcing_gather_kernel, grid, dim3(256), 0, s, raw, m, ndays, n_cells, pos, F,
                     n_cols, day0, sstride);
  return hipGetLastError();
}

// L11_runoff_acc with map_flag on a routing grid coarser than the L1 grid
// (mo_mrm_pre_routing.f90:110-126): qAcc(node) = 0, plus qAll(k) * area(k)
// for the node's L1 cells k in increasing reference order, then
// * 1000 / TST.  The cells of device node p are device cells
// [cstart[p], cstart[p + 1]) (grouped by node, reference order inside).  tot
// holds tot_rows rows of L1_total_runoff (row (t0 + j) mod tot_rows for step
// t0 + j); the step's qOUT goes to its rep ring rows at the node's lag, as the
// cell kernels write them on an L1 = L11 grid.  One thread per (node, set),
// blockIdx.z the step.
__global__ __launch_bounds__(256) void runoff_agg_kernel(
    const double *tot, int64_t tot_rows, const int32_t *cstart, const double *area,
    int64_t n_nodes, int64_t sstride, int64_t ld, double *ring, const uint8_t *lag,
    int64_t ring_len, int32_t rep, int64_t t0, double tst, double rtst) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n_nodes) return;
  const int64_t set0 = (int64_t)blockIdx.y * sstride;
  const int64_t t = t0 + blockIdx.z;
  const double *src = tot + (t % tot_rows) * ld + set0;
  double sum = 0.0;
  for (int32_t c = cstart[p]; c < cstart[p + 1]; ++c) sum = sum + src[c] * area[c];
  const double q = div_rcp(sum * 1000.0, tst, rtst);
  const int32_t g = lag ? lag[p] : 0;
  for (int32_t i = 0; i < rep; ++i) ring[ring_row(t * rep + i, g, ring_len) * ld + set0 + p] = q;
}

hipError_t launch_runoff_agg(const double *tot, int64_t tot_rows, const int32_t *cstart,
                             const double *area, int64_t n_nodes, int64_t sstride, int64_t ld,
                             int n_sets, double *ring, const uint8_t *lag, int64_t ring_len,
                             int32_t rep, int64_t t0, int32_t nsteps, double tst, hipStream_t s) {
  if (n_nodes < 1 || n_sets < 1 || nsteps < 1 || nsteps > 65535 || tot_rows < 1 || ring_len < 1 ||
      rep < 1 || !cstart || !tot || !ring || !(tst > 0.0))
    return hipErrorInvalidValue;
  const dim3 grid((unsigned)((n_nodes + 255) / 256), (unsigned)n_sets, (unsigned)nsteps);
  hipLaunchKernelGGL(runoff_agg_kernel, grid, dim3(256), 0, s, tot, tot_rows, cstart, area,
                     n_nodes, sstride, ld, ring, lag, ring_len, rep, t0, tst, 1.0 / tst);
  return hipGetLastError();
}

// Routing steps longer than the model step (processCase(8) = 2, 3 with
// tsRoutFactor >= 1, mo_mhm_interface_run.f90:494-512): every model step adds
// its L1_total_runoff to RunToRout [mm] (acc = acc + q from 0 after each
// routing); on a routing step L11_runoff_acc converts the sum with the routing
// step TS_rout (mo_mrm_pre_routing.f90:110-126: qAcc = 0 + RunToRout * area,
// then * 1000 / (HourSecs * TS_rout)) into the step's ring row (lag, as the
// cell kernels write it) and RunToRout starts again from 0.  One thread per
// (cell, set).
__global__ __launch_bounds__(256) void runoff_sum_kernel(const double *total, double *acc,
                                                         double *ring, const double *area,
                                                         const uint8_t *lag, int64_t n_cells,
                                                         int64_t sstride, int64_t ld, double tst,
                                                         int32_t route) {
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n_cells) return;
  const int64_t i = (int64_t)blockIdx.y * sstride + c;
  const double sum = acc[i] + total[i];
  if (route) {
    ring[(int64_t)lag[c] * ld + i] = ((0.0 + sum * area[c]) * 1000.0) / tst;
    acc[i] = 0.0;
  } else {
    acc[i] = sum;
  }
}

hipError_t launch_runoff_sum(const double *total, double *acc, double *ring, const double *area,
                             const uint8_t *lag, int64_t n_cells, int64_t sstride, int64_t ld,
                             int n_sets, double tst, bool route, hipStream_t s) {
  if (n_cells < 1 || n_sets < 1 || !lag) return hipErrorInvalidValue;
  const dim3 grid((unsigned)((n_cells + 255) / 256), (unsigned)n_sets);
  hipLaunchKernelGGL(runoff_sum_kernel, grid, dim3(256), 0, s, total, acc, ring, area, lag,
                     n_cells, sstride, ld, tst, route ? 1 : 0);
  return hipGetLastError();
}

// Inflow gauges for the tiled routing (add_inflow, mo_mrm_pre_routing.f90:
// 179-214, as route_node applies them): the qOUT of an inflow node, in the
// ring rows of steps [t_lo, t_hi), is replaced by the gauge's discharge, or
// increased by it for a headwater gauge, before the tiles read those rows.
// One thread per (step, set) applies the gauges in their order.
__global__ __launch_bounds__(256) void inflow_patch_kernel(RouteArgs r, double *ring,
                                                           const uint8_t *lag, int64_t t_lo,
                                                           int64_t t_hi, int32_t rep) {
  const int64_t t = t_lo + (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int32_t set = blockIdx.y;
  if (t >= t_hi) return;
  const int64_t ld = (int64_t)r.n_sets * r.sstride;
  for (int32_t g = 0; g < r.n_inflow; ++g) {
    const int32_t p = r.inflow_node[g];
    // each routing sub-step of a model step adds that step's inflow
    const double qi = r.inflow_q[(t - r.t_base) / rep * r.n_inflow + g];
    double &q = ring[ring_row(t, lag[p], r.ring_len) * ld + (int64_t)set * r.sstride + p];
    q = r.inflow_hw[g] ? q + qi : qi;
  }
}

// ---------------------------------------------------------------------------
// host launchers
template <int NH>
static hipError_t step_nh(const CellArgs &a, const StepDev &st, int64_t t, int block, int n_sets,
                          hipStream_t s) {
  dim3 grid((unsigned)((a.n_cells + block - 1) / block), (unsigned)n_sets);
  const bool out = a.out.sum != nullptr;
  if (a.jarvis && out)
    hipLaunchKernelGGL((cell_step_kernel<NH, true, true>), grid, dim3(block), 0, s, a, StepArgs{st, t});
  else if (a.jarvis)
    hipLaunchKernelGGL((cell_step_kernel<NH, true, false>), grid, dim3(block), 0, s, a, StepArgs{st, t});
  else if (out)
    hipLaunchKernelGGL((cell_step_kernel<NH, false, true>), grid, dim3(block), 0, s, a, StepArgs{st, t});
  else
    hipLaunchKernelGGL((cell_step_kernel<NH, false, false>), grid, dim3(block), 0, s, a, StepArgs{st, t});
  return hipGetLastError();
}

template <int NH>
static hipError_t fused_nh(const CellArgs &a, int64_t t0, int nsteps, int step0, int block,
                           int n_sets, hipStream_t s) {
  const bool out = a.out.sum != nullptr;
  const size_t lane = lane_slots(NH, a.jarvis != 0, out ? a.out.n : 0) * sizeof(double);
  // the lanes' LDS slots of a workgroup stay within 64 KB
  while (block * lane > 65536) block /= 2;
  const size_t shm = block * lane;
  dim3 grid((unsigned)((a.n_cells + block - 1) / block), (unsigned)n_sets);
  const FusedArgs f{t0, nsteps, step0};
  if (a.jarvis && out)
    hipLaunchKernelGGL((cell_fused_kernel<NH, true, true, false>), grid, dim3(block), shm, s, a, f);
  else if (out)
    hipLaunchKernelGGL((cell_fused_kernel<NH, false, true, false>), grid, dim3(block), shm, s, a, f);
  else if (a.jarvis && a.sun)
    hipLaunchKernelGGL((cell_fused_kernel<NH, true, false, true>), grid, dim3(block), shm, s, a, f);
  else if (a.jarvis)
    hipLaunchKernelGGL((cell_fused_kernel<NH, true, false, false>), grid, dim3(block), shm, s, a, f);
  else if (a.sun)
    hipLaunchKernelGGL((cell_fused_kernel<NH, false, false, true>), grid, dim3(block), shm, s, a, f);
  else
    hipLaunchKernelGGL((cell_fused_kernel<NH, false, false, false>), grid, dim3(block), shm, s, a, f);
  return hipGetLastError();
}

hipError_t launch_cell_step(int nh, const CellArgs &a, const StepDev &st, int64_t t, int block,
                            int n_sets, hipStream_t s) {
  switch (nh) {
    case 1: return step_nh<1>(a, st, t, block, n_sets, s);
    case 2: return step_nh<2>(a, st, t, block, n_sets, s);
    case 3: return step_nh<3>(a, st, t, block, n_sets, s);
    case 4: return step_nh<4>(a, st, t, block, n_sets, s);
    case 5: return step_nh<5>(a, st, t, block, n_sets, s);
    case 6: return step_nh<6>(a, st, t, block, n_sets, s);
  }
  return hipErrorInvalidValue;
}

hipError_t launch_cell_fused(int nh, const CellArgs &a, int64_t t0, int nsteps, int step0,
                             int block, int n_sets, hipStream_t s) {
  switch (nh) {
    case 1: return fused_nh<1>(a, t0, nsteps, step0, block, n_sets, s);
    case 2: return fused_nh<2>(a, t0, nsteps, step0, block, n_sets, s);
    case 3: return fused_nh<3>(a, t0, nsteps, step0, block, n_sets, s);
    case 4: return fused_nh<4>(a, t0, nsteps, step0, block, n_sets, s);
    case 5: return fused_nh<5>(a, t0, nsteps, step0, block, n_sets, s);
    case 6: return fused_nh<6>(a, t0, nsteps, step0, block, n_sets, s);
  }
  return hipErrorInvalidValue;
}

hipError_t launch_sun(const CellArgs &a, int step0, int nsteps, double *sun, hipStream_t s) {
  if (nsteps < 1 || nsteps > 65535 || a.pet_case != 1) return hipErrorInvalidValue;
  hipLaunchKernelGGL(sun_kernel, dim3((unsigned)((a.n_cells + 255) / 256), (unsigned)nsteps),
                     dim3(256), 0, s, a, step0, sun);
  return hipGetLastError();
}

hipError_t launch_route_diag(const RouteArgs &r, int64_t d, int64_t p_lo, int64_t p_hi,
                             hipStream_t s) {
  if (p_lo < 0 || p_hi > r.n_nodes || p_hi <= p_lo) return hipErrorInvalidValue;
  dim3 grid((unsigned)((p_hi - p_lo + 255) / 256), (unsigned)r.n_sets);
  hipLaunchKernelGGL(route_diag_kernel, grid, dim3(256), 0, s, r, d, (uint32_t)p_lo,
                     (uint32_t)p_hi);
  return hipGetLastError();
}

hipError_t launch_route_tile(const RouteArgs &r, const TileArgs &g, const WindowArgs &v,
                             int64_t bin_lo, int64_t bin_hi,
                             int64_t n_bins, int32_t L, hipStream_t s) {
  // a window's rows do not wrap (ring length and window starts are multiples
  // of B; the ring has kTileHeight rows past its length), and a ring row's
  // bytes fit the kernel's 32-bit stride
  if (bin_lo < 0 || bin_hi > n_bins || bin_hi <= bin_lo || v.B < 1 || v.B > v.bstride ||
      v.bstride > kTileWindowMax || v.nwin < 1 || r.ring_len % v.B != 0 || r.t_lo % v.B != 0 ||
      (uint64_t)r.n_sets * (uint64_t)r.sstride * 8u > 0xFFFFFFFFull)
    return hipErrorInvalidValue;
  dim3 grid((unsigned)(bin_hi - bin_lo), (unsigned)r.n_sets);
  const size_t base = sizeof(double) * 2 * (size_t)kTileBuf;
  const size_t stage = (size_t)v.out_rows * (sizeof(TileOutRow) + sizeof(double) * (v.B + 1)) +
                       sizeof(double) * kTileSlots;
  const bool st = base + stage <= kTileStageLds;
  const size_t shm = st ? base + stage : base;
  if (st && r.qacc)
    hipLaunchKernelGGL((route_tile_kernel<true, true>), grid, dim3(kTileSlots), shm, s, r, g, v, L,
                       (int32_t)bin_lo);
  else if (st)
    hipLaunchKernelGGL((route_tile_kernel<true, false>), grid, dim3(kTileSlots), shm, s, r, g, v, L,
                       (int32_t)bin_lo);
  else if (r.qacc)
    hipLaunchKernelGGL((route_tile_kernel<false, true>), grid, dim3(kTileSlots), shm, s, r, g, v, L,
                       (int32_t)bin_lo);
  else
    hipLaunchKernelGGL((route_tile_kernel<false, false>), grid, dim3(kTileSlots), shm, s, r, g, v, L,
                       (int32_t)bin_lo);
  return hipGetLastError();
}

namespace {
// a set's area holds the words of its boundary rows; 32-bit byte offsets
bool flow_fits(const RouteArgs &r, const TileArgs &g, const FlowArgs &f) {
  return f.n_bins >= 1 && f.area && f.fail && f.lag && f.astride >= kFlowHead + 2 * g.n_bnd &&
         (uint64_t)r.n_sets * (uint64_t)r.sstride * 8u <= 0xFFFFFFFFull;
}
}  // namespace

hipError_t launch_route_step(const RouteArgs &r, const TileArgs &g, const FlowArgs &f,
                             hipStream_t s) {
  // one step of a one-step ring
  if (!flow_fits(r, g, f) || r.ring_len != 1 || r.t_lo != 0 || r.t_hi != 1 || r.t_base != 0)
    return hipErrorInvalidValue;
  dim3 grid((unsigned)f.n_bins, (unsigned)r.n_sets);
  if (r.qacc)
    hipLaunchKernelGGL(route_step_kernel<true>, grid, dim3(kTileSlots), 0, s, r, g, f);
  else
    hipLaunchKernelGGL(route_step_kernel<false>, grid, dim3(kTileSlots), 0, s, r, g, f);
  return hipGetLastError();
}

hipError_t launch_route_stream(const RouteArgs &r, const TileArgs &g, const FlowArgs &f,
                               hipStream_t s) {
  // the steps' rows do not wrap (the ring has the tiles' height in rows past
  // its length), and the proxies and outputs of a bin have a lane each
  if (!flow_fits(r, g, f) || r.t_lo < 0 || r.t_hi <= r.t_lo || r.t_hi - r.t_lo > 0x3FFFFFFF ||
      r.t_lo % r.ring_len + (r.t_hi - r.t_lo) > r.ring_len || f.proxy_waves < 0 ||
      f.out_waves < 0 || f.proxy_waves > 4 || f.out_waves > 8)
    return hipErrorInvalidValue;
  dim3 grid((unsigned)f.n_bins, (unsigned)r.n_sets);
  dim3 block((unsigned)(kTileSlots + 64 * (f.proxy_waves + f.out_waves)));
  if (r.qacc)
    hipLaunchKernelGGL(route_stream_kernel<true>, grid, block, 0, s, r, g, f);
  else
    hipLaunchKernelGGL(route_stream_kernel<false>, grid, block, 0, s, r, g, f);
  return hipGetLastError();
}

hipError_t launch_inflow_patch(const RouteArgs &r, double *ring, const uint8_t *lag, int64_t t_lo,
                               int64_t t_hi, hipStream_t s, int32_t rep) {
  if (t_hi <= t_lo || t_lo < r.t_base || r.n_inflow < 1 || !lag || rep < 1)
    return hipErrorInvalidValue;
  dim3 grid((unsigned)((t_hi - t_lo + 255) / 256), (unsigned)r.n_sets);
  hipLaunchKernelGGL(inflow_patch_kernel, grid, dim3(256), 0, s, r, ring, lag, t_lo, t_hi, rep);
  return hipGetLastError();
}

hipError_t launch_route_wg(const RouteArgs &r, const int64_t *dom_start, const int32_t *dom_dmax,
                           int n_domains, int64_t d_lo, int64_t d_hi, int drain, int block,
                           hipStream_t s) {
  dim3 grid((unsigned)n_domains, (unsigned)r.n_sets);
  hipLaunchKernelGGL(route_wg_kernel, grid, dim3(block), 0, s, r, dom_start, dom_dmax, d_lo, d_hi,
                     drain);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// MPR-lite on the device: every parameter row of one set from its gamma
// vector (the order of mhmhip.h's MHMHIP_MPRLITE_* indices) and the cells'
// land-cover fractions, soil texture, aspect and latitude -- the synthetic
// domains' stand-in regionalisation, the same operations in the same order
// as its numpy statement (parameters.mpr_lite with static_fields and
// pet_radiation_params), so every row but the root fractions has the host's
// bits (those take c**(z/10) from the chain's power instead of libm's pow).
// The rows hold what mhmhip_set_cell_var stores for those fields: the
// degree-day rows times c2TSTu, the recession rows as c2TSTu / k.  The snow
// and sealed-threshold fields follow the reference's transfer functions
// (src/MPR/mo_multi_param_reg.f90:800-852, 883-894). One lane per cell.
__global__ __launch_bounds__(256) void mprlite_kernel(MprLiteArgs a, int32_t set) {
  mathtab_fill();  // the root fractions' power reads it (before any thread returns)
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= a.n_cells) return;
  const int64_t S = a.sstride;
  const double fF = a.in[c], fI = a.in[S + c], fP = a.in[2 * S + c];
  const double tx = a.in[3 * S + c], asp = a.in[4 * S + c];
  double *P = a.P + (int64_t)set * S + c;
  auto put = [&](int row, double v) { P[(int64_t)row * a.ld] = v; };
  const double *g = a.gamma;
  const int nh = a.nh;
  const double c2 = a.c2;
  put(PR_FS, fI);
  // snow_acc_melt_param: degree-day factors per cover class, then the
  // class-weighted cell values
  const double ddf_f = g[MHMHIP_MPRLITE_DDF_FOREST];
  const double ddf_p = ddf_f + g[MHMHIP_MPRLITE_DDF_PERVIOUS];
  const double ddf_i = ddf_p + g[MHMHIP_MPRLITE_DDF_IMPERVIOUS];
  const double max_f = ddf_f + g[MHMHIP_MPRLITE_MAXDDF_FOREST];
  const double max_i = ddf_i + g[MHMHIP_MPRLITE_MAXDDF_IMPERVIOUS];
  const double max_p = ddf_p + g[MHMHIP_MPRLITE_MAXDDF_PERVIOUS];
  put(PR_TTH, g[MHMHIP_MPRLITE_SNOW_TEMP]);
  put(PR_INCR, g[MHMHIP_MPRLITE_DDF_INCREASE]);
  put(PR_DNPS, (ddf_f * fF + ddf_i * fI + ddf_p * fP) * c2);
  put(PR_DMAXS, (max_f * fF + max_i * fI + max_p * fP) * c2);
  put(PR_SEALTHR, g[MHMHIP_MPRLITE_IMPERVIOUS_STORAGE]);
  // monthly leaf area index: interception capacity, PET-LAI factor and the
  // radiation cases' fields
  for (int m = 0; m < 12; ++m) {
    const double lai = fF * a.lai[m] + fI * a.lai[12 + m] + fP * a.lai[24 + m];
    put(pr_maxinter(nh) + m, g[MHMHIP_MPRLITE_CANOPY] * lai);
    put(pr_petlai(nh) + m, fmin(fmax(0.6 + 0.08 * lai, 0.3), 1.3));
    if (a.pet_case == 2) put(pr_prietay(nh) + m, 1.05 + 0.06 * lai);
    if (a.pet_case == 3) {
      put(pr_aero(nh) + m, 208.0 / (0.6 + 0.1 * lai));
      put(pr_surf(nh) + m, 40.0 + 120.0 / (1.0 + lai));
    }
  }
  // soil water contents per horizon
  const double poro = 0.38 + 0.12 * tx, fcr = 0.55 + 0.25 * (1.0 - tx);
  const double wpr = 0.30 + 0.25 * tx;
  const double sexp = g[MHMHIP_MPRLITE_INFIL_SHAPE] * (1.0 + 0.3 * tx);
  double rc = fF * g[MHMHIP_MPRLITE_ROOT_FOREST] + fI * g[MHMHIP_MPRLITE_ROOT_IMPERVIOUS] +
              fP * g[MHMHIP_MPRLITE_ROOT_PERVIOUS];
  rc = fmin(fmax(rc, 1e-3), 0.999);
  double fr[MHMHIP_MAX_HORIZONS];
  double cum_top = 0.0, fsum = 0.0, top = 0.0;
  for (int h = 0; h < nh; ++h) {
    const double dz = a.hd[h] - top;
    top = a.hd[h];
    const double sat = dz * poro, fc = sat * fcr;
    put(pr_sat(nh) + h, sat);
    put(pr_fc(nh) + h, fc);
    put(pr_wp(nh) + h, fc * wpr);
    put(pr_exp(nh) + h, sexp);
    // root fraction: cumulative 1 - c**(z / 10 mm), differenced, normalised
    const double cum = 1.0 - exp_ylogx(a.hd[h] / 10.0, rc);
    fr[h] = fmax(cum - cum_top, 0.0);
    cum_top = cum;
    fsum = fsum + fr[h];
  }
  const double fden = fmax(fsum, 1e-12);
  for (int h = 0; h < nh; ++h) put(pr_froots(nh) + h, fr[h] / fden);
  put(PR_JARVIS, g[MHMHIP_MPRLITE_JARVIS_C1]);
  // recession constants [d], stored as c2TSTu / k
  const double k1 = g[MHMHIP_MPRLITE_SLOW_KS] * (0.5 + tx);
  put(PR_K0S, c2 / (g[MHMHIP_MPRLITE_FAST_FOREST] * (1.0 + 0.5 * (1.0 - fF))));
  put(PR_K1S, c2 / k1);
  put(PR_KPS, c2 / fmax(g[MHMHIP_MPRLITE_RECHARGE] * (0.5 + tx), 2.0));
  put(PR_K2S, c2 / fmax(g[MHMHIP_MPRLITE_GEOPARAM] * (0.5 + 0.5 * tx), k1));
  put(PR_ALPHA, g[MHMHIP_MPRLITE_EXP_SLOW]);
  put(PR_KARST, 1.0);
  put(PR_UNSATTHR, g[MHMHIP_MPRLITE_INTERFLOW_CAPACITY] * (0.2 + 0.3 * tx));
  // PET aspect correction
  const double thr = g[MHMHIP_MPRLITE_ASPECT_THRESH], mn = g[MHMHIP_MPRLITE_PET_MIN];
  const double mx = g[MHMHIP_MPRLITE_PET_MAX];
  put(PR_FASP, asp < thr ? mn + mx * (thr - asp) / thr : mn + mx * (asp - thr) / (360.0 - thr));
  put(PR_HARSAM, g[MHMHIP_MPRLITE_HARGREAVES]);
  put(PR_TANLAT, a.in[5 * S + c]);
  put(PR_SINLAT, a.in[6 * S + c]);
  put(PR_COSLAT, a.in[7 * S + c]);
}

hipError_t launch_mprlite(const MprLiteArgs &a, int32_t set, hipStream_t s) {
  if (a.n_cells < 1 || a.nh < 1 || a.nh > MHMHIP_MAX_HORIZONS || !a.P || !a.in || set < 0)
    return hipErrorInvalidValue;
  hipLaunchKernelGGL(mprlite_kernel, dim3((unsigned)((a.n_cells + 255) / 256)), dim3(256), 0, s, a,
                     set);
  return hipGetLastError();
}

}  // namespace mhmhip
