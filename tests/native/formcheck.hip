// formcheck.hip -- the branch-free form of the cell chain (chain.h) beside its
// branches on the device, for tests of one step's values.  Not part of the
// model library: linked into libmhmcheck.so (mhm_amd/build.py).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "chain.h"

namespace {
using namespace mhmhip;

constexpr int NH = 3;
// inputs of a cell, in order: weather, month and step, parameters, states
enum In {
  I_PREC, I_TEMP, I_PET, I_MAXI, I_EVAP, I_FS, I_THRS, I_INCR, I_DMAX, I_DNP, I_TTH, I_K0, I_K1,
  I_K2, I_KP, I_KARST, I_ALPHA, I_THRU, I_C1, I_SAT, I_FR = I_SAT + NH, I_FC = I_FR + NH,
  I_WP = I_FC + NH, I_BEXP = I_WP + NH, I_INTER = I_BEXP + NH, I_PACK, I_SEAL, I_UNSAT, I_SATS,
  I_SM, I_COUNT = I_SM + NH
};
enum Out {
  O_THR, O_ECAN, O_INTER, O_DDF, O_MELT, O_PEFF, O_RAIN, O_SNOW, O_PACK, O_RSEAL, O_ASEAL, O_SEAL,
  O_INFIL, O_AET = O_INFIL + NH, O_SM = O_AET + NH, O_FAST = O_SM + NH, O_SLOW, O_PERC, O_UNSAT,
  O_SATS, O_BFLOW, O_TOTAL, O_COUNT
};

template <bool JV>
__device__ void step_branches(const double *v, double *o) {
  double inter = v[I_INTER], pack = v[I_PACK], seal = v[I_SEAL], unsat = v[I_UNSAT];
  double satS = v[I_SATS], sm[NH], infil[NH], aet[NH], frac[NH], rfw[NH];
  const double maxi = v[I_MAXI], revap = 1.0 / v[I_EVAP];
  for (int h = 0; h < NH; ++h) {
    sm[h] = v[I_SM + h];
    rfw[h] = 1.0 / (v[I_FC + h] - v[I_WP + h]);
    frac[h] = exp_ylogx(v[I_BEXP + h], div_rcp(sm[h], v[I_SAT + h], 1.0 / v[I_SAT + h]));
  }
  const double ratio = canopy_fill(maxi, 1.0 / maxi, v[I_PREC], inter, o[O_THR]);
  canopy_evap(v[I_PET], maxi, ratio, ratio > 0.0 ? pow23(ratio) : 0.0, inter, o[O_ECAN]);
  snow_accum_melt(v[I_INCR], v[I_DMAX], v[I_DNP], (v[I_DMAX] - v[I_DNP]) / v[I_INCR], v[I_PREC],
                  v[I_TEMP], v[I_TTH], o[O_THR], pack, o[O_DDF], o[O_MELT], o[O_PEFF], o[O_RAIN],
                  o[O_SNOW]);
  soil_moisture<NH, JV>(v[I_FS], v[I_THRS], 1.0 / v[I_THRS], v[I_PET], v[I_EVAP], revap,
                        v + I_SAT, v + I_FR, v + I_FC, v + I_WP, rfw, v[I_C1], o[O_ECAN],
                        o[O_PEFF], frac, o[O_RSEAL], seal, infil, sm, aet, o[O_ASEAL]);
  runoff_fast(v[I_K0], infil[NH - 1], v[I_THRU], unsat, o[O_FAST]);
  runoff_slow_perc(v[I_K1], v[I_KP], v[I_KARST],
                   unsat > 0.0 ? exp_ylogx(1.0 + v[I_ALPHA], unsat) : 0.0, satS, unsat, o[O_SLOW],
                   o[O_PERC]);
  runoff_sat_zone(v[I_K2], satS, o[O_BFLOW]);
  o[O_TOTAL] = total_runoff(v[I_FS], o[O_FAST], o[O_SLOW], o[O_BFLOW], o[O_RSEAL]);
  o[O_INTER] = inter, o[O_PACK] = pack, o[O_SEAL] = seal, o[O_UNSAT] = unsat, o[O_SATS] = satS;
  for (int h = 0; h < NH; ++h)
    o[O_INFIL + h] = infil[h], o[O_AET + h] = aet[h], o[O_SM + h] = sm[h];
}

template <bool JV>
__device__ void step_ordinary(const double *v, double *o) {
  double inter = v[I_INTER], pack = v[I_PACK], seal = v[I_SEAL], unsat = v[I_UNSAT];
  double satS = v[I_SATS], in = 0.0, used = 0.0;
  const double maxi = v[I_MAXI];
  canopy_ordinary(v[I_PET], maxi, maxi > kEps ? 1.0 / maxi : 0.0, v[I_PREC], inter, o[O_THR],
                  o[O_ECAN]);
  const SnowMeteo m = snow_meteo(v[I_INCR], v[I_DMAX], v[I_DNP], v[I_TTH], v[I_PREC], v[I_TEMP]);
  o[O_DDF] = m.ddf;
  snow_ordinary(m.melt, m.cold, o[O_THR], pack, o[O_MELT], o[O_PEFF], o[O_RAIN], o[O_SNOW]);
  sealed_ordinary(v[I_FS] > 0.0, v[I_THRS], 1.0 / v[I_THRS],
                  div_rcp(v[I_PET], v[I_EVAP], 1.0 / v[I_EVAP]), o[O_ECAN], o[O_PEFF], o[O_RSEAL],
                  seal, o[O_ASEAL]);
  for (int h = 0; h < NH; ++h) {
    const double sat = v[I_SAT + h], fc = v[I_FC + h], wp = v[I_WP + h], fr = v[I_FR + h];
    double sm = v[I_SM + h];
    const double frac =
        pow_v<1>(DV<1>{{256.0 * v[I_BEXP + h]}}, DV<1>{{div_rcp(sm, sat, 1.0 / sat)}}).v[0];
    in = infiltrate_ordinary(h ? in : o[O_PEFF], frac, sat, sm);
    const double range = (JV ? sat : fc) - wp;
    const double f = stress_ordinary<JV>(sm, wp, fr, (JV ? 1.0 : fr) / range, range, v[I_C1],
                                         1.0 / v[I_C1]);
    const double demand = v[I_PET] - o[O_ECAN];
    const double aet = evaporate_ordinary(h ? demand - used : demand, f, sm);
    used = h ? used + aet : aet;
    o[O_INFIL + h] = in, o[O_AET + h] = aet, o[O_SM + h] = sm;
  }
  runoff_fast_ordinary(v[I_K0], in, v[I_THRU], unsat, o[O_FAST]);
  const double pw = pow_v<1>(DV<1>{{256.0 * (1.0 + v[I_ALPHA])}},
                             DV<1>{{vmax_k(unsat, DBL_MIN)}}).v[0];
  runoff_slow_perc_ordinary(v[I_K1], v[I_KP], v[I_KARST], pw, satS, unsat, o[O_SLOW], o[O_PERC]);
  o[O_BFLOW] = v[I_K2] * satS;
  satS = satS - o[O_BFLOW];
  o[O_TOTAL] = total_runoff(v[I_FS], o[O_FAST], o[O_SLOW], o[O_BFLOW], o[O_RSEAL]);
  if (!(v[I_FS] > 0.0)) o[O_RSEAL] = o[O_ASEAL] = 0.0;
  o[O_INTER] = inter, o[O_PACK] = pack, o[O_SEAL] = seal, o[O_UNSAT] = unsat, o[O_SATS] = satS;
}

// ok[i]: the cell is an ordinary one
template <bool JV>
__global__ void forms_kernel(const double *in, double *branches, double *ordinary, int32_t *ok,
                             int64_t n) {
  mathtab_fill();
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double v[I_COUNT], a[O_COUNT], b[O_COUNT];
  for (int k = 0; k < I_COUNT; ++k) v[k] = in[i * I_COUNT + k];
  ok[i] = ordinary_params<NH, JV>(v[I_FS], v[I_THRS], v[I_INCR], v[I_DMAX], v[I_DNP], v[I_TTH],
                                  v[I_K0], v[I_K1], v[I_K2], v[I_KP], v[I_KARST], v[I_ALPHA],
                                  v[I_THRU], v + I_SAT, v + I_FR, v + I_FC, v + I_WP, v + I_BEXP,
                                  v[I_C1]) &&
          ordinary_states<NH>(v[I_INTER], v[I_PACK], v[I_SEAL], v[I_UNSAT], v[I_SATS], v + I_SM,
                              v + I_SAT) &&
          v[I_PREC] >= 0.0;
  step_branches<JV>(v, a);
  step_ordinary<JV>(v, b);
  for (int k = 0; k < O_COUNT; ++k) {
    branches[i * O_COUNT + k] = a[k];
    ordinary[i * O_COUNT + k] = b[k];
  }
}

__global__ void ratio_kernel(const double *x, double *out, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = pow23_ratio(x[i]);
}

}  // namespace

extern "C" int mhmhip_check_form_sizes(int *inputs, int *outputs) {
  *inputs = I_COUNT;
  *outputs = O_COUNT;
  return 0;
}

// One step of n cells in both forms on device 0: in[n][inputs], branches and
// ordinary [n][outputs], ok[n].
extern "C" int mhmhip_check_forms(int jarvis, const double *in, double *branches, double *ordinary,
                                  int32_t *ok, int64_t n) {
  if (n < 1 || !in || !branches || !ordinary || !ok) return -1;
  const size_t bi = sizeof(double) * I_COUNT * n, bo = sizeof(double) * O_COUNT * n;
  char *d = nullptr;
  if (hipMalloc(&d, bi + 2 * bo + sizeof(int32_t) * n) != hipSuccess) return -2;
  double *di = reinterpret_cast<double *>(d), *da = reinterpret_cast<double *>(d + bi);
  double *db = reinterpret_cast<double *>(d + bi + bo);
  int32_t *dk = reinterpret_cast<int32_t *>(d + bi + 2 * bo);
  int rc = 0;
  if (hipMemcpy(di, in, bi, hipMemcpyHostToDevice) != hipSuccess) {
    rc = -3;
  } else {
    const dim3 grid((unsigned)((n + 255) / 256));
    if (jarvis)
      hipLaunchKernelGGL(forms_kernel<true>, grid, dim3(256), 0, 0, di, da, db, dk, n);
    else
      hipLaunchKernelGGL(forms_kernel<false>, grid, dim3(256), 0, 0, di, da, db, dk, n);
    if (hipGetLastError() != hipSuccess || hipDeviceSynchronize() != hipSuccess ||
        hipMemcpy(branches, da, bo, hipMemcpyDeviceToHost) != hipSuccess ||
        hipMemcpy(ordinary, db, bo, hipMemcpyDeviceToHost) != hipSuccess ||
        hipMemcpy(ok, dk, sizeof(int32_t) * n, hipMemcpyDeviceToHost) != hipSuccess)
      rc = -4;
  }
  (void)hipFree(d);
  return rc;
}

// pow23_ratio of n values on device 0.
extern "C" int mhmhip_check_ratio(const double *x, double *out, int64_t n) {
  if (n < 1 || !x || !out) return -1;
  const size_t bytes = sizeof(double) * n;
  double *d = nullptr;
  if (hipMalloc(&d, 2 * bytes) != hipSuccess) return -2;
  int rc = 0;
  if (hipMemcpy(d, x, bytes, hipMemcpyHostToDevice) != hipSuccess) {
    rc = -3;
  } else {
    hipLaunchKernelGGL(ratio_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, 0, d, d + n,
                       n);
    if (hipGetLastError() != hipSuccess || hipDeviceSynchronize() != hipSuccess ||
        hipMemcpy(out, d + n, bytes, hipMemcpyDeviceToHost) != hipSuccess)
      rc = -4;
  }
  (void)hipFree(d);
  return rc;
}
