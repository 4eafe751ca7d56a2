// Fourier convergence of one item, shared by the symmetric path (k_converge) and
// the general path (k_bvp, k_rescue).
#pragma once
#include "rt_work.h"

namespace aa {

namespace {

constexpr double VLIDORT_ACCURACY_D = (double)0.0001f;   // V283/VLIDORT_Mod.F90:232

// Adds Fourier term M's component cum of one item to its TOA Stokes vector and
// tests the azimuth series (VLIDORT_CONVERGE_OBSGEO).  Writes the outputs of an
// item that is done; returns whether it goes on to the next term.
template <int N, int S>
__device__ __forceinline__ bool converge_term(const RTWork& W, int it, int obs, size_t oi, double ff, int M,
                                              const double (&cum)[S]) {
  const double flux_multiplier = (M == 0) ? 1.0 : 2.0;
  double* stk = W.stokes + (size_t)it * 3;
  bool done = false;
  double sf[S];
#pragma unroll
  for (int o = 0; o < S; ++o) sf[o] = flux_multiplier * cum[o];
  int testconv = W.testconv[it], fsaved = W.fsaved[it];
  if (M == 0) {
#pragma unroll
    for (int o = 0; o < S; ++o) stk[o] = sf[o] + W.ss[(size_t)it * 3 + o] + W.db[(size_t)it * 3 + o];
  } else {
    const double azm = W.raa[obs] * (double)M * DEG_TO_RAD;
    const double azmfac[3] = {cos(azm), cos(azm), sin(azm)};
    double tazm[S], tnew[S];
#pragma unroll
    for (int o = 0; o < S; ++o) { tazm[o] = azmfac[o] * sf[o]; tnew[o] = stk[o] + tazm[o]; }
    int count = 0;
    if (tazm[0] != 0.0) { const double accur = fabs(tazm[0] / tnew[0]); if (accur < VLIDORT_ACCURACY_D) count++; }
    else count++;
#pragma unroll
    for (int o = 0; o < S; ++o) stk[o] = tnew[o];
    if (count == 1) {
      testconv++;
      if (testconv == 2) { done = true; fsaved = M; }
    } else { testconv = 0; fsaved = 2 * N - 1; }
  }
  W.testconv[it] = testconv;
  W.fsaved[it] = fsaved;
  if (M >= W.nmoments) done = true;
  if (done) {
    const float pif = 4.0f * atanf(1.0f);
    const double pi = (double)pif;
    const double I = stk[0];
    W.radiance[oi] = I;
    W.reflectance[oi] = (pi * I) / (cos(W.sza[obs] * pi / (double)180.0f) * ff);
    if (S > 1) { W.qout[oi] = stk[1]; W.uout[oi] = stk[2]; }
    W.nfourier[oi] = fsaved + 1;
    return false;
  }
  return true;
}

}  // namespace
}  // namespace aa
