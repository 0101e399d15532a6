// ttc_lqr_sym.hpp -- what the symplectic sweeps share (ttc_lqr_sym16.hpp, ttc_lqr_symw.hpp): the
// certificate's thresholds, the intervals of the renormalisation and of the exact discounts, lane helpers.
#pragma once
#include "ttc_lqr_mfma16.hpp"

#ifndef TTC_SYM_RENORM
#define TTC_SYM_RENORM 8  // steps between power-of-2 renormalisations of the symplectic sweep
#endif

namespace ttc {

// Certificate of the symplectic sweep: the final solve P = Y1^{-1} Y2 is accepted when the
// condition number of Y1 (cond_inf at d = 32; at d = 16 and 64 its estimate ||Y1||_inf / min|u_kk|
// from the pivots of the same elimination) is <= kSymCondMax and max|P - P'| <= kSymAsymMax max|P|;
// problems that miss it are recomputed by the rescue pass.
constexpr float kSymCondMax = 1.0e7f;
// steps between exact (exp2) evaluations of the symplectic sweep's discount factors; the
// steps in between multiply the previous step's by a constant ratio
constexpr int kSymRefresh = 8;
constexpr float kSymAsymMax = 1.0e-6f;

// max over the D lanes of a problem (D = 16, 32, 64)
template <int D>
__device__ __forceinline__ float dgroup_max(float v) {
  v = fmaxf(v, ror16f<8>(v));
  v = fmaxf(v, ror16f<4>(v));
  v = fmaxf(v, ror16f<2>(v));
  v = fmaxf(v, ror16f<1>(v));
  if constexpr (D >= 32) v = fmaxf(v, __shfl_xor(v, 16, 64));
  if constexpr (D >= 64) v = fmaxf(v, __shfl_xor(v, 32, 64));
  return v;
}

// v of the lane whose byte address (4 * lane) is xaddr
__device__ __forceinline__ float lane_read(float v, int xaddr) {
  return __int_as_float(__builtin_amdgcn_ds_bpermute(xaddr, __float_as_int(v)));
}

}  // namespace ttc
