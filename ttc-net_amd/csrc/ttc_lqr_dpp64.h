// ttc_lqr_dpp64.h -- products of a 16 x 16 fp64 matrix held one row a lane with vectors held one
// entry a lane, as fused DPP multiply-adds.
//
// A d = 16 problem is one 16-lane row, and v_fmac_f64_dpp row_newbcast:c reads lane c of it, so
// a matrix-vector product is 16 instructions per vector and needs no broadcast through LDS.  In
// the fp64 row-layout backward kernels those broadcasts were the bound: a wave-step read 96 (the
// stable path's two passes) or 48 (the rollout) 16-byte rows of LDS, and the four waves of a
// workgroup share one LDS port.
//
// Every lane of the row must be active.  A DPP source must not be written by a VALU instruction in
// the two preceding wait states (the s_nop at either end; a statement never writes its sources).
#pragma once
#include <hip/hip_runtime.h>
#include "ttc_lqr_elim16.h"

namespace ttc {

#define TTC_DOT2(K, M)                                                                              \
  "v_fmac_f64_dpp %[a], %[x], %[m" #M "] row_newbcast:" #M " row_mask:0xf bank_mask:0xf\n\t"   \
  "v_fmac_f64_dpp %[b], %[y], %[m" #M "] row_newbcast:" #M " row_mask:0xf bank_mask:0xf\n\t"
#define TTC_OUT2(K, M)                                                                              \
  "v_fmac_f64_dpp %[g" #M "], %[x], %[s] row_newbcast:" #M " row_mask:0xf bank_mask:0xf\n\t"
#define TTC_OUT2Y(K, M)                                                                             \
  "v_fmac_f64_dpp %[g" #M "], %[y], %[t] row_newbcast:" #M " row_mask:0xf bank_mask:0xf\n\t"

// a += sum_c m[c] x[lane c],  b += sum_c m[c] y[lane c], in the order of c
__device__ __forceinline__ void dpp_dot2(double& a, double& b, const double (&m)[16], double x, double y) {
  asm volatile("s_nop 2\n\t" TTC_DOT2(0, 0) TTC_R1(TTC_DOT2, 0) "s_nop 2"
               : [a] "+&v"(a), [b] "+&v"(b)
               : [x] "v"(x), [y] "v"(y), [m0] "v"(m[0]), [m1] "v"(m[1]), [m2] "v"(m[2]), [m3] "v"(m[3]),
                 [m4] "v"(m[4]), [m5] "v"(m[5]), [m6] "v"(m[6]), [m7] "v"(m[7]), [m8] "v"(m[8]), [m9] "v"(m[9]),
                 [m10] "v"(m[10]), [m11] "v"(m[11]), [m12] "v"(m[12]), [m13] "v"(m[13]), [m14] "v"(m[14]),
                 [m15] "v"(m[15]));
}

// g[c] += x[lane c] s, then g[c] += y[lane c] t
__device__ __forceinline__ void dpp_outer2(double (&g)[16], double x, double s, double y, double t) {
#define TTC_G(i) [g##i] "+&v"(g[i])
  asm volatile("s_nop 2\n\t" TTC_OUT2(0, 0) TTC_R1(TTC_OUT2, 0) TTC_OUT2Y(0, 0) TTC_R1(TTC_OUT2Y, 0) "s_nop 2"
               : TTC_G(0), TTC_G(1), TTC_G(2), TTC_G(3), TTC_G(4), TTC_G(5), TTC_G(6), TTC_G(7), TTC_G(8), TTC_G(9),
                 TTC_G(10), TTC_G(11), TTC_G(12), TTC_G(13), TTC_G(14), TTC_G(15)
               : [x] "v"(x), [s] "v"(s), [y] "v"(y), [t] "v"(t));
#undef TTC_G
}

#undef TTC_DOT2
#undef TTC_OUT2
#undef TTC_OUT2Y

}  // namespace ttc
