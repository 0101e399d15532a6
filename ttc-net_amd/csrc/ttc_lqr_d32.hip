// ttc_lqr_d32.hip -- kernels instantiated for d = du = 32.
#include "ttc_lqr_kernels.hpp"

namespace ttc {

int launch_fwd_d32(const float* A, const float* B, const float* Q, const float* R, const float* Qf,
                  const float* lA, const float* lB, const float* lQ, const float* h0, int64_t P, int H, int T,
                  float* u, float* st_a, float* st_b, int sm, int32_t* status, hipStream_t s, int flags,
                  int64_t call, int32_t* rescue_ws) {
  // fp32 sweeps without per-step gains run on the matrix cores unless the row-layout kernel
  // is asked for: the certified symplectic sweep by default, per-step Riccati when asked for.
  // fp64 rescue of a symplectic sweep; without one (the stable backward's gains, row-layout or
  // Riccati-step kernels asked for) the sweep is fp64 throughout.  So it is at odd head counts under
  // TTC_LQR_FLAG_FP64_RESCUE itself (long horizons), which has always promised them that: 5 heads,
  // 64 tokens, T = 512 end 2e-8 (u) and 2e-7 (gradients) from 64 bits in 34.8 ms, where the certified
  // fp32 sweep of the even counts ends 1.4e-6 and 2.2e-6 away in 0.6 ms.
  const bool odd = H % 2 != 0 && !(flags & TTC_LQR_FLAG_FP64_FALLBACK);
  if ((flags & TTC_LQR_FLAG_FP64_RESCUE) &&
      (sm == STASH_GAINS || (flags & (TTC_LQR_FLAG_ROW_KERNEL | TTC_LQR_FLAG_RICCATI_STEPS)) || odd))
    flags |= TTC_LQR_FLAG_FP64_RICCATI;
  if (!(flags & (TTC_LQR_FLAG_FP64_RICCATI | TTC_LQR_FLAG_ROW_KERNEL)) && sm != STASH_GAINS)
    return launch_fwd_d32_mfma(A, B, Q, R, Qf, lA, lB, lQ, h0, P, H, T, u, st_a, st_b, sm, status, s,
                               !(flags & TTC_LQR_FLAG_RICCATI_STEPS), call,
                               (flags & TTC_LQR_FLAG_FP64_RESCUE) != 0, rescue_ws);
  return launch_fwd<32, true>(A, B, Q, R, Qf, lA, lB, lQ, h0, P, H, T, u, st_a, st_b, sm, status, s, flags);
}

int launch_bwd_d32(const float* A, const float* B, const float* Q, const float* R, const float* Qf,
                  const float* lA, const float* lB, const float* lQ, const float* h0, const float* dU,
                  const float* kst, const float* q0s, int64_t P, int H, int T, void* traj, bool fp64, float* gA,
                  float* gR, float* gQf, float* glA, float* glB, float* glQ, float* gh0, float* gBp,
                  float* gQp, float limit, int32_t* status, hipStream_t s) {
  if (fp64)
    return launch_bwd<32, double>(A, B, Q, R, Qf, lA, lB, lQ, h0, dU, kst, q0s, P, H, T, static_cast<double4*>(traj),
                                 gA, gR, gQf, glA, glB, glQ, gh0, gBp, gQp, limit, status, s);
  return launch_bwd<32>(A, B, Q, R, Qf, lA, lB, lQ, h0, dU, kst, q0s, P, H, T, static_cast<float4*>(traj), gA, gR,
                       gQf, glA, glB, glQ, gh0, gBp, gQp, limit, status, s);
}

int launch_ham_d32(const float* A, const float* B, const float* Q, const float* R, const float* Qf,
                  const float* lA, const float* lB, const float* lQ, const float* h0, const float* u0,
                  const float* dU, const float* v1s, const float* q0s, int64_t P, int H, int T, float tau,
                  float* gA, float* gR, float* gQf, float* glA, float* glB, float* glQ, float* gh0, float* gBp,
                  float* gQp, float limit, int32_t* fail_list, int32_t* fail_count, int32_t* status,
                  hipStream_t s, bool fp64, const int32_t* plist) {
  if (fp64)
    return launch_ham<32, double>(A, B, Q, R, Qf, lA, lB, lQ, h0, u0, dU, v1s, q0s, P, H, T, tau, gA, gR, gQf, glA, glB,
                       glQ, gh0, gBp, gQp, limit, fail_list, fail_count, status, s, plist);
  return launch_ham<32>(A, B, Q, R, Qf, lA, lB, lQ, h0, u0, dU, v1s, q0s, P, H, T, tau, gA, gR, gQf, glA, glB,
                       glQ, gh0, gBp, gQp, limit, fail_list, fail_count, status, s, plist);
}

}  // namespace ttc
