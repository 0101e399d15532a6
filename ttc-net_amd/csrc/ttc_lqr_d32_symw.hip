// ttc_lqr_d32_symw.hip -- the d = du = 32 symplectic sweep (ttc_lqr_symw.hpp), instantiated.
#include "ttc_lqr_symw.hpp"

namespace ttc {

int launch_symw_d32(const float* A, const float* B, const float* Q, const float* R, const float* Qf, const float* lA,
                    const float* lB, const float* lQ, const float* h0, int64_t P, int H, int T, float* u, float* st_a,
                    float* st_b, int sm, int32_t* status, hipStream_t s,
                    int64_t call) {
  if (sm == STASH_NONE)
    launch_symw<32, STASH_NONE, true>(A, B, Q, R, Qf, lA, lB, lQ, h0, P, H, T, u, st_a, st_b, status, s, call);
  else if (u != nullptr)
    launch_symw<32, STASH_V1, true>(A, B, Q, R, Qf, lA, lB, lQ, h0, P, H, T, u, st_a, st_b, status, s, call);
  else
    launch_symw<32, STASH_V1, false>(A, B, Q, R, Qf, lA, lB, lQ, h0, P, H, T, u, st_a, st_b, status, s, call);
  return hipGetLastError() == hipSuccess ? TTC_LQR_OK : TTC_LQR_ELAUNCH;
}

}  // namespace ttc
