#pragma once
// ttc_lqr_kernels.hpp -- row-layout gfx950 kernels of TTC-Net's batched receding-horizon LQR solve.
//
// Problem (one per token n and head h, P = N*H problems), restating
// ttc/solvers/torch_lqr.py:65-91 and ttc/solvers/lin_solver_lqr.py:113-212:
//   A_k  = diag(1 + a*exp(lgA*(k+1)))       B_k = B diag(exp(lgB*(k+1)))
//   Qc_k = diag(exp(lgQ*k)) Q diag(exp(lgQ*k)) (k >= 1)   R = diag(1/R_inv)
//   V_T = Q_f ;  for k = T-1..0:
//     W = V B_k,  Quu = R + B_k'W,  Qux = W'A_k,  K_k = -Quu^{-1} Qux,
//     V <- A_k V A_k + Qux' K_k + Qc_k
//   u0 = K_0 h0.
//
// Layout: one problem per D lanes of a wave (D = d = du in {16,32,64}); lane i owns
// row i of every D x D matrix (V, W, the augmented [Quu | Qux] row, gradient rows).
// Cross-lane traffic goes through wave-private LDS (write a row, read broadcast
// rows back) -- no workgroup barriers inside the time loop.  The token-shared B is
// staged once per block into LDS.  Gains are computed by Gauss-Jordan elimination
// with partial pivoting: Quu is SPD in exact arithmetic, but on long-horizon stress
// inputs fp32 rounding can make it indefinite, where Cholesky / unpivoted LDL' break
// down while pivoted elimination (what torch.linalg.solve does in the reference)
// stays accurate.
//
// Backward (gradients of sum(d_u * u0)): implicit differentiation of the KKT system
// (ttc/solvers/torch_lqr.py:34-63).  Primal and adjoint trajectories are rolled out
// with the stored gains, and costates are swept back with the closed-loop recursion
//   lambda_k = Qc_k h_k + A_k lambda_{k+1} + K_k'(R u_k + B_k' lambda_{k+1}),
// (the reference's open-loop recursion plus a term that is zero at the optimum),
// which is stable where the open-loop one amplifies rounding by prod(A_k).
#include <hip/hip_runtime.h>
#include <math.h>
#include <type_traits>
#include <stdint.h>

#include "ttc_lqr.h"
#include "ttc_lqr_internal.h"
#include "ttc_lqr_dpp64.h"


namespace ttc {

constexpr int kPad = 4;  // LDS row padding (floats): keeps rows 16-byte aligned, staggers banks

// Forward stash modes.
constexpr int STASH_NONE = 0;   // u only
constexpr int STASH_GAINS = 1;  // every gain K_t [P,T,du,d] + Quu_0 [P,du,du] (stable backward)
constexpr int STASH_V1 = 2;     // V_1 [P,d,d] + Quu_0 [P,du,du] (fast backward)

template <int D, int PPB_ = (D == 16) ? 16 : (D == 32 ? 4 : 1)>
struct Geo {
  static constexpr int PPB = PPB_;  // problems per block
  static constexpr int THREADS = PPB * D;
  static constexpr int LDM = D + kPad;                  // LDS row stride (elements)
  static constexpr int MAT = D * LDM;
  static constexpr int NVEC = 12;                       // D-element vector slots per problem
  static constexpr int PER_PROB = MAT + NVEC * D + 4;   // +4 elements: bank skew between problems
};

// The backward kernels' blocks.  In fp64 at d = 16 a block is one wave: the calls are short lists of
// problems, whose waves share a CU's load and LDS ports unless each gets a CU of its own (stable path
// of 32 problems x 1,024 steps 2.17 -> 1.52 ms).
template <int D, typename R>
using BwdGeo = std::conditional_t<D == 16 && std::is_same<R, double>::value, Geo<16, 4>, Geo<D>>;

// Order LDS traffic between lanes of one wave: stores before this point are
// visible to loads after it (LDS executes one wave's requests in order).
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// 16-byte vector moves of fp32 (4 per vector) or fp64 (2 per vector) rows.
template <typename R> struct V16;
template <> struct V16<float> {
  static constexpr int N = 4;
  __device__ static void ld(const float* s, float* o) {
    const float4 v = *reinterpret_cast<const float4*>(s);
    o[0] = v.x; o[1] = v.y; o[2] = v.z; o[3] = v.w;
  }
  __device__ static void st(float* s, const float* i) { *reinterpret_cast<float4*>(s) = make_float4(i[0], i[1], i[2], i[3]); }
};
template <> struct V16<double> {
  static constexpr int N = 2;
  __device__ static void ld(const double* s, double* o) {
    const double2 v = *reinterpret_cast<const double2*>(s);
    o[0] = v.x; o[1] = v.y;
  }
  __device__ static void st(double* s, const double* i) { *reinterpret_cast<double2*>(s) = make_double2(i[0], i[1]); }
};

template <int N, typename R>
__device__ __forceinline__ void ld_row(const R* s, R (&out)[N]) {
  static_assert(N % 4 == 0, "row length");
#pragma unroll
  for (int c = 0; c < N; c += V16<R>::N) V16<R>::ld(s + c, out + c);
}

template <int N, typename R>
__device__ __forceinline__ void st_row(R* s, const R (&in)[N]) {
#pragma unroll
  for (int c = 0; c < N; c += V16<R>::N) V16<R>::st(s + c, in + c);
}

template <int N>
__device__ __forceinline__ void ld_global_row(const float* __restrict__ g, float (&out)[N]) {
#pragma unroll
  for (int c = 0; c < N; c += 4) {
    const float4 v = *reinterpret_cast<const float4*>(g + c);
    out[c] = v.x; out[c + 1] = v.y; out[c + 2] = v.z; out[c + 3] = v.w;
  }
}

template <int N>
__device__ __forceinline__ void st_global_row(float* __restrict__ g, const float (&in)[N]) {
#pragma unroll
  for (int c = 0; c < N; c += 4)
    *reinterpret_cast<float4*>(g + c) = make_float4(in[c], in[c + 1], in[c + 2], in[c + 3]);
}

template <int N>
__device__ __forceinline__ void ld_global_row(const float* __restrict__ g, double (&out)[N]) {
#pragma unroll
  for (int c = 0; c < N; c += 4) {
    const float4 v = *reinterpret_cast<const float4*>(g + c);
    out[c] = v.x; out[c + 1] = v.y; out[c + 2] = v.z; out[c + 3] = v.w;
  }
}

template <int N>
__device__ __forceinline__ void st_global_row(float* __restrict__ g, const double (&in)[N]) {
#pragma unroll
  for (int c = 0; c < N; c += 4)
    *reinterpret_cast<float4*>(g + c) = make_float4((float)in[c], (float)in[c + 1], (float)in[c + 2], (float)in[c + 3]);
}

template <int N>
__device__ __forceinline__ void ld_global_row(const double* __restrict__ g, double (&out)[N]) {
#pragma unroll
  for (int c = 0; c < N; c += 2) {
    const double2 v = *reinterpret_cast<const double2*>(g + c);
    out[c] = v.x; out[c + 1] = v.y;
  }
}

template <int N>
__device__ __forceinline__ void st_global_row(double* __restrict__ g, const double (&in)[N]) {
#pragma unroll
  for (int c = 0; c < N; c += 2) *reinterpret_cast<double2*>(g + c) = make_double2(in[c], in[c + 1]);
}

// Max of a 32-bit key over the D lanes of a problem (all lanes get the result).
// bound_ctrl: a source lane the DPP move cannot read gives 0, the identity of the unsigned
// max, so the move may be folded into the max as its DPP operand (v_max_u32_dpp).
template <int N>
__device__ __forceinline__ unsigned ror16(unsigned v) {
  return __builtin_amdgcn_mov_dpp(v, 0x120 + N, 0xF, 0xF, true);  // row_ror:N
}
template <int D>
__device__ __forceinline__ unsigned group_max_u32(unsigned k) {
  k = max(k, ror16<8>(k));
  k = max(k, ror16<4>(k));
  k = max(k, ror16<2>(k));
  k = max(k, ror16<1>(k));
  if constexpr (D >= 32) k = max(k, (unsigned)__shfl_xor((int)k, 16, 64));
  if constexpr (D >= 64) k = max(k, (unsigned)__shfl_xor((int)k, 32, 64));
  return k;
}

template <int D, typename R = float>
__device__ __forceinline__ R group_sum(R v, R* scratch, int li) {
  // via LDS: every lane writes, everyone reads the D values
  wave_sync();
  scratch[li] = v;
  wave_sync();
  R vals[D];
  ld_row<D>(scratch, vals);
  R s = 0;
#pragma unroll
  for (int c = 0; c < D; ++c) s += vals[c];
  return s;
}

// max(a, b) that returns NaN when either is NaN (v_maximum3_f32 forms, with |x| as a free
// source modifier in absmax)
__device__ __forceinline__ float maxnan(float a, float b) { return __builtin_elementwise_maximum(a, b); }
__device__ __forceinline__ float absmax(float a, float b) { return maxnan(fabsf(a), fabsf(b)); }

// Monotone 32-bit key of |x| (fp64: its high word, sign cleared).
__device__ __forceinline__ unsigned mag_key(float x) { return __float_as_uint(fabsf(x)); }
__device__ __forceinline__ unsigned mag_key(double x) {
  return (unsigned)(__double_as_longlong(fabs(x)) >> 32);
}

// Reciprocal of a pivot: the hardware reciprocal (1 ulp) in fp32, a division in fp64
// (used for d = 16; the wider eliminations keep the division).
__device__ __forceinline__ float pivot_recip(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ double pivot_recip(double x) { return 1.0 / x; }

// In-place Gauss-Jordan elimination with partial pivoting on the D x D left block
// of the augmented rows `aug` (lane li owns row li, width W >= D).  On return the
// lane with pivot position `pos` holds row `pos` of (left^{-1} * right) scaled by
// `mypiv` (divide by it).  `prow` is W elements of this problem's LDS.
// CHUNK > 0 reads the pivot row CHUNK elements at a time, each chunk's loads followed by its
// updates (a scheduling barrier keeps the loads from being hoisted): fewer live registers
// for kernels whose peak is this elimination, one LDS latency per chunk instead of one per row.
// NC <= W: the columns that carry data (the rest is padding to whole 16-byte vectors and is
// left as it is).
template <int D, int W, int CHUNK = 0, int NC = W, typename R>
__device__ __forceinline__ void gauss_jordan(R (&aug)[W], int li, R* prow, R& mypiv, int& pos) {
  static_assert(NC > D && NC <= W, "data columns");
  constexpr unsigned kIdxBits = (D == 16) ? 4u : (D == 32 ? 5u : 6u);
  constexpr unsigned kIdxMask = (1u << kIdxBits) - 1u;
  constexpr int VN = V16<R>::N;
  bool done = false;
  mypiv = R(1);
  pos = 0;
#pragma unroll
  for (int k = 0; k < D; ++k) {
    // pivot = largest |aug[k]| among rows not yet used; ties -> lowest lane.
    // Key = magnitude bits with the low bits replaced by (D-1-lane).
    const unsigned key = done ? 0u : ((mag_key(aug[k]) & ~kIdxMask) | (unsigned)(D - 1 - li));
    const unsigned best = group_max_u32<D>(key);
    const int who = D - 1 - (int)(best & kIdxMask);
    const bool me = (who == li);
    constexpr int c0 = 0;
    (void)c0;
    const int cs = k & ~(VN - 1);
    if (me) {
#pragma unroll
      for (int c = (k & ~(VN - 1)); c < W; c += VN) V16<R>::st(prow + c, aug + c);
    }
    wave_sync();
    (void)cs;
    R pkv;  // the pivot
    if constexpr (CHUNK == 0) {
      R pr[W];
#pragma unroll
      for (int c = (k & ~(VN - 1)); c < W; c += VN) V16<R>::ld(prow + c, pr + c);
      pkv = pr[k];
      const R inv = D == 16 ? pivot_recip(pkv) : R(1) / pkv;  // (wider: register pressure)
      const R f = me ? R(0) : aug[k] * inv;
#pragma unroll
      for (int c = k + 1; c < NC; ++c) aug[c] = fma(-f, pr[c], aug[c]);
    } else {
      static_assert(CHUNK % VN == 0 && W % CHUNK == 0, "pivot-row chunks");
      pkv = prow[k];
      const R inv = D == 16 ? pivot_recip(pkv) : R(1) / pkv;
      const R f = me ? R(0) : aug[k] * inv;
#pragma unroll
      for (int c0 = k & ~(CHUNK - 1); c0 < W; c0 += CHUNK) {
        R pr[CHUNK];
#pragma unroll
        for (int c = 0; c < CHUNK; c += VN) V16<R>::ld(prow + c0 + c, pr + c);
#pragma unroll
        for (int c = 0; c < CHUNK; ++c)
          if (c0 + c > k && c0 + c < NC) aug[c0 + c] = fma(-f, pr[c], aug[c0 + c]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (me) { mypiv = pkv; pos = k; done = true; }
    wave_sync();  // next pivot row may overwrite prow
  }
}

// LU factorisation with partial pivoting of the D x D left block of the augmented rows,
// then back substitution: the same contract as gauss_jordan (the lane with pivot position
// `pos` ends with row `pos` of left^{-1} right in aug[D..W), times `mypiv`, here 1).
// Gauss-Jordan eliminates above the pivot too; its solutions are as accurate, but its
// residuals can be larger by a factor cond(left), and the Riccati update's Schur complement
// V - W Quu^{-1} W' inherits the residual: on long, barely discounted horizons with expensive
// control (cond(Quu) ~ 1e20) fp64 Gauss-Jordan lost two more digits of the gradients than
// LU.  The fp64 sweeps use this one.
template <int D, int W, typename R>
__device__ __forceinline__ void lu_rows(R (&aug)[W], int li, R* prow, R& mypiv, int& pos) {
  constexpr unsigned kIdxBits = (D == 16) ? 4u : (D == 32 ? 5u : 6u);
  constexpr unsigned kIdxMask = (1u << kIdxBits) - 1u;
  constexpr int VN = V16<R>::N;
  bool done = false;
  mypiv = R(1);
  pos = 0;
#pragma unroll
  for (int k = 0; k < D; ++k) {
    const unsigned key = done ? 0u : ((mag_key(aug[k]) & ~kIdxMask) | (unsigned)(D - 1 - li));
    const unsigned best = group_max_u32<D>(key);
    const bool me = (D - 1 - (int)(best & kIdxMask)) == li;
    if (me) {
#pragma unroll
      for (int c = (k & ~(VN - 1)); c < W; c += VN) V16<R>::st(prow + c, aug + c);
    }
    wave_sync();
    R pr[W];
#pragma unroll
    for (int c = (k & ~(VN - 1)); c < W; c += VN) V16<R>::ld(prow + c, pr + c);
    // rows already used as pivots keep their U row: only the remaining rows are eliminated
    const R f = (me || done) ? R(0) : aug[k] / pr[k];
#pragma unroll
    for (int c = k + 1; c < W; ++c) aug[c] = fma(-f, pr[c], aug[c]);
    if (me) { pos = k; done = true; }
    wave_sync();  // next pivot row may overwrite prow
  }
  // back substitution, last pivot first: x_k = (rhs_k - sum_{j>k} U_kj x_j) / U_kk
#pragma unroll
  for (int k = D - 1; k >= 0; --k) {
    if (pos == k) {
      const R iu = R(1) / aug[k];
#pragma unroll
      for (int c = D; c < W; ++c) aug[c] *= iu;
#pragma unroll
      for (int c = D; c < W; c += VN) V16<R>::st(prow + c, aug + c);
    }
    wave_sync();
    if (pos < k) {
      R x[W - D];
#pragma unroll
      for (int c = 0; c < W - D; c += VN) V16<R>::ld(prow + D + c, x + c);
      const R u = aug[k];  // U[pos][k]
#pragma unroll
      for (int c = 0; c < W - D; ++c) aug[D + c] = fma(-u, x[c], aug[D + c]);
    }
    wave_sync();
  }
}

// The pivoted solve of the row-layout kernels: LU in fp64, Gauss-Jordan in fp32.
template <int D, int W, typename R>
__device__ __forceinline__ void solve_rows(R (&aug)[W], int li, R* prow, R& mypiv, int& pos) {
  if constexpr (std::is_same<R, double>::value) lu_rows<D, W>(aug, li, prow, mypiv, pos);
  else gauss_jordan<D, W>(aug, li, prow, mypiv, pos);
}

// ---------------------------------------------------------------------------
// Row-layout Riccati sweep from step t_start down to 0: u0 and the stash of mode SM
// (STASH_NONE; STASH_GAINS: all gains K_t [P,T,du,d] into `kstash` and Quu_0; STASH_V1:
// V_1 [P,d,d] into `kstash` and Quu_0 -- the compact stash of the fast backward).
// R is the arithmetic type of the sweep (float, or double for long ill-conditioned
// horizons); inputs, u and the stash are fp32 in HBM.  The D lanes of a problem
// enter with V = V_{t_start+1} (lane li holds row li); Bs holds the problem's B
// (row stride Geo<D>::LDM) and S is the problem's Geo<D>::PER_PROB-element scratch.
// ---------------------------------------------------------------------------
template <int D, typename R, int SM, bool WRITE_U>
__device__ __forceinline__ void rpl_sweep(
    const float* __restrict__ A_diag, const float* __restrict__ Qg, const float* __restrict__ Rinv,
    const float* __restrict__ lgA, const float* __restrict__ lgB, const float* __restrict__ lgQ,
    const float* __restrict__ h0, const R* Bs, R* S, int li, int64_t p, bool valid, int64_t n, int T,
    int t_start, R (&V)[D], float* __restrict__ u_out, float* __restrict__ kstash,
    float* __restrict__ q0stash, int* __restrict__ status) {
  using G = Geo<D>;
  R* mat = S;
  R* vb = S + G::MAT;
  R* va = vb + D;
  R* vx = va + D;
  R* prow = vx + D;  // 2D elements

  const R a_i = A_diag[p * D + li];
  const R rr_i = R(1) / (R)Rinv[p * D + li];
  const R lgB_i = lgB[p * D + li];
  const R lgQ_i = lgQ[p * D + li];
  const R lgA_p = lgA[p];

  R Bcol[D], Qrow[D];
  {
    const float* qg = Qg + n * D * D;
#pragma unroll
    for (int c = 0; c < D; ++c) {
      Qrow[c] = R(0.5) * ((R)qg[li * D + c] + (R)qg[c * D + li]);
      Bcol[c] = Bs[c * G::LDM + li];
    }
  }

  for (int t = t_start; t >= 0; --t) {
    if (SM == STASH_V1 && t == 0 && valid) {
      float vrow[D];
#pragma unroll
      for (int c = 0; c < D; ++c) vrow[c] = (float)V[c];
      st_global_row<D>(kstash + (p * D + li) * D, vrow);
    }
    const R tp1 = (R)(t + 1);
    const R eA = exp(lgA_p * tp1);
    const R beta_i = exp(lgB_i * tp1);
    const R alpha_i = fma(a_i, eA, R(1));
    const R q_i = (t > 0) ? exp(lgQ_i * (R)t) : R(0);

    // W~ = V B (row li)
    R w[D];
#pragma unroll
    for (int k = 0; k < D; ++k) w[k] = R(0);
#pragma unroll
    for (int m = 0; m < D; ++m) {
      R brow[D];
      ld_row<D>(Bs + m * G::LDM, brow);
#pragma unroll
      for (int k = 0; k < D; ++k) w[k] = fma(V[m], brow[k], w[k]);
    }
    wave_sync();
    vb[li] = beta_i;
    va[li] = alpha_i;
    wave_sync();
    R beta[D], alpha[D];
    ld_row<D>(vb, beta);
    ld_row<D>(va, alpha);
#pragma unroll
    for (int k = 0; k < D; ++k) w[k] *= beta[k];  // W = V B_k
    st_row<D>(mat + li * G::LDM, w);
    wave_sync();

    // augmented row li: [Quu_li | Qux_li],  Quu = B_k'W + R,  Qux_lc = W_cl * alpha_c
    R aug[2 * D];
#pragma unroll
    for (int k = 0; k < D; ++k) aug[k] = R(0);
#pragma unroll
    for (int m = 0; m < D; ++m) {
      R wrow[D];
      ld_row<D>(mat + m * G::LDM, wrow);
#pragma unroll
      for (int k = 0; k < D; ++k) aug[k] = fma(Bcol[m], wrow[k], aug[k]);
    }
#pragma unroll
    for (int k = 0; k < D; ++k) aug[k] = aug[k] * beta_i + ((k == li) ? rr_i : R(0));
#pragma unroll
    for (int c = 0; c < D; ++c) aug[D + c] = mat[c * G::LDM + li] * alpha[c];
    if (SM != STASH_NONE && t == 0 && valid) {
      if constexpr (SM == STASH_GAINS && std::is_same<R, double>::value) {
        // the stable backward's adjoint solve w_0 = -Quu_0^{-1} d_u in the sweep's arithmetic
        R qrow[D];
#pragma unroll
        for (int k = 0; k < D; ++k) qrow[k] = aug[k];
        st_global_row<D>(reinterpret_cast<double*>(q0stash) + (p * D + li) * D, qrow);
      } else {
        float qrow[D];
#pragma unroll
        for (int k = 0; k < D; ++k) qrow[k] = (float)aug[k];
        st_global_row<D>(q0stash + (p * D + li) * D, qrow);
      }
    }

    R mypiv;
    int pos;
    solve_rows<D, 2 * D>(aug, li, prow, mypiv, pos);
    R x[D];  // row `pos` of X = Quu^{-1} Qux  (K = -X)
    const R ipiv = R(1) / mypiv;
#pragma unroll
    for (int c = 0; c < D; ++c) x[c] = aug[D + c] * ipiv;
    if (SM == STASH_GAINS && valid) {
      // gains in the sweep's arithmetic: on long horizons with expensive control |K|
      // reaches 1e19, and fp32-rounded gains make the closed-loop rollouts diverge
      R krow[D];
#pragma unroll
      for (int c = 0; c < D; ++c) krow[c] = -x[c];
      if constexpr (std::is_same<R, double>::value)
        st_global_row<D>(reinterpret_cast<double*>(kstash) + (((int64_t)p * T + t) * D + pos) * D, krow);
      else
        st_global_row<D>(kstash + (((int64_t)p * T + t) * D + pos) * D, krow);
    }
    if (t == 0) {
      // u0[pos] = K_0[pos,:] . h0
      R hv[D];
      wave_sync();
      vx[li] = (R)h0[p * D + li];
      wave_sync();
      ld_row<D>(vx, hv);
      R s = R(0);
#pragma unroll
      for (int c = 0; c < D; ++c) s = fma(x[c], hv[c], s);
      const float u0 = (float)(-s);
      if (WRITE_U && valid) u_out[p * D + pos] = u0;
      if (status != nullptr && valid && !isfinite(u0)) atomicOr(status, TTC_LQR_STATUS_NONFINITE);
      break;  // V_0 is not needed
    }
    // all lanes finished reading W during the elimination; publish X rows by position
    st_row<D>(mat + pos * G::LDM, x);
    wave_sync();
    // V <- alpha_i (alpha_m V_im - sum_j W_ij X_jm) + q_i q_m Q_im
    R acc[D];
#pragma unroll
    for (int m = 0; m < D; ++m) acc[m] = R(0);
#pragma unroll
    for (int j = 0; j < D; ++j) {
      R xrow[D];
      ld_row<D>(mat + j * G::LDM, xrow);
#pragma unroll
      for (int m = 0; m < D; ++m) acc[m] = fma(w[j], xrow[m], acc[m]);
    }
    R qv[D];
    vx[li] = q_i;
    wave_sync();
    ld_row<D>(vx, qv);
#pragma unroll
    for (int m = 0; m < D; ++m)
      V[m] = fma(alpha_i, fma(alpha[m], V[m], -acc[m]), (q_i * qv[m]) * Qrow[m]);
    // symmetrise: V_im = (V_im + V_mi) / 2
    wave_sync();
    st_row<D>(mat + li * G::LDM, V);
    wave_sync();
#pragma unroll
    for (int m = 0; m < D; ++m) V[m] = R(0.5) * (V[m] + mat[m * G::LDM + li]);
    wave_sync();
  }
}

// ---------------------------------------------------------------------------
// Forward kernel (row layout): stage B, V_T = sym(Q_f), full sweep.
// ---------------------------------------------------------------------------
template <int D, typename R, int SM, bool WRITE_U>
__global__ __launch_bounds__(Geo<D>::THREADS) void lqr_fwd_kernel(
    const float* __restrict__ A_diag, const float* __restrict__ Bg, const float* __restrict__ Qg,
    const float* __restrict__ Rinv, const float* __restrict__ Qf, const float* __restrict__ lgA,
    const float* __restrict__ lgB, const float* __restrict__ lgQ, const float* __restrict__ h0,
    int64_t P, int H, int T, int ntok_lds, float* __restrict__ u_out, float* __restrict__ kstash,
    float* __restrict__ q0stash, int* __restrict__ status) {
  using G = Geo<D>;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  R* smem = reinterpret_cast<R*>(smem_raw);
  const int li = threadIdx.x % D;
  const int pb = threadIdx.x / D;
  const int64_t p0 = (int64_t)blockIdx.x * G::PPB;
  int64_t p = p0 + pb;
  const bool valid = p < P;
  if (!valid) p = P - 1;  // idle lanes recompute a real problem, never store
  const int64_t n = p / H;
  const int64_t n0 = p0 / H;

  // stage the block's token-shared B matrices in LDS
  {
    const int64_t plast = (p0 + G::PPB - 1 < P) ? (p0 + G::PPB - 1) : (P - 1);
    const int ntok = (int)(plast / H - n0 + 1);
    for (int e = threadIdx.x; e < ntok * D * D; e += G::THREADS) {
      const int tk = e / (D * D), rem = e % (D * D);
      smem[(tk * D + rem / D) * G::LDM + rem % D] = (R)Bg[(n0 + tk) * D * D + rem];
    }
  }
  __syncthreads();
  const R* Bs = smem + (int)(n - n0) * G::MAT;
  R* S = smem + ntok_lds * G::MAT + pb * G::PER_PROB;

  R V[D];
  {
    const float* qf = Qf + p * D * D;
#pragma unroll
    for (int c = 0; c < D; ++c) V[c] = R(0.5) * ((R)qf[li * D + c] + (R)qf[c * D + li]);
  }
  rpl_sweep<D, R, SM, WRITE_U>(A_diag, Qg, Rinv, lgA, lgB, lgQ, h0, Bs, S, li, p, valid, n, T, T - 1, V,
                                  u_out, kstash, q0stash, status);
}

// ---------------------------------------------------------------------------
// Backward kernel: adjoint feed-forward, closed-loop rollouts of the primal and
// adjoint trajectories (forward in time, into `traj`), then the reverse costate
// sweep with all gradient accumulations.  grad_B / grad_Q are written per problem
// into gBp / gQp and summed over heads by headsum_kernel.
// ---------------------------------------------------------------------------
template <typename R> struct Traj4 { using type = float4; };
template <> struct Traj4<double> { using type = double4; };
template <typename R> __device__ __forceinline__ typename Traj4<R>::type mk4(R x, R y, R z, R w) {
  if constexpr (std::is_same<R, double>::value) return make_double4(x, y, z, w);
  else return make_float4(x, y, z, w);
}

template <int D>
__device__ __forceinline__ void flag_value(float v, float limit, int& flags) {
  if (!isfinite(v)) flags |= TTC_LQR_STATUS_NONFINITE;
  else if (fabsf(v) >= limit) flags |= TTC_LQR_STATUS_LARGE;
}
template <int D>
__device__ __forceinline__ void flag_value(double v, float limit, int& flags) {
  flag_value<D>((float)v, limit, flags);
}

// Steps whose gains the fp64 d = 16 kernel has in flight, phase 1 and 2.  Its bound is one wave's
// serial step (about 0.7 us for the two phases: 224 DPP multiply-adds, five library exponentials and
// the loads).  32 problems x 1,024 steps: 2.88 ms with the vectors broadcast through LDS by four
// waves of a workgroup, 2.36 with DPP, 1.52 with a wave per workgroup (its own CU's load port for the
// gains), 1.43 with 3 and 2 steps in flight, 1.51 with 4 and 3 (accumulator registers as spill space).
constexpr int kAhead1 = 3, kAhead2 = 2;

template <int D, typename R = float>
__global__ __launch_bounds__((BwdGeo<D, R>::THREADS)) void lqr_bwd_kernel(
    const float* __restrict__ A_diag, const float* __restrict__ Bg, const float* __restrict__ Qg,
    const float* __restrict__ Rinv, const float* __restrict__ Qf, const float* __restrict__ lgA,
    const float* __restrict__ lgB, const float* __restrict__ lgQ, const float* __restrict__ h0,
    const float* __restrict__ dU, const float* __restrict__ kstash, const float* __restrict__ q0stash,
    int64_t P, int H, int T, int ntok_lds, typename Traj4<R>::type* __restrict__ traj, float* __restrict__ gA,
    float* __restrict__ gRinv, float* __restrict__ gQf, float* __restrict__ glgA,
    float* __restrict__ glgB, float* __restrict__ glgQ, float* __restrict__ gh0,
    float* __restrict__ gBp, float* __restrict__ gQp, float grad_limit, int* __restrict__ status,
    const int32_t* __restrict__ gidx = nullptr, const double* __restrict__ gsl = nullptr,
    const double* __restrict__ q0sl = nullptr) {
  using G = BwdGeo<D, R>;
  extern __shared__ __align__(16) float smem_f[];
  R* const smem = reinterpret_cast<R*>(smem_f);
  const R* const kst = reinterpret_cast<const R*>(kstash);  // gains K_t in the forward sweep's type
  const int li = threadIdx.x % D;
  const int pb = threadIdx.x / D;
  const int64_t p0 = (int64_t)blockIdx.x * G::PPB;
  int64_t p = p0 + pb;
  const bool valid = p < P;
  if (!valid) p = P - 1;
  const int64_t n = p / H;
  const int64_t n0 = p0 / H;
  {
    const int64_t plast = (p0 + G::PPB - 1 < P) ? (p0 + G::PPB - 1) : (P - 1);
    const int ntok = (int)(plast / H - n0 + 1);
    for (int e = threadIdx.x; e < ntok * D * D; e += G::THREADS) {
      const int tk = e / (D * D), rem = e % (D * D);
      smem[(tk * D + rem / D) * G::LDM + rem % D] = Bg[(n0 + tk) * D * D + rem];
    }
  }
  __syncthreads();
  const R* Bs = smem + (int)(n - n0) * G::MAT;
  // this problem's gains [T][D][D] and Quu_0: the sweep's, or (fp64, gidx[p] >= 0) the forward
  // rescue's kept ones in slot gidx[p] (gains in gsl, Quu_0 after V_1 in q0sl)
  const R* kp = kst + (int64_t)p * T * D * D;
  const R* q0p = reinterpret_cast<const R*>(q0stash) + (int64_t)p * D * D;
  if constexpr (std::is_same<R, double>::value) {
    const int64_t k = gidx != nullptr ? (int64_t)gidx[p] : -1;
    if (k >= 0) {
      kp = gsl + k * T * D * D;
      q0p = q0sl + k * 2 * D * D + D * D;
    }
  }
  R* S = smem + ntok_lds * G::MAT + pb * G::PER_PROB;
  R* v0 = S + G::MAT;     // 8 vectors of D floats
  R* v1 = v0 + D;
  R* v2 = v1 + D;
  R* v3 = v2 + D;
  R* v4 = v3 + D;
  R* v5 = v4 + D;
  R* v6 = v5 + D;
  R* v7 = v6 + D;
  R* prow = v7 + D;       // D + 4 floats

  const R a_i = A_diag[p * D + li];
  const R rr_i = R(1) / Rinv[p * D + li];
  const R lgB_i = lgB[p * D + li];
  const R lgQ_i = lgQ[p * D + li];
  const R lgA_p = lgA[p];
  R Brow[D];
#pragma unroll
  for (int c = 0; c < D; ++c) Brow[c] = Bs[li * G::LDM + c];

  // adjoint feed-forward at t = 0: w0 = -Quu_0^{-1} d_u
  R w0_i;
  {
    R aug[D + 4];
    // Quu_0 as the forward sweep stored it (fp64 when it ran in fp64)
    ld_global_row<D>(q0p + li * D, *reinterpret_cast<R(*)[D]>(aug));
    aug[D] = dU[p * D + li];
    aug[D + 1] = aug[D + 2] = aug[D + 3] = R(0);
    R piv;
    int pos;
    solve_rows<D, D + 4>(aug, li, prow, piv, pos);
    v0[pos] = -aug[D] / piv;
    wave_sync();
    w0_i = v0[li];
    wave_sync();
  }

  // phase 1: rollouts, t = 0..T-1.  At d = 16 the gain rows are loaded ahead of their steps (in fp64 a
  // wave runs alone on its SIMD, so nothing else hides a load's latency): kAhead1 rows in flight in
  // fp64, one in fp32; at d = 32 / 64 the extra registers would spill.
  constexpr bool PF = D == 16;
  constexpr bool DPP = D == 16 && std::is_same<R, double>::value;  // products by DPP, not through LDS
  constexpr int A1 = DPP ? kAhead1 : 1, A2 = DPP ? kAhead2 : 1;
  R h_i = h0[p * D + li];
  R hb_i = R(0);
  R kn[A1][PF ? D : 1];
  if constexpr (PF) {
#pragma unroll
    for (int a = 0; a < A1; ++a) ld_global_row<D>(kp + ((int64_t)(a < T ? a : T - 1) * D + li) * D, kn[a]);
  }
  auto roll = [&](const int t, R(&next)[PF ? D : 1]) {
    const R tp1 = (R)(t + 1);
    const R alpha_i = fma(a_i, exp(lgA_p * tp1), R(1));
    const R beta_i = exp(lgB_i * tp1);
    R krow[D];
    if constexpr (PF) {
#pragma unroll
      for (int c = 0; c < D; ++c) krow[c] = next[c];
      if (t + A1 < T) ld_global_row<D>(kp + ((int64_t)(t + A1) * D + li) * D, next);
    }
    R u_i = R(0), w_i = (t == 0) ? w0_i : R(0);
    R hn = alpha_i * h_i, hbn = alpha_i * hb_i;
    if constexpr (DPP) {
      dpp_dot2(u_i, w_i, krow, h_i, hb_i);
      dpp_dot2(hn, hbn, Brow, beta_i * u_i, beta_i * w_i);
    } else {
      v0[li] = h_i;
      v1[li] = hb_i;
      wave_sync();
      R hv[D], hbv[D];
      ld_row<D>(v0, hv);
      ld_row<D>(v1, hbv);
      if constexpr (!PF) ld_global_row<D>(kp + ((int64_t)t * D + li) * D, krow);
#pragma unroll
      for (int c = 0; c < D; ++c) {
        u_i = fma(krow[c], hv[c], u_i);
        w_i = fma(krow[c], hbv[c], w_i);
      }
      v2[li] = beta_i * u_i;
      v3[li] = beta_i * w_i;
      wave_sync();
      R bu[D], bw[D];
      ld_row<D>(v2, bu);
      ld_row<D>(v3, bw);
#pragma unroll
      for (int j = 0; j < D; ++j) {
        hn = fma(Brow[j], bu[j], hn);
        hbn = fma(Brow[j], bw[j], hbn);
      }
    }
    if (valid) traj[((int64_t)p * T + t) * D + li] = mk4<R>(h_i, hb_i, u_i, w_i);
    h_i = hn;
    hb_i = hbn;
    if constexpr (!DPP) wave_sync();
  };
  for (int t0 = 0; t0 < T; t0 += A1) {
#pragma unroll
    for (int a = 0; a < A1; ++a)
      if (t0 + a < T) roll(t0 + a, kn[a]);  // uniform
  }

  R Bcol[D], Qrow[D];
  {
    const float* qg = Qg + n * D * D;
#pragma unroll
    for (int c = 0; c < D; ++c) {
      Bcol[c] = Bs[c * G::LDM + li];
      Qrow[c] = R(0.5) * (qg[li * D + c] + qg[c * D + li]);
    }
  }

  // phase 2: costates lambda_{t+1}, gradients, t = T-1..0
  int flags = 0;
  R lam_i, lamb_i;
  {
    v0[li] = h_i;
    v1[li] = hb_i;
    wave_sync();
    R hv[D], hbv[D], qf[D], gq[D];
    ld_row<D>(v0, hv);
    ld_row<D>(v1, hbv);
    const float* qfp = Qf + p * D * D;
    lam_i = R(0);
    lamb_i = R(0);
#pragma unroll
    for (int c = 0; c < D; ++c) {
      qf[c] = R(0.5) * (qfp[li * D + c] + qfp[c * D + li]);
      lam_i = fma(qf[c], hv[c], lam_i);
      lamb_i = fma(qf[c], hbv[c], lamb_i);
      gq[c] = R(0.5) * (h_i * hbv[c] + hb_i * hv[c]);
      flag_value<D>(gq[c], grad_limit, flags);
    }
    if (valid) st_global_row<D>(gQf + (p * D + li) * D, gq);
    wave_sync();
  }
  R gA_i = R(0), glgA_part = R(0), glgB_i = R(0), gr_i = R(0), glgQ_i = R(0), gh0_i = R(0);
  R gBrow[D], gQrow[D];
#pragma unroll
  for (int c = 0; c < D; ++c) { gBrow[c] = R(0); gQrow[c] = R(0); }

  // at d = 16 the steps' trajectory entries and gain columns are loaded ahead, as in phase 1
  typename Traj4<R>::type trn[A2];
  R kcn[A2][PF ? D : 1];
  if constexpr (PF) {
#pragma unroll
    for (int a = 0; a < A2; ++a) {
      const int64_t t = T - 1 - a > 0 ? T - 1 - a : 0;
      trn[a] = traj[((int64_t)p * T + t) * D + li];
#pragma unroll
      for (int c = 0; c < D; ++c) kcn[a][c] = kp[(t * D + c) * D + li];  // K_t[c, li]
    }
  }
  auto back = [&](const int t, typename Traj4<R>::type& trx, R(&next)[PF ? D : 1]) {
    const auto tr = PF ? trx : traj[((int64_t)p * T + t) * D + li];
    const R h_t = tr.x, hb_t = tr.y, u_i = tr.z, w_i = tr.w;
    R kcol[D];
    if constexpr (PF) {
#pragma unroll
      for (int c = 0; c < D; ++c) kcol[c] = next[c];
      if (t >= A2) {  // uniform
        trx = traj[((int64_t)p * T + (t - A2)) * D + li];
#pragma unroll
        for (int c = 0; c < D; ++c) next[c] = kp[((int64_t)(t - A2) * D + c) * D + li];
      }
    }
    const R tp1 = (R)(t + 1);
    const R eA = exp(lgA_p * tp1);
    const R alpha_i = fma(a_i, eA, R(1));
    const R beta_i = exp(lgB_i * tp1);
    // A: d/dA_t,i = h_t,i lamb_{t+1},i + hb_t,i lam_{t+1},i   (torch_lqr.py:51)
    const R gAt = fma(h_t, lamb_i, hb_t * lam_i);
    gA_i = fma(gAt, eA, gA_i);
    glgA_part = fma(gAt * a_i, tp1 * eA, glgA_part);
    // B: lamb u' + lam w' (torch_lqr.py:53), chained through B_t = B diag(beta_t)
    R btl = R(0), btlb = R(0);
    if constexpr (DPP) {
      dpp_dot2(btl, btlb, Bcol, lam_i, lamb_i);
      dpp_outer2(gBrow, beta_i * w_i, lam_i, beta_i * u_i, lamb_i);
    } else {
      v0[li] = lam_i;
      v1[li] = lamb_i;
      v2[li] = beta_i * u_i;
      v3[li] = beta_i * w_i;
      wave_sync();
      R lv[D], lbv[D], bu[D], bw[D];
      ld_row<D>(v0, lv);
      ld_row<D>(v1, lbv);
      ld_row<D>(v2, bu);
      ld_row<D>(v3, bw);
#pragma unroll
      for (int c = 0; c < D; ++c) {
        gBrow[c] = fma(lamb_i, bu[c], fma(lam_i, bw[c], gBrow[c]));
        btl = fma(Bcol[c], lv[c], btl);
        btlb = fma(Bcol[c], lbv[c], btlb);
      }
    }
    glgB_i = fma(tp1 * beta_i, fma(u_i, btlb, w_i * btl), glgB_i);
    // R = 1/R_inv:  d/dR_inv = -(u w) / R_inv^2   (torch_lqr.py:59)
    gr_i = fma(-u_i * w_i, rr_i * rr_i, gr_i);
    if (t >= 1) {
      const R q_i = exp(lgQ_i * (R)t);
      // closed-loop correction c = R u + B_t' lambda_{t+1}; Q_t = D_t Q D_t:  gradient
      // D_t sym(h hb') D_t  (torch_lqr.py:55)
      const R cu_i = fma(u_i, rr_i, beta_i * btl), cw_i = fma(w_i, rr_i, beta_i * btlb);
      R Qh = R(0), Qhb = R(0), kcu = R(0), kcw = R(0);
      if constexpr (DPP) {
        const R qh_i = q_i * h_t, qhb_i = q_i * hb_t;
        dpp_dot2(Qh, Qhb, Qrow, qh_i, qhb_i);
        dpp_dot2(kcu, kcw, kcol, cu_i, cw_i);
        dpp_outer2(gQrow, qh_i, R(0.5) * qhb_i, qhb_i, R(0.5) * qh_i);
      } else {
        v4[li] = q_i * h_t;
        v5[li] = q_i * hb_t;
        v6[li] = cu_i;
        v7[li] = cw_i;
        wave_sync();
        R qh[D], qhb[D], cu[D], cw[D];
        ld_row<D>(v4, qh);
        ld_row<D>(v5, qhb);
        ld_row<D>(v6, cu);
        ld_row<D>(v7, cw);
#pragma unroll
        for (int c = 0; c < D; ++c) {
          Qh = fma(Qrow[c], qh[c], Qh);
          Qhb = fma(Qrow[c], qhb[c], Qhb);
          gQrow[c] = fma(R(0.5) * q_i, fma(h_t, qhb[c], hb_t * qh[c]), gQrow[c]);
          const R kji = PF ? kcol[c] : kp[((int64_t)t * D + c) * D + li];  // K_t[c, li]
          kcu = fma(kji, cu[c], kcu);
          kcw = fma(kji, cw[c], kcw);
        }
      }
      Qh *= q_i;
      Qhb *= q_i;
      glgQ_i = fma((R)t, fma(h_t, Qhb, hb_t * Qh), glgQ_i);
      lam_i = Qh + fma(alpha_i, lam_i, kcu);
      lamb_i = Qhb + fma(alpha_i, lamb_i, kcw);
    } else {
      gh0_i = alpha_i * lamb_i;  // torch_lqr.py:61 (lambda_0 = A_0' lambda_1)
    }
    if constexpr (!DPP) wave_sync();
  };
  for (int t0 = T - 1; t0 >= 0; t0 -= A2) {
#pragma unroll
    for (int a = 0; a < A2; ++a)
      if (t0 - a >= 0) back(t0 - a, trn[a], kcn[a]);  // uniform
  }
  const R glgA_p = group_sum<D>(glgA_part, v0, li);
  // the reference's guard covers A_diag, B, Q, R_inv, Q_f and h0 (B and Q: the head sums,
  // checked by headsum_kernel), not the log-discounts
  flag_value<D>(gA_i, grad_limit, flags);
  flag_value<D>(gr_i, grad_limit, flags);
  flag_value<D>(gh0_i, grad_limit, flags);
  if (valid) {
    gA[p * D + li] = gA_i;
    gRinv[p * D + li] = gr_i;
    glgB[p * D + li] = glgB_i;
    glgQ[p * D + li] = glgQ_i;
    gh0[p * D + li] = gh0_i;
    if (li == 0) glgA[p] = glgA_p;
    st_global_row<D>(gBp + (p * D + li) * D, gBrow);
    st_global_row<D>(gQp + (p * D + li) * D, gQrow);
    if (flags && status != nullptr) atomicOr(status, flags);
  }
}

// exp2 and reciprocal in the rollout's arithmetic: the hardware instructions in fp32, the
// library functions in fp64.
__device__ __forceinline__ float exp2r(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ __forceinline__ double exp2r(double x) { return exp2(x); }
__device__ __forceinline__ float rcpr(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ double rcpr(double x) { return 1.0 / x; }

// ---------------------------------------------------------------------------
// Fast backward: forward Hamiltonian rollout with a terminal certificate.
//
// From V_1 and Quu_0 (the forward's compact stash) and the forward output u_0:
//   w_0 = -Quu_0^{-1} d_u,  h_1 = A_0 h_0 + B_0 u_0,  h~_1 = B_0 w_0,
//   lambda_1 = V_1 h_1,     lambda~_1 = V_1 h~_1,
// and for t = 1..T-1 the costate recursion of lin_solver_lqr.py:82-98 solved for
// lambda_{t+1}, with the stationarity condition R u_t + B_t' lambda_{t+1} = 0:
//   lambda_{t+1} = A_t^{-1} (lambda_t - Qc_t h_t),   u_t = -R^{-1} B_t' lambda_{t+1},
//   h_{t+1} = A_t h_t + B_t u_t                      (same for the adjoint, w_t).
// This is the reference's fused backward rollout (symplectic_iter.py:764-885):
// no per-step gains are needed and every gradient term of step t is formed when
// step t is rolled.  The recursion amplifies rounding along the unstable modes of
// the Hamiltonian map, so every problem carries a certificate: the terminal
// condition lambda_T = Q_f h_T must hold for both trajectories to relative
// accuracy `tau` (max-norm over the D entries, relative to |Q_f h_T| + |lambda_T|)
// and every gradient must be finite.  A problem that misses it writes nothing and is
// appended to fail_list (chunk-local index); the caller recomputes it with the
// stable path (stored gains, closed-loop costates).  grad_B / grad_Q partials go to
// gBp / gQp for headsum_kernel, as in lqr_bwd_kernel.
// LISTED == false: problems 0..P-1; LISTED: the P chunk-local problem indices plist[0..P-1] (the
// problems of head groups another rollout rejected).  fp64 and listed: a problem p with
// slot_of[p] >= 0 reads V_1 and Quu_0 in fp64 from slots[slot_of[p]] (256 doubles each, kept by
// the forward's fp64 rescue) instead of the fp32 v1s / q0s.  Every output, partial and fail_list
// entry is then at the listed problem's own index, and each problem reads its token's B
// from global memory instead of the block's LDS copy.
// ---------------------------------------------------------------------------
#ifndef TTC_HAM64_WAVES
#define TTC_HAM64_WAVES 2  // waves per SIMD of the fp64 rollout (registers capped; its loop keeps them all)
#endif
template <int D, typename R = float, bool LISTED = false>
__global__ __launch_bounds__((BwdGeo<D, R>::THREADS))
__attribute__((amdgpu_waves_per_eu(std::is_same<R, double>::value ? TTC_HAM64_WAVES : 1))) void lqr_ham_bwd_kernel(
    const float* __restrict__ A_diag, const float* __restrict__ Bg, const float* __restrict__ Qg,
    const float* __restrict__ Rinv, const float* __restrict__ Qf, const float* __restrict__ lgA,
    const float* __restrict__ lgB, const float* __restrict__ lgQ, const float* __restrict__ h0,
    const float* __restrict__ u0g, const float* __restrict__ dU, const float* __restrict__ v1s,
    const float* __restrict__ q0s, int64_t P, int H, int T, int ntok_lds, float tau, float* __restrict__ gA,
    float* __restrict__ gRinv, float* __restrict__ gQf, float* __restrict__ glgA, float* __restrict__ glgB,
    float* __restrict__ glgQ, float* __restrict__ gh0, float* __restrict__ gBp, float* __restrict__ gQp,
    float grad_limit, int* __restrict__ fail_list, int* __restrict__ fail_count, int* __restrict__ status,
    const int* __restrict__ plist, const int32_t* __restrict__ slot_of, const double* __restrict__ slots,
    int64_t nslot) {
  using G = BwdGeo<D, R>;
  extern __shared__ __align__(16) float smem_f[];
  R* const smem = reinterpret_cast<R*>(smem_f);
  const int li = threadIdx.x % D;
  const int pb = threadIdx.x / D;
  const int64_t p0 = (int64_t)blockIdx.x * G::PPB;
  const int64_t slot = p0 + pb;
  const bool valid = slot < P;
  // idle lanes recompute a real problem, never store
  int64_t p = valid ? slot : P - 1;
  if constexpr (LISTED) p = plist[p];
  const int64_t n = p / H;
  const int64_t n0 = p0 / H;
  if constexpr (!LISTED) {
    const int64_t plast = (p0 + G::PPB - 1 < P) ? (p0 + G::PPB - 1) : (P - 1);
    const int ntok = (int)(plast / H - n0 + 1);
    for (int e = threadIdx.x; e < ntok * D * D; e += G::THREADS) {
      const int tk = e / (D * D), rem = e % (D * D);
      smem[(tk * D + rem / D) * G::LDM + rem % D] = Bg[(n0 + tk) * D * D + rem];
    }
  }
  __syncthreads();
  R* S = smem + ntok_lds * G::MAT + pb * G::PER_PROB;
  R* v0 = S + G::MAT;  // 6 vectors of D floats, then the pivot row
  R* v1 = v0 + D;
  R* v2 = v1 + D;
  R* v3 = v2 + D;
  R* v4 = v3 + D;
  R* v5 = v4 + D;
  R* prow = v5 + D;    // D + 4 floats

  const R a_i = A_diag[p * D + li];
  const R r_i = Rinv[p * D + li];
  const R rr_i = R(1) / r_i;
  constexpr R kLog2e = R(1.4426950408889634);
  const R lgB_i = lgB[p * D + li];
  const R lgQ_i = lgQ[p * D + li];
  const R lgA_p = lgA[p];
  // discounts as exp2 of base-2 exponents, the arithmetic of the forward kernels
  const R lb2_i = lgB_i * kLog2e, lq2_i = lgQ_i * kLog2e, la2_p = lgA_p * kLog2e;
  R Brow[D], Bcol[D], Qrow[D];
  {
    const float* qg = Qg + n * D * D;
    if constexpr (!LISTED) {
      const R* Bs = smem + (int)(n - n0) * G::MAT;
#pragma unroll
      for (int c = 0; c < D; ++c) {
        Brow[c] = Bs[li * G::LDM + c];
        Bcol[c] = Bs[c * G::LDM + li];
      }
    } else {
      const float* bg = Bg + n * D * D;
#pragma unroll
      for (int c = 0; c < D; ++c) {
        Brow[c] = bg[li * D + c];
        Bcol[c] = bg[c * D + li];
      }
    }
#pragma unroll
    for (int c = 0; c < D; ++c) Qrow[c] = R(0.5) * (qg[li * D + c] + qg[c * D + li]);
  }

  // the forward's fp64 V_1 / Quu_0 of this problem, where it kept them
  int kslot = -1;
  if constexpr (LISTED && std::is_same<R, double>::value) {
    if (slot_of != nullptr) kslot = slot_of[p];
    if (kslot >= nslot) kslot = -1;  // an index beyond the slots is no slot (never read past them)
  }
  // t = 0: adjoint feed-forward w_0 = -Quu_0^{-1} d_u (pivoted elimination)
  R w_i;
  {
    R aug[D + 4];
    if constexpr (LISTED && std::is_same<R, double>::value) {
      if (kslot >= 0) ld_global_row<D>(slots + (int64_t)kslot * (2 * D * D) + D * D + li * D,
                                      *reinterpret_cast<R(*)[D]>(aug));
      else ld_global_row<D>(q0s + (p * D + li) * D, *reinterpret_cast<R(*)[D]>(aug));
    } else {
      ld_global_row<D>(q0s + (p * D + li) * D, *reinterpret_cast<R(*)[D]>(aug));
    }
    aug[D] = dU[p * D + li];
    aug[D + 1] = aug[D + 2] = aug[D + 3] = R(0);
    R piv;
    int pos;
    solve_rows<D, D + 4>(aug, li, prow, piv, pos);
    v0[pos] = -aug[D] / piv;
    wave_sync();
    w_i = v0[li];
    wave_sync();
  }

  R h_i = h0[p * D + li], hb_i = R(0), lam_i, lamb_i;
  R gA_i, glgA_part, glgB_i, gr_i, gh0_i, glgQ_i = R(0);
  R gBrow[D], gQrow[D];
  {
    const R u_i = u0g[p * D + li];
    const R eA = exp2r(la2_p);
    const R alpha_i = fma(a_i, eA, R(1));
    const R beta_i = exp2r(lb2_i);
    v2[li] = beta_i * u_i;
    v3[li] = beta_i * w_i;
    wave_sync();
    R bu[D], bw[D];
    ld_row<D>(v2, bu);
    ld_row<D>(v3, bw);
    R hn = alpha_i * h_i, hbn = R(0);
#pragma unroll
    for (int j = 0; j < D; ++j) {
      hn = fma(Brow[j], bu[j], hn);
      hbn = fma(Brow[j], bw[j], hbn);
    }
    v0[li] = hn;
    v1[li] = hbn;
    wave_sync();
    R hv[D], hbv[D], vrow[D];
    ld_row<D>(v0, hv);
    ld_row<D>(v1, hbv);
    if constexpr (LISTED && std::is_same<R, double>::value) {
      if (kslot >= 0) ld_global_row<D>(slots + (int64_t)kslot * (2 * D * D) + li * D, vrow);
      else ld_global_row<D>(v1s + (p * D + li) * D, vrow);
    } else {
      ld_global_row<D>(v1s + (p * D + li) * D, vrow);
    }
    R lam = R(0), lamb = R(0);
#pragma unroll
    for (int c = 0; c < D; ++c) {
      lam = fma(vrow[c], hv[c], lam);
      lamb = fma(vrow[c], hbv[c], lamb);
    }
    v4[li] = lam;
    v5[li] = lamb;
    wave_sync();
    R lv[D], lbv[D];
    ld_row<D>(v4, lv);
    ld_row<D>(v5, lbv);
    R btl = R(0), btlb = R(0);
#pragma unroll
    for (int c = 0; c < D; ++c) {
      gBrow[c] = fma(lamb, bu[c], lam * bw[c]);  // torch_lqr.py:53 chained through B_0 = B diag(beta_0)
      gQrow[c] = R(0);
      btl = fma(Bcol[c], lv[c], btl);
      btlb = fma(Bcol[c], lbv[c], btlb);
    }
    const R gAt = h_i * lamb;  // h~_0 = 0   (torch_lqr.py:51)
    gA_i = gAt * eA;
    glgA_part = gAt * a_i * eA;
    glgB_i = beta_i * fma(u_i, btlb, w_i * btl);
    gr_i = -u_i * w_i * rr_i * rr_i;  // d(1/R_inv)/dR_inv  (torch_lqr.py:59)
    gh0_i = alpha_i * lamb;           // torch_lqr.py:61
    h_i = hn;
    hb_i = hbn;
    lam_i = lam;
    lamb_i = lamb;
    wave_sync();
  }

  // products by DPP, not through LDS: 0.90 -> 0.60 ms for a short list's 1,024 steps
  constexpr bool DPP = D == 16 && std::is_same<R, double>::value;
  for (int t = 1; t < T; ++t) {
    const R tf = (R)t;
    // state cost on h_t:  Qc_t = D_t Q D_t,  D_t = diag(exp(lgQ t))   (torch_lqr.py:55 + chain rule)
    const R q_i = exp2r(lq2_i * tf);
    const R qh_i = q_i * h_i, qhb_i = q_i * hb_i;
    R Qh = R(0), Qhb = R(0);
    // with twice the symmetric gradient of Qc_t (halved after the loop)
    if constexpr (DPP) {
      dpp_dot2(Qh, Qhb, Qrow, qh_i, qhb_i);
      dpp_outer2(gQrow, qh_i, qhb_i, qhb_i, qh_i);
    } else {
      v0[li] = qh_i;
      v1[li] = qhb_i;
      wave_sync();
      R qh[D], qhb[D];
      ld_row<D>(v0, qh);
      ld_row<D>(v1, qhb);
#pragma unroll
      for (int c = 0; c < D; ++c) {
        Qh = fma(Qrow[c], qh[c], Qh);
        Qhb = fma(Qrow[c], qhb[c], Qhb);
        gQrow[c] = fma(qh_i, qhb[c], fma(qhb_i, qh[c], gQrow[c]));
      }
    }
    Qh *= q_i;
    Qhb *= q_i;
    glgQ_i = fma(tf, fma(h_i, Qhb, hb_i * Qh), glgQ_i);
    // step t dynamics
    const R tp1 = tf + R(1);
    const R eA = exp2r(la2_p * tp1);
    const R alpha_i = fma(a_i, eA, R(1));
    const R beta_i = exp2r(lb2_i * tp1);
    const R ia = rcpr(alpha_i);
    const R lam_n = (lam_i - Qh) * ia;
    const R lamb_n = (lamb_i - Qhb) * ia;
    R btl = R(0), btlb = R(0);
    if constexpr (DPP) {
      dpp_dot2(btl, btlb, Bcol, lam_n, lamb_n);
    } else {
      v2[li] = lam_n;
      v3[li] = lamb_n;
      wave_sync();
      R lv[D], lbv[D];
      ld_row<D>(v2, lv);
      ld_row<D>(v3, lbv);
#pragma unroll
      for (int c = 0; c < D; ++c) {
        btl = fma(Bcol[c], lv[c], btl);
        btlb = fma(Bcol[c], lbv[c], btlb);
      }
    }
    const R u_i = -r_i * beta_i * btl;
    const R w_i2 = -r_i * beta_i * btlb;
    R hn = alpha_i * h_i, hbn = alpha_i * hb_i;
    if constexpr (DPP) {
      const R bu_i = beta_i * u_i, bw_i = beta_i * w_i2;
      dpp_dot2(hn, hbn, Brow, bu_i, bw_i);
      dpp_outer2(gBrow, bw_i, lam_n, bu_i, lamb_n);
    } else {
      v4[li] = beta_i * u_i;
      v5[li] = beta_i * w_i2;
      wave_sync();
      R bu[D], bw[D];
      ld_row<D>(v4, bu);
      ld_row<D>(v5, bw);
#pragma unroll
      for (int j = 0; j < D; ++j) {
        hn = fma(Brow[j], bu[j], hn);
        hbn = fma(Brow[j], bw[j], hbn);
        gBrow[j] = fma(lamb_n, bu[j], fma(lam_n, bw[j], gBrow[j]));
      }
    }
    const R gAt = fma(h_i, lamb_n, hb_i * lam_n);
    gA_i = fma(gAt, eA, gA_i);
    glgA_part = fma(gAt * a_i, tp1 * eA, glgA_part);
    glgB_i = fma(tp1 * beta_i, fma(u_i, btlb, w_i2 * btl), glgB_i);
    gr_i = fma(-u_i * w_i2, rr_i * rr_i, gr_i);
    h_i = hn;
    hb_i = hbn;
    lam_i = lam_n;
    lamb_i = lamb_n;
    if constexpr (!DPP) wave_sync();
  }

#pragma unroll
  for (int c = 0; c < D; ++c) gQrow[c] *= R(0.5);

  // terminal cost: grad Q_f = sym(h_T h~_T'); certificate lambda_T = Q_f h_T
  R gq[D];
  R e1, e2, m1, m2, m3, m4;
  {
    v0[li] = h_i;
    v1[li] = hb_i;
    wave_sync();
    R hv[D], hbv[D];
    ld_row<D>(v0, hv);
    ld_row<D>(v1, hbv);
    const float* qfp = Qf + p * D * D;
    R fh = R(0), fhb = R(0);
#pragma unroll
    for (int c = 0; c < D; ++c) {
      const R qf = R(0.5) * (qfp[li * D + c] + qfp[c * D + li]);
      fh = fma(qf, hv[c], fh);
      fhb = fma(qf, hbv[c], fhb);
      gq[c] = R(0.5) * fma(h_i, hbv[c], hb_i * hv[c]);
    }
    e1 = fabs(lam_i - fh);
    e2 = fabs(lamb_i - fhb);
    m1 = fabs(fh) + fabs(lam_i);
    m2 = fabs(fhb) + fabs(lamb_i);
    wave_sync();
  }
  const R glgA_p = group_sum<D>(glgA_part, v0, li);
  // every accumulator finite <=> this sum is (a sum of finite values overflows only near 1e38)
  R fin = fabs(gA_i) + fabs(gr_i) + fabs(glgB_i) + fabs(glgQ_i) + fabs(gh0_i) + fabs(glgA_p);
#pragma unroll
  for (int c = 0; c < D; ++c) fin += fabs(gBrow[c]) + fabs(gQrow[c]) + fabs(gq[c]);
  // group maxima of non-negative floats via their bit patterns (NaN sorts above +inf)
  const float E1 = __uint_as_float(group_max_u32<D>(__float_as_uint((float)e1)));
  const float E2 = __uint_as_float(group_max_u32<D>(__float_as_uint((float)e2)));
  m3 = __uint_as_float(group_max_u32<D>(__float_as_uint((float)m1)));
  m4 = __uint_as_float(group_max_u32<D>(__float_as_uint((float)m2)));
  // finite as stored (fp32): an fp64 rollout can leave the fp32 range while staying finite
  const unsigned bad_lane = isfinite((float)fin) ? 0u : 1u;
  // magnitudes beyond the fp32 range fail: an fp64 trajectory can stay finite there while both
  // sides of the comparison round to +inf, and inf <= tau * inf would pass
  const bool ok = group_max_u32<D>(bad_lane) == 0u && E1 <= tau * m3 && E2 <= tau * m4 && isfinite(m3) &&
                  isfinite(m4);
  if (!valid) return;
  if (!ok) {
    if (li == 0) fail_list[atomicAdd(fail_count, 1)] = (int)p;
    return;
  }
  // the reference's guard covers A_diag, B, Q, R_inv, Q_f and h0 (B and Q: the head sums,
  // checked by headsum_kernel), not the log-discounts
  int flags = 0;
#pragma unroll
  for (int c = 0; c < D; ++c) flag_value<D>(gq[c], grad_limit, flags);
  flag_value<D>(gA_i, grad_limit, flags);
  flag_value<D>(gr_i, grad_limit, flags);
  flag_value<D>(gh0_i, grad_limit, flags);
  gA[p * D + li] = gA_i;
  gRinv[p * D + li] = gr_i;
  glgB[p * D + li] = glgB_i;
  glgQ[p * D + li] = glgQ_i;
  gh0[p * D + li] = gh0_i;
  if (li == 0) glgA[p] = glgA_p;
  st_global_row<D>(gQf + (p * D + li) * D, gq);
  st_global_row<D>(gBp + (p * D + li) * D, gBrow);
  st_global_row<D>(gQp + (p * D + li) * D, gQrow);
  if (flags && status != nullptr) atomicOr(status, flags);
}


// ---------------------------------------------------------------------------
// Rescue pass after a matrix-core forward: every problem whose marker is NaN (u[p][0],
// or Quu_0[p][0][0] in the stash when u is not written) is solved again from scratch
// with the row-layout sweep (pivoted Gauss-Jordan at every step).  The matrix-core
// kernels mark the problems whose Cholesky pivot broke down; a problem whose genuine
// result is NaN is recomputed too and keeps its NaN.  Each block of one wave walks the
// problems in strides of 64: one marker load per lane, a ballot, then PPW = 64 / D
// marked problems at a time (lane li of group qo owns row li of problem qo).  With a status
// word, the scan runs only when the forward set TTC_LQR_STATUS_RESCUED in it.
// ---------------------------------------------------------------------------
// One rescued problem per group of D lanes: stage its B, V_T = sym(Q_f), sweep from scratch.
template <int D, int SM, bool WRITE_U, typename R>
__device__ __forceinline__ void rescue_one(
    const float* __restrict__ A_diag, const float* __restrict__ Bg, const float* __restrict__ Qg,
    const float* __restrict__ Rinv, const float* __restrict__ Qf, const float* __restrict__ lgA,
    const float* __restrict__ lgB, const float* __restrict__ lgQ, const float* __restrict__ h0, int H, int T,
    float* __restrict__ u_out, float* __restrict__ kstash, float* __restrict__ q0stash, int* __restrict__ status,
    R* Bs, R* S, int li, int64_t p, bool valid) {
  const int64_t n = p / H;
  wave_sync();
#pragma unroll
  for (int c = 0; c < D; ++c) Bs[li * Geo<D>::LDM + c] = (R)Bg[n * D * D + li * D + c];
  R V[D];
  const float* qf = Qf + p * D * D;
#pragma unroll
  for (int c = 0; c < D; ++c) V[c] = R(0.5) * ((R)qf[li * D + c] + (R)qf[c * D + li]);
  wave_sync();
  rpl_sweep<D, R, SM, WRITE_U>(A_diag, Qg, Rinv, lgA, lgB, lgQ, h0, Bs, S, li, p, valid, n, T, T - 1, V, u_out,
                                kstash, q0stash, status);
}

template <int D, typename R = float>
struct Rescue {
  static constexpr int PPW = 64 / D;
  static constexpr int PER = Geo<D>::MAT + Geo<D>::PER_PROB;  // B rows + rpl_sweep scratch
  static constexpr size_t LDS_BYTES = sizeof(R) * (size_t)PPW * PER;
};

// R: the sweep's arithmetic (double after a long-horizon fp32 symplectic sweep, whose rejected
// problems are the ill-conditioned ones that need fp64)
template <int D, int SM, bool WRITE_U, typename R = float>
__global__ __launch_bounds__(64) void lqr_rescue_kernel(
    const float* __restrict__ A_diag, const float* __restrict__ Bg, const float* __restrict__ Qg,
    const float* __restrict__ Rinv, const float* __restrict__ Qf, const float* __restrict__ lgA,
    const float* __restrict__ lgB, const float* __restrict__ lgQ, const float* __restrict__ h0,
    int64_t P, int H, int T, float* __restrict__ u_out, float* __restrict__ kstash,
    float* __restrict__ q0stash, int* __restrict__ status) {
  constexpr int PPW = Rescue<D, R>::PPW;
  extern __shared__ __align__(16) float smem_rf[];
  R* const smem = reinterpret_cast<R*>(smem_rf);
  const int lane = threadIdx.x;
  const int qo = lane / D;
  const int li = lane % D;
  R* Bs = smem + qo * Rescue<D, R>::PER;
  R* S = Bs + Geo<D>::MAT;
  // nothing was marked (the forward sets the bit when it marks a problem)
  if (status != nullptr && !(__atomic_load_n(status, __ATOMIC_RELAXED) & TTC_LQR_STATUS_RESCUED)) return;
  const float* mark = WRITE_U ? u_out : q0stash;
  const int64_t mstride = WRITE_U ? D : (int64_t)D * D;
  for (int64_t base = (int64_t)blockIdx.x * 64; base < P; base += (int64_t)gridDim.x * 64) {
    const int64_t pl = base + lane;
    unsigned long long mask = __ballot(pl < P && isnan(mark[pl * mstride]));
    while (mask != 0ull) {
      // group qo takes the qo-th marked problem of the mask (if there is one)
      unsigned long long m = mask;
      for (int k = 0; k < qo && m != 0ull; ++k) m &= m - 1ull;
      const bool valid = m != 0ull;
      const int64_t p = base + (valid ? (__ffsll((long long)m) - 1) : (__ffsll((long long)mask) - 1));
      for (int k = 0; k < PPW && mask != 0ull; ++k) mask &= mask - 1ull;
      rescue_one<D, SM, WRITE_U, R>(A_diag, Bg, Qg, Rinv, Qf, lgA, lgB, lgQ, h0, H, T, u_out, kstash, q0stash,
                                    status, Bs, S, li, p, valid);
    }
  }
}

// The same rescue with one wave per group of PPW consecutive problems (a wave whose problems
// carry no marker returns at once): every marked problem's sweep runs concurrently.  For the
// fp64 sweeps after a long-horizon symplectic sweep, whose rejected problems cluster by token
// (a window of 64 could hold many, each window's sweeps running back to back).
template <int D, int SM, bool WRITE_U, typename R>
__global__ __launch_bounds__(64) void lqr_rescue_fine_kernel(
    const float* __restrict__ A_diag, const float* __restrict__ Bg, const float* __restrict__ Qg,
    const float* __restrict__ Rinv, const float* __restrict__ Qf, const float* __restrict__ lgA,
    const float* __restrict__ lgB, const float* __restrict__ lgQ, const float* __restrict__ h0,
    int64_t P, int H, int T, float* __restrict__ u_out, float* __restrict__ kstash,
    float* __restrict__ q0stash, int* __restrict__ status) {
  constexpr int PPW = Rescue<D, R>::PPW;
  extern __shared__ __align__(16) float smem_rf[];
  R* const smem = reinterpret_cast<R*>(smem_rf);
  const int lane = threadIdx.x;
  const int qo = lane / D;
  const int li = lane % D;
  R* Bs = smem + qo * Rescue<D, R>::PER;
  R* S = Bs + Geo<D>::MAT;
  if (status != nullptr && !(__atomic_load_n(status, __ATOMIC_RELAXED) & TTC_LQR_STATUS_RESCUED)) return;
  const float* mark = WRITE_U ? u_out : q0stash;
  const int64_t mstride = WRITE_U ? D : (int64_t)D * D;
  const int64_t base = (int64_t)blockIdx.x * PPW;
  const int64_t pq = base + qo;
  const bool valid = pq < P && isnan(mark[pq * mstride]);
  if (__ballot(valid) == 0ull) return;
  rescue_one<D, SM, WRITE_U, R>(A_diag, Bg, Qg, Rinv, Qf, lgA, lgB, lgQ, h0, H, T, u_out, kstash, q0stash, status,
                                Bs, S, li, valid ? pq : base, valid);
}

// The fp64 rescue with a workspace (ttc_lqr_forward_ws): the marked problems are listed first,
// then a grid of one wave per SIMD takes them PPW at a time, so that every sweep it runs is
// full (the clustered or sparse markers leave most groups of PPW consecutive problems
// part-filled).  The list's order is whatever the atomics give; each problem is solved on its
// own, so the results do not depend on it.  Workspace: [0] the count, [64..] the list.
static __global__ void rescue_list_reset_kernel(int32_t* __restrict__ ws) { ws[0] = 0; }

static __global__ __launch_bounds__(256) void rescue_list_kernel(int64_t P, const float* __restrict__ mark, int64_t mstride,
                                                          int32_t* __restrict__ ws, const int* __restrict__ status) {
  if (status != nullptr && !(__atomic_load_n(status, __ATOMIC_RELAXED) & TTC_LQR_STATUS_RESCUED)) return;
  const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const bool m = p < P && isnan(mark[p * mstride]);
  const unsigned long long b = __ballot(m);
  if (b == 0ull) return;  // uniform over the wave
  const int lane = threadIdx.x & 63;
  int base = 0;
  if (lane == 0) base = atomicAdd(ws, (int)__popcll(b));
  base = __shfl(base, 0, 64);
  if (m) ws[64 + base + (int)__popcll(b & ((1ull << lane) - 1ull))] = (int32_t)p;
}

template <int D, int SM, bool WRITE_U, typename R>
__global__ __launch_bounds__(64) void lqr_rescue_listed_kernel(
    const float* __restrict__ A_diag, const float* __restrict__ Bg, const float* __restrict__ Qg,
    const float* __restrict__ Rinv, const float* __restrict__ Qf, const float* __restrict__ lgA,
    const float* __restrict__ lgB, const float* __restrict__ lgQ, const float* __restrict__ h0,
    int H, int T, float* __restrict__ u_out, float* __restrict__ kstash, float* __restrict__ q0stash,
    int* __restrict__ status, const int32_t* __restrict__ ws) {
  constexpr int PPW = Rescue<D, R>::PPW;
  extern __shared__ __align__(16) float smem_rf[];
  R* const smem = reinterpret_cast<R*>(smem_rf);
  const int lane = threadIdx.x;
  const int qo = lane / D;
  const int li = lane % D;
  R* Bs = smem + qo * Rescue<D, R>::PER;
  R* S = Bs + Geo<D>::MAT;
  if (status != nullptr && !(__atomic_load_n(status, __ATOMIC_RELAXED) & TTC_LQR_STATUS_RESCUED)) return;
  const int64_t n = __builtin_amdgcn_readfirstlane(ws[0]);
  const int32_t* list = ws + 64;
  for (int64_t b0 = (int64_t)blockIdx.x * PPW; b0 < n; b0 += (int64_t)gridDim.x * PPW) {
    const int64_t k = b0 + qo;
    const bool valid = k < n;
    const int64_t p = list[valid ? k : b0];
    rescue_one<D, SM, WRITE_U, R>(A_diag, Bg, Qg, Rinv, Qf, lgA, lgB, lgQ, h0, H, T, u_out, kstash, q0stash, status,
                                  Bs, S, li, p, valid);
  }
}

// CUs of the current device (0 if unknown).
inline int device_cus() {
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
    return 0;
  return cus;
}

template <int D, int SM, bool WU, typename RT = float>
inline void launch_rescue_k(const float* A, const float* B, const float* Q, const float* R, const float* Qf,
                            const float* lA, const float* lB, const float* lQ, const float* h0, int64_t P, int H,
                            int T, float* u, float* st_a, float* st_b, int32_t* status, hipStream_t s,
                            int32_t* rescue_ws = nullptr) {
  const int cus = (std::is_same<RT, double>::value && rescue_ws != nullptr) ? device_cus() : 0;
  if (cus > 0 && P < ((int64_t)1 << 31)) {
    const float* mark = WU ? u : st_b;
    const int64_t mstride = WU ? D : (int64_t)D * D;
    hipLaunchKernelGGL(rescue_list_reset_kernel, dim3(1), dim3(1), 0, s, rescue_ws);
    hipLaunchKernelGGL(rescue_list_kernel, dim3((unsigned)((P + 255) / 256)), dim3(256), 0, s, P, mark, mstride,
                       rescue_ws, status);
    hipLaunchKernelGGL((lqr_rescue_listed_kernel<D, SM, WU, RT>), dim3((unsigned)(4 * cus)), dim3(64),
                       (Rescue<D, RT>::LDS_BYTES), s, A, B, Q, R, Qf, lA, lB, lQ, h0, H, T, u, st_a, st_b, status,
                       rescue_ws);
    return;
  }
  if (std::is_same<RT, double>::value) {
    const int64_t blocks = (P + Rescue<D, RT>::PPW - 1) / Rescue<D, RT>::PPW;
    hipLaunchKernelGGL((lqr_rescue_fine_kernel<D, SM, WU, RT>), dim3((unsigned)blocks), dim3(64),
                       (Rescue<D, RT>::LDS_BYTES), s, A, B, Q, R, Qf, lA, lB, lQ, h0, P, H, T, u, st_a, st_b, status);
    return;
  }
  int64_t blocks = (P + 63) / 64;
  if (blocks > 4096) blocks = 4096;
  hipLaunchKernelGGL((lqr_rescue_kernel<D, SM, WU, RT>), dim3((unsigned)blocks), dim3(64), (Rescue<D, RT>::LDS_BYTES),
                     s, A, B, Q, R, Qf, lA, lB, lQ, h0, P, H, T, u, st_a, st_b, status);
}

// ---------------------------------------------------------------------------
// launch helpers (instantiated per D in ttc_lqr_d*.hip)
// ---------------------------------------------------------------------------
template <typename G>
inline int ntok_lds_for(int H) {
  constexpr int PPB = G::PPB;
  const int span = (PPB - 1) / H + 2;
  return span < PPB ? span : PPB;
}

template <typename G>
inline size_t lds_bytes(int H, size_t elem = sizeof(float)) {
  return elem * ((size_t)ntok_lds_for<G>(H) * G::MAT + (size_t)G::PPB * G::PER_PROB);
}

template <int D, typename RT, int SM, bool WU>
inline void launch_fwd_k(const float* A, const float* B, const float* Q, const float* R, const float* Qf,
                         const float* lA, const float* lB, const float* lQ, const float* h0, int64_t P, int H,
                         int T, float* u, float* st_a, float* st_b, int32_t* status, hipStream_t s) {
  const dim3 grid((unsigned)((P + Geo<D>::PPB - 1) / Geo<D>::PPB)), block(Geo<D>::THREADS);
  hipLaunchKernelGGL((lqr_fwd_kernel<D, RT, SM, WU>), grid, block, lds_bytes<Geo<D>>(H, sizeof(RT)), s, A, B, Q, R, Qf,
                     lA, lB, lQ, h0, P, H, T, ntok_lds_for<Geo<D>>(H), u, st_a, st_b, status);
}

// Forward launch by stash mode: sm = STASH_NONE (u), STASH_GAINS (gains + Quu_0 into
// st_a / st_b, no u) or STASH_V1 (V_1 + Quu_0 into st_a / st_b, u when u != nullptr).
template <int D, typename RT>
inline int launch_fwd_t(const float* A, const float* B, const float* Q, const float* R, const float* Qf,
                        const float* lA, const float* lB, const float* lQ, const float* h0, int64_t P, int H,
                        int T, float* u, float* st_a, float* st_b, int sm, int32_t* status, hipStream_t s) {
  switch (sm) {
    case STASH_NONE:
      launch_fwd_k<D, RT, STASH_NONE, true>(A, B, Q, R, Qf, lA, lB, lQ, h0, P, H, T, u, st_a, st_b, status, s);
      break;
    case STASH_GAINS:
      launch_fwd_k<D, RT, STASH_GAINS, false>(A, B, Q, R, Qf, lA, lB, lQ, h0, P, H, T, u, st_a, st_b, status, s);
      break;
    case STASH_V1:
      if (u != nullptr)
        launch_fwd_k<D, RT, STASH_V1, true>(A, B, Q, R, Qf, lA, lB, lQ, h0, P, H, T, u, st_a, st_b, status, s);
      else
        launch_fwd_k<D, RT, STASH_V1, false>(A, B, Q, R, Qf, lA, lB, lQ, h0, P, H, T, u, st_a, st_b, status, s);
      break;
    default:
      return TTC_LQR_EINVAL;
  }
  return TTC_LQR_OK;
}

template <int D, bool HAS_FP64>
inline int launch_fwd(const float* A, const float* B, const float* Q, const float* R, const float* Qf,
                      const float* lA, const float* lB, const float* lQ, const float* h0, int64_t P, int H,
                      int T, float* u, float* st_a, float* st_b, int sm, int32_t* status, hipStream_t s, int flags) {
  if (P <= 0) return TTC_LQR_OK;
  int rc;
  if (flags & TTC_LQR_FLAG_FP64_RICCATI) {
    if constexpr (HAS_FP64)
      rc = launch_fwd_t<D, double>(A, B, Q, R, Qf, lA, lB, lQ, h0, P, H, T, u, st_a, st_b, sm, status, s);
    else
      return TTC_LQR_EUNSUPPORTED;
  } else {
    rc = launch_fwd_t<D, float>(A, B, Q, R, Qf, lA, lB, lQ, h0, P, H, T, u, st_a, st_b, sm, status, s);
  }
  if (rc != TTC_LQR_OK) return rc;
  return hipGetLastError() == hipSuccess ? TTC_LQR_OK : TTC_LQR_ELAUNCH;
}

template <int D, typename RT = float>
inline int launch_ham(const float* A, const float* B, const float* Q, const float* R, const float* Qf,
                      const float* lA, const float* lB, const float* lQ, const float* h0, const float* u0,
                      const float* dU, const float* v1s, const float* q0s, int64_t P, int H, int T, float tau,
                      float* gA, float* gR, float* gQf, float* glA, float* glB, float* glQ, float* gh0, float* gBp,
                      float* gQp, float limit, int32_t* fail_list, int32_t* fail_count, int32_t* status,
                      hipStream_t s, const int32_t* plist = nullptr, const int32_t* slot_of = nullptr,
                      const double* slots = nullptr, int64_t nslot = 0) {
  if (P <= 0) return TTC_LQR_OK;
  using G = BwdGeo<D, RT>;
  const dim3 grid((unsigned)((P + G::PPB - 1) / G::PPB)), block(G::THREADS);
  if (plist != nullptr)
    hipLaunchKernelGGL((lqr_ham_bwd_kernel<D, RT, true>), grid, block, lds_bytes<G>(H, sizeof(RT)), s, A, B, Q, R, Qf,
                       lA, lB, lQ, h0, u0, dU, v1s, q0s, P, H, T, ntok_lds_for<G>(H), tau, gA, gR, gQf, glA, glB, glQ,
                       gh0, gBp, gQp, limit, fail_list, fail_count, status, plist, slot_of, slots, nslot);
  else
    hipLaunchKernelGGL((lqr_ham_bwd_kernel<D, RT, false>), grid, block, lds_bytes<G>(H, sizeof(RT)), s, A, B, Q, R,
                       Qf, lA, lB, lQ, h0, u0, dU, v1s, q0s, P, H, T, ntok_lds_for<G>(H), tau, gA, gR, gQf, glA, glB,
                       glQ, gh0, gBp, gQp, limit, fail_list, fail_count, status, plist, nullptr, nullptr,
                       (int64_t)0);
  return hipGetLastError() == hipSuccess ? TTC_LQR_OK : TTC_LQR_ELAUNCH;
}

template <int D, typename RT = float>
inline int launch_bwd(const float* A, const float* B, const float* Q, const float* R, const float* Qf,
                      const float* lA, const float* lB, const float* lQ, const float* h0, const float* dU,
                      const float* kst, const float* q0s, int64_t P, int H, int T,
                      typename Traj4<RT>::type* traj, float* gA,
                      float* gR, float* gQf, float* glA, float* glB, float* glQ, float* gh0, float* gBp,
                      float* gQp, float limit, int32_t* status, hipStream_t s, const int32_t* gidx = nullptr,
                      const double* gsl = nullptr, const double* q0sl = nullptr) {
  if (P <= 0) return TTC_LQR_OK;
  using G = BwdGeo<D, RT>;
  const dim3 grid((unsigned)((P + G::PPB - 1) / G::PPB)), block(G::THREADS);
  hipLaunchKernelGGL((lqr_bwd_kernel<D, RT>), grid, block, lds_bytes<G>(H, sizeof(RT)), s, A, B, Q, R, Qf, lA, lB,
                     lQ, h0, dU,
                     kst, q0s, P, H, T, ntok_lds_for<G>(H), traj, gA, gR, gQf, glA, glB, glQ, gh0, gBp, gQp,
                     limit, status, gidx, gsl, q0sl);
  return hipGetLastError() == hipSuccess ? TTC_LQR_OK : TTC_LQR_ELAUNCH;
}

}  // namespace ttc
