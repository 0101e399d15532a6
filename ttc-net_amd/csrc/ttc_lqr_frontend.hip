// ttc_lqr_frontend.hip -- the layer's front-end between in_proj and the solver
// (ttc/layers/ttc_layer.py:110-135), forward and backward: one pass over the projection's rows
//   [head 0: h0 d | A d | R du | coeff_Qf rq | log_gammas 1 + du + d] ... [coeff_B rb | coeff_Q rq]
// that splits, normalises and writes the solver's inputs contiguously:
//   A = l2norm, R = max(l2norm(softplus), 1e-6), coeff_Qf / coeff_Q = l2norm(softplus),
//   coeff_B = l2norm, log_gammas = -softplus - relu(-bias),
// with l2norm(x) = x / sqrt(sum(x^2) + 1e-6) and torch's softplus (the identity above 20).
//
// Bound: launches.  As torch operators this is 35 kernels of 1.5-6 us forward and about 70
// backward (elementwise, one reduction per norm, a copy per strided output), which at 32 tokens is
// most of a decode step (160 us of kernels, 520 us with their dispatch) and at 2,048 tokens half of
// a training step; here it is one kernel each way.  One wave per (token, head) and one for the
// token's shared coefficients: a row's segments are read coalesced, their sums of squares reduced in
// the wave.  Large calls are not bound by memory either: 51 MB in 48 us (1,021 tokens of 32 heads, d =
// 32), 1.1 TB/s -- at d = 16 a segment fills 16 of the 64 lanes, the five norms' reductions depend on
// shuffles one after the other, and each softplus is evaluated again when its value is written.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "ttc_frontend.h"
#include "ttc_lqr.h"

namespace ttc {

struct FrontDims {
  int H, d, du, rb, rq;
  __host__ __device__ int head() const { return 3 * d + 2 * du + rq + 1; }
  __host__ __device__ int64_t row() const { return (int64_t)head() * H + rb + rq; }
};

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m, 64);
  return v;
}

__device__ __forceinline__ float softplus(float x) { return x > 20.0f ? x : log1pf(expf(x)); }

// d softplus(x) / dx
__device__ __forceinline__ float dsoftplus(float x) {
  if (x > 20.0f) return 1.0f;
  const float z = expf(x);
  return z / (z + 1.0f);
}

// dst = l2norm(f(src)) over n values, f the identity or softplus; CLAMP: at least 1e-6 (NaN kept)
template <bool SP, bool CLAMP>
__device__ __forceinline__ void norm_segment(const float* __restrict__ src, int n, int lane, float* __restrict__ dst) {
  float ss = 0.f;
  for (int i = lane; i < n; i += 64) {
    const float v = SP ? softplus(src[i]) : src[i];
    ss = fmaf(v, v, ss);
  }
  const float s = rsqrtf(wave_sum(ss) + 1e-6f);
  for (int i = lane; i < n; i += 64) {
    const float y = (SP ? softplus(src[i]) : src[i]) * s;
    dst[i] = (CLAMP && y < 1e-6f) ? 1e-6f : y;
  }
}

// its chain rule: dsrc from src and the gradient g of dst (nullptr: zero)
template <bool SP, bool CLAMP>
__device__ __forceinline__ void norm_segment_backward(const float* __restrict__ src, const float* __restrict__ g, int n,
                                                      int lane, float* __restrict__ dsrc) {
  if (g == nullptr) {
    for (int i = lane; i < n; i += 64) dsrc[i] = 0.f;
    return;
  }
  float ss = 0.f;
  for (int i = lane; i < n; i += 64) {
    const float v = SP ? softplus(src[i]) : src[i];
    ss = fmaf(v, v, ss);
  }
  const float s = rsqrtf(wave_sum(ss) + 1e-6f);
  auto grad = [&](int i, float v) { return (CLAMP && !(v * s >= 1e-6f)) ? 0.f : g[i]; };
  float vg = 0.f;
  for (int i = lane; i < n; i += 64) {
    const float v = SP ? softplus(src[i]) : src[i];
    vg = fmaf(v, grad(i, v), vg);
  }
  const float k = wave_sum(vg) * s * s * s;
  for (int i = lane; i < n; i += 64) {
    const float x = src[i], v = SP ? softplus(x) : x;
    const float dv = fmaf(s, grad(i, v), -v * k);
    dsrc[i] = SP ? dv * dsoftplus(x) : dv;
  }
}

__global__ __launch_bounds__(256) void front_end_kernel(const float* __restrict__ proj, const float* __restrict__ bias,
                                                        int64_t N, int64_t first, FrontDims D, float* __restrict__ A,
                                                        float* __restrict__ cB, float* __restrict__ cQ,
                                                        float* __restrict__ R, float* __restrict__ cQf,
                                                        float* __restrict__ lA, float* __restrict__ lB,
                                                        float* __restrict__ lQ, float* __restrict__ h0) {
  const int lane = threadIdx.x & 63;
  const int64_t unit = first + (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int64_t n = unit / (D.H + 1);
  if (n >= N) return;
  const int h = (int)(unit % (D.H + 1));
  const float* row = proj + n * D.row() + (int64_t)h * D.head();
  if (h == D.H) {  // the token's shared coefficients
    norm_segment<false, false>(row, D.rb, lane, cB + n * D.rb);
    norm_segment<true, false>(row + D.rb, D.rq, lane, cQ + n * D.rq);
    return;
  }
  const int64_t p = n * D.H + h;
  for (int i = lane; i < D.d; i += 64) h0[p * D.d + i] = row[i];
  row += D.d;
  norm_segment<false, false>(row, D.d, lane, A + p * D.d);
  row += D.d;
  norm_segment<true, true>(row, D.du, lane, R + p * D.du);
  row += D.du;
  norm_segment<true, false>(row, D.rq, lane, cQf + p * D.rq);
  row += D.rq;
  for (int i = lane; i < 1 + D.du + D.d; i += 64) {
    float v = -softplus(row[i]);
    if (bias != nullptr) {  // relu that keeps NaN, as torch's does (fmaxf(NaN, 0) is 0)
      const float m = -bias[i];
      v -= m < 0.f ? 0.f : m;
    }
    if (i == 0) lA[p] = v;
    else if (i <= D.du) lB[p * D.du + i - 1] = v;
    else lQ[p * D.d + i - 1 - D.du] = v;
  }
}

__global__ __launch_bounds__(256) void front_end_backward_kernel(
    const float* __restrict__ proj, int64_t N, int64_t first, FrontDims D, const float* __restrict__ gA,
    const float* __restrict__ gcB, const float* __restrict__ gcQ, const float* __restrict__ gR,
    const float* __restrict__ gcQf, const float* __restrict__ glA, const float* __restrict__ glB,
    const float* __restrict__ glQ, const float* __restrict__ gh0, float* __restrict__ dproj) {
  const int lane = threadIdx.x & 63;
  const int64_t unit = first + (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int64_t n = unit / (D.H + 1);
  if (n >= N) return;
  const int h = (int)(unit % (D.H + 1));
  const int64_t at = n * D.row() + (int64_t)h * D.head();
  const float* row = proj + at;
  float* out = dproj + at;
  auto seg = [](const float* g, int64_t k) { return g == nullptr ? nullptr : g + k; };
  if (h == D.H) {
    norm_segment_backward<false, false>(row, seg(gcB, n * D.rb), D.rb, lane, out);
    norm_segment_backward<true, false>(row + D.rb, seg(gcQ, n * D.rq), D.rq, lane, out + D.rb);
    return;
  }
  const int64_t p = n * D.H + h;
  for (int i = lane; i < D.d; i += 64) out[i] = gh0 == nullptr ? 0.f : gh0[p * D.d + i];
  row += D.d, out += D.d;
  norm_segment_backward<false, false>(row, seg(gA, p * D.d), D.d, lane, out);
  row += D.d, out += D.d;
  norm_segment_backward<true, true>(row, seg(gR, p * D.du), D.du, lane, out);
  row += D.du, out += D.du;
  norm_segment_backward<true, false>(row, seg(gcQf, p * D.rq), D.rq, lane, out);
  row += D.rq, out += D.rq;
  for (int i = lane; i < 1 + D.du + D.d; i += 64) {
    const float* g = i == 0 ? seg(glA, p) : i <= D.du ? seg(glB, p * D.du + i - 1) : seg(glQ, p * D.d + i - 1 - D.du);
    out[i] = g == nullptr ? 0.f : -g[0] * dsoftplus(row[i]);
  }
}

// A launch takes at most 2^32 - 1 threads: units (one wave each) beyond that go in further launches.
constexpr int64_t kFrontUnits = 4 * (((int64_t)1 << 24) - 1);

// Any sizes whose element offsets fit 64 bits.
static bool front_args_ok(int64_t n, int64_t H, int64_t d, int64_t du, int64_t rb, int64_t rq) {
  if (n < 0 || H < 1 || d < 0 || du < 0 || rb < 0 || rq < 0) return false;
  constexpr int64_t lim = (int64_t)1 << 31;
  const int64_t head = 3 * d + 2 * du + rq + 1;
  if (H + 1 >= lim || head >= lim || rb + rq >= lim) return false;
  return n <= ((int64_t)1 << 62) / (head * H + rb + rq);
}

static bool given(const void* p, int64_t elements) { return elements == 0 || p != nullptr; }

template <typename F>
static int front_launches(int64_t units, F&& launch) {
  for (int64_t first = 0; first < units; first += kFrontUnits) {
    const int64_t left = units - first, now = left < kFrontUnits ? left : kFrontUnits;
    launch(first, dim3((unsigned)((now + 3) / 4)));
    if (hipGetLastError() != hipSuccess) return TTC_LQR_ELAUNCH;
  }
  return TTC_LQR_OK;
}

}  // namespace ttc

using namespace ttc;

extern "C" {

int ttc_lqr_front_end(const float* proj, const float* gamma_bias, int64_t n_tokens, int32_t heads, int32_t d,
                      int32_t du, int32_t b_rank, int32_t q_rank, float* A_diag, float* coeff_B, float* coeff_Q,
                      float* R_inv, float* coeff_Qf, float* log_gamma_A, float* log_gamma_B, float* log_gamma_Q,
                      float* h0, void* stream) {
  if (!front_args_ok(n_tokens, heads, d, du, b_rank, q_rank)) return TTC_LQR_EINVAL;
  if (n_tokens == 0) return TTC_LQR_OK;
  if (!proj || !given(A_diag, d) || !given(coeff_B, b_rank) || !given(coeff_Q, q_rank) || !given(R_inv, du) ||
      !given(coeff_Qf, q_rank) || !log_gamma_A || !given(log_gamma_B, du) || !given(log_gamma_Q, d) || !given(h0, d))
    return TTC_LQR_EINVAL;
  return front_launches(n_tokens * ((int64_t)heads + 1), [&](int64_t first, dim3 grid) {
    hipLaunchKernelGGL(front_end_kernel, grid, dim3(256), 0, reinterpret_cast<hipStream_t>(stream), proj, gamma_bias,
                       n_tokens, first, FrontDims{heads, d, du, b_rank, q_rank}, A_diag, coeff_B, coeff_Q, R_inv,
                       coeff_Qf, log_gamma_A, log_gamma_B, log_gamma_Q, h0);
  });
}

int ttc_lqr_front_end_backward(const float* proj, int64_t n_tokens, int32_t heads, int32_t d, int32_t du,
                               int32_t b_rank, int32_t q_rank, const float* grad_A_diag, const float* grad_coeff_B,
                               const float* grad_coeff_Q, const float* grad_R_inv, const float* grad_coeff_Qf,
                               const float* grad_log_gamma_A, const float* grad_log_gamma_B,
                               const float* grad_log_gamma_Q, const float* grad_h0, float* grad_proj, void* stream) {
  if (!front_args_ok(n_tokens, heads, d, du, b_rank, q_rank)) return TTC_LQR_EINVAL;
  if (n_tokens == 0) return TTC_LQR_OK;
  if (!proj || !grad_proj) return TTC_LQR_EINVAL;
  return front_launches(n_tokens * ((int64_t)heads + 1), [&](int64_t first, dim3 grid) {
    hipLaunchKernelGGL(front_end_backward_kernel, grid, dim3(256), 0, reinterpret_cast<hipStream_t>(stream), proj,
                       n_tokens, first, FrontDims{heads, d, du, b_rank, q_rank}, grad_A_diag, grad_coeff_B,
                       grad_coeff_Q, grad_R_inv, grad_coeff_Qf, grad_log_gamma_A, grad_log_gamma_B, grad_log_gamma_Q,
                       grad_h0, grad_proj);
  });
}

}  // extern "C"
