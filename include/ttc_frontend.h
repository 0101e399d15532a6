/* ttc_frontend.h -- C ABI of libttc_lqr.so around the solver: the layer's front-end and the padding of
 * the solver's tensors (status codes: ttc_lqr.h).  Device pointers, contiguous arrays; work is enqueued
 * on `stream` (a hipStream_t). */
#ifndef TTC_FRONTEND_H
#define TTC_FRONTEND_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* ---- Layer front-end: the solver inputs from the input projection (ttc/layers/ttc_layer.py:110-135) ----
 * proj [n_tokens, row] holds per token, for each head, h0 [d], A [d], R [du], coeff_Qf [q_rank] and
 * log_gammas [1 + du + d], then coeff_B [b_rank] and coeff_Q [q_rank].  Writes the solver's inputs:
 * l2norm(A), l2norm(coeff_B), l2norm(softplus(.)) of coeff_Q, R (at least 1e-6) and coeff_Qf, the
 * log-discounts -softplus(.) - relu(-gamma_bias) (gamma_bias [1 + du + d] or NULL), and h0.  Any
 * d, du and ranks >= 0 (outputs without elements may be NULL).  The backward writes grad_proj from the
 * gradients of the outputs (NULL: zero); grad_proj covers every element of proj. */
int ttc_lqr_front_end(const float* proj, const float* gamma_bias, int64_t n_tokens, int32_t heads, int32_t d,
                      int32_t du, int32_t b_rank, int32_t q_rank, float* A_diag, float* coeff_B, float* coeff_Q,
                      float* R_inv, float* coeff_Qf, float* log_gamma_A, float* log_gamma_B, float* log_gamma_Q,
                      float* h0, void* stream);
int ttc_lqr_front_end_backward(const float* proj, int64_t n_tokens, int32_t heads, int32_t d, int32_t du,
                               int32_t b_rank, int32_t q_rank, const float* grad_A_diag, const float* grad_coeff_B,
                               const float* grad_coeff_Q, const float* grad_R_inv, const float* grad_coeff_Qf,
                               const float* grad_log_gamma_A, const float* grad_log_gamma_B,
                               const float* grad_log_gamma_Q, const float* grad_h0, float* grad_proj, void* stream);

/* Matrices padded from rows x cols (0 or more) to padded rows x padded cols (powers of two, columns at
 * least 4), up to 12 arrays in one launch: shapes[5 k ..] = {matrices, rows, cols, padded rows, padded
 * cols} of array k, fill[k] the value of its new elements (bytes 2: 0 or 1), src (NULL if without
 * elements) / dst (16-byte aligned) their device pointers; `src`, `dst`, `shapes` and `fill` themselves
 * are host arrays.  bytes: 4 (fp32) or 2 (bf16). */
int ttc_lqr_pad(const void* const* src, void* const* dst, const int64_t* shapes, const float* fill, int32_t count,
                int32_t bytes, void* stream);

#ifdef __cplusplus
}
#endif

#endif /* TTC_FRONTEND_H */
