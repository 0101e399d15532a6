// ttc_lqr_sym16.hpp -- d = du = 16 forward: the certified symplectic sweep on the fp32 matrix cores,
// then the final solve and Riccati step 0.
//
// One wave holds PPW problems -- with TOK heads of one token and one register copy of B, B' and -sym(Q),
// else any consecutive problems with a copy each -- as Y-hat = [Y1'; Y2'] in the MFMA C layout: lane
// 16 g + c holds rows 4 g + r of column c.  Per step
//   M = R^{-1} B_k' Y2'      Y1' <- A_k^{-1} (Y1' + B_k M)      Y2' <- A_k Y2' + Qc_k Y1'
// (the reference's transposed row-block update, symplectic_iter.py:226-251, with V_t = Y1^{-1} Y2) is
// three products of four v_mfma_f32_16x16x4f32; 12 and about 33 vector instructions per problem.  Fp32
// matrix and vector instructions do not overlap on gfx950, so the sweep is bound by their sum (2.1 M
// problems, T = 64: 79 % of the fp32 matrix peak).  The three-way bf16 splits of the wider sweeps
// (ttc_lqr_split.hpp) do not pay here: splitting a 4-register operand takes 22 vector instructions
// (81 cycles) and its products three matrix instructions that occupy the vector ALU for 36-51 more,
// against 128 cycles for the four fp32 ones.
//
// PPW = 4 fills the chip's latencies from one wave (six waves per SIMD at 80 registers: the final
// solve stages Y1 and -Y2 one at a time through a 16 x 20 region per problem, R_inv and the previous
// step's factors wait in LDS; three per SIMD with a copy of the operands per problem).  Small batches
// take 2 or 1 problems a wave: a step of one problem has a quarter of the instructions, and the chip
// has the SIMDs to spare.
#pragma once
#include "ttc_lqr_sym.hpp"

namespace ttc {

template <int PPW, bool TOK>
struct Sym16 {
  static_assert(PPW == 1 || PPW == 2 || PPW == 4, "problems per wave");
  static constexpr int NBQ = TOK ? 1 : PPW;  // register copies of the operands
  static constexpr int LDX = 16 + kPad;
  static constexpr int REG = 16 * LDX;     // per problem: 16 rows; the pivot row of the final solve (32)
  static constexpr int VEC = 4 * 16;       // alpha, q, -beta^2 R^{-1}, 1 / alpha
  static constexpr size_t LDS_BYTES = sizeof(float) * PPW * (REG + VEC);
  static constexpr int MINW = PPW < 4 ? 4 : TOK ? 6 : 3;  // waves per SIMD the registers must allow
};

template <int PPW, bool TOK, int SM, bool WRITE_U>
__global__ __launch_bounds__(64)
__attribute__((amdgpu_waves_per_eu(Sym16<PPW, TOK>::MINW, Sym16<PPW, TOK>::MINW))) void
lqr_sym16_kernel(const float* __restrict__ A_diag, const float* __restrict__ Bg, const float* __restrict__ Qg,
                 const float* __restrict__ Rinv, const float* __restrict__ Qf, const float* __restrict__ lgA,
                 const float* __restrict__ lgB, const float* __restrict__ lgQ, const float* __restrict__ h0,
                 int64_t P, int H, int T, int PB, float* __restrict__ u_out, float* __restrict__ kstash,
                 float* __restrict__ q0stash, int* __restrict__ status) {
  using G = Sym16<PPW, TOK>;
  constexpr int D = 16, LDX = G::LDX, NBQ = G::NBQ;
  extern __shared__ __align__(16) float sm[];
  constexpr float kLog2e = 1.4426950408889634f;
  const int lane = threadIdx.x;
  const int g = lane >> 4, c = lane & 15;
  // XCD-aware block order (consecutive workgroups go round-robin to the 8 XCDs, each with its own
  // L2): a contiguous run of waves per XCD, so that those of one token share an L2
  const unsigned nblk = gridDim.x, bid = blockIdx.x;
  const unsigned lblk = (nblk % 8u == 0u) ? (bid % 8u) * (nblk / 8u) + bid / 8u : bid;
  // my problems: up to PB heads of one token, or PPW consecutive problems
  const unsigned groups = TOK ? (unsigned)((H + PB - 1) / PB) : 1u;
  const int head0 = TOK ? (int)(lblk % groups) * PB : 0;
  const int64_t pbase = TOK ? (int64_t)(lblk / groups) * H + head0 : (int64_t)lblk * PPW;
  const int64_t left = TOK ? H - head0 : P - pbase;
  const int most = TOK ? PB : PPW;
  const int nq = left < most ? (int)left : most;  // (the slots beyond: the last problem again, unstored)
  auto clampq = [&](int q) { return q < nq ? q : nq - 1; };
  auto region = [&](int q) { return sm + q * G::REG; };
  auto vecs = [&](int q) { return sm + PPW * G::REG + q * G::VEC; };

  // row layout: lane c of group g owns row c of problem qr (groups beyond PPW repeat the last one)
  const int qr = g < PPW ? g : PPW - 1;
  const int64_t po = pbase + clampq(qr);
  const float a_l = A_diag[po * D + c];
  const float lb2_l = lgB[po * D + c] * kLog2e, lq2_l = lgQ[po * D + c] * kLog2e;
  const float la2_l = lgA[po] * kLog2e;

  // B, B' and -sym(Q) as operands; Y1' = I and -Y2' = -sym(Q_f)
  float Bm[NBQ][4], Bt[NBQ][4], Qn[NBQ][4];
  auto bqi = [](int q) { return NBQ == 1 ? 0 : q; };
  v4f Y1[PPW], NV[PPW];
  {
#pragma unroll
    for (int q = 0; q < NBQ; ++q) {
      const int64_t n = (pbase + clampq(q)) / H;
      const float* bq = Bg + n * D * D;
      const float* qq = Qg + n * D * D;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = 4 * g + r;
        Bm[q][r] = bq[i * D + c];
        Bt[q][r] = bq[c * D + i];
        Qn[q][r] = -0.5f * (qq[i * D + c] + qq[c * D + i]);
      }
    }
#pragma unroll
    for (int q = 0; q < PPW; ++q) {
      const float* fq = Qf + (pbase + clampq(q)) * D * D;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = 4 * g + r;
        NV[q][r] = -0.5f * (fq[i * D + c] + fq[c * D + i]);
        Y1[q][r] = (i == c) ? 1.0f : 0.0f;
      }
    }
  }
  // step ratios of the sweep's discount factors (t runs down): q(t-1) = q(t) 2^{-lq2},
  // beta(t-1)^2 = beta(t)^2 2^{-2 lb2}, each as a pair hi + lo of floats from a double exp2
  // (the multiplications add only their rounding, no drift from a rounded ratio)
  float rQ, rQe, rB2, rB2e;
  {
    const double x = exp2((double)-lq2_l), y = exp2((double)(-2.0f * lb2_l));
    rQ = (float)x;
    rQe = (float)(x - (double)rQ);
    rB2 = (float)y;
    rB2e = (float)(y - (double)rB2);
  }
  const int x16 = (lane ^ 16) << 2, x32 = (lane ^ 32) << 2;
  region(qr)[c] = Rinv[po * D + c];  // the sweep leaves the regions unused until its final solve
  wave_sync();

  for (int t = T - 1; t >= 1; --t) {
    // the discount factors from the previous step's times the step ratios, recomputed exactly every
    // kSymRefresh steps (e_A stays an exp2 every step: by recurrence it moved the gradients' largest
    // error against fp64 from 1.3e-6 to 1.7e-6, for 0.6 % of the sweep)
    {
      float* v = vecs(qr);
      const float eA = __builtin_amdgcn_exp2f(la2_l * (float)(t + 1));
      float q, nb2;
      if ((T - 1 - t) % kSymRefresh == 0) {
        const float beta = __builtin_amdgcn_exp2f(lb2_l * (float)(t + 1));
        q = __builtin_amdgcn_exp2f(lq2_l * (float)t);
        nb2 = -(beta * beta) * region(qr)[c];
      } else {
        const float q0 = v[D + c], n0 = v[2 * D + c];
        q = fmaf(q0, rQ, q0 * rQe);
        nb2 = fmaf(n0, rB2, n0 * rB2e);
      }
      const float alpha = fmaf(a_l, eA, 1.0f);
      v[c] = alpha;
      v[D + c] = q;
      v[2 * D + c] = nb2;
      v[3 * D + c] = __builtin_amdgcn_rcpf(alpha);
    }
    wave_sync();
    const bool renorm = (T - 1 - t) % TTC_SYM_RENORM == TTC_SYM_RENORM - 1;
#pragma unroll
    for (int q = 0; q < PPW; ++q) {
      const float* v = vecs(q);
      // M = (B' N) diag-row(-beta^2 R^{-1}) = R^{-1} B_k' Y2'
      v4f M = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < 4; ++s) M = mfma16x16x4(Bm[bqi(q)][s], NV[q][s], M);
      const v4f nf = ld4(v + 2 * D + 4 * g);
#pragma unroll
      for (int r = 0; r < 4; ++r) M[r] *= nf[r];
      // Y1' <- A^{-1} (Y1' + B M)
#pragma unroll
      for (int s = 0; s < 4; ++s) Y1[q] = mfma16x16x4(Bt[bqi(q)][s], M[s], Y1[q]);
      const v4f ia = ld4(v + 3 * D + 4 * g);
      const v4f al = ld4(v + 4 * g);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        Y1[q][r] *= ia[r];
        NV[q][r] *= al[r];
      }
      // -Y2' <- -A Y2' - Qc Y1'  (operand -Qc[c][4g+s] = q_c (-Q)[4g+s][c] q_{4g+s})
      const float qc = v[D + c];
      const v4f qrw = ld4(v + D + 4 * g);
      float op[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) op[s] = Qn[bqi(q)][s] * (qc * qrw[s]);
#pragma unroll
      for (int s = 0; s < 4; ++s) NV[q] = mfma16x16x4(op[s], Y1[q][s], NV[q]);
      if (renorm) {  // columns of Y-hat (rows of Y, which leave Y1^{-1} Y2 unchanged), by powers of 2
        const v4f& y = Y1[q];
        const v4f& z = NV[q];
        float mk = maxnan(absmax(y[0], z[0]), fabsf(y[1]));
        mk = maxnan(maxnan(mk, fabsf(z[1])), fabsf(y[2]));
        mk = maxnan(maxnan(mk, fabsf(z[2])), fabsf(y[3]));
        mk = maxnan(mk, fabsf(z[3]));
        mk = maxnan(mk, lane_read(mk, x16));
        mk = maxnan(mk, lane_read(mk, x32));
        const int e = 1 - __builtin_amdgcn_frexp_expf(mk);  // m * 2^e in [1, 2)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          Y1[q][r] = __builtin_amdgcn_ldexpf(Y1[q][r], e);
          NV[q][r] = __builtin_amdgcn_ldexpf(NV[q][r], e);
        }
      }
    }
    wave_sync();
  }

  // ---- final solve: -V_1 = Y1^{-1} (-Y2) by pivoted Gauss-Jordan on the rows [Y1 | -Y2], staged one
  // at a time through each problem's region (row c of Y1 = column c of Y1'), which then holds the
  // pivot row and the solution; the certificate; N = sym(-V_1) in the C layout -------------------
  float* buf = region(qr);
  float aug[2 * D];
#pragma unroll
  for (int mtx = 0; mtx < 2; ++mtx) {
    wave_sync();  // the previous rows have been read
#pragma unroll
    for (int q = 0; q < PPW; ++q) st4(region(q) + c * LDX + 4 * g, mtx == 0 ? Y1[q] : NV[q]);
    wave_sync();
    ld_row<D>(buf + c * LDX, *reinterpret_cast<float(*)[D]>(aug + mtx * D));
  }
  float rs = 0.f;
#pragma unroll
  for (int k = 0; k < D; ++k) rs += fabsf(aug[k]);
  const float n1 = dgroup_max<D>(rs);  // ||Y1||_inf
  wave_sync();  // every row read before the pivot-row buffer (aliasing them) is written
  unsigned okbits = 0u;
  {
    float piv;
    int pos;
    gauss_jordan<D, 2 * D, 8>(aug, c, buf, piv, pos);
    const float ip = 1.0f / piv;
    float pn[D];
#pragma unroll
    for (int k = 0; k < D; ++k) pn[k] = aug[D + k] * ip;
    // the condition number from the pivots, the diagonal of U in Y1 = L U:
    // ||Y1||_inf / min|u_kk| <= n cond_inf(Y1) (|l_ij| <= 1 under partial pivoting); the
    // asymmetry test below is the one that separates the inaccurate problems
    const float n2 = dgroup_max<D>(fabsf(ip));
    st_row<D>(buf + pos * LDX, pn);
    wave_sync();
    float da = 0.f, mx = 0.f;
#pragma unroll
    for (int k = 0; k < D; ++k) {
      da = fmaxf(da, fabsf(pn[k] - buf[k * LDX + pos]));
      mx = fmaxf(mx, fabsf(pn[k]));
    }
    da = dgroup_max<D>(da);
    mx = dgroup_max<D>(mx);
    const bool ok = (n1 * n2 <= kSymCondMax) && (da <= kSymAsymMax * mx);  // false on NaN
    const unsigned long long bal = __ballot(ok);
#pragma unroll
    for (int q = 0; q < PPW; ++q) okbits |= (unsigned)((bal >> (q * D)) & 1ull) << q;
#pragma unroll
    for (int q = 0; q < PPW; ++q) {
      const float* b = region(q);
#pragma unroll
      for (int r = 0; r < 4; ++r) NV[q][r] = 0.5f * (b[(4 * g + r) * LDX + c] + b[c * LDX + 4 * g + r]);
    }
    wave_sync();
  }

  // ---- step 0: stash V_1, W_0 = V_1 B_0, Quu_0 = R + B_0' W_0, u0 = -Quu_0^{-1} W_0' (alpha_0 h0) ----
  // (the row-layout problem indices once more, from an opaque copy of the lane index: after the
  // sweep's loop, which needs every register, they are cheaper to recompute than to keep across it)
  int64_t po0;
  bool own0;
  {
    int ln = lane;
    asm volatile("" : "+v"(ln));
    const int q = ln / D;
    own0 = q < PPW && q < nq;
    po0 = pbase + (own0 ? q : nq - 1);
  }
  {
    float* v = vecs(qr);
    const float alpha = fmaf(a_l, __builtin_amdgcn_exp2f(la2_l), 1.0f);
    v[D + c] = alpha * h0[po0 * D + c];             // (A_0 h0)_c
    v[2 * D + c] = __builtin_amdgcn_exp2f(lb2_l);  // beta_0
  }
  wave_sync();
  v4f nQ[PPW];
#pragma unroll
  for (int q = 0; q < PPW; ++q) {
    const int64_t pid = pbase + clampq(q);
    if (SM == STASH_V1 && q < nq && ((okbits >> q) & 1u)) {
      float* vp = kstash + pid * D * D;
#pragma unroll
      for (int r = 0; r < 4; ++r) vp[(4 * g + r) * D + c] = -NV[q][r];
    }
    const float* v = vecs(q);
    const float bj = v[2 * D + c];
    float Bk[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) Bk[s] = Bm[bqi(q)][s] * bj;
    v4f nW = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 4; ++s) nW = mfma16x16x4(NV[q][s], Bk[s], nW);
    const float rr = 1.0f / Rinv[pid * D + c];
#pragma unroll
    for (int r = 0; r < 4; ++r) nQ[q][r] = (4 * g + r == c) ? -rr : 0.0f;
#pragma unroll
    for (int s = 0; s < 4; ++s) nQ[q] = mfma16x16x4(Bk[s], nW[s], nQ[q]);
    // -y = -W' A_0 h0
    const v4f ah = ld4(v + D + 4 * g);
    float ny = 0.f;
#pragma unroll
    for (int r = 0; r < 4; ++r) ny = fmaf(nW[r], ah[r], ny);
    ny += __shfl_xor(ny, 16, 64);
    ny += __shfl_xor(ny, 32, 64);
    wave_sync();  // every lane has read alpha*h0 and beta before the rhs overwrites the beta slot
    if (g == 0) vecs(q)[2 * D + c] = -ny;  // y
  }
  wave_sync();
#pragma unroll
  for (int q = 0; q < PPW; ++q)
#pragma unroll
    for (int r = 0; r < 4; ++r) region(q)[(4 * g + r) * LDX + c] = -nQ[q][r];
  wave_sync();
  float row[D + 4];
  ld_row<D>(buf + c * LDX, *reinterpret_cast<float(*)[D]>(row));
  row[D] = vecs(qr)[2 * D + c];
  row[D + 1] = row[D + 2] = row[D + 3] = 0.f;
  const bool store = own0 && ((okbits >> qr) & 1u);
  if (SM == STASH_V1 && store)
    st_global_row<D>(q0stash + (po0 * D + c) * D, *reinterpret_cast<float(*)[D]>(row));
  wave_sync();  // all rows read before the pivot-row buffer (aliasing them) is written
  float piv;
  int pos = c;
  {
    // Quu_0 is positive definite for a certified problem: elimination without row exchanges by DPP
    // broadcasts; a problem where a pivot says otherwise is solved again with partial pivoting (by the
    // whole wave, taken by that problem alone: no problem's bits depend on its wave-mates)
    float x[17], xpiv;
#pragma unroll
    for (int k = 0; k < 17; ++k) x[k] = row[k];
    bool bad;  // the same on a problem's 16 lanes
    gj_spd16x1(x, c, xpiv, bad);
    if (__any(bad)) gauss_jordan<D, D + 4, 4, D + 1>(row, c, buf, piv, pos);
    if (!bad) row[D] = x[16], piv = xpiv, pos = c;
  }
  const float u0 = -row[D] / piv;
  if (store) {
    if (WRITE_U) u_out[po0 * D + pos] = u0;
    if (status != nullptr && !isfinite(u0)) atomicOr(status, TTC_LQR_STATUS_NONFINITE);
  }
  // problems that were not certified: marked for the rescue pass
  if (lane < nq && !((okbits >> lane) & 1u)) {
    const float nan = __builtin_nanf("");
    if (WRITE_U) u_out[(pbase + lane) * D] = nan;
    else q0stash[(pbase + lane) * D * D] = nan;
    if (status != nullptr) atomicOr(status, TTC_LQR_STATUS_RESCUED);
  }
}

template <int PPW, bool TOK, int SM, bool WU>
inline void launch_sym16_ppw(const float* A, const float* B, const float* Q, const float* R, const float* Qf,
                             const float* lA, const float* lB, const float* lQ, const float* h0, int64_t P, int H,
                             int T, float* u, float* st_a, float* st_b, int32_t* status, hipStream_t s) {
  // as many heads a wave as even out over a token's waves
  const int waves = (H + PPW - 1) / PPW, PB = (H + waves - 1) / waves;
  const int64_t blocks = TOK ? P / H * ((H + PB - 1) / PB) : (P + PPW - 1) / PPW;
  hipLaunchKernelGGL((lqr_sym16_kernel<PPW, TOK, SM, WU>), dim3((unsigned)blocks), dim3(64),
                     (Sym16<PPW, TOK>::LDS_BYTES), s, A, B, Q, R, Qf, lA, lB, lQ, h0, P, H, T, PB, u, st_a, st_b,
                     status);
}

// Problems per wave, by what 1,024 SIMDs have to do for the whole call's problems (these P may be a chunk of
// them, and the forms give the same bits only as far as the compiler treats them alike).  Whole call,
// T = 64: one up to 2,048 problems (512: 115 us against 133 with two and 168 with four), two up to 4,096
// (162 / 178 us with four; odd head counts one, 164), four above (8,160: 226 us against 222 with two,
// 65,280: 960 / 1,020), sharing the token's operands when the head count is a multiple of four; otherwise
// a copy each, since waves with idle slots cost more (524,280 problems: 7.2 ms; by token 7.3 with 2
// heads, 7.1 with 3 and 6, 8.2 with 1 and 5; shared by four 6.7).
template <int SM, bool WU>
inline void launch_sym16(const float* A, const float* B, const float* Q, const float* R, const float* Qf,
                         const float* lA, const float* lB, const float* lQ, const float* h0, int64_t P, int H, int T,
                         float* u, float* st_a, float* st_b, int32_t* status, hipStream_t s, int64_t call) {
  if (call <= 2048 || (call <= 4096 && H % 2 != 0))
    launch_sym16_ppw<1, true, SM, WU>(A, B, Q, R, Qf, lA, lB, lQ, h0, P, H, T, u, st_a, st_b, status, s);
  else if (call <= 4096)
    launch_sym16_ppw<2, true, SM, WU>(A, B, Q, R, Qf, lA, lB, lQ, h0, P, H, T, u, st_a, st_b, status, s);
  else if (H % 4 == 0)
    launch_sym16_ppw<4, true, SM, WU>(A, B, Q, R, Qf, lA, lB, lQ, h0, P, H, T, u, st_a, st_b, status, s);
  else
    launch_sym16_ppw<4, false, SM, WU>(A, B, Q, R, Qf, lA, lB, lQ, h0, P, H, T, u, st_a, st_b, status, s);
}

}  // namespace ttc
