// ttc_lqr_symw.hpp -- d = du = 32 / 64 forward: the certified symplectic sweep on the bf16 matrix
// cores with three-way splits (ttc_lqr_split.hpp), then the final solve and Riccati step 0.
//
// The sweep (the reference's transposed row-block update, symplectic_iter.py:226-251) keeps
// Y-hat = [Y1'; Y2'] with V_t = Y1^{-1} Y2 and per step forms
//   M = R^{-1} B_k' Y2'      Y1' <- A_k^{-1} (Y1' + B_k M)      Y2' <- A_k Y2' + Qc_k Y1'
// Only left products, so the columns of Y-hat are independent: a wave owns CW = 32 of them (16 for
// small batches) -- a whole problem at d = 32, half of one at d = 64 -- and no wave waits for another
// inside the loop.  32 columns let one 32 x 32 x 16 instruction read each A operand once (half the LDS
// traffic of 16 columns, which at d = 64 is nearly as long as the matrix work), and hold the state of a
// wave in 64 registers at d = 64 (32 at d = 32), so two waves share a SIMD there (four at d = 32).
// The A operands B', B and -sym(Q) are the token's, the same for every head: split once into LDS
// (72 KB at d = 64, 18 KB at d = 32), in the order a lane reads them (16 bytes per lane and part).
//
// 32 x 32 tile in the MFMA C layout: lane l = 32 h + m holds, in register r, row
// 8 (r >> 2) + 4 h + (r & 3) of column m.  Registers 8 b .. 8 b + 7 are the rows 16 b + 8 (j >> 2)
// + 4 h + (j & 3) of k-block b: a C tile is a B operand as it stands, with the A operand's k
// permuted the same way.  (16 x 16 tiles: lane 16 g + m, rows 4 g + r; one 16 x 16 x 32 instruction takes
// two tiles.)  In both, group v of four registers is the rows row(v) .. + 3 and a k-block is two groups.
//
// Bound at d = 64: 288 matrix instructions per problem-step (9,200 busy cycles per SIMD) beside about
// 1,550 vector instructions (its share of the final solve included), and the power they draw: at
// 131,072 problems x 128 steps the matrix cores are busy 68 % of the time at 1.38 PFLOP/s (bf16), and
// the clock averages 1.95 of 2.4 GHz, so that fewer cycles (dot-product residuals, 6.55e7, against
// masked subtractions and interleaved issue, 5.64e7, at 32,768 problems) gave the same time.  47.1 -> 30.5 ms there against the fp32 matrix cores
// (90 % of their peak); with 16 columns a wave 256 problems 1.65 -> 0.42 ms, and one head (1,024
// problems), which ran Riccati steps, 3.87 -> 1.16 ms.  Problems that the certificate rejects pay for
// this sweep and then for Riccati steps, at every head count: where a fifth of the problems are
// rejected (token scales spread by e^N(0,1.5), T = 256) a head count that ran Riccati steps alone loses,
// 4.4 -> 6.0 ms with 3 heads x 256 tokens and 4.3 -> 5.3 with one head x 512; with 12 heads x 128, a
// multiple of 4, which had an fp32 sweep before, 13.9 -> 7.5 ms.
// At d = 32 the matrix cores (36 instructions of 34 cycles per problem-step) and the vector ALU (375
// instructions) bound it together, and the waves to overlap them decide: 131,072 problems x 256 steps
// 36.8 ms with two waves per SIMD (workgroups of 8 waves), 30.6 with three of 4 waves, 29.4 with
// four, 29.6 with five; 48.5 ms on the fp32 matrix cores.
#pragma once
#include "ttc_lqr_sym.hpp"
#include "ttc_lqr_split.hpp"

namespace ttc {

template <int D, int CW>
struct SymW {
  static_assert((D == 32 || D == 64) && (CW == 16 || CW == 32), "wide symplectic sweep");
  using Tile = typename SplitTile<CW>::T;
  static constexpr int NI = D / CW;            // CW x CW tiles of my columns
  static constexpr int NK = CW == 32 ? D / 16 : D / 32;  // matrix instructions over k per term
  static constexpr int NV = 2 * NK;            // 4-row groups of a column block
  static constexpr int NB = D / 16;            // 16 x 16 tiles per dimension (step 0)
  static constexpr int WPP = D / CW;           // waves per problem
  static constexpr int WPS = 64 / CW;          // waves of 64 rows of Y (the row layout of one wave) ...
  static constexpr int RPP = 64 / D;           // ... which are RPP problems
  static constexpr int MAXPB = 4 / WPP;        // problems per workgroup (four waves)
  static constexpr int LDX = D + kPad;
  static constexpr int REG = D * LDX;          // per problem, after the sweep: D rows
  static constexpr int FRAG = 9 * NI * NK * 256;  // floats of the split operands [matrix][part][I][kb][lane]
  static constexpr int VEC = 4 * D;            // per wave: alpha, q, -beta^2 R^{-1}, 1 / alpha
  static constexpr int AUGW = D == 32 ? 3 * D : 2 * D;  // final solve: [Y1 | -Y2 | I] (d = 64: no identity)
  static constexpr int MINW = D == 32 && CW == 32 ? 4 : 2;  // waves per SIMD the registers must allow
  static_assert(REG >= AUGW + 4, "pivot row fits a problem's region");
  // problems of a workgroup rounded up to whole row-layout waves
  __host__ __device__ static constexpr int regions(int PB) { return (PB + RPP - 1) / RPP * RPP; }
  __host__ __device__ static constexpr int body(int PB) {
    return FRAG > regions(PB) * REG ? FRAG : regions(PB) * REG;
  }
  static size_t lds_bytes(int PB) {
    return sizeof(float) * (size_t)(body(PB) + regions(PB) * WPP * VEC + regions(PB));
  }
};

template <int D, int CW, int SM, bool WRITE_U>
__global__ __launch_bounds__((64 * SymW<D, CW>::WPP * SymW<D, CW>::MAXPB))
__attribute__((amdgpu_waves_per_eu(SymW<D, CW>::MINW, SymW<D, CW>::MINW))) void
lqr_symw_kernel(const float* __restrict__ A_diag, const float* __restrict__ Bg, const float* __restrict__ Qg,
                const float* __restrict__ Rinv, const float* __restrict__ Qf, const float* __restrict__ lgA,
                const float* __restrict__ lgB, const float* __restrict__ lgQ, const float* __restrict__ h0, int H,
                int T, int PB, float* __restrict__ u_out, float* __restrict__ kstash, float* __restrict__ q0stash,
                int* __restrict__ status) {
  using G = SymW<D, CW>;
  using Tile = typename G::Tile;
  constexpr int NI = G::NI, NK = G::NK, NV = G::NV, NB = G::NB, WPP = G::WPP, LDX = G::LDX, RPP = G::RPP;
  extern __shared__ __align__(16) float sm[];
  constexpr float kLog2e = 1.4426950408889634f;
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int cc = lane % CW, hg = lane / CW;   // CW x CW tiles: column, row group
  const int g = lane >> 4, c = lane & 15;     // 16 x 16 tiles (step 0)
  auto row = [](int v, int hgrp) { return (CW == 32 ? 8 : 16) * v + 4 * hgrp; };  // first row of group v
  const int li = lane % D;                    // row layout
  // XCD-aware block order (consecutive workgroups go round-robin to the 8 XCDs, each with its own
  // L2): a contiguous run of workgroups per XCD, so that those of one token share an L2
  const unsigned nblk = gridDim.x, bid = blockIdx.x;
  const unsigned lblk = (nblk % 8u == 0u) ? (bid % 8u) * (nblk / 8u) + bid / 8u : bid;
  const int groups = (H + PB - 1) / PB;
  const int64_t n = lblk / (unsigned)groups;
  const int head0 = (int)(lblk % (unsigned)groups) * PB;
  const int pb = wv / WPP;                    // my problem of the workgroup
  const int ch = wv % WPP;                    // my CW columns of it
  const int64_t pid = n * H + (head0 + pb < H ? head0 + pb : H - 1);  // idle: recompute, never store
  const float* bq = Bg + n * D * D;
  const float* qq = Qg + n * D * D;
  float* vec = sm + G::body(PB) + wv * G::VEC;
  float* okf = sm + G::body(PB) + G::regions(PB) * WPP * G::VEC;

  // split operands of the token: matrix 0: B' , 1: B, 2: -sym(Q); lane (m, hg), slot j holds
  // X[CW I + m][row(2 kb + (j >> 2)) + (j & 3)]
  v8bf* frag = reinterpret_cast<v8bf*>(sm);
  for (int e = threadIdx.x; e < 3 * NI * NK * 64; e += blockDim.x) {
    const int ln = e & 63, kb = (e >> 6) % NK, I = (e >> 6) / NK % NI, mat = (e >> 6) / (NK * NI);
    const int m = CW * I + ln % CW;
    float x[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int k = row(2 * kb + (j >> 2), ln / CW) + (j & 3);
      x[j] = mat == 0 ? bq[k * D + m] : mat == 1 ? bq[m * D + k] : -0.5f * (qq[m * D + k] + qq[k * D + m]);
    }
    const Split8 s = split8(v4f{x[0], x[1], x[2], x[3]}, v4f{x[4], x[5], x[6], x[7]});
    const int at = ((mat * 3 * NI + I) * NK + kb) * 64 + ln;
    frag[at] = s.hi;
    frag[at + NI * NK * 64] = s.mid;
    frag[at + 2 * NI * NK * 64] = s.lo;
  }

  // my columns of Y1' = I and of -Y2' = -sym(Q_f)
  Tile Y1[NI], N2[NI];
  // rows row(v) .. + 3 of my column
  auto get4 = [](const Tile(&x)[NI], int v) {
    if constexpr (CW == 32) {
      const Tile& t = x[v >> 2];
      const int i = 4 * (v & 3);
      return v4f{t[i], t[i + 1], t[i + 2], t[i + 3]};
    } else {
      return x[v];
    }
  };
  auto put4 = [](Tile(&x)[NI], int v, const v4f y) {
    if constexpr (CW == 32) {
      Tile& t = x[v >> 2];
      const int i = 4 * (v & 3);
      t[i] = y[0], t[i + 1] = y[1], t[i + 2] = y[2], t[i + 3] = y[3];
    } else {
      x[v] = y;
    }
  };
  auto clear = [](Tile(&x)[NI]) {
#pragma unroll
    for (int I = 0; I < NI; ++I)
#pragma unroll
      for (int r = 0; r < CW * CW / 64; ++r) x[I][r] = 0.f;
  };
  {
    const float* fq = Qf + pid * D * D;
    const int j = CW * ch + cc;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      v4f y, z;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = row(v, hg) + r;
        z[r] = -0.5f * (fq[i * D + j] + fq[j * D + i]);
        y[r] = (i == j) ? 1.0f : 0.0f;
      }
      put4(Y1, v, y);
      put4(N2, v, z);
    }
  }
  const float a_l = A_diag[pid * D + li];
  const float lb2_l = lgB[pid * D + li] * kLog2e, lq2_l = lgQ[pid * D + li] * kLog2e;
  const float la2_l = lgA[pid] * kLog2e;
  const float rinv_l = Rinv[pid * D + li];
  // step ratios of the discount factors (t runs down): q(t-1) = q(t) 2^{-lq2} and
  // beta(t-1)^2 = beta(t)^2 2^{-2 lb2}, as pairs hi + lo from a double exp2 (no drift)
  float rQ, rQe, rB2, rB2e;
  {
    const double x = exp2((double)-lq2_l), y = exp2((double)(-2.0f * lb2_l));
    rQ = (float)x;
    rQe = (float)(x - (double)rQ);
    rB2 = (float)y;
    rB2e = (float)(y - (double)rB2);
  }
  __syncthreads();  // operands written

  auto operand = [&](int mat, int I, int kb) {
    const v8bf* f = frag + ((mat * 3 * NI + I) * NK + kb) * 64 + lane;
    return Split8{f[0], f[NI * NK * 64], f[2 * NI * NK * 64]};
  };
  // acc[I] += X S for one matrix X; src(v): rows row(v) .. + 3 of my column of S
  // (software pipelined: the operands and the split of k-block kb + 1 are issued between the matrix
  // instructions of kb, so that one wave keeps both units busy)
  auto product = [&](int mat, auto&& src, Tile(&acc)[NI]) {
    Split8 b = split8(src(0), src(1)), a[NI];
#pragma unroll
    for (int I = 0; I < NI; ++I) a[I] = operand(mat, I, 0);
#pragma unroll
    for (int kb = 0; kb < NK; ++kb) {
      Split8 an[NI], bn = b;
      if (kb + 1 < NK) {
#pragma unroll
        for (int I = 0; I < NI; ++I) an[I] = operand(mat, I, kb + 1);
        bn = split8(src(2 * kb + 2), src(2 * kb + 3));
      }
      mfma_split<CW>(a, b, acc);
      if (kb + 1 < NK) {
#pragma unroll
        for (int i = 0; i < 3 * NI; ++i) {  // matrix instruction, LDS read, vector instructions
          __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x2, 4, 0);
        }
#pragma unroll
        for (int i = 0; i < 3 * NI; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x2, 4, 0);
        }
#pragma unroll
        for (int I = 0; I < NI; ++I) a[I] = an[I];
        b = bn;
      }
    }
  };
  auto rowvec = [&](int which, int v) { return ld4(vec + which * D + row(v, hg)); };  // of the wave's vectors

  float q_l = 0.f, nb2_l = 0.f;
  for (int t = T - 1; t >= 1; --t) {
    // e_A is an exp2 every step (by recurrence it costs the gradients accuracy), the other
    // factors one every kSymRefresh steps
    if ((T - 1 - t) % kSymRefresh == 0) {
      const float beta = __builtin_amdgcn_exp2f(lb2_l * (float)(t + 1));
      q_l = __builtin_amdgcn_exp2f(lq2_l * (float)t);
      nb2_l = -(beta * beta) * rinv_l;
    } else {
      q_l = fmaf(q_l, rQ, q_l * rQe);
      nb2_l = fmaf(nb2_l, rB2, nb2_l * rB2e);
    }
    const float alpha = fmaf(a_l, __builtin_amdgcn_exp2f(la2_l * (float)(t + 1)), 1.0f);
    wave_sync();  // the previous step's reads
    vec[li] = alpha;
    vec[D + li] = q_l;
    vec[2 * D + li] = nb2_l;
    vec[3 * D + li] = __builtin_amdgcn_rcpf(alpha);
    wave_sync();
    Tile M[NI], P[NI];
    clear(M);
    // M = diag(-beta^2 R^{-1}) B' (-Y2')
    product(0, [&](int v) { return get4(N2, v); }, M);
#pragma unroll
    for (int v = 0; v < NV; ++v) put4(M, v, get4(M, v) * rowvec(2, v));
    // Y1' <- A^{-1} (Y1' + B M)
    product(1, [&](int v) { return get4(M, v); }, Y1);
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      put4(Y1, v, get4(Y1, v) * rowvec(3, v));
      put4(N2, v, get4(N2, v) * rowvec(0, v));
    }
    // -Y2' <- -A Y2' + q o (-Q (q o Y1'))
    clear(P);
    product(2, [&](int v) { return get4(Y1, v) * rowvec(1, v); }, P);
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const v4f s = rowvec(1, v), x = get4(P, v);
      v4f y = get4(N2, v);
#pragma unroll
      for (int r = 0; r < 4; ++r) y[r] = fmaf(s[r], x[r], y[r]);
      put4(N2, v, y);
    }
    // columns of Y-hat (rows of Y, which leave Y1^{-1} Y2 unchanged) rescaled by powers of 2
    if ((T - 1 - t) % TTC_SYM_RENORM == TTC_SYM_RENORM - 1) {
      float mk = 0.f;
#pragma unroll
      for (int I = 0; I < NI; ++I)
#pragma unroll
        for (int r = 0; r < CW * CW / 64; ++r) mk = maxnan(mk, absmax(Y1[I][r], N2[I][r]));
      if (CW == 16) mk = maxnan(mk, lane_read(mk, (lane ^ 16) << 2));
      mk = maxnan(mk, lane_read(mk, (lane ^ 32) << 2));
      const int e = 1 - __builtin_amdgcn_frexp_expf(mk);  // m * 2^e in [1, 2)
#pragma unroll
      for (int I = 0; I < NI; ++I)
#pragma unroll
        for (int r = 0; r < CW * CW / 64; ++r) {
          Y1[I][r] = __builtin_amdgcn_ldexpf(Y1[I][r], e);
          N2[I][r] = __builtin_amdgcn_ldexpf(N2[I][r], e);
        }
    }
  }

  // ---- final solve: -V_1 = Y1^{-1} (-Y2) by pivoted Gauss-Jordan, in the row layout (the first
  // wave of each 64 rows, D lanes per problem), and the certificate -----------------------------
  float* region = sm + pb * G::REG;             // my problem's rows
  const bool solver = wv % G::WPS == 0;         // one wave per 64 rows
  const int spb = wv / G::WPS * RPP + lane / D; // my lanes' problem in the row layout
  float* sreg = sm + spb * G::REG;
  const bool svalid = spb < PB && head0 + spb < H;
  const int64_t spid = n * H + (svalid ? head0 + spb : H - 1);
  float aug[G::AUGW];
#pragma unroll
  for (int mtx = 0; mtx < 2; ++mtx) {
    __syncthreads();  // the operands / the previous rows have been read
    const Tile(&X)[NI] = mtx == 0 ? Y1 : N2;    // column m of Y-hat = row m of Y
#pragma unroll
    for (int v = 0; v < NV; ++v) st4(region + (CW * ch + cc) * LDX + row(v, hg), get4(X, v));
    __syncthreads();
    if (solver) {
      float yr[D];
      ld_row<D>(sreg + li * LDX, yr);
#pragma unroll
      for (int k = 0; k < D; ++k) aug[mtx * D + k] = yr[k];
    }
  }
  if (solver) {
    if constexpr (D == 32) {
#pragma unroll
      for (int k = 0; k < D; ++k) aug[2 * D + k] = (k == li) ? 1.0f : 0.0f;
    }
    float rs = 0.f;
#pragma unroll
    for (int k = 0; k < D; ++k) rs += fabsf(aug[k]);
    const float n1 = dgroup_max<D>(rs);  // ||Y1||_inf
    wave_sync();  // every row read before the pivot-row buffer (aliasing them) is written
    float piv;
    int pos;
    gauss_jordan<D, G::AUGW, 8>(aug, li, sreg, piv, pos);
    const float ip = 1.0f / piv;
    float pn[D];
#pragma unroll
    for (int k = 0; k < D; ++k) pn[k] = aug[D + k] * ip;  // row pos of -V_1
    float n2;
    if constexpr (D == 32) {
      float ri = 0.f;
#pragma unroll
      for (int k = 0; k < D; ++k) ri += fabsf(aug[2 * D + k]);
      n2 = dgroup_max<D>(ri * fabsf(ip));  // ||Y1^{-1}||_inf
    } else {
      // the spread of the pivots (the diagonal of U in Y1 = L U), ||Y1||_inf for the largest
      n2 = dgroup_max<D>(fabsf(ip));
    }
    st_row<D>(sreg + pos * LDX, pn);
    wave_sync();
    float da = 0.f, mx = 0.f;
#pragma unroll
    for (int k = 0; k < D; ++k) {
      da = fmaxf(da, fabsf(pn[k] - sreg[k * LDX + pos]));
      mx = fmaxf(mx, fabsf(pn[k]));
    }
    da = dgroup_max<D>(da);
    mx = dgroup_max<D>(mx);
    const bool ok = (n1 * n2 <= kSymCondMax) && (da <= kSymAsymMax * mx);  // false on NaN
    if (li == 0) okf[spb] = ok ? 1.0f : 0.0f;
    if (li == 0 && svalid && !ok) {  // marked for the rescue pass
      const float nan = __builtin_nanf("");
      if (WRITE_U) u_out[spid * D] = nan;
      else q0stash[spid * D * D] = nan;
      if (status != nullptr) atomicOr(status, TTC_LQR_STATUS_RESCUED);
    }
  }
  __syncthreads();

  // ---- step 0: stash V_1, W_0 = V_1 B_0 and Quu_0 = R + B_0' W_0 on 16 x 16 tiles (fp32 matrix
  // cores; my two tile columns J), u0 = -Quu_0^{-1} W_0' (alpha_0 h0) ----------------------------
  const bool store = head0 + pb < H && okf[pb] != 0.0f;
  constexpr int JW = NB / WPP;
  const int J0 = ch * JW;
  v4f N[NB][NB];  // -V_1, symmetrised: tile (I, J) holds rows 16 I + 4 g + r of column 16 J + c
#pragma unroll
  for (int I = 0; I < NB; ++I)
#pragma unroll
    for (int J = 0; J < NB; ++J) {
      const v4f tr = ld4(region + (16 * J + c) * LDX + 16 * I + 4 * g);
#pragma unroll
      for (int r = 0; r < 4; ++r) N[I][J][r] = 0.5f * (region[(16 * I + 4 * g + r) * LDX + 16 * J + c] + tr[r]);
    }
  const float al0 = fmaf(a_l, __builtin_amdgcn_exp2f(la2_l), 1.0f);
  vec[li] = al0 * h0[pid * D + li];                // (A_0 h0)_li
  vec[D + li] = __builtin_amdgcn_exp2f(lb2_l);     // beta_0
  wave_sync();
  if (SM == STASH_V1 && store) {
    float* vp = kstash + pid * D * D;
#pragma unroll
    for (int I = 0; I < NB; ++I)
#pragma unroll
      for (int J = 0; J < NB; ++J)
        if (J >= J0 && J < J0 + JW) {
#pragma unroll
          for (int r = 0; r < 4; ++r) vp[(16 * I + 4 * g + r) * D + 16 * J + c] = -N[I][J][r];
        }
  }
  v4f nW[NB][JW], nQ[NB][JW];
#pragma unroll
  for (int I = 0; I < NB; ++I)
#pragma unroll
    for (int jj = 0; jj < JW; ++jj) {
      const int j = 16 * (J0 + jj) + c;
      const float rr = 1.0f / Rinv[pid * D + j];
      nW[I][jj] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int r = 0; r < 4; ++r) nQ[I][jj][r] = (16 * I + 4 * g + r == j) ? -rr : 0.0f;
    }
#pragma unroll
  for (int K = 0; K < NB; ++K) {
    float Bk[JW][4];
#pragma unroll
    for (int jj = 0; jj < JW; ++jj)
#pragma unroll
      for (int s = 0; s < 4; ++s)
        Bk[jj][s] = bq[(16 * K + 4 * g + s) * D + 16 * (J0 + jj) + c] * vec[D + 16 * (J0 + jj) + c];
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int I = 0; I < NB; ++I)
#pragma unroll
        for (int jj = 0; jj < JW; ++jj) nW[I][jj] = mfma16x16x4(N[K][I][s], Bk[jj][s], nW[I][jj]);
  }
#pragma unroll
  for (int K = 0; K < NB; ++K)
#pragma unroll
    for (int I = 0; I < NB; ++I) {
      float Bk[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) Bk[s] = bq[(16 * K + 4 * g + s) * D + 16 * I + c] * vec[D + 16 * I + c];
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int jj = 0; jj < JW; ++jj) nQ[I][jj] = mfma16x16x4(Bk[s], nW[K][jj][s], nQ[I][jj]);
    }
  // y = W' A_0 h0, to the third vector slot of the problem's first wave
  float* yv = sm + G::body(PB) + pb * WPP * G::VEC + 2 * D;
#pragma unroll
  for (int jj = 0; jj < JW; ++jj) {
    float ny = 0.f;
#pragma unroll
    for (int I = 0; I < NB; ++I) {
      const v4f ah = ld4(vec + 16 * I + 4 * g);
#pragma unroll
      for (int r = 0; r < 4; ++r) ny = fmaf(nW[I][jj][r], ah[r], ny);
    }
    ny += __shfl_xor(ny, 16, 64);
    ny += __shfl_xor(ny, 32, 64);
    if (g == 0) yv[16 * (J0 + jj) + c] = -ny;
  }
  __syncthreads();  // every wave has read N
  // rows of Quu_0, the lower tiles mirrored from the upper ones
#pragma unroll
  for (int I = 0; I < NB; ++I)
#pragma unroll
    for (int jj = 0; jj < JW; ++jj) {
      const int J = J0 + jj;
      if (I > J) continue;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float x = -nQ[I][jj][r];
        region[(16 * I + 4 * g + r) * LDX + 16 * J + c] = x;
        if (I < J) region[(16 * J + c) * LDX + 16 * I + 4 * g + r] = x;
      }
    }
  __syncthreads();
  if (!solver) return;
  float qr[D + 4];
  ld_row<D>(sreg + li * LDX, *reinterpret_cast<float(*)[D]>(qr));
  qr[D] = sm[G::body(PB) + spb * WPP * G::VEC + 2 * D + li];
  qr[D + 1] = qr[D + 2] = qr[D + 3] = 0.f;
  const bool sstore = svalid && okf[spb] != 0.0f;
  if (SM == STASH_V1 && sstore)
    st_global_row<D>(q0stash + (spid * D + li) * D, *reinterpret_cast<float(*)[D]>(qr));
  wave_sync();  // all rows read before the pivot-row buffer (aliasing them) is written
  float piv;
  int pos;
  gauss_jordan<D, D + 4, (D + 4) % 8 == 0 ? 8 : 4, D + 1>(qr, li, sreg, piv, pos);
  const float u0 = -qr[D] / piv;
  if (sstore) {
    if (WRITE_U) u_out[spid * D + pos] = u0;
    if (status != nullptr && !isfinite(u0)) atomicOr(status, TTC_LQR_STATUS_NONFINITE);
  }
}

// Workgroups of four waves of one token: two problems at d = 64, where two workgroups' copies of the
// operands fill a CU's LDS, up to four at d = 32 (eight measured 1.5 % slower, two 0.5 %), evened out
// over the token's workgroups; half as many with 16 columns a wave.
template <int D, int CW, int SM, bool WU>
inline void launch_symw_cw(const float* A, const float* B, const float* Q, const float* R, const float* Qf,
                           const float* lA, const float* lB, const float* lQ, const float* h0, int64_t P, int H, int T,
                           float* u, float* st_a, float* st_b, int32_t* status, hipStream_t s) {
  using G = SymW<D, CW>;
  const int groups = (H + G::MAXPB - 1) / G::MAXPB, PB = (H + groups - 1) / groups;
  hipLaunchKernelGGL((lqr_symw_kernel<D, CW, SM, WU>), dim3((unsigned)(P / H * ((H + PB - 1) / PB))),
                     dim3(64 * G::WPP * PB), G::lds_bytes(PB), s, A, B, Q, R, Qf, lA, lB, lQ, h0, H, T, PB, u, st_a,
                     st_b, status);
}

template <int D, int SM, bool WU>
inline void launch_symw(const float* A, const float* B, const float* Q, const float* R, const float* Qf,
                        const float* lA, const float* lB, const float* lQ, const float* h0, int64_t P, int H, int T,
                        float* u, float* st_a, float* st_b, int32_t* status, hipStream_t s, int64_t call) {
  // (by the whole call's problems: the two forms round differently, and a call's chunks must not)
  // 16 columns a wave: twice the waves, each with half the work, for batches that would leave most
  // SIMDs idle or with one wave (measured, T = 128, whole call: d = 64, 256 problems 476 against 644 us,
  // 512 663 / 677, 1,024 1,157 / 1,097; d = 32, 512 problems 248 / 318, 1,024 301 / 325, 2,048 482 /
  // 443); the operands are read from LDS twice as often, which costs 9 % when the chip is full, so at
  // d = 64 also for the odd head counts whose idle waves cost more (30,000 problems, narrow / wide: 1 head
  // 29.1 / 38.2 ms, 3 heads 29.2 / 35.6, 5 heads 28.9 / 31.9, 7 heads 29.3 / 30.3, 9 heads 29.2 / 29.9,
  // 11 heads 29.2 / 28.9; the wide form's idle half problem is one part in H + 1 of its work)
  if (call * D <= 32768 || (D == 64 && H % 2 != 0 && H <= 9))
    launch_symw_cw<D, 16, SM, WU>(A, B, Q, R, Qf, lA, lB, lQ, h0, P, H, T, u, st_a, st_b, status, s);
  else
    launch_symw_cw<D, 32, SM, WU>(A, B, Q, R, Qf, lA, lB, lQ, h0, P, H, T, u, st_a, st_b, status, s);
}

}  // namespace ttc
