// ttc_lqr_mfma_blk.hpp -- d = du in {32, 64} forward kernel: the Riccati sweep as 16x16
// tiles on the matrix cores (v_mfma_f32_16x16x4f32), with a blocked Cholesky.
//
// A wave holds PPW problems; every D x D matrix is NB x NB tiles (NB = D/16), each tile
// in the MFMA C/D layout: lane 16g + c holds X[4g + r][c], r = 0..3.  For a product
// C = X Y the A operand of lane (g, c) is X[c][4g + s] and the B operand Y[4g + s][c]
// (instruction s of 4 covers k = 4g + s), so a C-layout tile serves directly as a B
// operand, and as an A operand when X is the transpose of a tile we hold (X_IK = T_KI').
// Per Riccati step t >= 1 and problem:
//   B_k = B diag(beta)                      the MFMA operand, scaled per block-row
//   -W = N B_k           (N = -V)           NB^3 * 4 MFMA
//   -Quu = B_k'(-W) - R, upper tiles        NB(NB+1)/2 * NB * 4 MFMA
//   -W' from -W through LDS (tile transpose)
//   blocked Cholesky of S' = [Quu | W'] by 16-row panels j:
//     -L_jj^{-T} from a 16x16 DPP elimination of [-Quu_jj; -I] (row layout),
//     panel   P'_ji = L_jj^{-1} S'_ji       4 MFMA per tile
//     trailing -S'_Ji += P'_jJ' P'_ji      4 MFMA per tile
//   so that the W' tiles end as M' = L^{-1} W' (M = W L^{-T}, W Quu^{-1} W' = M M');
//   N + M M' = -(V - W Quu^{-1} W'), upper tiles, one operand -> exactly symmetric
//   N <- diag(a)(N + M M')diag(a) - diag(q) Q diag(q), lower tiles mirrored via LDS.
// Step 0 forms W and Quu the same way and solves Quu_0 z = W_0' A_0 h0 (u0 = -z) by
// Gauss-Jordan with partial pivoting in the row layout (lane li owns row li); it also writes
// the stash V_1 / Quu_0.
//
// Multi-wave workgroups (and every d = 64 launch) keep B and -sym(Q) in LDS, shared by the
// WPB waves of the workgroup: its WPB * PPW problems are consecutive heads of one token
// (the launcher guarantees it).  That leaves the registers to N and the step's products,
// so two waves share each SIMD.  One-wave d = 32 workgroups keep B and Q in registers.
//
// Breakdown guard: in exact arithmetic every Cholesky pivot of Quu = R + B'VB is at least
// min_j 1/R_inv_j (Quu >= R); a pivot below half of that, or not finite, means rounding
// made V indefinite.  The wave then stops and marks its problems with a NaN (u[p][0], or
// Quu_0[p][0][0] when u is not written); lqr_rescue_kernel recomputes every marked problem
// with the row-layout sweep (pivoted Gauss-Jordan at every step).
#pragma once
#include "ttc_lqr_mfma16.hpp"

namespace ttc {

template <int D, int PPW_, int WPB_>
struct MB {
  static constexpr int NB = D / 16;                 // tiles per dimension
  static constexpr int PPW = PPW_;                  // problems per wave
  static constexpr int WPB = WPB_;                  // waves per workgroup
  static constexpr int GPP = 4 / PPW;               // 16-lane groups per problem in the 16x16 elimination
  static constexpr int RPP = 64 / D;                // problems per row-layout pass (D lanes each)
  static constexpr int NPASS = PPW / RPP;           // row-layout passes over the wave's problems
  static_assert(PPW % RPP == 0 && PPW <= 4, "problems per wave");
  static constexpr int NT = NB * (NB + 1) / 2;      // upper tiles (I <= J)
  static constexpr int LDX = D + kPad;              // LDS row stride of D-wide rows
  static constexpr int LDG = 20;                    // LDS row stride of a 16 x 16 tile
  // B and -sym(Q) in LDS, shared by the workgroup (d = 64 always; d = 32 with several waves)
  static constexpr bool BQ_LDS = D == 64 || WPB > 1;
  // workgroup-shared region: [B' (column-major B) | -sym(Q) fragments]
  static constexpr int OFF_Q = D * LDX;
  static constexpr int SH = BQ_LDS ? OFF_Q + NT * 256 : 0;
  // per-problem region: transpose buffer (CH block-rows per round), also the 16x16 tile
  // buffer and the step-0 row buffer
  static constexpr int CH = BQ_LDS ? NB / 2 : NB;
  static constexpr int XROWS = CH * 16;
  static constexpr int REG = XROWS * LDX;
  static_assert(REG % 4 == 0 && REG >= 16 * LDG && REG >= D + 4, "per-problem LDS region");
  // per-problem vectors: alpha, q (step 0: alpha*h0), beta (step 0: rhs)
  static constexpr int VEC = 3 * D;
  static constexpr int PER_WAVE = PPW * (REG + VEC);
  static constexpr int THREADS = 64 * WPB;
  // two waves per SIMD, except with four problems per wave that keep B and Q in registers
  static constexpr int MINW = (PPW == 4 && !BQ_LDS) ? 1 : 2;
  static constexpr size_t LDS_BYTES = sizeof(float) * ((size_t)SH + (size_t)WPB * PER_WAVE);
};

// upper tile (I, J), I <= J, in row-major order of the upper triangle
template <int NB>
__host__ __device__ constexpr int utile(int I, int J) {
  return I * NB - I * (I - 1) / 2 + (J - I);
}

// RESC_: rescue pass after the symplectic sweep: a workgroup runs only when
// one of its problems carries the NaN marker, and stores the marked problems only.
template <int D, int PPW_, int WPB_, int SM, bool WRITE_U, bool RESC_ = false>
__global__ __launch_bounds__(64 * WPB_)
__attribute__((amdgpu_waves_per_eu(MB<D, PPW_, WPB_>::MINW, MB<D, PPW_, WPB_>::MINW))) void
lqr_fwd_blk_kernel(const float* __restrict__ A_diag, const float* __restrict__ Bg, const float* __restrict__ Qg,
                   const float* __restrict__ Rinv, const float* __restrict__ Qf, const float* __restrict__ lgA,
                   const float* __restrict__ lgB, const float* __restrict__ lgQ, const float* __restrict__ h0,
                   int64_t P, int H, int T, float* __restrict__ u_out, float* __restrict__ kstash,
                   float* __restrict__ q0stash, int* __restrict__ status) {
  using G = MB<D, PPW_, WPB_>;
  constexpr int NB = G::NB, PPW = G::PPW, NT = G::NT, LDX = G::LDX, LDG = G::LDG;
  constexpr int NBQ = G::BQ_LDS ? 1 : PPW;  // register copies of B / Q
  auto bqi = [](int q) { return NBQ == 1 ? 0 : q; };
  constexpr int RPP = G::RPP, NPASS = G::NPASS;
  constexpr bool BQL = G::BQ_LDS;
  extern __shared__ __align__(16) float sm[];
  constexpr float kLog2e = 1.4426950408889634f;
  const int lane = threadIdx.x & 63;
  const int wv = G::WPB == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave of the workgroup (uniform)
  const int g = lane >> 4;          // lane group: MFMA row block
  const int c = lane & 15;          // MFMA column; row of the 16x16 elimination
  const int qe = g / G::GPP;        // my problem in the 16x16 elimination
  const int li = lane % D;          // my row (of D) in the row layout
  // XCD-aware block order: the hardware deals consecutive workgroups round-robin to the 8 XCDs,
  // each with its own L2; give each XCD a contiguous run of problems instead, so that the
  // workgroups of one token (which read its B and Q) share an L2
  const unsigned nblk = gridDim.x, bid = blockIdx.x;
  const unsigned lblk = (nblk % 8u == 0u) ? (bid % 8u) * (nblk / 8u) + bid / 8u : bid;
  const int64_t pbase = ((int64_t)lblk * G::WPB + wv) * PPW;

  int64_t pid[PPW];
#pragma unroll
  for (int q = 0; q < PPW; ++q) pid[q] = (pbase + q < P) ? (pbase + q) : (P - 1);  // idle: recompute, never store
  unsigned marked = ~0u;  // the problems this launch may store
  if constexpr (RESC_) {
    // the same decision in every wave of the workgroup, before its only barrier
    if (status != nullptr && !(__atomic_load_n(status, __ATOMIC_RELAXED) & TTC_LQR_STATUS_RESCUED)) return;
    bool mk = false;
    if (lane < PPW && pbase + lane < P) {
      const float m = WRITE_U ? u_out[(pbase + lane) * D] : q0stash[(pbase + lane) * D * D];
      mk = m != m;  // NaN marker of the sweep before
    }
    marked = (unsigned)(__ballot(mk) & ((1ull << PPW) - 1ull));
    if (__syncthreads_or(marked != 0u) == 0) return;
  }
  float* shb = sm;             // shared B' (d = 64)
  float* shq = sm + G::OFF_Q;  // shared -sym(Q) fragments (d = 64)
  float* wbase = sm + G::SH + wv * G::PER_WAVE;
  auto region = [&](int q) { return wbase + q * G::REG; };
  float* vecs = wbase + PPW * G::REG;  // [q][alpha D | q D | beta D]

  // row layout, pass pa: lane li of problem qr = pa * RPP + lane / D
  int qr[NPASS];
  int64_t po[NPASS];
  bool own_valid[NPASS];
  float a_l[NPASS], lb2_l[NPASS], lq2_l[NPASS], la2_o[NPASS];
#pragma unroll
  for (int pa = 0; pa < NPASS; ++pa) {
    qr[pa] = pa * RPP + lane / D;
    po[pa] = (pbase + qr[pa] < P) ? (pbase + qr[pa]) : (P - 1);
    own_valid[pa] = pbase + qr[pa] < P;
    a_l[pa] = A_diag[po[pa] * D + li];
    lb2_l[pa] = lgB[po[pa] * D + li] * kLog2e;
    lq2_l[pa] = lgQ[po[pa] * D + li] * kLog2e;
    la2_o[pa] = lgA[po[pa]] * kLog2e;
  }

  // C-layout state: N = -V (all tiles); B and -sym(Q) (registers, or shared LDS for d = 64)
  v4f NV[PPW][NB][NB];
  float Bm[NBQ][NB][NB][4];
  v4f Qn[NBQ][NT];
  float rr[PPW][NB];  // 1 / R_inv[16I + c]
  if constexpr (BQL) {
    // the workgroup's token: B column-major, -sym(Q) as per-lane C-layout fragments
    const int64_t n = pid[0] / H;
    const float* bq = Bg + n * D * D;
    const float* qq = Qg + n * D * D;
    for (int e = threadIdx.x; e < D * D; e += G::THREADS) {
      const int i = e / D, j = e % D;
      shb[j * LDX + i] = bq[e];
    }
    for (int e = threadIdx.x; e < NT * 64; e += G::THREADS) {
      const int tile = e >> 6, ln = e & 63;
      int I = 0, rem = tile;
      while (rem >= NB - I) {
        rem -= NB - I;
        ++I;
      }
      const int J = I + rem;
      v4f qn;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = 16 * I + 4 * (ln >> 4) + r, j = 16 * J + (ln & 15);
        qn[r] = -0.5f * (qq[i * D + j] + qq[j * D + i]);
      }
      st4(shq + e * 4, qn);
    }
  }
#pragma unroll
  for (int q = 0; q < PPW; ++q) {
    const int64_t n = pid[q] / H;
    const float* bq = Bg + n * D * D;
    const float* qq = Qg + n * D * D;
    const float* fq = Qf + pid[q] * D * D;
#pragma unroll
    for (int I = 0; I < NB; ++I) {
#pragma unroll
      for (int J = 0; J < NB; ++J) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = 16 * I + 4 * g + r, j = 16 * J + c;
          NV[q][I][J][r] = -0.5f * (fq[i * D + j] + fq[j * D + i]);
          if (!BQL && q < NBQ) {
            Bm[bqi(q)][I][J][r] = bq[i * D + j];
            if (I <= J) Qn[bqi(q)][utile<NB>(I, J)][r] = -0.5f * (qq[i * D + j] + qq[j * D + i]);
          }
        }
      }
    }
  }
  // R = 1 / R_inv per problem, and the pivot floor of my elimination problem: half of
  // min_j 1 / R_inv_j
  float piv_floor = 0.f;
  {
#pragma unroll
    for (int q = 0; q < PPW; ++q)
#pragma unroll
      for (int I = 0; I < NB; ++I) rr[q][I] = 1.0f / Rinv[pid[q] * D + 16 * I + c];
#pragma unroll
    for (int q = 0; q < PPW; ++q) {
      float m = rr[q][0];
#pragma unroll
      for (int I = 1; I < NB; ++I) m = fminf(m, rr[q][I]);
      m = 0.5f * row16_min(m);
      if (q == qe) piv_floor = m;
    }
  }
  if constexpr (BQL) __syncthreads();  // shared B / Q written (the only workgroup barrier)

  // B_k = B diag(beta), block-row K: Bk[J][s] = B[16K + 4g + s][16J + c] beta[16J + c]
  auto load_bk_row = [&](int q, int K, float (&Bk)[NB][4]) {
    const float* v = vecs + q * G::VEC;
#pragma unroll
    for (int J = 0; J < NB; ++J) {
      const float bj = v[2 * D + 16 * J + c];
      if constexpr (BQL) {
        const v4f b4 = ld4(shb + (16 * J + c) * LDX + 16 * K + 4 * g);
#pragma unroll
        for (int s = 0; s < 4; ++s) Bk[J][s] = b4[s] * bj;
      } else {
#pragma unroll
        for (int s = 0; s < 4; ++s) Bk[J][s] = Bm[bqi(q)][K][J][s] * bj;
      }
    }
  };
  // -W = N B_k and the upper tiles of -Quu = B_k'(-W) - R
  auto w_quu = [&](int q, v4f (&nW)[NB][NB], v4f (&nQ)[NT]) {
#pragma unroll
    for (int I = 0; I < NB; ++I)
#pragma unroll
      for (int J = 0; J < NB; ++J) nW[I][J] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int K = 0; K < NB; ++K) {
      float Bk[NB][4];
      load_bk_row(q, K, Bk);
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int I = 0; I < NB; ++I)
#pragma unroll
          for (int J = 0; J < NB; ++J) nW[I][J] = mfma16x16x4(NV[q][K][I][s], Bk[J][s], nW[I][J]);
    }
#pragma unroll
    for (int I = 0; I < NB; ++I)
#pragma unroll
      for (int J = I; J < NB; ++J) {
        v4f acc = v4f{0.f, 0.f, 0.f, 0.f};
        if (I == J) {
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[r] = (4 * g + r == c) ? -rr[q][I] : 0.0f;
        }
        nQ[utile<NB>(I, J)] = acc;
      }
#pragma unroll
    for (int K = 0; K < NB; ++K) {
      float Bk[NB][4];
      load_bk_row(q, K, Bk);
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int I = 0; I < NB; ++I)
#pragma unroll
          for (int J = I; J < NB; ++J)
            nQ[utile<NB>(I, J)] = mfma16x16x4(Bk[I][s], nW[K][J][s], nQ[utile<NB>(I, J)]);
    }
  };

  // One matrix-core Riccati step t >= 1.  Returns true when the breakdown guard fired
  // (N is then unchanged: the guard is evaluated before N is touched).
  auto step = [&](const int t) -> bool {
    const float tp1 = (float)(t + 1);
#pragma unroll
    for (int pa = 0; pa < NPASS; ++pa) {
      float* v = vecs + qr[pa] * G::VEC;
      v[li] = fmaf(a_l[pa], __builtin_amdgcn_exp2f(la2_o[pa] * tp1), 1.0f);  // alpha
      v[D + li] = __builtin_amdgcn_exp2f(lq2_l[pa] * (float)t);              // q
      v[2 * D + li] = __builtin_amdgcn_exp2f(lb2_l[pa] * tp1);               // beta
    }
    wave_sync();

    v4f nWt[PPW][NB][NB];  // -W' tiles (C layout), later M'
    v4f nQ[PPW][NT];       // -Quu upper tiles, later the L' panels
#pragma unroll
    for (int q = 0; q < PPW; ++q) {
      v4f nW[NB][NB];
      w_quu(q, nW, nQ[q]);
      // -W -> LDS row-major, read back as -W' (CH block-rows per round)
      float* xb = region(q);
#pragma unroll
      for (int h = 0; h < NB; h += G::CH) {
#pragma unroll
        for (int I = h; I < h + G::CH; ++I)
#pragma unroll
          for (int J = 0; J < NB; ++J)
#pragma unroll
            for (int r = 0; r < 4; ++r) xb[(16 * (I - h) + 4 * g + r) * LDX + 16 * J + c] = nW[I][J][r];
        wave_sync();
#pragma unroll
        for (int I = h; I < h + G::CH; ++I)
#pragma unroll
          for (int J = 0; J < NB; ++J) nWt[q][J][I] = ld4(xb + (16 * (I - h) + c) * LDX + 16 * J + 4 * g);
        wave_sync();
      }
    }

    // ---- blocked Cholesky of S' = [Quu | W'] by 16-row panels --------------------------
    bool bad = false;
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      // diagonal tile -Quu_jj (symmetric: the column fragment is a row fragment)
#pragma unroll
      for (int q = 0; q < PPW; ++q) st4(region(q) + c * LDG + 4 * g, nQ[q][utile<NB>(j, j)]);
      wave_sync();
      float* tb = region(qe);
      float qrow[16], irow[16];
      ld_row<16>(tb + c * LDG, qrow);
#pragma unroll
      for (int k = 0; k < 16; ++k) irow[k] = (k == c) ? -1.0f : 0.0f;
      // elimination of the rows [-Quu_jj; -I]: the -I rows end as -L_jj^{-T}
      static_for<16>([&](auto kc) {
        constexpr int k = decltype(kc)::value;
        const float npiv = bcast16<k>(qrow[k]);  // -d_k
        bad |= !(-npiv >= piv_floor);            // also catches NaN
        const float rs = __builtin_amdgcn_rsqf(-npiv);
        const float ip = rs * rs;
        const float ni = irow[k] * ip;
        if constexpr (k < 15) {
          const float nq = qrow[k] * ip;
          Elim16<k>::qw(qrow, irow, nq, ni);
        }
        irow[k] *= rs;
      });
      wave_sync();
      st_row<16>(tb + c * LDG, irow);  // rows of -L_jj^{-T} (groups of one problem write equal values)
      wave_sync();
#pragma unroll
      for (int q = 0; q < PPW; ++q) {
        const float* ub = region(q);
        float nU[4];  // A operand of -L_jj^{-1}: -L^{-T}[4g + s][c]
#pragma unroll
        for (int s = 0; s < 4; ++s) nU[s] = ub[(4 * g + s) * LDG + c];
        // panel: P'_ji = (-L^{-1})(-S'_ji)
#pragma unroll
        for (int i = j + 1; i < NB; ++i) {
          v4f acc = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int s = 0; s < 4; ++s) acc = mfma16x16x4(nU[s], nQ[q][utile<NB>(j, i)][s], acc);
          nQ[q][utile<NB>(j, i)] = acc;
        }
#pragma unroll
        for (int i = 0; i < NB; ++i) {
          v4f acc = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int s = 0; s < 4; ++s) acc = mfma16x16x4(nU[s], nWt[q][j][i][s], acc);
          nWt[q][j][i] = acc;
        }
        // trailing: -S'_Ji += P'_jJ' P'_ji
#pragma unroll
        for (int J = j + 1; J < NB; ++J) {
#pragma unroll
          for (int s = 0; s < 4; ++s) {
#pragma unroll
            for (int i = J; i < NB; ++i)
              nQ[q][utile<NB>(J, i)] =
                  mfma16x16x4(nQ[q][utile<NB>(j, J)][s], nQ[q][utile<NB>(j, i)][s], nQ[q][utile<NB>(J, i)]);
#pragma unroll
            for (int i = 0; i < NB; ++i)
              nWt[q][J][i] = mfma16x16x4(nQ[q][utile<NB>(j, J)][s], nWt[q][j][i][s], nWt[q][J][i]);
          }
        }
      }
      wave_sync();  // the tile buffer is rewritten by the next panel
    }
    if (__any(bad)) return true;

    // ---- N + M M' (upper tiles), scaling, mirror ----------------------------------------
#pragma unroll
    for (int q = 0; q < PPW; ++q) {
#pragma unroll
      for (int kb = 0; kb < NB; ++kb)
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
          for (int I = 0; I < NB; ++I)
#pragma unroll
            for (int J = I; J < NB; ++J) NV[q][I][J] = mfma16x16x4(nWt[q][kb][I][s], nWt[q][kb][J][s], NV[q][I][J]);
      const float* v = vecs + q * G::VEC;
#pragma unroll
      for (int I = 0; I < NB; ++I) {
        const v4f arow = ld4(v + 16 * I + 4 * g);
        const v4f qrw = ld4(v + D + 16 * I + 4 * g);
#pragma unroll
        for (int J = I; J < NB; ++J) {
          const float acol = v[16 * J + c];
          const float qcol = v[D + 16 * J + c];
          v4f qn;
          if constexpr (BQL) qn = ld4(shq + (utile<NB>(I, J) * 64 + lane) * 4);
          else qn = Qn[bqi(q)][utile<NB>(I, J)];
#pragma unroll
          for (int r = 0; r < 4; ++r) NV[q][I][J][r] = fmaf(arow[r] * acol, NV[q][I][J][r], (qrw[r] * qcol) * qn[r]);
        }
      }
      // lower tiles from the upper ones (CH block-rows per round)
      float* xb = region(q);
#pragma unroll
      for (int h = 0; h < NB - 1; h += G::CH) {
#pragma unroll
        for (int I = h; I < h + G::CH && I < NB - 1; ++I)
#pragma unroll
          for (int J = I + 1; J < NB; ++J)
#pragma unroll
            for (int r = 0; r < 4; ++r) xb[(16 * (I - h) + 4 * g + r) * LDX + 16 * J + c] = NV[q][I][J][r];
        wave_sync();
#pragma unroll
        for (int I = h; I < h + G::CH && I < NB - 1; ++I)
#pragma unroll
          for (int J = I + 1; J < NB; ++J) NV[q][J][I] = ld4(xb + (16 * (I - h) + c) * LDX + 16 * J + 4 * g);
        wave_sync();
      }
    }
    return false;
  };

  unsigned okbits = marked;  // problems whose results are stored (rescue: marked)

  // Step 0: stash V_1, form W_0 and Quu_0, u0 = -Quu_0^{-1} W_0' (alpha_0 * h0).
  auto step0 = [&]() {
#pragma unroll
    for (int pa = 0; pa < NPASS; ++pa) {
      float* v = vecs + qr[pa] * G::VEC;
      const float alpha = fmaf(a_l[pa], __builtin_amdgcn_exp2f(la2_o[pa]), 1.0f);
      v[li] = alpha;
      v[D + li] = alpha * h0[po[pa] * D + li];            // (A_0 h0)_li
      v[2 * D + li] = __builtin_amdgcn_exp2f(lb2_l[pa]);  // beta_0
    }
    wave_sync();
    v4f nQ[PPW][NT];
#pragma unroll
    for (int q = 0; q < PPW; ++q) {
      if (SM == STASH_V1 && pbase + q < P && ((okbits >> q) & 1u)) {
        float* vp = kstash + pid[q] * D * D;
#pragma unroll
        for (int I = 0; I < NB; ++I)
#pragma unroll
          for (int J = 0; J < NB; ++J)
#pragma unroll
            for (int r = 0; r < 4; ++r) vp[(16 * I + 4 * g + r) * D + 16 * J + c] = -NV[q][I][J][r];
      }
      v4f nW[NB][NB];
      w_quu(q, nW, nQ[q]);
      // -y = -W' A_0 h0: -y[16J + c] = sum_{I,r} (-W)[16I+4g+r][16J+c] ah[16I+4g+r]
      const float* v = vecs + q * G::VEC;
      float ny[NB];
#pragma unroll
      for (int J = 0; J < NB; ++J) ny[J] = 0.f;
#pragma unroll
      for (int I = 0; I < NB; ++I) {
        const v4f ah = ld4(v + D + 16 * I + 4 * g);
#pragma unroll
        for (int J = 0; J < NB; ++J)
#pragma unroll
          for (int r = 0; r < 4; ++r) ny[J] = fmaf(nW[I][J][r], ah[r], ny[J]);
      }
#pragma unroll
      for (int J = 0; J < NB; ++J) {
        ny[J] += __shfl_xor(ny[J], 16, 64);
        ny[J] += __shfl_xor(ny[J], 32, 64);
      }
      wave_sync();  // every lane has read alpha*h0 and beta before the rhs overwrites the beta slot
      if (g == 0) {
#pragma unroll
        for (int J = 0; J < NB; ++J) vecs[q * G::VEC + 2 * D + 16 * J + c] = -ny[J];  // y
      }
    }
    // rows of Quu_0 to the row layout, XROWS rows per round through the transpose buffer
#pragma unroll
    for (int pa = 0; pa < NPASS; ++pa) {
      float aug[D + 4];
#pragma unroll
      for (int k = 0; k < D + 4; ++k) aug[k] = 0.f;
#pragma unroll
      for (int h = 0; h < D; h += G::XROWS) {
        wave_sync();
#pragma unroll
        for (int q = pa * RPP; q < pa * RPP + RPP; ++q) {
          float* xb = region(q);
#pragma unroll
          for (int I = 0; I < NB; ++I)
#pragma unroll
            for (int J = I; J < NB; ++J)
#pragma unroll
              for (int r = 0; r < 4; ++r) {
                const float x = -nQ[q][utile<NB>(I, J)][r];
                if (16 * I >= h && 16 * I < h + G::XROWS) xb[(16 * I - h + 4 * g + r) * LDX + 16 * J + c] = x;
                if (J > I && 16 * J >= h && 16 * J < h + G::XROWS)
                  xb[(16 * J - h + c) * LDX + 16 * I + 4 * g + r] = x;
              }
        }
        wave_sync();
        if (li >= h && li < h + G::XROWS)
          ld_row<D>(region(qr[pa]) + (li - h) * LDX, *reinterpret_cast<float(*)[D]>(aug));
      }
      aug[D] = vecs[qr[pa] * G::VEC + 2 * D + li];
      const bool store = own_valid[pa] && ((okbits >> qr[pa]) & 1u);
      if (SM == STASH_V1 && store)
        st_global_row<D>(q0stash + (po[pa] * D + li) * D, *reinterpret_cast<float(*)[D]>(aug));
      wave_sync();  // all rows read before the pivot-row buffer (aliasing them) is written
      float piv;
      int pos;
      gauss_jordan<D, D + 4, (D + 4) % 8 == 0 ? 8 : 4, D + 1>(aug, li, region(qr[pa]), piv, pos);
      const float u0 = -aug[D] / piv;
      if (store) {
        if (WRITE_U) u_out[po[pa] * D + pos] = u0;
        if (status != nullptr && !isfinite(u0)) atomicOr(status, TTC_LQR_STATUS_NONFINITE);
      }
    }
  };

  int t = T - 1;
  bool failed = false;
  while (!failed && t >= 1) {
    failed = step(t);
    --t;
  }
  if (!failed) step0();
  else okbits = 0u;
  // problems whose sweep broke down: mark them for lqr_rescue_kernel
  if (lane < PPW && pbase + lane < P && ((marked >> lane) & 1u) && !((okbits >> lane) & 1u)) {
    const float nan = __builtin_nanf("");
    if (WRITE_U) u_out[(pbase + lane) * D] = nan;
    else q0stash[(pbase + lane) * D * D] = nan;
    if (status != nullptr) atomicOr(status, TTC_LQR_STATUS_RESCUED);
  }
}

}  // namespace ttc
