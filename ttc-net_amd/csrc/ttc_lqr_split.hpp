// ttc_lqr_split.hpp -- fp32 matrix products on the bf16 matrix cores by exact three-way splits.
//
// A float has a 24-bit significand and a bf16 number an 8-bit one with the same exponent range, so
// x = hi + mid + lo with hi = bf16(x), mid = bf16(x - hi), lo = bf16(x - hi - mid): both
// differences are exact in fp32, and round-to-nearest leaves |mid| <= 2^-9 |x| and a remainder of
// at most 6 bits for lo, so the sum is exact -- where all three are normal bf16 numbers: below about
// 2^-108 first lo, then mid fall under 2^-126 and |x| keeps fewer bits, and above 3.39e38 hi rounds to
// infinity (the sweeps' certificate then fails on the NaN that follows, and the problem is recomputed
// in fp32 or fp64).  The sweeps rescale their columns to [1, 2) every 8 steps, so only state costs that
// are all that small reach the lower range.  A product of two such numbers keeps the six terms
//   hi hi, hi mid, mid hi, hi lo, mid mid, lo hi
// (each exact in the fp32 accumulator's product) and drops mid lo + lo mid + lo lo, below
// 2^-26 |x y|: under the half ulp of the fp32 product that one fused multiply-add rounds.  The sum
// over k then rounds once per matrix instruction instead of once per product, so the error
// against fp64 is smaller than the fp32 matrix instruction's (measured, normal inputs: 4.9e-8
// against 7.4e-8 relative over k = 16, 1.18e-7 against 1.45e-7 over k = 64).
//
// Why: on gfx950 v_mfma_f32_16x16x4f32 runs at 64 flop per cycle and SIMD (32 cycles) and shares
// its multipliers with the vector ALU -- the two do not overlap -- while the bf16 matrix cores run
// at 1024 (measured: 16x16x32 17 cycles, 32x32x16 34) and leave the vector ALU about half of
// those.  Six products cost 6/16 of the fp32 instruction's time, and the splits 5.5 vector
// instructions per element of the varying operand.
#pragma once
#include "ttc_lqr_mfma16.hpp"

namespace ttc {

typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));

// Two floats to packed bf16, round to nearest even (v_cvt_pk_bf16_f32).
__device__ __forceinline__ unsigned cvt_bf16x2(float a, float b) {
  return __builtin_bit_cast(unsigned, __builtin_convertvector((v2f{a, b}), v2bf));
}

// a - h[0] and b - h[1] for a packed pair h (exact).  (v_dot2_f32_bf16 with (-1, 0) does each in
// one instruction, but it runs on the matrix pipe: 64 of them beside 4 matrix instructions took the
// sum of both times, shifts, masks and subtractions 60 % of it.)
__device__ __forceinline__ void residual2(float& a, float& b, unsigned h) {
  a -= __uint_as_float(h << 16);
  b -= __uint_as_float(h & 0xffff0000u);
}

// hi, mid, lo of a pair of floats, packed.
__device__ __forceinline__ void split2(float a, float b, unsigned& h, unsigned& m, unsigned& l) {
  h = cvt_bf16x2(a, b);
  residual2(a, b, h);
  m = cvt_bf16x2(a, b);
  residual2(a, b, m);
  l = cvt_bf16x2(a, b);
}

// Eight floats as three matrix operands.
struct Split8 {
  v8bf hi, mid, lo;
};

__device__ __forceinline__ Split8 split8(const v4f x, const v4f y) {
  unsigned h[4], m[4], l[4];
  split2(x[0], x[1], h[0], m[0], l[0]);
  split2(x[2], x[3], h[1], m[1], l[1]);
  split2(y[0], y[1], h[2], m[2], l[2]);
  split2(y[2], y[3], h[3], m[3], l[3]);
  return Split8{__builtin_bit_cast(v8bf, v4u{h[0], h[1], h[2], h[3]}),
                __builtin_bit_cast(v8bf, v4u{m[0], m[1], m[2], m[3]}),
                __builtin_bit_cast(v8bf, v4u{l[0], l[1], l[2], l[3]})};
}

// CW x CW tiles (16 or 32): the accumulator of a lane, and the matrix instruction over 16 k (CW = 32)
// or 32 k (CW = 16).
template <int CW> struct SplitTile;
template <> struct SplitTile<32> {
  using T = v16f;
  static __device__ __forceinline__ T mfma(v8bf a, v8bf b, T c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
};
template <> struct SplitTile<16> {
  using T = v4f;
  static __device__ __forceinline__ T mfma(v8bf a, v8bf b, T c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
};

// acc[I] += A_I B, the small terms first; the accumulators of one term are independent.
template <int CW, int NI>
__device__ __forceinline__ void mfma_split(const Split8 (&a)[NI], const Split8& b, typename SplitTile<CW>::T (&acc)[NI]) {
  auto term = [&](auto&& x, const v8bf& y) {
#pragma unroll
    for (int I = 0; I < NI; ++I) acc[I] = SplitTile<CW>::mfma(x(a[I]), y, acc[I]);
  };
  term([](const Split8& v) { return v.lo; }, b.hi);
  term([](const Split8& v) { return v.hi; }, b.lo);
  term([](const Split8& v) { return v.mid; }, b.mid);
  term([](const Split8& v) { return v.mid; }, b.hi);
  term([](const Split8& v) { return v.hi; }, b.mid);
  term([](const Split8& v) { return v.hi; }, b.hi);
}

}  // namespace ttc
