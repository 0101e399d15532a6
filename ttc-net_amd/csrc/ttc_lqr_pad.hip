// ttc_lqr_pad.hip -- zero-padding of the solver's tensors from (d, du) to the kernels' state size (16,
// 32 or 64), all of a call in one launch (up to 64 GB).  As torch operators each tensor is a fill and a copy: 16
// launches and their dispatch were 85 us of a small call; here it is one launch of about 5 us, one
// write per output element (four a thread, 16 bytes) and one read per input element.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "ttc_frontend.h"
#include "ttc_lqr.h"

namespace ttc {

struct PadJobs {
  static constexpr int MAX = 12;
  const void* src[MAX];
  void* dst[MAX];
  int64_t M[MAX];        // matrices
  int rows[MAX], cols[MAX];
  int lrows[MAX], lcols[MAX];  // log2 of the padded rows and columns
  float fill[MAX];
  unsigned first[MAX];
  int count;
};

__device__ __forceinline__ void put(float* o, const float (&v)[4]) {
  *reinterpret_cast<float4*>(o) = make_float4(v[0], v[1], v[2], v[3]);
}
// bf16 bit patterns: the values are bf16 (or the fill, 0 or 1), so their upper halves are exact
__device__ __forceinline__ void put(uint16_t* o, const float (&v)[4]) {
  *reinterpret_cast<uint2*>(o) = make_uint2((__float_as_uint(v[0]) >> 16) | (__float_as_uint(v[1]) & 0xffff0000u),
                                            (__float_as_uint(v[2]) >> 16) | (__float_as_uint(v[3]) & 0xffff0000u));
}
__device__ __forceinline__ float get(const float* p) { return *p; }
__device__ __forceinline__ float get(const uint16_t* p) { return __uint_as_float((uint32_t)*p << 16); }

template <typename T>
__global__ __launch_bounds__(256) void pad_kernel(const PadJobs jobs, unsigned block0) {
  const unsigned block = block0 + blockIdx.x;
  int k = 0;
  while (k + 1 < jobs.count && block >= jobs.first[k + 1]) ++k;  // uniform
  const int lr = jobs.lrows[k], lc = jobs.lcols[k], rows = jobs.rows[k], cols = jobs.cols[k];
  const int64_t e = ((int64_t)(block - jobs.first[k]) * 256 + threadIdx.x) * 4;
  const int64_t m = e >> (lr + lc);
  if (m >= jobs.M[k]) return;
  const int j = (int)(e & ((1 << lc) - 1)), i = (int)((e >> lc) & ((1 << lr) - 1));
  const T* in = static_cast<const T*>(jobs.src[k]) + (m * rows + i) * cols;
  float v[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) v[t] = (i < rows && j + t < cols) ? get(in + j + t) : jobs.fill[k];
  put(static_cast<T*>(jobs.dst[k]) + e, v);
}

}  // namespace ttc

using namespace ttc;

extern "C" int ttc_lqr_pad(const void* const* src, void* const* dst, const int64_t* shapes, const float* fill,
                           int32_t count, int32_t bytes, void* stream) {
  if (count < 0 || count > PadJobs::MAX || (bytes != 2 && bytes != 4)) return TTC_LQR_EINVAL;
  if (count > 0 && (!src || !dst || !shapes || !fill)) return TTC_LQR_EINVAL;
  auto log2of = [](int64_t v) {
    int l = 0;
    while (((int64_t)1 << l) < v && l < 30) ++l;
    return ((int64_t)1 << l) == v ? l : -1;
  };
  PadJobs jobs{};
  int64_t blocks = 0;
  for (int k = 0; k < count; ++k) {
    const int64_t* s = shapes + 5 * k;  // matrices, rows, cols, padded rows, padded cols
    const int lr = log2of(s[3]), lc = log2of(s[4]);
    if (s[0] < 0 || s[1] < 0 || s[2] < 0 || s[1] > s[3] || s[2] > s[4] || lr < 0 || lc < 2) return TTC_LQR_EINVAL;
    if (s[0] == 0) continue;
    if ((!src[k] && s[1] > 0 && s[2] > 0) || !dst[k]) return TTC_LQR_EINVAL;
    const int c = jobs.count++;
    jobs.src[c] = src[k];
    jobs.dst[c] = dst[k];
    jobs.M[c] = s[0];
    jobs.rows[c] = (int)s[1];
    jobs.cols[c] = (int)s[2];
    jobs.lrows[c] = lr;
    jobs.lcols[c] = lc;
    jobs.fill[c] = fill[k];
    jobs.first[c] = (unsigned)blocks;
    blocks += ((s[0] << (lr + lc)) + 1023) / 1024;
    if (blocks > 0x7fffffff) return TTC_LQR_EINVAL;
  }
  if (jobs.count == 0) return TTC_LQR_OK;
  // a launch takes at most 2^32 - 1 threads (64 GB of fp32 outputs): the rest in further launches
  constexpr int64_t kMostBlocks = ((int64_t)1 << 24) - 1;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  for (int64_t b = 0; b < blocks; b += kMostBlocks) {
    const dim3 grid((unsigned)(blocks - b < kMostBlocks ? blocks - b : kMostBlocks)), block(256);
    if (bytes == 4) hipLaunchKernelGGL(pad_kernel<float>, grid, block, 0, st, jobs, (unsigned)b);
    else hipLaunchKernelGGL(pad_kernel<uint16_t>, grid, block, 0, st, jobs, (unsigned)b);
    if (hipGetLastError() != hipSuccess) return TTC_LQR_ELAUNCH;
  }
  return TTC_LQR_OK;
}
