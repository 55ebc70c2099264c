// Products that write fp32 (gemm16_kernel.h, gemm16s_kernel.h): split ones on 256
// x 256 tiles, fp32 ones over three bf16 planes per operand, and the kernel that
// makes the planes.

#include "gemm16s_kernel.h"

namespace cpt {
namespace gemm {

CPT_ST16_INST_X3(CPT_ST16_DEFINE)
template int launch_nt16_f32<true, true, false, 8>(KArgs, hipStream_t);
template int launch_nt16_f32<true, false, false, 8>(KArgs, hipStream_t);
template int launch_nt16_f32<false, false, false, 8>(KArgs, hipStream_t);
template int launch_nt16_f32<false, true, false, 8>(KArgs, hipStream_t);
template int launch_nt16_f32<true, true, true, 8>(KArgs, hipStream_t);
template int launch_nt16_f32<true, false, true, 8>(KArgs, hipStream_t);
template int launch_nt16_f32<false, false, true, 8>(KArgs, hipStream_t);
template int launch_nt16_f32<false, true, true, 8>(KArgs, hipStream_t);
template int launch_nt16_f32<true, true, true, 6>(KArgs, hipStream_t);
template int launch_nt16_f32<true, false, true, 6>(KArgs, hipStream_t);
template int launch_nt16_f32<false, false, true, 6>(KArgs, hipStream_t);
template int launch_nt16_f32<false, true, true, 6>(KArgs, hipStream_t);

// planes[0..2] = bf16 h, m, l with h = bf16(x), m = bf16(x - h), l = bf16(x - h
// - m): round-to-nearest each, both differences exact, so x = h + m + l to 24
// bits.  *flag is set when some x is not in that range: not finite, above 2^55
// (so no product or sum of the planes overflows where fp32's would not), or
// below 2^-100 but not 0 (whose l would be subnormal or lost).  One such element
// sends every product of its operand to the general-layout kernel, the splitting
// paid for nothing: a full fine-tune step of 2048 tokens at 2048 x 5632 takes 2.31
// ms, 4.36 with one in x and grad_y, 5.59 with one in every operand (5.25 without
// planes at all).  HBM-bound: 4
// bytes read and 6 written per element (2048 x 5632: 24 us, 4.8 TB/s).  rows of
// `cols` elements (a multiple of 8), ld apart; one thread per 8 columns.
__global__ __launch_bounds__(256) void split_f32_kernel(const float* __restrict__ x, int64_t ld,
                                                        int64_t rows, int64_t cols,
                                                        uint16_t* __restrict__ planes, int* flag) {
  const int64_t c8 = cols >> 3;
  const int64_t n = rows * c8;
  const int64_t plane = rows * cols;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const int64_t r = i / c8, c = (i - r * c8) * 8;
  float v[8];
  const float4 a = *reinterpret_cast<const float4*>(x + r * ld + c);
  const float4 b = *reinterpret_cast<const float4*>(x + r * ld + c + 4);
  v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
  v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
  bool bad = false;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float m = fabsf(v[e]);
    bad |= !(m <= 0x1p55f) || (m < 0x1p-100f && m != 0.0f);
  }
  if (bad) __hip_atomic_store(flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
  for (int p = 0; p < 3; ++p) {
    const uint32_t w[4] = {pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]),
                           pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7])};
    *reinterpret_cast<uint4*>(planes + p * plane + r * cols + c) =
        make_uint4(w[0], w[1], w[2], w[3]);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] -= __uint_as_float(e & 1 ? w[e >> 1] & 0xFFFF0000u : w[e >> 1] << 16);
  }
}

}  // namespace gemm
}  // namespace cpt

using namespace cpt;

extern "C" int cpt_split_f32(const void* x, int64_t ld, int64_t rows, int64_t cols, void* planes,
                             void* flag, void* stream) {
  if (rows < 0 || cols < 0) return kErrShape;
  if (rows == 0 || cols == 0) return kOk;
  if (!x || !planes || !flag) return kErrShape;
  if (!aligned16(x) || !aligned16(planes) || (ld & 3) || (cols & 7) || ld < cols ||
      ((uintptr_t)flag & 3))
    return kErrAlign;
  const int64_t blocks = (rows * (cols >> 3) + 255) / 256;
  if (blocks > 0x7FFFFFFF) return kErrTooLarge;
  hipLaunchKernelGGL(gemm::split_f32_kernel, dim3((unsigned)blocks), dim3(256), 0,
                     (hipStream_t)stream, (const float*)x, ld, rows, cols, (uint16_t*)planes,
                     (int*)flag);
  return hipGetLastError() == hipSuccess ? kOk : kErrLaunch;
}
