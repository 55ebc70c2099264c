// Split products on the 128 x 128 tiles of the 16x16x32 loop
// (gemm16s_kernel.h): the kernels that write fp32 partials, and the kernel
// that sums them and runs the epilogue.

#include "gemm16s_kernel.h"

namespace cpt {
namespace gemm {

CPT_ST16_INST_F32(CPT_ST16_DEFINE, kBF16)
CPT_ST16_INST_F32(CPT_ST16_DEFINE, kF16)

namespace st16 {

// l[e] = sum_k P_t[m][k] Q_t[k][n + e] in fp32 (the products are exact)
template <int DT>
__device__ __forceinline__ void lora8(const KArgs& A, int t, int64_t m, int64_t n, bool vec,
                                      float (&l)[8]) {
#pragma unroll
  for (int e = 0; e < 8; ++e) l[e] = 0.0f;
  const int r = A.lrank;
  for (int k0 = 0; k0 < r; k0 += 8) {
    float p[8];
    wide8<DT>(*reinterpret_cast<const uint4*>(A.lp[t] + m * A.lldp + k0), p);
    if (A.lq_km) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float q[8];
        wide8<DT>(*reinterpret_cast<const uint4*>(A.lq[t] + (n + e) * r + k0), q);
#pragma unroll
        for (int k = 0; k < 8; ++k) l[e] += p[k] * q[k];
      }
    } else {
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const uint16_t* row = A.lq[t] + (k0 + k) * A.lldq + n;
        float q[8];
        if (vec) {
          wide8<DT>(*reinterpret_cast<const uint4*>(row), q);
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e) q[e] = wide16<DT>(row[e], 0);
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) l[e] += p[k] * q[e];
      }
    }
  }
}

// One thread per 8 columns of one row.  HBM-bound on the partials (they mostly
// sit in the last-level cache): the loads of 4 splits are in flight together,
// added in split order.
__device__ __forceinline__ void sum8(const float* p, int64_t stride, int splits, float (&v)[8]) {
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = 0.0f;
  int s = 0;
  for (; s + 4 <= splits; s += 4) {
    f32x4 w[8];
#pragma unroll
    for (int j = 0; j < 8; ++j)
      w[j] = reinterpret_cast<const f32x4*>(p + (s + (j >> 1)) * stride)[j & 1];
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) v[4 * (j & 1) + e] += w[j][e];
  }
  for (; s < splits; ++s)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const f32x4 w = reinterpret_cast<const f32x4*>(p + s * stride)[j];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[4 * j + e] += w[e];
    }
}

template <int DT>
__device__ __forceinline__ void add_term(const KArgs& A, int t, int64_t m, int64_t n, bool vec,
                                         float (&v)[8]) {
  if (!A.lp[t]) return;
  float l[8];
  lora8<DT>(A, t, m, n, vec, l);
#pragma unroll
  for (int e = 0; e < 8; ++e)
    v[e] = round16<DT>(round16<DT>(v[e]) + round16<DT>(A.lalpha[t] * round16<DT>(l[e])));
}

template <int DT, bool DUAL>
__global__ __launch_bounds__(256) void reduce_kernel(const KArgs A, int terms, int64_t ldo,
                                                     bool vec) {
  const int64_t cols = (DUAL ? A.D : A.N) / 8;
  const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= A.M * cols) return;
  const int64_t m = e / cols, n = (e - m * cols) * 8;
  const float* p = A.ws + m * A.ldc + n;
  const int64_t stride = A.M * A.ldc;
  float v[8];
  sum8(p, stride, A.ksplit, v);
  if constexpr (!DUAL) {
    for (int t = 0; t < terms; ++t) add_term<DT>(A, t, m, n, vec, v);
    *reinterpret_cast<uint4*>(A.C + m * ldo + n) = pack8<DT>(v);
  } else {
    float u[8], h[8];
    sum8(p + A.D, stride, A.ksplit, u);
    if (terms > 0) add_term<DT>(A, 0, m, n, vec, v);
    if (terms > 1) add_term<DT>(A, 1, m, n, vec, u);
    const uint4 wg = pack8<DT>(v), wu = pack8<DT>(u);
    const int64_t off = m * A.D + n;
    if (A.h_mid) {
      wide8<DT>(wg, v);
      wide8<DT>(wu, u);
#pragma unroll
      for (int i = 0; i < 8; ++i) h[i] = silu_mul1(v[i], u[i]);
      *reinterpret_cast<uint4*>(A.h_mid + off) = pack8<DT>(h);
    }
    if (A.h_gate) {
      *reinterpret_cast<uint4*>(A.h_gate + off) = wg;
      *reinterpret_cast<uint4*>(A.h_up + off) = wu;
    }
  }
}

// The same for larger outputs with adapter terms.  A wave owns 16 rows x 64
// columns in the MFMA's output layout (lane l: row l % 16, columns 16 i + 4
// (l / 16) ..), so a term of a 16 x 16 block is one MFMA (two above rank 16) on
// P's rows and Q's columns, as in the unsplit products' epilogue.  The partials
// bind it; a thread per 8 columns is bound by the terms there, reading 8 columns
// of Q for one row: 2048 x 4096, rank 16, 2 ranges, mean of one and two terms: 63
// us, here 25.
template <int DT, bool DUAL>
__global__ __launch_bounds__(256) void reduce_lora_kernel(const KArgs A, int terms, int64_t ldo) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t cols = DUAL ? A.D : A.N;
  const int64_t cb = (cols + 255) / 256;
  const int64_t mb = blockIdx.x / cb;
  const int64_t n0 = (blockIdx.x - mb * cb) * 256 + wave * 64;
  if (n0 >= cols) return;   // the whole wave
  const int64_t m = mb * 16 + (lane & 15);
  const bool mok = m < A.M;
  const int r = A.lrank, k0 = 4 * (lane >> 4);
  int64_t n[4];
  bool nok[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    n[i] = n0 + 16 * i + 4 * (lane >> 4);
    nok[i] = n[i] < cols;   // cols % 8 == 0: a lane's 4 are all in or all out
  }
  // lanes past the output read its first elements
  const float* const row = A.ws + (mok ? m : 0) * A.ldc;
  const int64_t stride = A.M * A.ldc;
  auto sums = [&](const float* base, f32x4 (&v)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    int s = 0;
    for (; s + 4 <= A.ksplit; s += 4) {
      f32x4 w[4][4];
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          w[j][i] = *reinterpret_cast<const f32x4*>(base + (s + j) * stride + (nok[i] ? n[i] : 0));
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] += w[j][i];
    }
    for (; s < A.ksplit; ++s)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        v[i] += *reinterpret_cast<const f32x4*>(base + s * stride + (nok[i] ? n[i] : 0));
  };
  auto k4 = [](const uint16_t* p, bool ok) {
    return ok ? *reinterpret_cast<const s16x4*>(p) : s16x4{0, 0, 0, 0};
  };
  auto term = [&](int t, f32x4 (&v)[4]) {
    if (!A.lp[t]) return;
    f32x4 l[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) l[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    for (int kb = 0; kb < r; kb += 16) {
      const int k = kb + k0;   // r % 8 == 0: a lane's 4 ranks are all in or all out
      const s16x4 pf = k4(A.lp[t] + m * A.lldp + k, mok && k < r);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int64_t c = n0 + 16 * i + (lane & 15);
        const bool ok = c < cols && k < r;
        s16x4 qf = {0, 0, 0, 0};
        if (DUAL || A.lq_km) {
          qf = k4(A.lq[t] + c * r + k, ok);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (ok) qf[e] = (short)A.lq[t][(k + e) * A.lldq + c];
        }
        l[i] = mfma16<DT>(qf, pf, l[i]);
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        v[i][e] = round16<DT>(round16<DT>(v[i][e]) +
                              round16<DT>(A.lalpha[t] * round16<DT>(l[i][e])));
  };
  auto pack4 = [](const f32x4& v) {
    return make_uint2(pack16<DT>(v[0], v[1]), pack16<DT>(v[2], v[3]));
  };
  f32x4 v[4];
  sums(row, v);
  if constexpr (!DUAL) {
    for (int t = 0; t < terms; ++t) term(t, v);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (mok && nok[i]) *reinterpret_cast<uint2*>(A.C + m * ldo + n[i]) = pack4(v[i]);
  } else {
    f32x4 u[4];
    sums(row + A.D, u);
    term(0, v);
    if (terms > 1) term(1, u);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (!(mok && nok[i])) continue;
      const int64_t off = m * A.D + n[i];
      if (A.h_mid) {
        f32x4 h;
#pragma unroll
        for (int e = 0; e < 4; ++e)
          h[e] = silu_mul1(round16<DT>(v[i][e]), round16<DT>(u[i][e]));
        *reinterpret_cast<uint2*>(A.h_mid + off) = pack4(h);
      }
      if (A.h_gate) {
        *reinterpret_cast<uint2*>(A.h_gate + off) = pack4(v[i]);
        *reinterpret_cast<uint2*>(A.h_up + off) = pack4(u[i]);
      }
    }
  }
}

// fp32 outputs of a split fp32 product: c = alpha * sum
__global__ __launch_bounds__(256) void reduce_f32_kernel(const KArgs A, float* c, int64_t ldo) {
  const int64_t cols = A.N / 8;
  const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= A.M * cols) return;
  const int64_t m = e / cols, n = (e - m * cols) * 8;
  float v[8];
  sum8(A.ws + m * A.ldc + n, A.M * A.ldc, A.ksplit, v);
#pragma unroll
  for (int j = 0; j < 2; ++j)
    *reinterpret_cast<f32x4*>(c + m * ldo + n + 4 * j) =
        f32x4{A.alpha * v[4 * j], A.alpha * v[4 * j + 1], A.alpha * v[4 * j + 2],
              A.alpha * v[4 * j + 3]};
}

}  // namespace st16

int st16_reduce(int dt, bool dual, const KArgs& A, int terms, int64_t ldo, hipStream_t st) {
  const int64_t n = A.M * ((dual ? A.D : A.N) / 8);
  const int64_t blocks = (n + 255) / 256;
  if (blocks <= 0) return kOk;
  if (blocks > 0x7FFFFFFF) return kErrTooLarge;
  if (dt == kF32) {
    hipLaunchKernelGGL(st16::reduce_f32_kernel, dim3((unsigned)blocks), dim3(256), 0, st, A,
                       (float*)A.C, ldo);
    return hipGetLastError() == hipSuccess ? kOk : kErrLaunch;
  }
  // The MFMA form from 2^23 multiply-adds of a term on.  Measured, us on it against
  // a thread per 8 columns: 4 x 2048, rank 8, 14 ranges 12.1 / 6.2 (too few waves for
  // the ranges' latency); 512 x 2048, rank 8, 4 ranges 9.6 / 9.0; 2048 x 4096, rank
  // 16, 2 ranges 25 / 63.
  if (terms > 0 && A.M * (dual ? A.D : A.N) * A.lrank > (1 << 23)) {
    const int64_t grid = (A.M + 15) / 16 * (((dual ? A.D : A.N) + 255) / 256);
    if (grid > 0x7FFFFFFF) return kErrTooLarge;
#define CPT_ST16_RED(DT, DUAL)                                                                    \
  hipLaunchKernelGGL((st16::reduce_lora_kernel<DT, DUAL>), dim3((unsigned)grid), dim3(256), 0, \
                     st, A, terms, ldo)
    if (dt == kBF16) {
      if (dual) CPT_ST16_RED(kBF16, true); else CPT_ST16_RED(kBF16, false);
    } else {
      if (dual) CPT_ST16_RED(kF16, true); else CPT_ST16_RED(kF16, false);
    }
#undef CPT_ST16_RED
    return hipGetLastError() == hipSuccess ? kOk : kErrLaunch;
  }
  // 16-byte reads of Q's rows when they all start on 16 bytes
  bool vec = (A.lldq & 7) == 0;
  for (int t = 0; t < terms; ++t) vec = vec && aligned16(A.lq[t]);
#define CPT_ST16_RED(DT, DUAL)                                                                   \
  hipLaunchKernelGGL((st16::reduce_kernel<DT, DUAL>), dim3((unsigned)blocks), dim3(256), 0, st, A, \
                     terms, ldo, vec)
  if (dt == kBF16) {
    if (dual) CPT_ST16_RED(kBF16, true); else CPT_ST16_RED(kBF16, false);
  } else {
    if (dual) CPT_ST16_RED(kF16, true); else CPT_ST16_RED(kF16, false);
  }
#undef CPT_ST16_RED
  return hipGetLastError() == hipSuccess ? kOk : kErrLaunch;
}

}  // namespace gemm
}  // namespace cpt
