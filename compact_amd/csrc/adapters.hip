// Memory-bound kernels of the adapter path (DoRA / VeRA / AdaLoRA / DyLoRA on
// the FlashFFN v3 cache), reference src/flashffn.py:1697-2230.  VeRA, AdaLoRA
// and DyLoRA enter the Function as composed or sliced thin factors, so only
// DoRA's magnitude needs kernels of its own:
//
//   dora_scale     out[i, j] = rd(x[i, j] * rd(m[j] / nu[j]))   the post-bypass
//                  column scale c = m / nu (:1967-1975) and its chain rule
//                  g * c (:2054, :2128-2130).  out may alias x.
//   col_dot_div    out[j] = rd((sum_i rd(a[i, j] * b[i, j])) / den[j]), the sum
//                  in fp32 over fixed row chunks, then the chunks in order:
//                  the magnitude gradients (:2086-2089, :2112-2125).
//   dora_col_norm  nu[j] = ||W_j + s (B A)_j||_2 through the Gram identity
//                  nu^2 = ||W_j||^2 + 2s sum_k B_jk (W A^T)_jk
//                         + s^2 sum_l (B G)_jl B_jl,   G = A A^T,
//                  all in fp32, never forming B A (:1824-1840).
// rd() rounds to the tensors' storage dtype (round to nearest even), which is
// how the reference's eager bf16 ops round each result.

#include <type_traits>

#include "common.h"
#include "compact_amd.h"

namespace cpt {
namespace adapters {

constexpr int kBlock = 256;
constexpr int kDotThreads = 64;    // col_dot: one wavefront per column strip
constexpr int kDotRows = 128;      // rows per partial of cpt_col_dot_div
constexpr int kDotUnroll = 8;      // rows in flight per lane
constexpr int kRowsPerWave = 4;    // dora_rows: rows of W one wavefront owns
constexpr int kRankTile = 8;       // dora_rows: columns of W A^T per block

template <int DT> using St = typename Elem<DT>::T;

template <int DT>
__device__ __forceinline__ float rd(float v) {
  St<DT> t;
  Elem<DT>::st(&t, v);
  return Elem<DT>::ld(&t);
}

// ---------------------------------------------------------------------------
// dora_scale
// ---------------------------------------------------------------------------

template <int DT>
__global__ __launch_bounds__(kBlock) void dora_scale_vec_kernel(const void* x, const St<DT>* m,
                                                                const St<DT>* nu, void* out,
                                                                int64_t n8, int64_t d) {
  const int64_t e8 = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (e8 >= n8) return;
  const int64_t j0 = (e8 * 8) % d;   // d % 8 == 0: the 8 elements share a row
  float v[8];
  Vec8<DT>::ld(x, e8, v);
#pragma unroll
  for (int t = 0; t < 8; ++t) {
    const float c = rd<DT>(Elem<DT>::ld(m + j0 + t) / Elem<DT>::ld(nu + j0 + t));
    v[t] = v[t] * c;
  }
  Vec8<DT>::st(out, e8, v);
}

template <int DT>
__global__ __launch_bounds__(kBlock) void dora_scale_kernel(const St<DT>* x, const St<DT>* m,
                                                            const St<DT>* nu, St<DT>* out,
                                                            int64_t total, int64_t d) {
  const int64_t e = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (e >= total) return;
  const int64_t j = e % d;
  const float c = rd<DT>(Elem<DT>::ld(m + j) / Elem<DT>::ld(nu + j));
  Elem<DT>::st(out + e, Elem<DT>::ld(x + e) * c);
}

// ---------------------------------------------------------------------------
// col_dot_div
// ---------------------------------------------------------------------------

// VEC consecutive columns per lane; grid (column strips, chunks of `rows` rows).
// HBM-bound: 8 rows of both operands are loaded before any is added, in row
// order, and a chunk is short enough that 2048 rows make 64 waves a strip.
// 2048 x 11008 bf16 (90 MB): 78 us with 128-row chunks one row at a time
// (1.2 TB/s), 19-20 us so (4.6 TB/s).
template <int DT, int VEC>
__global__ __launch_bounds__(kDotThreads) void col_dot_partial_kernel(
    const St<DT>* __restrict__ a, const St<DT>* __restrict__ b, float* __restrict__ partial,
    int64_t n, int64_t d, int64_t rows) {
  const int64_t col = ((int64_t)blockIdx.x * kDotThreads + threadIdx.x) * VEC;
  if (col >= d) return;
  const int64_t r0 = (int64_t)blockIdx.y * rows;
  const int64_t r1 = r0 + rows < n ? r0 + rows : n;
  float acc[VEC];
#pragma unroll
  for (int t = 0; t < VEC; ++t) acc[t] = 0.0f;
  auto batch = [&](int64_t r, auto uc) {
    constexpr int U = decltype(uc)::value;
    float va[U][VEC], vb[U][VEC];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if constexpr (VEC == 8) {
        Vec8<DT>::ld(a, ((r + u) * d + col) / 8, va[u]);
        Vec8<DT>::ld(b, ((r + u) * d + col) / 8, vb[u]);
      } else {
        va[u][0] = Elem<DT>::ld(a + (r + u) * d + col);
        vb[u][0] = Elem<DT>::ld(b + (r + u) * d + col);
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int t = 0; t < VEC; ++t) acc[t] += rd<DT>(va[u][t] * vb[u][t]);
  };
  int64_t r = r0;
  for (; r + kDotUnroll <= r1; r += kDotUnroll) batch(r, std::integral_constant<int, kDotUnroll>{});
  for (; r < r1; ++r) batch(r, std::integral_constant<int, 1>{});
  float* p = partial + (int64_t)blockIdx.y * d + col;
#pragma unroll
  for (int t = 0; t < VEC; ++t) p[t] = acc[t];
}

template <int DT>
__global__ __launch_bounds__(kBlock) void col_dot_finish_kernel(const float* __restrict__ partial,
                                                                const St<DT>* __restrict__ den,
                                                                St<DT>* __restrict__ out,
                                                                int64_t d, int64_t chunks) {
  const int64_t col = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (col >= d) return;
  float acc = 0.0f;
  int64_t c = 0;
  for (; c + 8 <= chunks; c += 8) {   // 8 chunks' loads together, added in order
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = partial[(c + j) * d + col];
#pragma unroll
    for (int j = 0; j < 8; ++j) acc += v[j];
  }
  for (; c < chunks; ++c) acc += partial[c * d + col];
  Elem<DT>::st(out + col, acc / Elem<DT>::ld(den + col));
}

// ---------------------------------------------------------------------------
// dora_col_norm
// ---------------------------------------------------------------------------

// Per row j of W [rows, cols]: w2[j] = sum_i W_ji^2 (blockIdx.y == 0 only) and
// wa[j, k] = sum_i W_ji A_ki for the kRankTile ranks k of blockIdx.y.  Each
// wavefront owns kRowsPerWave rows, so one load of A serves all of them.
template <int DT, int VEC>
__global__ __launch_bounds__(kBlock) void dora_rows_kernel(const St<DT>* __restrict__ w,
                                                           const St<DT>* __restrict__ a,
                                                           int64_t rows, int64_t cols, int r,
                                                           float* __restrict__ w2,
                                                           float* __restrict__ wa) {
  const int wave = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  const int64_t row0 = ((int64_t)blockIdx.x * (kBlock / 64) + wave) * kRowsPerWave;
  if (row0 >= rows) return;
  const int k0 = blockIdx.y * kRankTile;
  const bool do_sq = blockIdx.y == 0;
  float acc[kRowsPerWave][kRankTile];
  float sq[kRowsPerWave];
#pragma unroll
  for (int q = 0; q < kRowsPerWave; ++q) {
    sq[q] = 0.0f;
#pragma unroll
    for (int k = 0; k < kRankTile; ++k) acc[q][k] = 0.0f;
  }
  for (int64_t i = (int64_t)lane * VEC; i < cols; i += 64 * VEC) {
    float wv[kRowsPerWave][VEC];
#pragma unroll
    for (int q = 0; q < kRowsPerWave; ++q) {
      const int64_t row = row0 + q;
      if (row < rows) {
        if constexpr (VEC == 8) {
          Vec8<DT>::ld(w, (row * cols + i) / 8, wv[q]);
        } else {
          wv[q][0] = Elem<DT>::ld(w + row * cols + i);
        }
      } else {
#pragma unroll
        for (int t = 0; t < VEC; ++t) wv[q][t] = 0.0f;
      }
      if (do_sq) {
#pragma unroll
        for (int t = 0; t < VEC; ++t) sq[q] += wv[q][t] * wv[q][t];
      }
    }
#pragma unroll
    for (int k = 0; k < kRankTile; ++k) {
      if (k0 + k >= r) break;
      float av[VEC];
      if constexpr (VEC == 8) {
        Vec8<DT>::ld(a, ((int64_t)(k0 + k) * cols + i) / 8, av);
      } else {
        av[0] = Elem<DT>::ld(a + (int64_t)(k0 + k) * cols + i);
      }
#pragma unroll
      for (int q = 0; q < kRowsPerWave; ++q) {
#pragma unroll
        for (int t = 0; t < VEC; ++t) acc[q][k] += wv[q][t] * av[t];
      }
    }
  }
#pragma unroll
  for (int q = 0; q < kRowsPerWave; ++q) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) sq[q] += __shfl_xor(sq[q], off);
#pragma unroll
    for (int k = 0; k < kRankTile; ++k) {
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) acc[q][k] += __shfl_xor(acc[q][k], off);
    }
  }
  if (lane != 0) return;
#pragma unroll
  for (int q = 0; q < kRowsPerWave; ++q) {
    const int64_t row = row0 + q;
    if (row >= rows) break;
    if (do_sq) w2[row] = sq[q];
#pragma unroll
    for (int k = 0; k < kRankTile; ++k) {
      if (k0 + k < r) wa[row * r + k0 + k] = acc[q][k];
    }
  }
}

// G[k, l] = sum_i A_ki A_li, one block per (k, l)
template <int DT>
__global__ __launch_bounds__(kBlock) void gram_kernel(const St<DT>* __restrict__ a, int64_t cols,
                                                      int r, float* __restrict__ g) {
  const int k = blockIdx.x / r;
  const int l = blockIdx.x % r;
  float acc = 0.0f;
  for (int64_t i = threadIdx.x; i < cols; i += kBlock)
    acc += Elem<DT>::ld(a + (int64_t)k * cols + i) * Elem<DT>::ld(a + (int64_t)l * cols + i);
  for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off);
  __shared__ float part[kBlock / 64];
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) g[blockIdx.x] = (part[0] + part[1]) + (part[2] + part[3]);
}

// nu[j] = sqrt(max((w2 + 2s * sum_k B_jk wa_jk) + s^2 * sum_l (B G)_jl B_jl, 0))
template <int DT, int OUT_DT>
__global__ __launch_bounds__(kBlock) void dora_finish_kernel(const float* __restrict__ w2,
                                                             const float* __restrict__ wa,
                                                             const St<DT>* __restrict__ b,
                                                             const float* __restrict__ g,
                                                             float two_s, float s_sq,
                                                             int64_t rows, int r,
                                                             St<OUT_DT>* __restrict__ nu) {
  const int64_t j = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (j >= rows) return;
  const St<DT>* bj = b + j * r;
  float cross = 0.0f;
  for (int k = 0; k < r; ++k) cross += Elem<DT>::ld(bj + k) * wa[j * r + k];
  float quad = 0.0f;
  for (int l = 0; l < r; ++l) {
    float t = 0.0f;
    for (int k = 0; k < r; ++k) t += Elem<DT>::ld(bj + k) * g[k * r + l];
    quad += t * Elem<DT>::ld(bj + l);
  }
  const float v = (w2[j] + two_s * cross) + s_sq * quad;
  Elem<OUT_DT>::st(nu + j, sqrtf(v > 0.0f ? v : 0.0f));
}

// ---------------------------------------------------------------------------
// dora_col_norm for 16-bit W with a rank of whole 8s up to 32: one pass over W
// on the matrix cores.
// ---------------------------------------------------------------------------
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

template <int DT>
__device__ __forceinline__ f32x4 mfma32(const uint4& a, const uint4& b, const f32x4& c) {
  if constexpr (DT == kBF16)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

// wa[s][row][k] = sum over split s of W_row,i A_k,i and w2[s][row] = sum of
// W_row,i^2, for the rows of W and then, as rows `rows` .. `rows` + r - 1, those
// of A itself (their wa is the Gram matrix).  One wavefront owns 16 rows and
// loads them straight into the MFMA operand layout (lane l: row l % 16, k
// 8 (l / 16) ..), 128 k in flight; the squares come from the same registers.
// Grid (16-row groups of 4, splits), kchunk % 128 == 0, cols % 8 == 0.
// HBM-bound on W: 11008 x 4096 bf16 at rank 16 took 69 us on the vector ALUs with
// two passes, one per 8 ranks; 28 us so (4096 x 11008: 90 and 30).
template <int DT, int NB>
__global__ __launch_bounds__(kBlock) void dora_rows16_kernel(const uint16_t* __restrict__ w,
                                                             const uint16_t* __restrict__ a,
                                                             int64_t rows, int64_t cols, int r,
                                                             int64_t kchunk,
                                                             float* __restrict__ w2,
                                                             float* __restrict__ wa) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t row0 = ((int64_t)blockIdx.x * 4 + wave) * 16;
  const int64_t wrows = (rows + 15) / 16 * 16;      // A's rows follow W's groups
  const int64_t arow = row0 - wrows;
  if (arow >= r) return;
  const bool own = arow < 0;
  const uint16_t* base = own ? w : a;
  const int64_t lim = own ? rows : r, first = own ? row0 : arow;
  const int64_t k_begin = blockIdx.y * kchunk;
  const int64_t k_end = k_begin + kchunk < cols ? k_begin + kchunk : cols;
  const int kq = 8 * (lane >> 4);
  const int64_t myrow = first + (lane & 15);
  const bool rok = myrow < lim;
  const uint16_t* pw = base + (rok ? myrow : 0) * cols + kq;
  f32x4 acc[NB];
#pragma unroll
  for (int t = 0; t < NB; ++t) acc[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  float sq = 0.0f;
  const uint4 zero = make_uint4(0, 0, 0, 0);
  for (int64_t k = k_begin; k < k_end; k += 128) {
    uint4 wv[4], av[4][NB];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      // cols % 8 == 0: a lane's 8 k are all in or all out
      const bool ok = k + 32 * u + kq < k_end;
      wv[u] = ok && rok ? *reinterpret_cast<const uint4*>(pw + k + 32 * u) : zero;
#pragma unroll
      for (int t = 0; t < NB; ++t) {
        const int rk = t * 16 + (lane & 15);
        av[u][t] = ok && rk < r
                       ? *reinterpret_cast<const uint4*>(a + (int64_t)rk * cols + k + 32 * u + kq)
                       : zero;
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
#pragma unroll
      for (int t = 0; t < NB; ++t) acc[t] = mfma32<DT>(wv[u], av[u][t], acc[t]);
      float v[8];
      Vec8<DT>::ld(&wv[u], 0, v);
#pragma unroll
      for (int e = 0; e < 8; ++e) sq += v[e] * v[e];
    }
  }
  sq += __shfl_xor(sq, 16);
  sq += __shfl_xor(sq, 32);
  const int64_t total = rows + r;
  const int64_t out0 = blockIdx.y * total + (own ? first : rows + first);
  if (lane < 16 && rok) w2[out0 + lane] = sq;
  // lane holds rows 4 (l / 16) + i, rank t * 16 + l % 16
#pragma unroll
  for (int t = 0; t < NB; ++t) {
    const int rk = t * 16 + (lane & 15);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int rr = 4 * (lane >> 4) + i;
      if (first + rr < lim && rk < r) wa[(out0 + rr) * r + rk] = acc[t][i];
    }
  }
}

// The split sums in order, then nu as dora_finish_kernel: LPR lanes per row (the
// rank rounded up to 8, 16 or 32), lane l holding rank l; G, summed once per
// block, and the block's B rows in LDS.  (One thread per row walked r^2 loads in
// a chain: 37 us for 11008 rows; 8 us so.)
template <int DT, int OUT_DT, int LPR>
__global__ __launch_bounds__(kBlock) void dora_finish16_kernel(
    const float* __restrict__ w2, const float* __restrict__ wa, const uint16_t* __restrict__ b,
    float two_s, float s_sq, int64_t rows, int r, int splits, St<OUT_DT>* __restrict__ nu) {
  constexpr int RPB = kBlock / LPR;
  __shared__ float g[32 * 33];
  __shared__ float bl[RPB][LPR + 1];
  const int tid = threadIdx.x, l = tid % LPR, q = tid / LPR;
  const int64_t total = rows + r;
  for (int e = tid; e < r * r; e += kBlock) {
    float v = 0.0f;
    for (int s = 0; s < splits; ++s) v += wa[(s * total + rows) * r + e];
    g[(e / r) * 33 + e % r] = v;
  }
  const int64_t row = (int64_t)blockIdx.x * RPB + q;
  const bool ok = row < rows && l < r;
  float bv = 0.0f, x = 0.0f;
  if (ok) {
    bv = Elem<DT>::ld(b + row * r + l);
    for (int s = 0; s < splits; ++s) x += wa[(s * total + row) * r + l];
  }
  bl[q][l] = bv;
  __syncthreads();
  float t = 0.0f;
  for (int k = 0; k < r; ++k) t += bl[q][k] * g[k * 33 + l];
  float cross = bv * x, quad = l < r ? t * bv : 0.0f;
#pragma unroll
  for (int off = LPR / 2; off > 0; off >>= 1) {
    cross += __shfl_xor(cross, off);
    quad += __shfl_xor(quad, off);
  }
  if (l != 0 || row >= rows) return;
  float n2 = 0.0f;
  for (int s = 0; s < splits; ++s) n2 += w2[s * total + row];
  const float v = (n2 + two_s * cross) + s_sq * quad;
  Elem<OUT_DT>::st(nu + row, sqrtf(v > 0.0f ? v : 0.0f));
}

// k ranges of the one-pass norm: ~1024 blocks of 64 rows, ranges of whole 128s
// and at least 256
inline int64_t norm_splits(int64_t rows, int64_t cols) {
  const int64_t blk = (rows + 63) / 64 > 0 ? (rows + 63) / 64 : 1;
  int64_t s = (1024 + blk - 1) / blk;
  if (s > cols / 256) s = cols / 256;
  return s < 1 ? 1 : s;
}
inline unsigned blocks(int64_t items, int per) { return (unsigned)((items + per - 1) / per); }
inline int launched() { return hipGetLastError() == hipSuccess ? kOk : kErrLaunch; }
inline bool dtype_ok(int dt) { return dt == kF32 || dt == kF16 || dt == kBF16; }

template <int DT>
bool vec8_ok(const void* p, int64_t d) {
  return d % 8 == 0 && aligned16(p);
}

inline int64_t dot_chunks(int64_t n, int64_t rows = kDotRows) { return (n + rows - 1) / rows; }

template <int DT>
int dora_scale_t(const void* x, const void* m, const void* nu, int64_t n, int64_t d, void* out,
                 hipStream_t st) {
  const int64_t total = n * d;
  if (vec8_ok<DT>(x, d) && aligned16(out)) {
    dora_scale_vec_kernel<DT><<<blocks(total / 8, kBlock), kBlock, 0, st>>>(
        x, (const St<DT>*)m, (const St<DT>*)nu, out, total / 8, d);
  } else {
    dora_scale_kernel<DT><<<blocks(total, kBlock), kBlock, 0, st>>>(
        (const St<DT>*)x, (const St<DT>*)m, (const St<DT>*)nu, (St<DT>*)out, total, d);
  }
  return launched();
}

template <int DT>
int col_dot_t(const void* a, const void* b, const void* den, int64_t n, int64_t d, int64_t rows,
              void* workspace, void* out, hipStream_t st) {
  const int64_t chunks = dot_chunks(n, rows);
  float* partial = (float*)workspace;
  if (chunks > 0) {
    if (vec8_ok<DT>(a, d) && aligned16(b)) {
      col_dot_partial_kernel<DT, 8><<<dim3(blocks(d / 8, kDotThreads), (unsigned)chunks),
                                      kDotThreads, 0, st>>>((const St<DT>*)a, (const St<DT>*)b,
                                                            partial, n, d, rows);
    } else {
      col_dot_partial_kernel<DT, 1><<<dim3(blocks(d, kDotThreads), (unsigned)chunks),
                                      kDotThreads, 0, st>>>((const St<DT>*)a, (const St<DT>*)b,
                                                            partial, n, d, rows);
    }
  }
  col_dot_finish_kernel<DT><<<blocks(d, kBlock), kBlock, 0, st>>>(partial, (const St<DT>*)den,
                                                                  (St<DT>*)out, d, chunks);
  return launched();
}

template <int DT, int OUT_DT>
void dora_finish_t(const float* w2, const float* wa, const void* b, const float* g, double s,
                   int64_t rows, int r, void* nu, hipStream_t st) {
  dora_finish_kernel<DT, OUT_DT><<<blocks(rows, kBlock), kBlock, 0, st>>>(
      w2, wa, (const St<DT>*)b, g, (float)(2.0 * s), (float)(s * s), rows, r, (St<OUT_DT>*)nu);
}

template <int DT, int OUT_DT>
void dora_finish16_t(const float* w2, const float* wa, const void* b, double s, int64_t rows,
                     int r, int splits, void* nu, hipStream_t st) {
  const int lpr = r <= 8 ? 8 : r <= 16 ? 16 : 32;
  const auto kern = r <= 8    ? dora_finish16_kernel<DT, OUT_DT, 8>
                    : r <= 16 ? dora_finish16_kernel<DT, OUT_DT, 16>
                              : dora_finish16_kernel<DT, OUT_DT, 32>;
  kern<<<blocks(rows, kBlock / lpr), kBlock, 0, st>>>(w2, wa, (const uint16_t*)b, (float)(2.0 * s),
                                                      (float)(s * s), rows, r, splits,
                                                      (St<OUT_DT>*)nu);
}

template <int DT>
int dora_col_norm16_t(const void* w, const void* a, const void* b, int64_t rows, int64_t cols,
                      int r, double s, void* workspace, void* nu, int nu_dtype, hipStream_t st) {
  int64_t splits = norm_splits(rows, cols);
  const int64_t kchunk = ((cols + splits - 1) / splits + 127) / 128 * 128;
  splits = (cols + kchunk - 1) / kchunk;
  float* w2 = (float*)workspace;
  float* wa = w2 + splits * (rows + r);
  const int64_t groups = (rows + 15) / 16 + (r + 15) / 16;
  const dim3 grid(blocks(groups, 4), (unsigned)splits);
  const auto kern = r <= 16 ? dora_rows16_kernel<DT, 1> : dora_rows16_kernel<DT, 2>;
  kern<<<grid, kBlock, 0, st>>>((const uint16_t*)w, (const uint16_t*)a, rows, cols, r, kchunk, w2,
                                wa);
  switch (nu_dtype) {
    case kF32: dora_finish16_t<DT, kF32>(w2, wa, b, s, rows, r, (int)splits, nu, st); break;
    case kF16: dora_finish16_t<DT, kF16>(w2, wa, b, s, rows, r, (int)splits, nu, st); break;
    default: dora_finish16_t<DT, kBF16>(w2, wa, b, s, rows, r, (int)splits, nu, st); break;
  }
  return launched();
}

template <int DT>
int dora_col_norm_t(const void* w, const void* a, const void* b, int64_t rows, int64_t cols,
                    int r, double s, void* workspace, void* nu, int nu_dtype, hipStream_t st) {
  float* w2 = (float*)workspace;
  float* wa = w2 + rows;
  float* g = wa + rows * r;
  const unsigned row_blocks = blocks(rows, (kBlock / 64) * kRowsPerWave);
  const unsigned rank_tiles = r > 0 ? (unsigned)((r + kRankTile - 1) / kRankTile) : 1u;
  if (vec8_ok<DT>(w, cols) && aligned16(a)) {
    dora_rows_kernel<DT, 8><<<dim3(row_blocks, rank_tiles), kBlock, 0, st>>>(
        (const St<DT>*)w, (const St<DT>*)a, rows, cols, r, w2, wa);
  } else {
    dora_rows_kernel<DT, 1><<<dim3(row_blocks, rank_tiles), kBlock, 0, st>>>(
        (const St<DT>*)w, (const St<DT>*)a, rows, cols, r, w2, wa);
  }
  if (r > 0) gram_kernel<DT><<<(unsigned)(r * r), kBlock, 0, st>>>((const St<DT>*)a, cols, r, g);
  switch (nu_dtype) {
    case kF32: dora_finish_t<DT, kF32>(w2, wa, b, g, s, rows, r, nu, st); break;
    case kF16: dora_finish_t<DT, kF16>(w2, wa, b, g, s, rows, r, nu, st); break;
    default: dora_finish_t<DT, kBF16>(w2, wa, b, g, s, rows, r, nu, st); break;
  }
  return launched();
}

}  // namespace adapters
}  // namespace cpt

using namespace cpt;
using namespace cpt::adapters;

extern "C" {

int cpt_dora_scale(const void* x, const void* m, const void* nu, int64_t n, int64_t d, int dtype,
                   void* out, void* stream) {
  if (!dtype_ok(dtype)) return kErrDType;
  if (n < 0 || d < 0) return kErrShape;
  if (n == 0 || d == 0) return kOk;
  if (!x || !m || !nu || !out) return kErrShape;
  hipStream_t st = (hipStream_t)stream;
  switch (dtype) {
    case kF32: return dora_scale_t<kF32>(x, m, nu, n, d, out, st);
    case kF16: return dora_scale_t<kF16>(x, m, nu, n, d, out, st);
    default: return dora_scale_t<kBF16>(x, m, nu, n, d, out, st);
  }
}

int64_t cpt_col_dot_workspace_bytes(int64_t n, int64_t d) {
  if (n < 0 || d < 0) return -1;
  const int64_t chunks = dot_chunks(n);
  return (chunks > 0 ? chunks : 1) * d * (int64_t)sizeof(float);
}

int cpt_col_dot_div(const void* a, const void* b, const void* den, int64_t n, int64_t d,
                    int dtype, void* workspace, void* out, void* stream) {
  return cpt_col_dot_div_rows(a, b, den, n, d, kDotRows, dtype, workspace, out, stream);
}

int cpt_col_dot_div_rows(const void* a, const void* b, const void* den, int64_t n, int64_t d,
                         int64_t rows, int dtype, void* workspace, void* out, void* stream) {
  if (!dtype_ok(dtype)) return kErrDType;
  if (n < 0 || d < 0 || rows < 1) return kErrShape;
  if (d == 0) return kOk;
  if (!den || !out || (n > 0 && (!a || !b || !workspace))) return kErrShape;
  if (dot_chunks(n, rows) > 65535) return kErrTooLarge;
  hipStream_t st = (hipStream_t)stream;
  switch (dtype) {
    case kF32: return col_dot_t<kF32>(a, b, den, n, d, rows, workspace, out, st);
    case kF16: return col_dot_t<kF16>(a, b, den, n, d, rows, workspace, out, st);
    default: return col_dot_t<kBF16>(a, b, den, n, d, rows, workspace, out, st);
  }
}

int64_t cpt_dora_col_norm16_workspace_bytes(int64_t rows, int64_t cols, int64_t r) {
  if (rows < 0 || cols < 0 || r < 0) return -1;
  return norm_splits(rows, cols) * (rows + r) * (r + 1) * (int64_t)sizeof(float);
}

int cpt_dora_col_norm16(const void* w, const void* a, const void* b, int64_t rows, int64_t cols,
                        int64_t r, double s, int dtype, void* workspace, void* nu, int nu_dtype,
                        void* stream) {
  if ((dtype != kBF16 && dtype != kF16) || !dtype_ok(nu_dtype)) return kErrDType;
  if (rows < 0 || cols < 0 || r < 0) return kErrShape;
  if (rows == 0) return kOk;
  if (!w || !a || !b || !nu || !workspace || r == 0 || r > 32 || (r & 7) || cols == 0)
    return kErrShape;
  if ((cols & 7) || !aligned16(w) || !aligned16(a) || ((uintptr_t)workspace & 3)) return kErrAlign;
  if (rows > ((int64_t)1 << 34)) return kErrTooLarge;
  hipStream_t st = (hipStream_t)stream;
  return dtype == kBF16 ? dora_col_norm16_t<kBF16>(w, a, b, rows, cols, (int)r, s, workspace, nu,
                                                   nu_dtype, st)
                        : dora_col_norm16_t<kF16>(w, a, b, rows, cols, (int)r, s, workspace, nu,
                                                  nu_dtype, st);
}

int64_t cpt_dora_col_norm_workspace_bytes(int64_t rows, int64_t r) {
  if (rows < 0 || r < 0) return -1;
  return (rows + rows * r + r * r) * (int64_t)sizeof(float);
}

int cpt_dora_col_norm(const void* w, const void* a, const void* b, int64_t rows, int64_t cols,
                      int64_t r, double s, int dtype, void* workspace, void* nu, int nu_dtype,
                      void* stream) {
  if (!dtype_ok(dtype) || !dtype_ok(nu_dtype)) return kErrDType;
  if (rows < 0 || cols < 0 || r < 0) return kErrShape;
  if (rows == 0) return kOk;
  if (!w || !nu || !workspace || (r > 0 && (!a || !b))) return kErrShape;
  if (r > 4096 || rows > ((int64_t)1 << 40)) return kErrTooLarge;
  hipStream_t st = (hipStream_t)stream;
  switch (dtype) {
    case kF32: return dora_col_norm_t<kF32>(w, a, b, rows, cols, (int)r, s, workspace, nu, nu_dtype, st);
    case kF16: return dora_col_norm_t<kF16>(w, a, b, rows, cols, (int)r, s, workspace, nu, nu_dtype, st);
    default: return dora_col_norm_t<kBF16>(w, a, b, rows, cols, (int)r, s, workspace, nu, nu_dtype, st);
  }
}

}  // extern "C"
