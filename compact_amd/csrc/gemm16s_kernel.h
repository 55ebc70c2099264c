// The 16x16x32 loop on small tiles: 128 x 128 outputs per block instead of the
// 256 x 256 of gemm16_kernel.h, for products whose 256 x 256 tiles are too few
// to fill the chip (a few hundred to a few thousand tokens, or a d_model-wide
// output).  Each output is the same chain of v_mfma_f32_16x16x32 over k in the
// same order, so a product is bit-identical on either tile size.
//
// Block: 256 threads (4 waves, 2 x 2), 128 x 128 outputs, k steps of 64; wave w
// owns rows 64 (w / 2) .. +63 and columns 64 (w % 2) .. +63 as 4 x 4 blocks of
// 16 x 16 (64 accumulator registers).
//
// LDS: S stages x 2 operands x [128][64] elements, 32 KiB a stage.  K-major
// tiles are swizzled as in gemm16_kernel.h (row r's chunk c at c ^ (r & 6));
// MN-major tiles are [64 k][128 mn], 256-byte rows, chunk c of row k at
// c ^ mn_swz(k).
//
// Schedule of one k-tile kt over its 32 MFMA slots, one barrier per k-tile:
//   slots 0..15   sub-step 0 (k 0..31) on fragment set F0, reading F1 of kt;
//                 the last 4 loads of tile kt - 1 + S
//   after slot 15 wait (own loads of tile kt + 1 landed: vmcnt; F1 read:
//                 lgkmcnt(0)), barrier: stage kt % S is free, tile kt + 1 whole
//   slots 16..31  sub-step 1 on F1, reading F0 of kt + 1; the first 4 loads of
//                 tile kt + S into stage kt % S
// Bound: with one block per CU (S = 4, 128 KiB) the k-tile costs 0.42 us (1 to
// 128 blocks; 0.50 to 0.55 with 256), the 32 KiB it loads at the latency of three
// tiles in flight, against 0.21 us of MFMAs; a full grid reaches 1.07 PFLOP/s (2048 x 2048, k 5632: 44.0 us, where
// 64 tiles of 256 x 256 took 96.2).  S = 2 (64 KiB) lets two blocks share a CU:
// the second block's MFMAs cover the first one's barrier, prologue and epilogue
// (2048 x 4096, k 11008: 161.5 us against 202.7).

//
// Element types: bf16 and fp16 operands (v_mfma_f32_16x16x32_bf16 / _f16, the
// same rates), fp32 accumulation.  A split product (EPI_F32, A.ksplit > 1)
// writes fp32 partials of a k range; st16_reduce sums them in split order and
// runs the epilogue.  An operand pair that is MN-major on both sides (the
// weight gradients, k = tokens) may end in a partial k-tile: its buffers then
// start at that tile, so the rows past K read zero.

//
// fp32 products (DT = kF32): each operand comes as three bf16 planes that sum
// to it (split_f32_kernel: 8 + 8 + 8 significant bits), and the k loop runs
// over six pairs of planes, the smallest products first: h l, l h, m m, h m,
// m h, h h.  The three left out are below 2^-24 of the product; every partial
// product is exact in fp32 and the sums are fp32, with one rounding per 32 k
// where v_mfma_f32_32x32x2_f32 rounds every 2.  The 256 x 256 tiles carry the
// same loop (nt16_f32_kernel); figures beside x3_gemm_impl in gemm.hip.

#pragma once

#include "gemm16_kernel.h"

namespace cpt {
namespace gemm {
namespace st16 {

using nt16::f32x4;
using nt16::i32x4;
using nt16::kBK;
using nt16::kThreads;
using nt16::load_lds;
using nt16::mn_swz;
using nt16::rsrc_sgpr;
using nt16::lora4_km;
using nt16::lora4_mn;
using nt16::s16x4;

constexpr int kT = 128;                       // tile rows and columns
constexpr int kOp = kT * kBK;                 // elements of one operand in one stage
constexpr int kLdOut = kT + 8;                // staged output rows (elements)
constexpr int kGluLdS = kT / 2 + 8;           // staged gate / up rows
constexpr int kGroup = 8;                     // tile rows an XCD runs together
template <int S> constexpr int lds_bytes() { return S * 2 * kOp * 2; }
static_assert(kT * kLdOut * 2 <= lds_bytes<2>(), "staged output tile");
static_assert(2 * kT * kGluLdS * 2 <= lds_bytes<2>(), "staged gate and up tiles");

// 4 x 4 blocks, block n = max(i, j) ascending: the first MFMAs need only the
// first fragments read
struct Order4 {
  uint8_t i[16], j[16];
  constexpr Order4() : i(), j() {
    int t = 0;
    for (int n = 0; n < 4; ++n) {
      for (int q = 0; q < n; ++q) { i[t] = n; j[t] = q; ++t; }
      for (int q = 0; q < n; ++q) { i[t] = q; j[t] = n; ++t; }
      i[t] = n; j[t] = n; ++t;
    }
  }
};

__device__ __forceinline__ void tile_of(int b, int nb, int tiles_m, int tiles_n, int& tm, int& tn) {
  // contiguous logical tiles per XCD, kGroup tile rows at a time
  const int xcd = b & 7, idx = b >> 3;
  const int base = nb >> 3, extra = nb & 7;
  const int logical = xcd * base + min(xcd, extra) + idx;
  const int per_group = kGroup * tiles_n;
  const int g = logical / per_group;
  const int rows = min(kGroup, tiles_m - g * kGroup);
  const int in = logical - g * per_group;
  tm = g * kGroup + in % rows;
  tn = in / rows;
}

// Rounding to, packing and widening the 16-bit element types
template <int DT> __device__ __forceinline__ uint32_t pack16(float a, float b) {
  if constexpr (DT == kBF16) return pack_bf16x2(a, b);
  else return (uint32_t)f32_to_f16_bits(a) | ((uint32_t)f32_to_f16_bits(b) << 16);
}
template <int DT> __device__ __forceinline__ float wide16(uint32_t w, int hi) {
  if constexpr (DT == kBF16) return __uint_as_float(hi ? w & 0xFFFF0000u : w << 16);
  else return f16_bits_to_f32((uint16_t)(hi ? w >> 16 : w & 0xFFFFu));
}
template <int DT> __device__ __forceinline__ float round16(float x) {
  if constexpr (DT == kBF16) return round_bf16(x);
  else return (float)(_Float16)x;
}
template <int DT> __device__ __forceinline__ uint4 pack8(const float (&v)[8]) {
  return make_uint4(pack16<DT>(v[0], v[1]), pack16<DT>(v[2], v[3]), pack16<DT>(v[4], v[5]),
                    pack16<DT>(v[6], v[7]));
}
template <int DT> __device__ __forceinline__ void wide8(const uint4& w, float (&v)[8]) {
  const uint32_t a[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = wide16<DT>(a[e >> 1], e & 1);
}

template <int DT> __device__ __forceinline__ void mfma32(f32x4& c, const bf16x8& a, const bf16x8& b) {
  if constexpr (DT == kBF16) nt16::mfma(c, a, b);
  else if constexpr (DT == kF32) nt16::mfma(c, a, b);   // bf16 planes
  else asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
}
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
template <int DT>
__device__ __forceinline__ f32x4 mfma16(const s16x4& a, const s16x4& b, const f32x4& c) {
  if constexpr (DT == kBF16) return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
  else return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(f16x4, a),
                                                    __builtin_bit_cast(f16x4, b), c, 0, 0, 0);
}

struct Lora {
  s16x4 p[2][4], q[2][4], ph[2][4], qh[2][4];
};

template <bool DUAL, int LT>
__device__ __forceinline__ void lora_load(const KArgs& A, int64_t m0, int64_t n0, int wm, int wn,
                                          int lane, Lora& F) {
  const int r = A.lrank;
  const bool hi = r > 16;
#pragma unroll
  for (int t = 0; t < LT; ++t) {
    const __amdgpu_buffer_rsrc_t rp = make_rsrc(A.lp[t], A.lp[t] ? A.M * A.lldp * 2 : 0);
    const int64_t qb = DUAL ? A.D * r * 2 : A.lq_km ? A.N * r * 2 : (int64_t)r * A.lldq * 2;
    const __amdgpu_buffer_rsrc_t rq = make_rsrc(A.lq[t], A.lq[t] ? qb : 0);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int64_t m = m0 + wm * 64 + 16 * j + (lane & 15);
      F.p[t][j] = lora4_km(rp, A.lldp, m, r, lane);
      F.ph[t][j] = s16x4{0, 0, 0, 0};
      if (hi) F.ph[t][j] = lora4_km(rp, A.lldp, m, r, lane, 16);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (DUAL && (i >> 1) != t) continue;
      F.qh[t][i] = s16x4{0, 0, 0, 0};
      if (DUAL || A.lq_km) {
        const int64_t n = DUAL ? (n0 >> 1) + wn * 32 + 16 * (i & 1) + (lane & 15)
                               : n0 + wn * 64 + 16 * i + (lane & 15);
        F.q[t][i] = lora4_km(rq, r, n, r, lane);
        if (hi) F.qh[t][i] = lora4_km(rq, r, n, r, lane, 16);
      } else {
        const int64_t n = n0 + wn * 64 + 16 * i + (lane & 15);
        F.q[t][i] = lora4_mn(rq, A.lldq, n, r, lane);
        if (hi) F.qh[t][i] = lora4_mn(rq, A.lldq, n, r, lane, 16);
      }
    }
  }
}

template <int DT, bool DUAL, int LT>
__device__ __forceinline__ f32x4 acc_lora(const KArgs& A, const f32x4& a, const Lora& F, int i,
                                          int j) {
  f32x4 v = a;
#pragma unroll
  for (int t = 0; t < LT; ++t) {
    if (DUAL && (i >> 1) != t) continue;
    f32x4 l = mfma16<DT>(F.q[t][i], F.p[t][j], f32x4{0.0f, 0.0f, 0.0f, 0.0f});
    if (A.lrank > 16) l = mfma16<DT>(F.qh[t][i], F.ph[t][j], l);
#pragma unroll
    for (int r = 0; r < 4; ++r)
      v[r] = round16<DT>(round16<DT>(v[r]) + round16<DT>(A.lalpha[t] * round16<DT>(l[r])));
  }
  return v;
}

template <int DT, bool AK, bool BK, int EPI, int CACHE, int LT, int S>
__global__ __launch_bounds__(kThreads, S == 2 ? 2 : 1) void st16_kernel(const KArgs A) {
  static_assert(LT == 0 || AK, "adapter terms ride with a K-major A (P's rows are tokens)");
  // EPI_F32 with CACHE_NONE / CACHE_BF16: partials of a plain / dual product
  constexpr bool DUAL = EPI == EPI_GLU || (EPI == EPI_F32 && CACHE == CACHE_BF16);
  constexpr bool TAIL = !AK && !BK;
  constexpr bool X3 = DT == kF32;
  static_assert(!X3 || EPI == EPI_F32, "fp32 products write fp32");
  if constexpr (X3)
    if (any_flag(A.flags)) return;
  static_assert(!DUAL || (AK && BK), "F1's operands are K-major");
  extern __shared__ __attribute__((aligned(16))) uint16_t lds[];
  const int tiles = A.tiles_m * A.tiles_n;
  const int split = EPI == EPI_F32 ? blockIdx.x / tiles : 0;
  int tm, tn;
  tile_of(blockIdx.x - split * tiles, tiles, A.tiles_m, A.tiles_n, tm, tn);
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave & 1, wm = wave >> 1;
  const int64_t m0 = (int64_t)tm * kT, n0 = (int64_t)tn * kT;
  const int64_t lda = A.a[0].ld, ldb = A.b[0].ld;   // pair 1 shares them (host check)
  const int64_t nb0 = DUAL ? n0 / 2 : n0;
  const int64_t nrows = DUAL ? A.D : A.N;

  // Loads.  Load i of an operand fills 1 KiB block q = 4 i + wave of its stage:
  //   K-major: rows 8 q .. + 7, lane l row 8 q + l / 8, chunk (l % 8) ^ (row & 6)
  //     (DUAL B: each wave's 64 columns are 32 gate and the same 32 up rows, so
  //     tile row r is gate or up by its bit 5, which is bit 0 of i);
  //   MN-major: k-rows 4 q .. + 3, lane l k-row 4 q + l / 16, chunk
  //     (l % 16) ^ mn_swz(k-row).
  // Past an edge the VGPR offset decides (num_records, or kOOB), as in
  // gemm16_kernel.h; past the last k-tile num_records is 0.
  uint32_t oa[4], ob[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int q = 4 * i + wave;
    const int ck = (lane & 7) ^ ((lane >> 3) & 6);
    const int r = 8 * q + (lane >> 3);
    const int rw = DUAL ? 32 * (i >> 1) + 8 * wave + (lane >> 3) : r;
    const int kr = 4 * q + (lane >> 4);
    const int cm = (lane & 15) ^ mn_swz(kr);
    oa[i] = AK ? (uint32_t)(((int64_t)r * lda + ck * 8) * 2)
               : m0 + cm * 8 < A.M ? (uint32_t)(((int64_t)kr * lda + cm * 8) * 2) : kOOB;
    ob[i] = BK ? (uint32_t)(((int64_t)rw * ldb + ck * 8) * 2)
               : n0 + cm * 8 < A.N ? (uint32_t)(((int64_t)kr * ldb + cm * 8) * 2) : kOOB;
  }
  const uint32_t stepa = AK ? (uint32_t)(kBK * 2) : (uint32_t)(kBK * lda * 2);
  const uint32_t stepb = BK ? (uint32_t)(kBK * 2) : (uint32_t)(kBK * ldb * 2);
  // Segments of the k loop: the operand pairs, or (X3) the six plane products
  // of each pair
  const int nseg = X3 ? 6 * A.npairs : A.npairs;
  auto pair_of = [&](int sg) { return X3 ? (A.npairs == 2 ? sg & 1 : 0) : sg; };
  auto ktiles = [&](int sg) { return (int)((A.K[pair_of(sg)] + kBK - 1) / kBK); };
  int nk_all = ktiles(0) + (A.npairs == 2 ? ktiles(1) : 0);
  if (X3) nk_all *= 6;
  const int kb = EPI == EPI_F32 ? min(nk_all, split * A.kt_per_split) : 0;
  const int nk = EPI == EPI_F32 ? min(nk_all - kb, A.kt_per_split) : nk_all;
  // the k-tile being loaded: its segment's buffers and byte deltas, the k-tiles
  // left in the segment and in the block's range
  i32x4 ra, rb, rbu;
  uint32_t da, db;
  int left, rem = nk, seg = 0;
  auto open = [&](int sg, int lk) {
    const int pr = pair_of(sg);
    const uint16_t* pa = A.a[pr].p;
    const uint16_t* pb = A.b[pr].p;
    if constexpr (X3) {
      // planes (A, B) of term t: (0,2) (2,0) (1,1) (0,1) (1,0) (0,0)
      const int t4 = 4 * (A.npairs == 2 ? sg >> 1 : sg);
      pa += ((0x010120 >> t4) & 15) * A.plane_a[pr];
      pb += ((0x001102 >> t4) & 15) * A.plane_b[pr];
    }
    // a partial last k-tile: the buffers start at its first row (TAIL)
    const int64_t k0 = TAIL && ((int64_t)lk + 1) * kBK > A.K[pr] ? (int64_t)lk * kBK : 0;
    ra = AK ? rsrc_sgpr(pa + m0 * lda, (A.M - m0) * lda * 2)
            : rsrc_sgpr(pa + k0 * lda + m0, ((A.K[pr] - k0) * lda - m0) * 2);
    rb = BK ? rsrc_sgpr(pb + nb0 * ldb, (nrows - nb0) * ldb * 2)
            : rsrc_sgpr(pb + k0 * ldb + n0, ((A.K[pr] - k0) * ldb - n0) * 2);
    rbu = DUAL ? rsrc_sgpr(A.b_up + nb0 * ldb, (nrows - nb0) * ldb * 2) : rb;
    da = TAIL && k0 ? 0 : (uint32_t)lk * stepa;
    db = TAIL && k0 ? 0 : (uint32_t)lk * stepb;
    left = ktiles(sg) - lk;
  };
  int lk0 = kb;
  while (seg + 1 < nseg && lk0 >= ktiles(seg)) lk0 -= ktiles(seg++);
  open(seg, lk0);
  auto advance = [&]() {
    da += stepa;
    db += stepb;
    --left;
    if (--rem <= 0) {
      ra[2] = rb[2] = rbu[2] = 0;
      da = db = 0;
    } else if (left == 0) {
      open(++seg, 0);
    } else if (TAIL && left == 1) {
      open(seg, ktiles(seg) - 1);
    }
  };
  // load p (0..7): even p -> A block p / 2, odd -> B
  auto issue = [&](int p, int st) {
    const int i = p >> 1;
    uint16_t* dst = lds + (st * 2 + (p & 1)) * kOp + (4 * i + wave) * 512;
    if (p & 1) load_lds(DUAL && (i & 1) ? rbu : rb, dst, ob[i], db);
    else load_lds(ra, dst, oa[i], da);
  };

  f32x4 acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  // fragment q of sub-step s: even q -> B (n block q / 2), odd q -> A (m block q / 2)
  const int nof = nt16::lds_off(wn * 64 + (lane & 15), lane >> 4);
  const int mof = nt16::lds_off(wm * 64 + (lane & 15), lane >> 4);
  const int nof1 = nt16::lds_off(wn * 64 + (lane & 15), (lane >> 4) + 4);
  const int mof1 = nt16::lds_off(wm * 64 + (lane & 15), (lane >> 4) + 4);
  const int mnk = 8 * (lane >> 4) + ((lane & 15) >> 2);     // k-row of the first read
  const int mn_lane = mnk * kT + ((lane & 3) >> 1) * 8 + (lane & 1) * 4;
  const int mn_fx = 8 * mn_swz(mnk);                        // XOR on the column (multiples of 16)
  bf16x8 f0[8], f1[8];
  auto rd = [&](int st, int s, int q) -> bf16x8 {
    const uint16_t* base = lds + st * 2 * kOp;
    const bool bside = (q & 1) == 0;
    if ((bside && BK) || (!bside && AK)) {
      const int o = bside ? kOp + (s ? nof1 : nof) : (s ? mof1 : mof);
      return *reinterpret_cast<const bf16x8*>(base + o + (q >> 1) * 16 * kBK);
    }
    const uint16_t* p = base + (bside ? kOp : 0) + mn_lane + s * 32 * kT +
                        (((bside ? 64 * wn : 64 * wm) + 16 * (q >> 1)) ^ mn_fx);
    const i16x4 lo = lds_read_tr(p);
    const i16x4 hi = lds_read_tr(p + 4 * kT);
    return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  };

  // prologue: tiles 0 .. S - 2 and half of tile S - 1; F0 of tile 0
#pragma unroll
  for (int st = 0; st < S; ++st) {
#pragma unroll
    for (int p = 0; p < (st == S - 1 ? 4 : 8); ++p) issue(p, st);
    if (st < S - 1) advance();
  }
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((S - 2) * 8 + 4) : "memory");
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    f0[q] = rd(0, 0, q);
    __builtin_amdgcn_sched_barrier(0);
  }

  constexpr Order4 ord;
  int cur = 0, prev = S - 1;
  for (int kt = 0; kt < nk; ++kt) {
    const int next = cur + 1 == S ? 0 : cur + 1;
    static_for<0, 32>([&](auto tc) {
      constexpr int t = decltype(tc)::value;
      if constexpr (t < 16) {
        constexpr int i = ord.i[t], j = ord.j[t];
        mfma32<DT>(acc[i][j], f0[2 * i], f0[2 * j + 1]);
        if constexpr (t < 8) f1[t] = rd(cur, 1, t);
        if constexpr (t >= 3 && (t - 3) % 4 == 0) issue(4 + (t - 3) / 4, prev);
        if constexpr (t == 15) {
          asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((S - 2) * 8)
                       : "memory");
          advance();
        }
      } else {
        constexpr int i = ord.i[t - 16], j = ord.j[t - 16];
        mfma32<DT>(acc[i][j], f1[2 * i], f1[2 * j + 1]);
        if constexpr (t < 24) f0[t - 16] = rd(next, 0, t - 16);
        if constexpr ((t - 19) % 4 == 0 && t >= 19) issue((t - 19) / 4, cur);
      }
      __builtin_amdgcn_sched_barrier(0);
    });
    prev = cur;
    cur = next;
  }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");

  // lane holds tile column 64 wn + 16 i + 4 (lane / 16) + 0..3 of tile row
  // 64 wm + 16 j + lane % 16 in acc[i][j] (DUAL: i < 2 gate column 32 wn + 16 i
  // + .., i >= 2 the same up column)
  const int etid = epi_tid();
  const int el = etid & 63;
  if constexpr (EPI == EPI_F32) {
    // partials [split][M][ldc] fp32; DUAL: up columns start at column D
    float* const out = A.ws + (int64_t)split * A.M * A.ldc;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int64_t n = (DUAL ? nb0 + wn * 32 + 16 * (i & 1) : n0 + wn * 64 + 16 * i) + 4 * (el >> 4);
      if (n >= nrows) continue;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int64_t m = m0 + wm * 64 + 16 * j + (el & 15);
        f32x4 v = acc[i][j];
        asm volatile("" : "+v"(v));
        if constexpr (X3) v *= A.alpha;   // 1 for partials
        if (m < A.M) *reinterpret_cast<f32x4*>(out + m * A.ldc + (DUAL && i >= 2 ? A.D : 0) + n) = v;
      }
    }
    return;
  } else {
  Lora F;
  if constexpr (LT > 0) lora_load<DUAL, LT>(A, m0, n0, wm, wn, el, F);
  if constexpr (!DUAL) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        f32x4 base = acc[i][j];
        asm volatile("" : "+v"(base));
        const f32x4 v = LT > 0 ? acc_lora<DT, false, LT>(A, base, F, i, j) : base;
        *reinterpret_cast<uint2*>(lds + (wm * 64 + 16 * j + (el & 15)) * kLdOut + wn * 64 + 16 * i +
                                  4 * (el >> 4)) =
            make_uint2(pack16<DT>(v[0], v[1]), pack16<DT>(v[2], v[3]));
      }
    __syncthreads();
    const int cl = (etid & 15) * 8;
    const int64_t n = n0 + cl;
    const bool nok = n < A.N;
    if constexpr (EPI == EPI_STORE) {
#pragma unroll
      for (int p = 0; p < 8; ++p) {
        const int r = p * 16 + (etid >> 4);
        const uint4 w = *reinterpret_cast<const uint4*>(lds + r * kLdOut + cl);
        if (nok && m0 + r < A.M) *reinterpret_cast<uint4*>(A.C + (m0 + r) * A.ldc + n) = w;
      }
    } else {
      // B1 on a 16-bit cache: SwiGLU backward of the staged grad_h_mid.  Every
      // load of a pass precedes its stores (the outputs may lie over the cache)
      static_assert(EPI == EPI_DGLU && CACHE == CACHE_BF16, "B1 on a 16-bit cache");
#pragma unroll 2
      for (int p = 0; p < 8; ++p) {
        const int r = p * 16 + (etid >> 4);
        if (!nok || m0 + r >= A.M) continue;
        const int64_t off = (m0 + r) * A.D + n;
        float dh[8], hg[8], hu[8], og[8], ou[8], oh[8];
        wide8<DT>(*reinterpret_cast<const uint4*>(lds + r * kLdOut + cl), dh);
        wide8<DT>(*reinterpret_cast<const uint4*>(A.h_gate + off), hg);
        wide8<DT>(*reinterpret_cast<const uint4*>(A.h_up + off), hu);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          float hact;
          swiglu_bwd1(dh[e], hg[e], hu[e], og[e], ou[e], hact);
          oh[e] = hact * hu[e];
        }
        *reinterpret_cast<uint4*>(A.grad_gate + off) = pack8<DT>(og);
        *reinterpret_cast<uint4*>(A.grad_up + off) = pack8<DT>(ou);
        if (A.h_mid_hat) *reinterpret_cast<uint4*>(A.h_mid_hat + off) = pack8<DT>(oh);
      }
    }
  } else {
    // F1 with no codec
    uint16_t* sg = lds;
    uint16_t* su = lds + kT * kGluLdS;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        f32x4 base = acc[i][j];
        asm volatile("" : "+v"(base));
        const f32x4 v = LT > 0 ? acc_lora<DT, true, LT>(A, base, F, i, j) : base;
        *reinterpret_cast<uint2*>((i < 2 ? sg : su) + (wm * 64 + 16 * j + (el & 15)) * kGluLdS +
                                  wn * 32 + 16 * (i & 1) + 4 * (el >> 4)) =
            make_uint2(pack16<DT>(v[0], v[1]), pack16<DT>(v[2], v[3]));
      }
    __syncthreads();
    const int cl = (etid & 7) * 8;
    const int64_t d = (n0 >> 1) + cl;
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const int r = p * 32 + (etid >> 3);
      if (d >= A.D || m0 + r >= A.M) continue;
      const uint4 wg = *reinterpret_cast<const uint4*>(sg + r * kGluLdS + cl);
      const uint4 wu = *reinterpret_cast<const uint4*>(su + r * kGluLdS + cl);
      const int64_t off = (m0 + r) * A.D + d;
      if (A.h_mid) {
        float g[8], u[8], h[8];
        wide8<DT>(wg, g);
        wide8<DT>(wu, u);
#pragma unroll
        for (int e = 0; e < 8; ++e) h[e] = silu_mul1(g[e], u[e]);
        *reinterpret_cast<uint4*>(A.h_mid + off) = pack8<DT>(h);
      }
      if constexpr (CACHE == CACHE_BF16) {
        *reinterpret_cast<uint4*>(A.h_gate + off) = wg;
        *reinterpret_cast<uint4*>(A.h_up + off) = wu;
      }
    }
  }
  }
}

}  // namespace st16

// The same product as launch_nt16's, on 128 x 128 tiles (A.tiles_m / tiles_n
// are recounted here; A.ksplit blocks per tile for EPI_F32).
template <int DT, bool AK, bool BK, int EPI, int CACHE, int LT, int S>
int launch_st16(KArgs A, hipStream_t st) {
  auto kern = st16::st16_kernel<DT, AK, BK, EPI, CACHE, LT, S>;
  static bool attr_set = false;   // per instantiation
  if (!attr_set) {
    if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                            st16::lds_bytes<S>()) != hipSuccess)
      return kErrLaunch;
    attr_set = true;
  }
  A.tiles_m = (int)((A.M + st16::kT - 1) / st16::kT);
  A.tiles_n = (int)((A.N + st16::kT - 1) / st16::kT);
  const int64_t blocks = (int64_t)A.tiles_m * A.tiles_n * (EPI == EPI_F32 ? A.ksplit : 1);
  if (blocks <= 0) return kOk;
  if (blocks > 0x7FFFFFFF) return kErrTooLarge;
  hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(st16::kThreads), st16::lds_bytes<S>(), st,
                     A);
  return hipGetLastError() == hipSuccess ? kOk : kErrLaunch;
}

}  // namespace gemm
}  // namespace cpt
