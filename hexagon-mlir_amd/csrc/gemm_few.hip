// C[M,N] = A[M,K] * op(B) where tiles of 128 x 128 would leave compute units without work (fp16 / bf16 in, fp32 sums): tiles of
// 16 x 16 to 128 x 64 and 96 x 96 in one round, a workgroup of eight waves to a tile; and parts of a long K (plan_gemm_parts).
//
// What bounds it: a CU takes in about 90 GB/s through L2 whatever it does with it, and a tile of BM x BN asks for (BM + BN) x K
// operands. 128 x 128 tiles run at that rate (0.31 us per 64 of K, K = 3072), so what is left is to have every CU take in a share:
// a smaller tile reads each operand more often, but all of the chip reads. Per slab the LDS is the next limit (128 bytes a
// clock): waves side by side read the same rows, so the shapes below give a wave 32 x 32 to 64 x 64 of the tile and let wave
// groups take the 32-k steps of a slab in turn; their sums meet in LDS at the end, where the tile leaves in whole rows. Eight
// waves with small accumulators beat four that own all of the tile (64 x 64, K = 3072: 11.5 against 17.5 us, a slab's reads
// and multiplications of one wave per SIMD have nothing to run beside). Cold weights, bf16, us, before (128 x 128 tiles, for [N,K]
// weights up to 64 rows gemm_skinny.hip) -> now:
//   [K,N]  16 rows: 768 x 768 8.8 -> 4.3, 4096 x 4096 30 -> 18;  64 rows: 768 x 3072 20 -> 8.8, 4096 x 4096 35 -> 19
//   [K,N]  N = 768, K = 3072: 256 rows 20.7 -> 9.3, 1000 rows 21 -> 12, 2000 rows 21.7 -> 17.4;  K = 768, 2000 rows 9.9 -> 7.8
//   [N,K]  N = 4096, K = 4096: 64 rows 14.5 -> 12, 128 rows 37.7 -> 16, 256 rows 37 -> 20, 500 rows 37 -> 27
#include <algorithm>
#include <type_traits>

#include "hexmi_common.h"

namespace hexmi {
namespace {

__device__ __attribute__((aligned(16))) unsigned g_few_zeros[4];      // where a copy of a chunk past K points

__device__ __forceinline__ f32x4 mfma16(const f16x8& b, const f16x8& a, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(b, a, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mfma16(const bf16x8& b, const bf16x8& a, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(b, a, c, 0, 0, 0);
}
template <typename T> struct Frag8;
template <> struct Frag8<f16> { typedef f16x8 V; };
template <> struct Frag8<bf16> { typedef bf16x8 V; };

// TM x TN: 16 x 16 tiles of a wave; SM x SN waves side by side; KH wave groups share the 32-k steps of a slab, STEPS (one or two) each.
template <int TM_, int TN_, int SM_, int SN_, int KH_, int STEPS_ = 1>
struct Shape {
  static constexpr int TM = TM_, TN = TN_, SM = SM_, SN = SN_, KH = KH_, STEPS = STEPS_, kWaves = SM * SN * KH, kThreads = kWaves * kWave;
  static constexpr int BM = SM * TM * 16, BN = SN * TN * 16, BK = KH * STEPS * 32;
  static constexpr int kStage = (BM + BN) * BK;                  // elements of a stage: rows of A, then B
};

// chunk c (16 bytes) of row r of a K-contiguous tile of BK elements a row sits at c ^ swz_row(r): sixteen rows of one chunk
// then cover all banks
template <int BK> __device__ __forceinline__ int swz_row(int r) { return BK == 64 ? (r >> 1) & 7 : r & 15; }
// N-contiguous tile of BN columns a row of k: the 32 lanes of a transposing read touch k % 4, k / 8 % 2 x 32 bytes, which the
// XOR spreads over the eight 32-byte slots of all banks
template <int BN> __device__ __forceinline__ int swz_col(int k) {
  if (BN == 96) return ((k >> 3) & 1) << 1;                     // (rows of three quarters of the banks: four start on different ones)
  if (BN == 128) return ((k & 3) | (((k >> 3) & 1) << 2)) << 1;
  return BN == 64 ? (((k >> 1) & 1) | (((k >> 3) & 1) << 1)) << 1 : ((k >> 3) & 1) << 1;
}

// Elements of K from a slab on, zero and less for slabs past the last one. The difference fits where slab * BK passes 2^31: near the
// longest K a slab past the last one wrapped round and was read from 2^31 elements before its row.
__host__ __device__ constexpr int rest_of(int K, int slab, int BK) { return (int)((unsigned)K - (unsigned)slab * (unsigned)BK); }
constexpr int kAnyMaxK = 0x7fffffff - 64;                        // the longest K of launch_gemm_any
static_assert(rest_of(kAnyMaxK, kAnyMaxK / 256, 256) == kAnyMaxK % 256 && rest_of(kAnyMaxK, kAnyMaxK / 256 + 4, 256) < 0 &&
              rest_of(kAnyMaxK, kAnyMaxK / 64 + 4, 64) < 0 && rest_of(kAnyMaxK, 0, 256) == kAnyMaxK, "slabs past the last one are past K");

// NS stages of a slab of KH * 32 k: copies fill all but one while that one is read; one barrier a slab. K % 8 == 0, operand rows
// on 16-byte boundaries ([K,N]: N % 8 == 0 too). runs: the output (and bias and residual) in runs of eight columns on
// 16-byte boundaries; otherwise they go by elements.
// ANY: operand rows at any alignment, any K and N ([K,N] weights with an odd N, views). A copy into LDS needs its 16 bytes on a
// boundary, a load into registers does not: two slabs are on their way in registers while a third is multiplied from one of two
// stages; tiles of 128 x 128 have one slab on its way, so that two fit a CU. Bound by the latency of a slab's loads as the copies are, so
// no load waits for a choice: a chunk that reaches past the end of K or of a [K,N] row is read as the last eight elements before it and
// shifted into place, with zeros behind K, on its way into LDS, in the last slab and the last column of tiles only. Rows of fewer than
// eight columns are read with the end of the row before (the first of B from its start); fewer than eight of K are one chunk, put
// together from elements. The last turns ask for no slab; the result leaves by up to eight elements of a thread at a time.
// us on 128 x 128 tiles that put such chunks together from elements under a branch of every load, a slab's one latency after the other /
// here ([K,N]): 128 x 7219 x 6656 299 / 47, 640 x 7031 x 3584 322 / 74, 16 x 4097 x 4096 120 / 18.5, 50 x 1001 x 768 48 / 5.3, 4000 x
// 4001 x 2048 160 / 96, 1021 x 50257 x 768 174 / 143; aligned neighbours with copies into LDS take 43, 61, 18, 5, 48 and 102. Few columns
// or little of K, there / by elements throughout / here: 65536 x 1 x 4096 203 / 866 / 132, 65536 x 7 x 768 57 / 167 / 29, 4096 x 4096 x 7
// 20 / 36 / 13. Short K on many tiles, there / with slabs of zeros asked for and one element after the other / here: 1021 x 50257 x 64
// 50 / 73 / 53, 65536 x 257 x 9 21 / 36 / 24, 20000 x 33 x 33 7.7 / 10.5 / 7.0. What alignment itself costs is a tenth to a fifth: rows on
// the boundaries / off them, [N,K] 128 x 7224 x 6651 37 / 43, [K,N] 44 / 47, 1021 x 50264 x 763 138 / 145. Two slabs on their way in
// 128 x 128 tiles leave one to a CU: 1021 x 50257 x 768 211, 640 x 7031 x 3584 140.
// PARTS: blockIdx.y takes a part of K; a form of its own, since working the part out first cost every small product of [K,N] weights a
// fortieth (3.10 us where it now takes 3.03).
template <typename T, typename OutT, typename S, int NS, bool TRANS_B, bool ANY, bool PARTS = false>
__global__ __launch_bounds__(S::kThreads, S::STEPS == 2 ? 4 : 2)
void gemm_few_kernel(const T* __restrict__ A, const T* __restrict__ B, OutT* C, int M, int N, int K, int64_t lda, int64_t ldb,
                     int64_t ldc, const OutT* __restrict__ bias, const OutT* resid, int64_t ldr, int tiles_m, int tiles_n,
                     int runs, int part) {
  constexpr int TM = S::TM, TN = S::TN, BM = S::BM, BN = S::BN, BK = S::BK, KH = S::KH, kWaves = S::kWaves, kThreads = S::kThreads;
  constexpr int kA = BM * BK / 512 / kWaves, kB = BN * BK / 512 / kWaves, kCopies = kA + kB;   // a wave's copies (1 KiB) of a slab
  static_assert(ANY || S::STEPS == 1, "a slab is one step of a wave");
  static_assert(kA * kWaves * 512 == BM * BK && kB * kWaves * 512 == BN * BK, "whole copies");
  constexpr int kStageBytes = S::kStage * 2, kPitch = BN + 4;    // pitch of the sums on their way out
  constexpr int kLds = std::max((ANY ? 2 : NS) * kStageBytes, KH * BM * kPitch * 4);
  __shared__ __attribute__((aligned(16))) char lds[kLds];

  const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int r16 = lane % 16, kg = lane / 16;
  int tm, tn;
  tile_of_block<8>(blockIdx.x, tiles_m, tiles_n, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;
  if constexpr (PARTS) {                                         // the part of K, whole slabs, whose sums go to a C of its own
    const int k0 = blockIdx.y * part;
    A += k0;
    B += TRANS_B ? (int64_t)k0 : k0 * ldb;
    C += blockIdx.y * (int64_t)M * ldc;
    K = K - k0 < part ? K - k0 : part;
  }

  // copy i of a slab moves chunks [i * 512 + wave * 64, + 64) of the tile: A's kA, then B's kB
  int voff[kCopies], kc[kCopies];
  const T* ptr[ANY ? kCopies : 1];
  int by[ANY ? kCopies : 1];                                     // ANY, [K,N]: columns the chunk was moved back to end at N
  if constexpr (ANY) {
#pragma unroll
    for (int i = 0; i < kCopies; ++i) {
      const int chunk = (i < kA ? i : i - kA) * kThreads + threadIdx.x;
      if (i < kA || TRANS_B) {
        const int row = chunk / (BK / 8), c = (chunk % (BK / 8)) ^ swz_row<BK>(row);
        const int left = (i < kA ? M - m0 : N - n0) - 1;
        ptr[i] = (i < kA ? A + (int64_t)m0 * lda : B + (int64_t)n0 * ldb) + (int64_t)(row < left ? row : left) * (i < kA ? lda : ldb) + c * 8;
        kc[i] = c * 8;
        by[i] = 0;
      } else {
        const int k = chunk / (BN / 8), c = (chunk % (BN / 8)) ^ swz_col<BN>(k);
        const int col = n0 + c * 8, at = col + 8 <= N ? col : N - 8;
        ptr[i] = B + (int64_t)k * ldb + at;
        kc[i] = k;
        by[i] = (col - at) & 7;                                  // (columns past N: anything, they are not stored)
      }
    }
  }
#pragma unroll
  for (int i = 0; i < (ANY ? 0 : kCopies); ++i) {
    const int chunk = (i < kA ? i : i - kA) * kThreads + threadIdx.x;
    if (i < kA || TRANS_B) {
      const int row = chunk / (BK / 8), c = (chunk % (BK / 8)) ^ swz_row<BK>(row);
      const int left = (i < kA ? M - m0 : N - n0) - 1;           // past the edge: the last row again, not stored
      voff[i] = (int)((int64_t)(row < left ? row : left) * (i < kA ? lda : ldb) * 2 + c * 16);
      kc[i] = c * 8;
    } else {
      const int k = chunk / (BN / 8), c = (chunk % (BN / 8)) ^ swz_col<BN>(k);
      const int left = N - n0 - 8;
      voff[i] = (int)((int64_t)k * ldb * 2 + (c * 8 < left ? c * 8 : left) * 2);
      kc[i] = k;
    }
  }
  const char* a_base = reinterpret_cast<const char*>(A + (int64_t)m0 * lda);
  const char* b_base = reinterpret_cast<const char*>(TRANS_B ? B + (int64_t)n0 * ldb : B + n0);
  const int64_t b_step = (TRANS_B ? BK : BK * ldb) * 2;
  const int slabs = (int)(((unsigned)K + BK - 1) / BK);
  auto copy = [&](int slab, int stage, auto ragged) __attribute__((always_inline)) {
    const char* a_from = a_base + (int64_t)slab * (BK * 2);
    const char* b_from = b_base + slab * b_step;
    char* to = lds + stage * kStageBytes + wave * 1024;
#pragma unroll
    for (int i = 0; i < kCopies; ++i) {
      const char* from = i < kA ? a_from : b_from;
      if constexpr (decltype(ragged)::value) {                   // the slab that reaches past K: zeros there
        const char* src = slab * BK + kc[i] < K ? from + voff[i] : reinterpret_cast<const char*>(g_few_zeros);
        copy_ptr_to_lds_asm(src, to + i * (kWaves * 1024));
      } else {
        copy_to_lds_asm(from, voff[i], to + i * (kWaves * 1024));
      }
    }
  };
  const int full = K / BK;
  auto copy_any = [&](int slab, int stage) __attribute__((always_inline)) {
    if (slab < full) copy(slab, stage, std::false_type{}); else copy(slab, stage, std::true_type{});
  };

  // this lane's fragments of a stage: wave group kh takes the slab's step kh (32 of K)
  const int kh = wave / (S::SM * S::SN), wm = wave % (S::SM * S::SN) / S::SN, wn = wave % S::SN;
  const int arow = wm * TM * 16 + r16;
  const int a_at = (arow * BK + ((kh * 4 + kg) ^ swz_row<BK>(arow)) * 8) * 2;
  int b_at[TN];
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    if (TRANS_B) {
      const int row = (wn * TN + j) * 16 + r16;
      b_at[j] = (BM * BK + row * BK + ((kh * 4 + kg) ^ swz_row<BK>(row)) * 8) * 2;
    } else {                                                     // lane i of 16: row i / 4, columns 4 (i % 4) .. + 3
      const int k = kh * 32 + kg * 8 + r16 / 4, col = (wn * TN + j) * 16 + (r16 & 3) * 4;
      b_at[j] = (BM * BK + k * BN + ((col / 8) ^ swz_col<BN>(k)) * 8 + col % 8) * 2;
    }
  }

  // bias and residual of this thread's runs of eight columns of the result, under the K walk
  constexpr int kRuns = (BM * BN / 8 + kThreads - 1) / kThreads;
  struct alignas(16) Run { OutT v[8]; };
  constexpr bool kEarly = !ANY || kRuns <= 2;                    // (128 x 128, two to a CU: no registers for them)
  Run add_b[kRuns], add_r[kRuns];
  auto ask = [&](int p) __attribute__((always_inline)) {
    const int idx = threadIdx.x + p * kThreads, row = idx / (BN / 8) % BM, col = idx % (BN / 8) * 8;
    const int gm = m0 + row < M ? m0 + row : M - 1, gn = n0 + col < N ? n0 + col : N - 8;
    if (bias) add_b[p] = *reinterpret_cast<const Run*>(bias + gn);
    if (resid) add_r[p] = *reinterpret_cast<const Run*>(resid + (int64_t)gm * ldr + gn);
  };
  if (kEarly && runs) {
#pragma unroll
    for (int p = 0; p < kRuns; ++p) ask(p);
  }

  f32x4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  typedef typename Frag8<T>::V Frag;
  struct Step { Frag a[TM], b[TN]; };
  auto read = [&](int stage, int st, Step& f) __attribute__((always_inline)) {   // st: step of the wave, KH * 32 of K apart
    const char* from = lds + stage * kStageBytes;
    const int far = st * (KH * 64), far_b = TRANS_B ? 0 : st * (KH * 32 * BN * 2);
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      if constexpr (TRANS_B) {
        f.b[j] = *reinterpret_cast<const Frag*>(from + (b_at[j] ^ far));
      } else {                                                   // four k on: the same place in its row
        union { i16x4 h[2]; Frag v; } u;
#pragma unroll
        for (int p = 0; p < 2; ++p)
          u.h[p] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4*)(from + b_at[j] + far_b + p * (4 * BN * 2)));
        f.b[j] = u.v;
      }
    }
#pragma unroll
    for (int i = 0; i < TM; ++i) f.a[i] = *reinterpret_cast<const Frag*>(from + (a_at ^ far) + i * (16 * BK * 2));   // the swizzle repeats
  };
  auto multiply = [&](const Step& f) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = mfma16(f.b[j], f.a[i], acc[i][j]);
  };
#define HEXMI_FENCE __builtin_amdgcn_sched_barrier(0)
  // The copies are assembly: the compiler would wait for all of them before any LDS read. Here a wave waits until at most `newer`
  // slabs of its own are in flight and its reads of the slab before have returned, then for every other wave.
  auto landed = [&](auto newer) __attribute__((always_inline)) {
    HEXMI_FENCE;
    __builtin_amdgcn_s_waitcnt(waitcnt_imm(decltype(newer)::value * kCopies));
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    HEXMI_FENCE;
  };
  if constexpr (ANY) {
    constexpr int kSets = S::STEPS == 2 ? 1 : 2;                 // slabs on their way
    u32x4 set[kSets][kCopies];
    // PLAIN: every chunk lies inside its row and K. The other form takes any slab, one past the last too (zeros).
    // first: the slab at the start of B, whose first rows, where they are shorter than a chunk, are read from there on: so many elements
    // on from where the chunk's end would be the row's
    auto ahead_of = [&](int i) __attribute__((always_inline)) {
      const int ahead = 8 - N - (kc[i] < 8 ? kc[i] : 8) * (ldb < 8 ? (int)ldb : 8);
      return !TRANS_B && i >= kA && ahead > 0 ? ahead : 0;
    };
    auto fetch = [&](int slab, u32x4 (&to)[kCopies], auto plain, auto first) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < kCopies; ++i) {
        if constexpr (decltype(plain)::value) {
          __builtin_memcpy(&to[i], ptr[i] + (i < kA || TRANS_B ? (int64_t)slab * BK : (int64_t)slab * BK * ldb), 16);
        } else {
          const int left = rest_of(K, slab, BK) - kc[i];         // elements or rows before the end of K; from the slab's start on where
                                                                 // eight (one) are left, and before the end of K otherwise
          const int k0 = (int)((unsigned)slab * (unsigned)BK);   // (slabs past the last one: any)
          if (i < kA || TRANS_B) __builtin_memcpy(&to[i], ptr[i] + (left > 8 ? k0 : K - 8 - kc[i]), 16);
          else __builtin_memcpy(&to[i], ptr[i] + (int64_t)(left > 1 ? k0 : K - 1 - kc[i]) * ldb + (decltype(first)::value ? ahead_of(i) : 0), 16);
        }
      }
    };
    auto put = [&](const u32x4 (&from)[kCopies], int slab, int stage, auto plain, auto first) __attribute__((always_inline)) {
      char* to = lds + stage * kStageBytes + threadIdx.x * 16;
#pragma unroll
      for (int i = 0; i < kCopies; ++i) {
        u32x4 v = from[i];
        if constexpr (!decltype(plain)::value) {
          const int left = rest_of(K, slab, BK) - kc[i];
          const u32x4 zero = {0u, 0u, 0u, 0u};
          v = shift_columns(v, zero, i < kA || TRANS_B ? (left < 8 ? 8 - left : 0) & 7 : by[i] - (decltype(first)::value ? ahead_of(i) : 0));
          v = left > 0 ? v : zero;
        }
        *reinterpret_cast<u32x4*>(to + (i < kA ? i * kThreads * 16 : BM * BK * 2 + (i - kA) * kThreads * 16)) = v;
      }
    };
    auto meet = [&]() __attribute__((always_inline)) {           // every wave's writes and reads of LDS are done; loads stay in flight
      HEXMI_FENCE;
      __builtin_amdgcn_s_waitcnt(waitcnt_imm(63));
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      HEXMI_FENCE;
    };
    if (K < 8) {                                                 // rows of A shorter than a chunk: chunk 0 by elements, zeros for the rest
      if (K > 0) {
        typedef unsigned short E;
        constexpr int kLoadsA = (BM * 8 + kThreads - 1) / kThreads, kLoadsB = (BN * 8 + kThreads - 1) / kThreads;
        E va[kLoadsA], vb[kLoadsB];
        const int last_m = M - m0 - 1, last_n = N - n0 - 1;
#pragma unroll
        for (int t = 0; t < kLoadsA; ++t) {
          const int e = threadIdx.x + t * kThreads, row = e / 8, k = e % 8;
          va[t] = reinterpret_cast<const E*>(A)[(int64_t)(m0 + (row < last_m ? row : last_m)) * lda + (k < K ? k : K - 1)];
        }
#pragma unroll
        for (int t = 0; t < kLoadsB; ++t) {
          const int e = threadIdx.x + t * kThreads, n = TRANS_B ? e / 8 : e % BN, k = TRANS_B ? e % 8 : e / BN;
          const int64_t gn = n0 + (n < last_n ? n : last_n), gk = k < K ? k : K - 1;
          vb[t] = reinterpret_cast<const E*>(B)[TRANS_B ? gn * ldb + gk : gk * ldb + gn];
        }
        for (int e = threadIdx.x; e < kStageBytes / 16; e += kThreads) reinterpret_cast<u32x4*>(lds)[e] = u32x4{0u, 0u, 0u, 0u};
        __syncthreads();
        E* st = reinterpret_cast<E*>(lds);
#pragma unroll
        for (int t = 0; t < kLoadsA; ++t) {
          const int e = threadIdx.x + t * kThreads, row = e / 8, k = e % 8;
          if (row < BM && k < K) st[row * BK + swz_row<BK>(row) * 8 + k] = va[t];
        }
#pragma unroll
        for (int t = 0; t < kLoadsB; ++t) {
          const int e = threadIdx.x + t * kThreads, n = TRANS_B ? e / 8 : e % BN, k = TRANS_B ? e % 8 : e / BN;
          if (n < BN && k < K)
            st[BM * BK + (TRANS_B ? n * BK + swz_row<BK>(n) * 8 + k : k * BN + ((n / 8) ^ swz_col<BN>(k)) * 8 + n % 8)] = vb[t];
        }
        __syncthreads();
        Step f;                                                  // (the slab's second step would multiply zeros)
        read(0, 0, f);
        multiply(f);
      }
    } else {
      constexpr std::true_type kPlain{}, kFirst{}, kEnd{};
      constexpr std::false_type kAny{};
      // slab j from its stage; slab j + 1 from its set into the other stage, which slab j - 1 has left; the next slab into that set.
      // kEnd: the last turns, nothing further to ask for
      auto turn = [&](int j, int stage, u32x4 (&next)[kCopies], auto plain, auto end) __attribute__((always_inline)) {
        meet();
#pragma unroll
        for (int st = 0; st < S::STEPS; ++st) {
          Step f;
          read(stage, st, f);
          if (st == 0) {
            if constexpr (decltype(end)::value) {
              if (j + 1 < slabs) put(next, j + 1, stage ^ 1, kAny, kAny);
            } else {
              put(next, j + 1, stage ^ 1, plain, kAny);
              fetch(j + 1 + kSets, next, plain, kAny);
            }
            HEXMI_FENCE;
          }
          multiply(f);
        }
      };
      fetch(0, set[0], kAny, kFirst);
      if constexpr (kSets > 1) fetch(1, set[1], kAny, kAny);
      put(set[0], 0, 0, kAny, kFirst);
      int j = 0;
      if (slabs > kSets) {
        fetch(kSets, set[0], kAny, kAny);
        if (TRANS_B || n0 + BN <= N) {
          const int whole = K / BK;
          for (; j + 2 + kSets < whole; j += 2) {
            turn(j, 0, set[kSets - 1], kPlain, kAny);
            turn(j + 1, 1, set[0], kPlain, kAny);
          }
        }
        for (; slabs - j > kSets + 1; j += 2) {                  // (the last slab but one: zeros asked for that no turn takes)
          turn(j, 0, set[kSets - 1], kAny, kAny);
          turn(j + 1, 1, set[0], kAny, kAny);
        }
      }
      turn(j, 0, set[kSets - 1], kAny, kEnd);
      if (j + 1 < slabs) turn(j + 1, 1, set[0], kAny, kEnd);
      if (kSets > 1 && j + 2 < slabs) turn(j + 2, 0, set[kSets - 1], kAny, kEnd);
    }
  } else {
    HEXMI_FENCE;
#pragma unroll
    for (int j = 0; j < NS - 1; ++j)
      if (j < slabs) copy_any(j, j);
    int stage = 0, j = 0;
    auto step = [&](auto newer, auto next) __attribute__((always_inline)) {   // next: the copies that follow into the free stage
      landed(newer);
      next();
      HEXMI_FENCE;
      Step f;
      read(stage, 0, f);
      multiply(f);
      stage = stage == NS - 1 ? 0 : stage + 1;
      ++j;
    };
    auto free_stage = [&]() { return stage == 0 ? NS - 1 : stage - 1; };
    constexpr std::integral_constant<int, NS - 2> kBehind{};
    while (j + NS - 1 < full) step(kBehind, [&]() __attribute__((always_inline)) { copy(j + NS - 1, free_stage(), std::false_type{}); });
    if (j + NS - 1 < slabs) step(kBehind, [&]() __attribute__((always_inline)) { copy(j + NS - 1, free_stage(), std::true_type{}); });
    auto last = [&](auto left) __attribute__((always_inline)) {    // left: slabs behind this one
      if (j + decltype(left)::value < slabs) step(left, []() __attribute__((always_inline)) {});
    };
    if constexpr (NS > 7) last(std::integral_constant<int, 6>{});
    if constexpr (NS > 6) last(std::integral_constant<int, 5>{});
    if constexpr (NS > 5) last(std::integral_constant<int, 4>{});
    if constexpr (NS > 4) last(std::integral_constant<int, 3>{});
    if constexpr (NS > 3) last(std::integral_constant<int, 2>{});
    if constexpr (NS > 2) last(std::integral_constant<int, 1>{});
    last(std::integral_constant<int, 0>{});
    static_assert(NS >= 2 && NS <= 8, "the ladder above");
  }
#undef HEXMI_FENCE

  // the wave groups' sums meet in LDS and leave in rows
  __syncthreads();
  float* red = reinterpret_cast<float*>(lds);
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int jj = 0; jj < TN; ++jj)                              // a lane: row lane % 16, columns 4 (lane / 16) .. + 3
      *reinterpret_cast<f32x4*>(red + (kh * BM + (wm * TM + i) * 16 + r16) * kPitch + (wn * TN + jj) * 16 + kg * 4) = acc[i][jj];
  __syncthreads();
  if (runs) {
#pragma unroll
    for (int p = 0; p < kRuns; ++p) {
      const int idx = threadIdx.x + p * kThreads, row = idx / (BN / 8), col = idx % (BN / 8) * 8;
      if (BM * BN / 8 % kThreads && row >= BM) break;
      if (!kEarly) ask(p);
      f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = s0;
#pragma unroll
      for (int h = 0; h < KH; ++h) {
        const float* from = red + (h * BM + row) * kPitch + col;
        s0 += *reinterpret_cast<const f32x4*>(from);
        s1 += *reinterpret_cast<const f32x4*>(from + 4);
      }
      Run out;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float v = e < 4 ? s0[e % 4] : s1[e % 4];
        if (bias) v += to_f32<OutT>(add_b[p].v[e]);
        if (resid) v += to_f32<OutT>(add_r[p].v[e]);
        out.v[e] = from_f32<OutT>(v);
      }
      if (m0 + row < M && n0 + col < N) *reinterpret_cast<Run*>(C + (int64_t)(m0 + row) * ldc + n0 + col) = out;
    }
  } else {
    // By elements, up to eight of a thread at a time. (A residual that is the output itself: an element is read and written by one thread.)
    constexpr int kEach = (BM * BN + kThreads - 1) / kThreads, kAtOnce = kEach % 8 == 0 ? 8 : kEach % 6 == 0 ? 6 : kEach % 4 == 0 ? 4 : kEach;
    static_assert(kAtOnce <= 8 && (kEach == 1 || kEach * kThreads == BM * BN), "whole groups");
#pragma unroll 1
    for (int base = threadIdx.x; base < BM * BN; base += kAtOnce * kThreads) {
      float v[kAtOnce];
#pragma unroll
      for (int u = 0; u < kAtOnce; ++u) {
        const int idx = base + u * kThreads;
        v[u] = 0.f;
#pragma unroll
        for (int h = 0; h < KH; ++h) v[u] += red[(h * BM + idx / BN) * kPitch + idx % BN];
      }
      auto row_of = [&](int u) { const int row = m0 + (base + u * kThreads) / BN; return row < M ? row : M - 1; };
      auto col_of = [&](int u) { const int col = n0 + (base + u * kThreads) % BN; return col < N ? col : N - 1; };
      if (bias) {
#pragma unroll
        for (int u = 0; u < kAtOnce; ++u) v[u] += to_f32<OutT>(bias[col_of(u)]);
      }
      if (resid) {
#pragma unroll
        for (int u = 0; u < kAtOnce; ++u) v[u] += to_f32<OutT>(resid[(int64_t)row_of(u) * ldr + col_of(u)]);
      }
#pragma unroll
      for (int u = 0; u < kAtOnce; ++u) {
        const int idx = base + u * kThreads, row = m0 + idx / BN, col = n0 + idx % BN;
        if (row < M && col < N) C[(int64_t)row * ldc + col] = from_f32<OutT>(v[u]);
      }
    }
  }
}

template <int BM, int BN> struct FewShape;                       // waves, stages: what measured fastest of two to five forms each
template <> struct FewShape<16, 16> { typedef Shape<1, 1, 1, 1, 8> S; static constexpr int NS = 8; };
template <> struct FewShape<16, 32> { typedef Shape<1, 2, 1, 1, 8> S; static constexpr int NS = 6; };
template <> struct FewShape<32, 32> { typedef Shape<2, 2, 1, 1, 8> S; static constexpr int NS = 5; };
template <> struct FewShape<32, 64> { typedef Shape<2, 2, 1, 2, 4> S; static constexpr int NS = 6; };
template <> struct FewShape<64, 64> { typedef Shape<2, 4, 2, 1, 4> S; static constexpr int NS = 4; };
template <> struct FewShape<128, 64> { typedef Shape<4, 4, 2, 1, 4> S; static constexpr int NS = 3; };
template <> struct FewShape<48, 32> { typedef Shape<3, 2, 1, 1, 8> S; static constexpr int NS = 4; };
template <> struct FewShape<96, 64> { typedef Shape<3, 4, 2, 1, 4> S; static constexpr int NS = 3; };
template <> struct FewShape<64, 96> { typedef Shape<4, 3, 1, 2, 4> S; static constexpr int NS = 3; };
template <> struct FewShape<96, 96> { typedef Shape<3, 6, 2, 1, 4> S; static constexpr int NS = 3; };
template <> struct FewShape<16, 64> { typedef Shape<1, 4, 1, 1, 8> S; static constexpr int NS = 4; };      // parts of K only,
template <> struct FewShape<16, 128> { typedef Shape<1, 8, 1, 1, 8> S; static constexpr int NS = 2; };     // these two
typedef Shape<4, 2, 2, 4, 1, 2> AnyShape128;                     // 128 x 128, ANY: two to a CU

// C[M,N] = the sums of the parts of K, in their order, + bias + residual: one rounding. A row of the sums is pitch floats, whole eights.
template <typename OutT>
__global__ __launch_bounds__(128)
void gemm_merge_kernel(const float* __restrict__ sums, OutT* C, int M, int N, int pitch, int parts, int64_t ldc,
                       const OutT* __restrict__ bias, const OutT* resid, int64_t ldr) {
  const int at = blockIdx.x * 128 + threadIdx.x, per_row = pitch / 4, row = at / per_row, col = at % per_row * 4;
  if (row >= M) return;
  const int64_t all = (int64_t)M * pitch;
  const float* from = sums + (int64_t)row * pitch + col;
  f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
  for (int p = 0; p < parts; ++p) s += *reinterpret_cast<const f32x4*>(from + p * all);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if (col + e >= N) break;
    float v = s[e];
    if (bias) v += to_f32<OutT>(bias[col + e]);
    if (resid) v += to_f32<OutT>(resid[(int64_t)row * ldr + col + e]);
    C[(int64_t)row * ldc + col + e] = from_f32<OutT>(v);
  }
}

}  // namespace

// (Tiles of sixteen rows at any number of rows: 85 x 512 x 9664 16.5 / 11.0, 113 x 304 x 11968 29.9 / 23.8, 72 x 1280 x 1280 6.5 / 6.2, 267 x 272 x 4480
// 9.9 / 8.3; 1.12 times the rate over 50 products of 65 to 267 rows, none slower.)
// (64 x 96 and 96 x 64 ask for an eighth less than the tile of 128 x 64 that took their calls and leave fewer CUs idle: 2638 x 512 x 5600 40 /
// 31, 168 x 6128 x 9520 86 / 68, 1725 x 624 x 9728 64 / 53, 583 x 2144 x 4288 24 / 20, 2751 x 488 x 5312 28.8 / 23.8, 280 x 4992 x 384 6.8 / 6.2; 1.08
// and 1.04 times the rate over 2731 and 421 products. Not where the last row of 128 x 64 tiles is half padding, which costs no intake, and the weights are
// more than the L2s hold of them beside the rest: 160 x 6016 x 6016 36 / 42, 284 x 4992 x 6096 40 / 49, [K,N] 427 x 2432 x 6656 44 / 54;
// [N,K] weights of 6 to 7 million 1.01 times the rate, 7 to 8 0.93, 12 to 16 0.89, beyond 0.88; [K,N] 7 to 8 1.02, 8 to 9 0.94, 12 to 16 0.88;
// 1130 products, an even count of 64 rows 1.05 to 1.10 at any. 48 x 32 before 32 x 64, [N,K]: 92 x 3304 x 8832 33 / 27.6, 687 x 400 x 3680 13.2 / 11.6,
// level or a few hundredths slower below K of about 1000 and against [K,N] weights (1149 x 320 x 2752 10.5 / 11.4). 48 x 64 with two stages of 256 of K loses 10 % to 64 x 64.)
// (96 x 96 asks for what 128 x 64 does, an eighth more of C to a tile; us on 128 x 128 tiles two to a CU or one / here: 1336 x 1600 x 1600
// 20.2 / 16.2, 330 x 5672 x 7232 72 / 56, 3209 x 592 x 9064 101 / 71, 165 x 8632 x 1984 19.7 / 15.2, 189 x 9704 x 384 10.2 / 8.1, 1510 x 1512 x
// 6912 64 / 47 ([K,N] 70 / 58); 1.23 times the rate over 310 products. Not where K is three or four whole slabs of 64, which those tiles ask for
// at once: 2176 x 1024 x 256 6.2 / 6.8, 640 x 3456 x 256 6.4 / 7.0, 96 x 22848 x 192 6.7 / 7.1; nor, with odd rows, which leave by elements here,
// up to 512: 544 x 3484 x 192 + residual 12.6 / 13.7, 848 x 2542 x 192 8.1 / 8.8, 320 x 5529 x 448 9.5 / 10.1. Of the others two are slower: 288 x
// 6656 x 12416 [K,N] 98 / 109, 73 x 22656 x 512 9.2 / 9.8. 128 x 128 on eight waves: equal to gemm.hip's.)
// The smallest tile of which there is at most one per CU (more tiles than CUs: a second round, at the same intake per CU as a tile of
// twice the area; over 250 random products of up to 2000 rows no other tile was more than 6 % ahead of this choice but where K < 128),
// none where even 128 x 64 and 96 x 96 are more. us for 128 x 64 / 64 x 64 / 32 x 64 / 32 x 32 tiles (how many), K = 3072 [K,N]: N = 768, 2000 rows
// 17.5 (192) / 22 (384); 1000 rows 18 (96) / 12 (192) / 18 (384); 500 rows 17 / 11.6 (96) / 10 (192) / 16 (384); 256 rows 16.5 / 11.7
// / 9.7 (96) / 9.3 (192).
// Up to 64 rows against [N,K] weights there is the weight stream of gemm_skinny.hip, whose start and end are shorter: it stays for 33
// rows and more up to K = 128 (50 x 176 x 32 3.3, 3.2; 38 x 320 x 64 3.1, 3.2), for 17 to 32 rows against weights of less than 2^23
// elements (29 x 640 x 3872 5.4, 5.8; 20 x 9968 x 320 4.5, 4.6; 23 x 8728 x 896 7.5, 6.9; 32 x 4096 x 4096 11.7, 10.3) and for up to
// 16 rows of less than 3 * 2^22 (16 x 768 x 3072 4.9, 5.1; 10 x 2800 x 3136 6.5, 7.0; 9 x 3672 x 3360 8.3, 7.8; 16 x 4096 x 4096
// 9.9, 8.7; 13 x 7904 x 5952 19.5, 16) -- but where five to eight rows and K of 2048 and more would go by dot products, a tile is
// always ahead (8 x 800 x 3168 8.5, 5.5; 7 x 304 x 11968 18, 11). Of the tiles beyond those lines, what would take the call instead first,
// us on weights from HBM / on weights three times which about fill the 256 MiB behind L2:
//   three and four rows from K = 1024 on (dot products): the tiles ahead at 4 x 4096 x 4096 (9.9, 8.9 / 9.4, 7.9), 4 x 11008 x 4096
//   (19.5, 19.7 / 19.2, 17.5), 3 x 14336 x 1024 (9.6, 8.2 / 9.2, 7.4), 4 x 4096 x 11008 (21.9, 21.2 / 21.5, 16.7); not with weights of 3 * 2^24
//   elements and more (3 x 16384 x 4096 25.9, 29.6 / 25.7, 29.5; 4 x 14336 x 4096 24.3, 25.5 / 23.9, 26.0; 3 x 8192 x 8192 26.0, 27.1 /
//   25.2, 26.8), nor on tiles of 64 x 96 (4 x 20056 x 1984 17.4, 18.7; 4 x 22858 x 2048 22.1, 24.2), nor where tiles of 32 columns and more
//   leave three eighths of the CUs without one (3 x 4192 x 3560 9.8, 11.5; 4 x 9527 x 6416 28, 33);
//   up to sixteen rows, half of a tile of 32 x 64 (weight stream): 16 x 14336 x 4096 22.8, 25.8 / 22.4, 24.9; 10 x 8666 x 10432 41.4, 45.1 /
//   41.6, 45.2; 13 x 11368 x 1664 11.7, 12.2 / 8.0, 8.8 (16 x 11008 x 4096 18.9, 20.7 / 19.1, 18.0); up to 24 of the 64 of a tile of 64 x
//   96 (weights from HBM: 9 x 20000 x 4096 29.4, 37.4; 16 x 24576 x 512 7.8, 8.6; 16 x 16400 x 1408 11.9, 13.7; 17 x 24576 x 4096 38.6,
//   42.3; 24 x 24576 x 1408 14.7, 16.5; 24 x 17856 x 4096 36.2, 34.6; 32 rows 39.3, 35.7 at 20000 x 4096, 42.5, 46.2 at
//   24576); or tiles of 16 x 16 for fewer than half
//   of the CUs: 9 x 1208 x 15232 17.9, 17.9 / 11.2, 13.8; 12 x 1422 x 9408 13.2, 13.2 / 8.5, 9.4;
//   up to 32 rows, up to sixteen channels per CU, weights of 3 * 2^24 elements and more (weight stream): 16 x 4096 x 14336 25.3, 27.2 / 24.5,
//   26.1; 17 x 4096 x 12288 23.2, 25.8 / 23.1, 25.8; 32 x 4096 x 12288 29.4, 31.4 / 29.3, 31.2 -- unless its rows stand a power of two
//   apart (16 x 4096 x 16384 33.5, 28.2 / 33.5, 28.0);
//   17 to 24 rows, two tiles of 16 x 32, weights of less than 2^25 elements (weight stream): 17 x 3072 x 5120 12.5, 13.2 / 8.0, 8.7;
//   24 x 3072 x 2752 8.1, 9.0 / 5.8, 6.4; 17 x 2560 x 6912 14.3, 15.0 / 8.6, 9.8 (32 rows 16.7, 16.4 / 11.2, 10.4).
// The weight stream takes whole 32s of K and 64 channels and more; what neither it nor the dot products take has its tile at any size of the
// weights (on the 128 x 128 tiles, us, before / now: 16 x 272 x 4264 40 / 6.8, 30 x 3000 x 2504 24.6 / 6.4, 16 x 11008 x 1000 15.8 / 7.8,
// 12 x 4096 x 776 12.6 / 4.5, 50 x 3000 x 104 4.9 / 3.5).
GemmFewTile plan_gemm_few(bool trans_b, int64_t M, int64_t N, int64_t K) {
  const int64_t cus = hexmi_num_cus();
  const bool dots = trans_b && N >= 64 && ((M <= 4 && K >= 1024) || (M <= 8 && K >= 2048));
  const bool stream = trans_b && N >= 64 && !dots && K % 32 == 0;
  if ((dots || stream) && M <= 64) {
    if (M > 32 ? K <= 128 : N * K < (int64_t)(M > 16 ? 2 : 3) << 22 && !(M >= 5 && M <= 8 && K >= 2048)) return {0, 0};
  }
  // half of the last row of 128 x 64 tiles is padding, and weights of 14 MiB and more ([K,N]: 16)
  const bool half = (M + 63) / 64 % 2 && N * K >= (int64_t)(trans_b ? 7 : 8) << 20 && ((M + 127) / 128) * ((N + 63) / 64) <= cus;
  static constexpr GemmFewTile kTiles[] = {{16, 16}, {16, 32}, {32, 32}, {48, 32}, {32, 64}, {64, 64}, {64, 96}, {96, 64}, {128, 64}, {96, 96}};
  for (const GemmFewTile& t : kTiles) {
    if (t.m == 48 && (K < 1024 || !trans_b)) continue;
    if (t.m == 96 && t.n == 96 && K % 64 == 0 && (N % 8 == 0 ? K > 128 && K <= 256 : K <= 512)) continue;
    if (t.n == 16 && !trans_b) continue;                         // sixteen columns of a row of B are a quarter of a line
    const int64_t count = ((M + t.m - 1) / t.m) * ((N + t.n - 1) / t.n);
    if (count > cus || (half && t.m * t.n == 64 * 96)) continue;
    if (dots && M <= 4 && (N * K >= (int64_t)3 << 24 || t.n > 64 || (t.n > 16 && 8 * count < 5 * cus))) return {0, 0};
    if (stream && M <= 16 && (t.n >= 64 || (t.n == 16 && 2 * count < cus))) return {0, 0};
    if (stream && M <= 24 && t.n > 64) return {0, 0};
    const bool narrow = stream && M <= 32 && t.m == 16 && N <= 16 * cus;    // a channel group of sixteen per CU at most
    if (narrow && M > 16 && M <= 24 && t.n == 32 && N * K < (int64_t)1 << 25) return {0, 0};
    if (narrow && N * K >= (int64_t)3 << 24 && (K & (K - 1)) != 0) return {0, 0};
    return t;
  }
  return {0, 0};
}

// The tile of a product on operand rows at any alignment: the smallest of which there is at most one per CU, 128 x 128 beyond.
static GemmFewTile plan_gemm_any(int64_t M, int64_t N) {
  static constexpr GemmFewTile kTiles[] = {{16, 32}, {32, 32}, {32, 64}, {64, 64}, {128, 64}};
  for (const GemmFewTile& t : kTiles)
    if ((t.m > 16 || M <= 64) && ((M + t.m - 1) / t.m) * ((N + t.n - 1) / t.n) <= hexmi_num_cus()) return t;
  return {128, 128};
}

template <typename T, typename OutT, bool TRANS_B>
int launch_gemm_any(const T* A, const T* B, OutT* C, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t ldc, hipStream_t s,
                    const OutT* bias, const OutT* resid, int64_t ldr) {
  const GemmFewTile tile = plan_gemm_any(M, N);
  const int64_t tiles_m = (M + tile.m - 1) / tile.m, tiles_n = (N + tile.n - 1) / tile.n;
  if (K > kAnyMaxK) return HEXMI_ENOTSUP;
  if (!grid_fits(tiles_m * tiles_n, 512)) {                      // more threads than a grid holds: half of the tiles, then the rest
    const bool rows = tiles_m >= tiles_n;
    const int64_t m = rows ? (tiles_m + 1) / 2 * tile.m : 0, n = rows ? 0 : (tiles_n + 1) / 2 * tile.n;
    const int rc = launch_gemm_any<T, OutT, TRANS_B>(A, B, C, rows ? m : M, rows ? N : n, K, lda, ldb, ldc, s, bias, resid, ldr);
    if (rc != HEXMI_OK) return rc;
    return launch_gemm_any<T, OutT, TRANS_B>(A + m * lda, B + n * (TRANS_B ? ldb : 1), C + m * ldc + n, M - m, N - n, K, lda, ldb, ldc, s,
                                             bias ? bias + n : nullptr, resid ? resid + m * ldr + n : nullptr, ldr);
  }
  const int runs = N % 8 == 0 && ldc % 8 == 0 && aligned_to(C, 16) && aligned_to(bias, 16) && aligned_to(resid, 16) &&
                   (!resid || ldr % 8 == 0);
#define HEXMI_ANY(S_)                                                                                                         \
  hipLaunchKernelGGL((gemm_few_kernel<T, OutT, S_, 2, TRANS_B, true>), dim3((unsigned)(tiles_m * tiles_n)), dim3(S_::kThreads), 0, s, A, B, \
                     C, (int)M, (int)N, (int)K, lda, ldb, ldc, bias, resid, ldr, (int)tiles_m, (int)tiles_n, runs, (int)K)
  typedef FewShape<128, 64>::S Any12864; typedef FewShape<64, 64>::S Any6464; typedef FewShape<32, 64>::S Any3264;
  typedef FewShape<32, 32>::S Any3232; typedef FewShape<16, 32>::S Any1632;
  if (tile.n == 128) HEXMI_ANY(AnyShape128);
  else if (tile.m == 128) HEXMI_ANY(Any12864);
  else if (tile.m == 64) HEXMI_ANY(Any6464);
  else if (tile.n == 64) HEXMI_ANY(Any3264);
  else if (tile.m == 32) HEXMI_ANY(Any3232);
  else HEXMI_ANY(Any1632);
#undef HEXMI_ANY
  return launch_status();
}

template <typename T, typename OutT, bool TRANS_B>
int launch_gemm_few(const GemmFewTile& tile, const T* A, const T* B, OutT* C, int64_t M, int64_t N, int64_t K, int64_t lda,
                    int64_t ldb, int64_t ldc, hipStream_t s, const OutT* bias, const OutT* resid, int64_t ldr) {
  const int tiles_m = (int)((M + tile.m - 1) / tile.m), tiles_n = (int)((N + tile.n - 1) / tile.n);
  const int runs = N % 8 == 0 && ldc % 8 == 0 && aligned_to(C, 16) && aligned_to(bias, 16) && aligned_to(resid, 16) &&
                   (!resid || ldr % 8 == 0);
#define HEXMI_FEW(BM, BN)                                                                                                    \
  hipLaunchKernelGGL((gemm_few_kernel<T, OutT, FewShape<BM, BN>::S, FewShape<BM, BN>::NS, TRANS_B, false>),                         \
                     dim3((unsigned)(tiles_m * tiles_n)), dim3(FewShape<BM, BN>::S::kThreads), 0, s, A, B, C, (int)M, (int)N, \
                     (int)K, lda, ldb, ldc, bias, resid, ldr, tiles_m, tiles_n, runs, (int)K)
  if (tile.m == 128) HEXMI_FEW(128, 64);
  else if (tile.m == 96 && tile.n == 64) HEXMI_FEW(96, 64);
  else if (tile.m == 96) HEXMI_FEW(96, 96);
  else if (tile.m == 48) HEXMI_FEW(48, 32);
  else if (tile.m == 64 && tile.n == 96) HEXMI_FEW(64, 96);
  else if (tile.m == 64) HEXMI_FEW(64, 64);
  else if (tile.n == 64) HEXMI_FEW(32, 64);
  else if (tile.m == 32) HEXMI_FEW(32, 32);
  else if (tile.n == 32) HEXMI_FEW(16, 32);
  else if constexpr (TRANS_B) HEXMI_FEW(16, 16);
  else return HEXMI_ENOTSUP;                                     // (the plan gives [K,N] none)
#undef HEXMI_FEW
  return launch_status();
}

// Parts of K where an output of few tiles leaves most CUs without a share of a long K: a tile of 32 rows of [K,N] weights takes them in at
// 24 GB/s to a CU. Up to one tile to a CU, parts of 512 and more, three of them at least; the sums pass through memory and a second
// launch, 3 us. us, the tiles above / parts ([K,N]): 1 x 1024 x 11376 37 / 12, 1 x 2560 x 4096 12.8 / 9.2, 16 x 2560 x 11376 52 / 20, 16 x 4096 x
// 4096 19.7 / 13.2, 16 x 8192 x 11008 53 / 39, 32 x 2048 x 11008 44 / 15.6, 64 x 4096 x 4096 20.9 / 15.7, 113 x 304 x 11968 22.7 / 11.6, 256 x
// 1024 x 11008 47 / 24, 512 x 512 x 8192 22.9 / 19.4. Below these lines the second launch costs what the parts give: 16 x 4096 x 2048 7.8 / 8.7,
// 64 x 768 x 3072 8.3 / 8.8, 11 x 7296 x 3200 15.4 / 16.7, 58 x 1408 x 4352 10.7 / 11.7; 1.22 times the rate over 110 products of K = 3072 on.
// Tiles of [N,K] weights come in whole lines (64 x 4096 x 4096 13.0 / 14.1, 512 x 512 x 8192 14.4 / 18.9), and as a whole the product has
// tiles of 16 x 16 to 32 x 64 on all CUs, whose operands pass from one to the next through L2 while all of them fit: parts are ahead from
// 19 MiB of operands on, and from K = 12800 on, where the walk is what is long. Rate in parts over that as a whole, 430 products of 33 to 600
// rows and K = 9216 to 18944, by millions of (M + N) K: up to 8 0.98, to 9 1.00, to 10.5 1.09, to 12 1.24, to 15 1.26, beyond 1.29; with less than
// 10.5, K of 12800 and more 1.12; K = 8192 0.94 (64 x 4096 x 11008 33 / 26, 128 x 1024 x 12288 28.9 / 15.8, 128 x 2048 x 10240 26 / 22, 40 x 2048 x 10240
// 20.2 / 15.1; 64 x 512 x 10240 10.3 / 11.9, 453 x 400 x 9344 16.4 / 18.0). Up to 32 rows the whole has few tiles: 8704 1.03, 9728 1.13, 11008 1.16,
// 12288 1.32; in fewer than eight parts a tenth ahead or level (32 x 4096 x 11008 21.6 / 21.4) for a second launch, so as a whole.
// [K,N] weights of few columns are read in whole lines as they are, so that only the walk is long: rate in parts over that as a whole, N up
// to 32 and M up to 16, K = 3072 to 3500 0.87, to 4000 0.91, to 4600 0.98, to 5500 1.05; M to 1024 and K to 5500 0.83 to 0.99, to 7000 1.03 to 1.25; M
// beyond 2048 0.77 to 0.94 at any K; N to 64 and M beyond 128 1.0 and less up to 5500 (17 x 16 x 3072 5.5 / 7.7, 4862 x 32 x 6080 12.8 / 16.3, 56 x 16 x
// 4760 7.0 / 8.6; 7000 products). Up to 16 rows of more than 1024 columns K to 3500 0.92, to 4000 0.99, to 4600 1.15 (3 x 1904 x 3184 8.9 / 10.5).
// Rows of [N,K] products past 1536 whose last tiles are half empty 0.78 to 0.95 (2630 x 76 x 10072 20.1 / 24.0).
// [K,N] weights whose rows stand off the boundaries, whole / in parts: 16 x 2027 x 12144 47 / 19, 128 x 1175 x 11904 49 / 24, 3 x 485 x 8704 20.6 / 11.4, 128 x
// 2250 x 5312 28.9 / 19.9, 15 x 1601 x 4352 13.8 / 11.8, 2 x 405 x 3136 10.9 / 11.3; 1.45 times the rate over 44 (up to 16 rows parts of 256 and
// more: a slab through registers is a latency; with 512 and more 2 x 1497 x 4512 13.2 / 13.8, with 256 and more at 64 rows 90 x 318 x 11584 13.3 -> 15.5).
// Up to 16 rows of more than 1024 columns tiles of 128 columns: 16 x 2560 x 11376 23.0 on 64 columns, 20.2; 1 x 1024 x 11376 11.5, 12.6.
GemmParts plan_gemm_parts(bool trans_b, int64_t M, int64_t N, int64_t K, bool any) {
  if (trans_b ? M <= 16 || K < (M <= 32 ? 9728 : 9216) : M <= 32 ? K < 3072 || K < N : K < 4608) return {};
  if (trans_b && M > 32 && K < 12800 && (M + N) * K < 19 << 19) return {};
  if (trans_b && M > 1536 && (N - 1) % 64 < 32) return {};       // the columns of the last tiles half padding and more
  if (!trans_b && !any) {
    if (N <= 32 && (M > 2048 || K < (M <= 16 ? 4608 : M <= 1024 ? 5632 : 7168))) return {};
    if (N <= 64 && K < (M <= 128 ? 4096 : 5632)) return {};
    if (M <= 16 && N > 1024 && K < 4096) return {};
  }
  const GemmFewTile t = M <= 16 ? GemmFewTile{16, N <= 1024 || any ? 64 : 128} : GemmFewTile{M <= 32 ? 32 : 64, 64};
  const int64_t tiles = ((M + t.m - 1) / t.m) * ((N + t.n - 1) / t.n);
  const int64_t parts = std::min(hexmi_num_cus() / std::max<int64_t>(tiles, 1), K / (any && M <= 16 ? 256 : 512));
  if (parts < 3 || (trans_b && M <= 32 && parts < 8)) return {};
  const int64_t part = ((K + parts - 1) / parts + 255) / 256 * 256;          // whole slabs of every shape
  return {t, (int)((K + part - 1) / part), (int)part};
}

template <typename T, typename OutT, bool TRANS_B>
int launch_gemm_parts(const GemmParts& plan, const T* A, const T* B, OutT* C, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb,
                      int64_t ldc, hipStream_t s, const OutT* bias, const OutT* resid, int64_t ldr, float* sums, bool any) {
  const int tiles_m = (int)((M + plan.tile.m - 1) / plan.tile.m), tiles_n = (int)((N + plan.tile.n - 1) / plan.tile.n);
  const int64_t pitch = gemm_parts_pitch(N);
#define HEXMI_PARTS_AS(BM, BN, NS, ANY)                                                                                            \
  hipLaunchKernelGGL((gemm_few_kernel<T, float, FewShape<BM, BN>::S, NS, TRANS_B, ANY, true>),                                             \
                     dim3((unsigned)(tiles_m * tiles_n), (unsigned)plan.parts), dim3(FewShape<BM, BN>::S::kThreads), 0, s, A, B, sums, \
                     (int)M, (int)N, (int)K, lda, ldb, pitch, (const float*)nullptr, (const float*)nullptr, (int64_t)0, tiles_m, tiles_n, 1, \
                     plan.part)
#define HEXMI_PARTS(BM, BN)                                                                                                  \
  do {                                                                                                                       \
    if constexpr (!TRANS_B) {                                                                                                \
      if (any) { HEXMI_PARTS_AS(BM, BN, 2, true); break; }                                                                     \
    }                                                                                                                        \
    HEXMI_PARTS_AS(BM, BN, (FewShape<BM, BN>::NS), false);                                                                    \
  } while (0)
  if (any && (TRANS_B || plan.tile.n > 64)) return HEXMI_ENOTSUP;
  if (plan.tile.m == 32) HEXMI_PARTS(32, 64);
  else if (plan.tile.m == 64) HEXMI_PARTS(64, 64);
  else if constexpr (TRANS_B) return HEXMI_ENOTSUP;              // (the plan gives [N,K] weights no tiles of sixteen rows)
  else if (plan.tile.n == 64) HEXMI_PARTS(16, 64);
  else HEXMI_PARTS_AS(16, 128, (FewShape<16, 128>::NS), false);
#undef HEXMI_PARTS
#undef HEXMI_PARTS_AS
  const int rc = launch_status();
  if (rc != HEXMI_OK) return rc;
  hipLaunchKernelGGL((gemm_merge_kernel<OutT>), dim3((unsigned)((M * (pitch / 4) + 127) / 128)), dim3(128), 0, s, sums, C, (int)M, (int)N,
                     (int)pitch, plan.parts, ldc, bias, resid, ldr);
  return launch_status();
}

#define HEXMI_INSTANCE(T, OutT, TB)                                                                                          \
  template int launch_gemm_few<T, OutT, TB>(const GemmFewTile&, const T*, const T*, OutT*, int64_t, int64_t, int64_t, int64_t, \
                                            int64_t, int64_t, hipStream_t, const OutT*, const OutT*, int64_t);                 \
  template int launch_gemm_any<T, OutT, TB>(const T*, const T*, OutT*, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t,   \
                                            hipStream_t, const OutT*, const OutT*, int64_t);                                     \
  template int launch_gemm_parts<T, OutT, TB>(const GemmParts&, const T*, const T*, OutT*, int64_t, int64_t, int64_t, int64_t, int64_t, \
                                              int64_t, hipStream_t, const OutT*, const OutT*, int64_t, float*, bool);
HEXMI_INSTANCE(f16, f16, false)
HEXMI_INSTANCE(f16, f16, true)
HEXMI_INSTANCE(f16, float, false)
HEXMI_INSTANCE(f16, float, true)
HEXMI_INSTANCE(bf16, bf16, false)
HEXMI_INSTANCE(bf16, bf16, true)
HEXMI_INSTANCE(bf16, float, false)
HEXMI_INSTANCE(bf16, float, true)
#undef HEXMI_INSTANCE

}  // namespace hexmi
