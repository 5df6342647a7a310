// C[M,N] = (A[M,K] * (W[N,K] - zero)^T) * scales for three to some hundred rows against int8 weights: tiles of one round over the
// CUs, a workgroup of eight waves to a tile.
//
// What bounds it: a slab of a tile is read from LDS once per wave side by side, copied into LDS, widened and multiplied, and at one
// workgroup per CU none of the four hides behind another entirely: an earlier form of 64 x 192 tiles took 34 us for 256 x 11008 x 4096
// on cold weights, 27 without the copies, 26 without the matrix instructions, 29 without the widening and 29 without the reads (this one 31). So: eight waves; the weights
// stay int8 in LDS and a wave widens its own channels only, waves standing side by side along the channels (64 rows to a tile) so
// that each weight is widened once; a slab of the larger tiles multiplies from registers while the next is read; the wave groups that take the 64-k parts of
// a slab add up in LDS at the end; scales are fetched under the K walk (at the end, by the threads that store, they cost 1 to 3 us
// of a call). A tile of every CU's own, down to 16 x 16, is what most shapes gain by: 128 x 128 tiles left two thirds and more of the CUs
// idle (256 x 4096 x 4096: 64 tiles), the chunked kernel of w8a16.hip pulls all rows into every CU.
#include <algorithm>
#include <type_traits>

#include "hexmi_common.h"

namespace hexmi {
namespace {

__device__ __attribute__((aligned(16))) unsigned g_w8_zeros[4];       // where a copy of a chunk past K points

// TM x TN: 16 x 16 tiles of a wave; SM x SN waves side by side; KH wave groups take the 64-k parts of a slab; NS stages.
template <int TM_, int TN_, int SM_, int SN_, int KH_, int NS_>
struct Shape {
  static constexpr int TM = TM_, TN = TN_, SM = SM_, SN = SN_, KH = KH_, NS = NS_;
  static constexpr int kWaves = SM * SN * KH, kThreads = kWaves * kWave;
  static constexpr bool kAhead = KH < 4;                         // the next slab is read while one multiplies
  static constexpr int BM = SM * TM * 16, BN = SN * TN * 16, BK = KH * 64;
  static constexpr int kStage = BM * BK * 2 + BN * BK;           // bytes of a stage: rows of A, then rows of W
};

// 16-byte chunk c of a row sits at c ^ swz(row): sixteen rows of one chunk then cover all banks
template <int PITCH> __device__ __forceinline__ int swz_row(int r) { return PITCH == 64 ? (r >> 1) & 3 : PITCH == 128 ? (r >> 1) & 7 : r & 15; }

// K % 16 == 0, operands on 16-byte boundaries. runs: the output in runs of eight columns on 16-byte boundaries. ZP: zero points.
// pt: one scale (and zero point) for all channels.
template <typename S, bool ZP>
__global__ __launch_bounds__(S::kThreads)
void w8a16_few_kernel(const f16* __restrict__ A, const int8_t* __restrict__ W, const f16* __restrict__ scales,
                      const int8_t* __restrict__ zp, f16* __restrict__ C, int M, int N, int K, int tiles_m, int tiles_n, int pt,
                      int runs) {
  constexpr int TM = S::TM, TN = S::TN, BM = S::BM, BN = S::BN, BK = S::BK, KH = S::KH, NS = S::NS, kThreads = S::kThreads;
  constexpr int kA = BM * BK * 2 / 16 / kThreads, kB = BN * BK / 16 / kThreads, kCopies = kA + kB;   // a wave's copies of a slab
  static_assert(kA * kThreads * 16 == BM * BK * 2 && kB * kThreads * 16 == BN * BK, "whole copies");
  constexpr int kPitch = BN + 4;                                 // pitch of the sums on their way out
  __shared__ __attribute__((aligned(16))) char lds[std::max(NS * S::kStage, KH * BM * kPitch * 4)];
  __shared__ __attribute__((aligned(16))) float lds_scale[BN];

  const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int r16 = lane % 16, kg = lane / 16;
  int tm, tn;
  tile_of_block<8>(blockIdx.x, tiles_m, tiles_n, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;

  // copy i of a slab moves chunks [i * kThreads + wave * 64, + 64) of the stage: A's kA, then W's kB
  int voff[kCopies], kc[kCopies];
#pragma unroll
  for (int i = 0; i < kCopies; ++i) {
    const bool a = i < kA;
    const int chunk = (a ? i : i - kA) * kThreads + threadIdx.x, per_row = a ? BK / 8 : BK / 16;
    const int row = chunk / per_row, c = (chunk % per_row) ^ (a ? swz_row<BK * 2>(row) : swz_row<BK>(row));
    const int left = (a ? M - m0 : N - n0) - 1;                  // past the edge: the last row again, not stored
    voff[i] = (row < left ? row : left) * (a ? 2 * K : K) + c * 16;
    kc[i] = c * (a ? 8 : 16);
  }
  const char* a_base = reinterpret_cast<const char*>(A + (int64_t)m0 * K);
  const char* w_base = reinterpret_cast<const char*>(W + (int64_t)n0 * K);
  const int slabs = (K + BK - 1) / BK, full = K / BK;
  auto copy = [&](int slab, int stage, auto ragged) __attribute__((always_inline)) {
    const char* a_from = a_base + (int64_t)slab * (BK * 2);
    const char* w_from = w_base + (int64_t)slab * BK;
    char* to = lds + stage * S::kStage + wave * 1024;
#pragma unroll
    for (int i = 0; i < kCopies; ++i) {
      const char* from = i < kA ? a_from : w_from;
      if constexpr (decltype(ragged)::value) {                   // the slab that reaches past K: zeros there
        const char* src = slab * BK + kc[i] < K ? from + voff[i] : reinterpret_cast<const char*>(g_w8_zeros);
        copy_ptr_to_lds_asm(src, to + i * (kThreads * 16));
      } else {
        copy_to_lds_asm(from, voff[i], to + i * (kThreads * 16));
      }
    }
  };

  // this lane's fragments of a stage: wave group kh takes 64 k, a lane of K group kg the sixteen at kh * 64 + kg * 16 (one
  // read of W, two of A), eight per matrix instruction
  const int kh = wave / (S::SM * S::SN), wm = wave % (S::SM * S::SN) / S::SN, wn = wave % S::SN;
  const int arow = wm * TM * 16 + r16, brow = wn * TN * 16 + r16;       // the swizzles repeat every sixteen rows
  int a_at[2];
#pragma unroll
  for (int p = 0; p < 2; ++p) a_at[p] = arow * (BK * 2) + ((kh * 8 + kg * 2 + p) ^ swz_row<BK * 2>(arow)) * 16;
  const int b_at = BM * BK * 2 + brow * BK + ((kh * 4 + kg) ^ swz_row<BK>(brow)) * 16;

  // zero points of this lane's channels
  f16 zero[ZP ? TN : 1];
  if constexpr (ZP) {
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int ch = n0 + brow + j * 16;
      zero[j] = (f16)(float)zp[pt ? 0 : ch < N ? ch : N - 1];
    }
  }

  // the scale of channel n0 + this thread, under the K walk (loads at the end would be a latency of their own)
  static_assert(BN <= kThreads, "a channel a thread");
  const int scale_at = n0 + (int)threadIdx.x < N ? n0 + (int)threadIdx.x : N - 1;
  const f16 scale = scales[pt ? 0 : scale_at];

  // Partial sums of an element over K, one to four of a wave group each: sixteen on tiles of sixteen rows and of 32 x 32, four on the
  // others. One chain of K / 32 additions would round more than the chunked kernel's sums, one for each 64 k of a chunk: twelve, six or
  // four by the channel tiles of a workgroup up to 16 rows, six or four up to 32, four up to 64, two beyond.
  constexpr int kParts = TM == 1 ? 16 / KH : KH == 4 ? 1 : 2;
  f32x4 acc[kParts][TM][TN];
#pragma unroll
  for (int p = 0; p < kParts; ++p)
#pragma unroll
    for (int m = 0; m < TM; ++m)
#pragma unroll
      for (int n = 0; n < TN; ++n) acc[p][m][n] = f32x4{0.f, 0.f, 0.f, 0.f};
#define HEXMI_FENCE __builtin_amdgcn_sched_barrier(0)
  typedef std::integral_constant<int, 0> Part0;
  typedef std::integral_constant<int, 1> Part1;
  struct Slab { u32x4 w[TN]; f16x8 a[2][TM]; };
  auto read = [&](int stage, Slab& f) __attribute__((always_inline)) {
    const char* from = lds + stage * S::kStage;
#pragma unroll
    for (int n = 0; n < TN; ++n) f.w[n] = *reinterpret_cast<const u32x4*>(from + b_at + n * (16 * BK));
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int m = 0; m < TM; ++m) f.a[p][m] = *reinterpret_cast<const f16x8*>(from + a_at[p] + m * (16 * BK * 2));
  };
  auto multiply = [&](const Slab& f, auto part) __attribute__((always_inline)) {      // part: of four sums, which two take this slab
    constexpr int kFirst = kParts == 4 ? 2 * decltype(part)::value : 0, kSecond = kParts == 1 ? 0 : kFirst + 1;
#pragma unroll
    for (int n = 0; n < TN; ++n) {
      f16x8 b0, b1;
      cvt16(f.w[n], b0, b1);
      if constexpr (ZP) {                                        // whole numbers of up to 255: exact
        b0 -= zero[n];
        b1 -= zero[n];
      }
#pragma unroll
      for (int m = 0; m < TM; ++m) {
        f32x4& c = acc[kFirst][m][n];
        c = __builtin_amdgcn_mfma_f32_16x16x32_f16(b0, f.a[0][m], c, 0, 0, 0);
      }
#pragma unroll
      for (int m = 0; m < TM; ++m) {
        f32x4& c = acc[kSecond][m][n];
        c = __builtin_amdgcn_mfma_f32_16x16x32_f16(b1, f.a[1][m], c, 0, 0, 0);
      }
    }
  };
  // The copies are assembly: the compiler would wait for all of them before any LDS read. Here a wave waits until at most `newer`
  // slabs of its own are in flight and its reads of the slab before have returned, then for every other wave.
  auto landed = [&](int newer) __attribute__((always_inline)) {
    HEXMI_FENCE;
    switch (newer) {
      case 0: __builtin_amdgcn_s_waitcnt(waitcnt_imm(0)); break;
      case 1: __builtin_amdgcn_s_waitcnt(waitcnt_imm(kCopies)); break;
      case 2: __builtin_amdgcn_s_waitcnt(waitcnt_imm(2 * kCopies)); break;
      default: __builtin_amdgcn_s_waitcnt(waitcnt_imm(3 * kCopies)); break;
    }
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    HEXMI_FENCE;
  };
  static_assert(NS >= 2 && NS <= 4 && 3 * kCopies < 64, "the waits above");
  int stage = 0, j = 0;
  auto copy_any = [&](int slab, int into) __attribute__((always_inline)) {
    if (slab < full) copy(slab, into, std::false_type{});
    else if (slab < slabs) copy(slab, into, std::true_type{});
  };
  HEXMI_FENCE;
#pragma unroll
  for (int s = 0; s < NS - 1; ++s) copy_any(s, s);
  if constexpr (S::kAhead) {
    // Slab j multiplies from registers while slab j + 1 is read and slabs up to j + NS are copied: its own stage is free once every
    // wave has read it. steady: slab j + NS is a whole one.
    auto step = [&](const Slab& now, Slab& next, auto steady) __attribute__((always_inline)) {
      constexpr bool kSteady = decltype(steady)::value;
      const int after = stage == NS - 1 ? 0 : stage + 1;
      if (kSteady || j + 1 < slabs) {
        landed(kSteady ? NS - 2 : std::min(NS - 2, slabs - 2 - j));
        if (kSteady) copy(j + NS, stage, std::false_type{}); else copy_any(j + NS, stage);
        HEXMI_FENCE;
        read(after, next);
        HEXMI_FENCE;
      }
      multiply(now, Part0{});
      stage = after;
      ++j;
    };
    landed(std::min(NS - 1, slabs) - 1);
    copy_any(NS - 1, NS - 1);                                    // (behind the first slab: it would hold that up)
    HEXMI_FENCE;
    Slab even, odd;
    read(0, even);
    while (j + NS + 1 < full) {
      step(even, odd, std::true_type{});
      step(odd, even, std::true_type{});
    }
    while (j < slabs) {
      step(even, odd, std::false_type{});
      if (j < slabs) step(odd, even, std::false_type{});
    }
  } else {
    // The short slabs of the small tiles gain nothing by that and K is mostly the stages' own: the last slabs in a row, each
    // with its wait known (512 x 1024 x 1024 5.5 -> 5.0 us, 66 x 1696 x 816 5.1 -> 4.6; 294 x 688 x 9600 17.9 -> 18.7).
    auto step = [&](int newer, auto part, auto next) __attribute__((always_inline)) {   // next: the copies that follow into the free stage
      landed(newer);
      next(stage == 0 ? NS - 1 : stage - 1);
      HEXMI_FENCE;
      Slab now;
      read(stage, now);
      multiply(now, part);
      stage = stage == NS - 1 ? 0 : stage + 1;
      ++j;
    };
    auto whole = [&](int into) __attribute__((always_inline)) { copy(j + NS - 1, into, std::false_type{}); };
    if constexpr (kParts == 4) {
      while (j + NS < full) {
        step(NS - 2, Part0{}, whole);
        step(NS - 2, Part1{}, whole);
      }
    }
    while (j + NS - 1 < full) step(NS - 2, Part0{}, whole);
    if (j + NS - 1 < slabs) step(NS - 2, Part1{}, [&](int into) __attribute__((always_inline)) { copy(j + NS - 1, into, std::true_type{}); });
#pragma unroll
    for (int left = NS - 2; left >= 0; --left)                   // slabs behind this one
      if (j + left < slabs) {
        if (left & 1) step(left, Part1{}, [](int) __attribute__((always_inline)) {});
        else step(left, Part0{}, [](int) __attribute__((always_inline)) {});
      }
  }
#undef HEXMI_FENCE

  // the wave groups' sums meet in LDS and leave in rows, scaled, rounded once
  __syncthreads();
  float* red = reinterpret_cast<float*>(lds);
#pragma unroll
  for (int m = 0; m < TM; ++m)
#pragma unroll
    for (int n = 0; n < TN; ++n) {                               // a lane: row lane % 16, columns 4 (lane / 16) .. + 3
      f32x4 sum = acc[0][m][n];
      if constexpr (kParts >= 2) sum += acc[1][m][n];
      if constexpr (kParts == 4) sum += acc[2][m][n] + acc[3][m][n];
      *reinterpret_cast<f32x4*>(red + (kh * BM + (wm * TM + m) * 16 + r16) * kPitch + (wn * TN + n) * 16 + kg * 4) = sum;
    }
  if (threadIdx.x < BN) lds_scale[threadIdx.x] = (float)scale;
  __syncthreads();
  if (runs) {
    for (int idx = threadIdx.x; idx < BM * BN / 8; idx += kThreads) {
      const int row = idx / (BN / 8), col = idx % (BN / 8) * 8;
      if (m0 + row >= M || n0 + col >= N) continue;
      f32x4 s[2] = {};
#pragma unroll
      for (int h = 0; h < KH; ++h)
#pragma unroll
        for (int p = 0; p < 2; ++p) s[p] += *reinterpret_cast<const f32x4*>(red + (h * BM + row) * kPitch + col + 4 * p);
      f16x8 out;
#pragma unroll
      for (int e = 0; e < 8; ++e) out[e] = (f16)(s[e / 4][e % 4] * lds_scale[col + e]);
      *reinterpret_cast<f16x8*>(C + (int64_t)(m0 + row) * N + n0 + col) = out;
    }
  } else {
    for (int idx = threadIdx.x; idx < BM * BN; idx += kThreads) {
      const int row = idx / BN, col = idx % BN;
      if (m0 + row >= M || n0 + col >= N) continue;
      float v = 0.f;
#pragma unroll
      for (int h = 0; h < KH; ++h) v += red[(h * BM + row) * kPitch + col];
      C[(int64_t)(m0 + row) * N + n0 + col] = (f16)(v * lds_scale[col]);
    }
  }
}

template <int BM, int BN> struct FewShape;                       // waves, stages
template <> struct FewShape<16, 16> { typedef Shape<1, 1, 1, 1, 8, 4> S; };
template <> struct FewShape<16, 32> { typedef Shape<1, 2, 1, 1, 8, 4> S; };
template <> struct FewShape<32, 32> { typedef Shape<2, 2, 1, 1, 8, 3> S; };
template <> struct FewShape<16, 64> { typedef Shape<1, 2, 1, 2, 4, 4> S; };
template <> struct FewShape<32, 64> { typedef Shape<2, 2, 1, 2, 4, 4> S; };
template <> struct FewShape<48, 64> { typedef Shape<3, 2, 1, 2, 4, 3> S; };
template <> struct FewShape<32, 96> { typedef Shape<2, 3, 1, 2, 4, 3> S; };
template <> struct FewShape<64, 64> { typedef Shape<4, 2, 1, 2, 4, 3> S; };
template <> struct FewShape<64, 96> { typedef Shape<4, 3, 1, 2, 4, 2> S; };
template <> struct FewShape<64, 128> { typedef Shape<4, 2, 1, 4, 2, 4> S; };
template <> struct FewShape<64, 192> { typedef Shape<4, 3, 1, 4, 2, 3> S; };

}  // namespace

// The smallest tile of which there is at most one per CU. us for 32 x 64 / 64 x 64 / 64 x 128 / 64 x 192 tiles (how many; cold weights)
// and what took these calls before there were any: 128 x 4096 x 4096 10.8 (256) / 13.3 (128) / 20 (64) / 25, 22.4; 256 x 4096 x 4096 19.8
// (512) / 14.6 (256) / 21.5 / 25.7, 27.3; 512 x 4096 x 4096 - / 26.7 (512) / 22.2 (256) / 26.6, 31.4; 256 x 11008 x 4096 - / 44 (688) /
// 44 (344) / 31 (232), 36.3. Tiles of 16 x 16 to 16 x 64 and the three between (us for these / the smallest of the four above or the
// chunked kernel of w8a16.hip): 16 x 4096 x 4096 5.7 (16 x 16) / 7.4, 32 x 4096 x 4096 6.6 (16 x 32) / 9.6, 64 x 4096 x 11008 22.6 (32 x 32 and
// 16 x 64) / 27.9, 95 x 912 x 3872 8.1 / 12.9, 45 x 1328 x 6464 7.0 / 15.5, 47 x 4330 x 7936 16.7 (16 x 64) / 22.7, 149 x 1504 x 8256 13.2
// (32 x 32) / 18.2, 80 x 6272 x 10624 31.9 (48 x 64) / 38.0, 339 x 2144 x 3840 12.8 (32 x 96) / 13.9, 289 x 4223 x 3072 17.0 (64 x 96) / 23.1.
// 16 x 64 copies fewer rows of A a CU than 32 x 32 and more of W: ahead up to K = 2048 (32 x 8192 x 2048 6.2 / 7.0, x 4096 12.3 / 12.6).
// 64 x 96 has two stages of 56 KiB where 64 x 128 has four of 24: ahead where K is short, or not long and the weights come through L2
// for many rows (284 x 4352 x 3968 22.6 / 26.2, 352 x 2816 x 2688 13.7 / 15.9; 600 x 1792 x 7040 35.9 / 34.0, 160 x 6992 x 3712 22.1 / 20.4).
// (128 x 128 tiles, 1000 x 4096 x 4096: 35.1, gemm.hip's 34.5. 48 x 32, 16 x 48, 32 x 48, 48 x 96, 96 x 64 and 32 x 128 tiles: nowhere ahead of
// both neighbours by more than 2 %.)
// The chunked kernel, a workgroup per CU with all rows and up to 48 channels, reads each weight once: it stays ahead where the weights are
// what counts (us there / on the tile; 4500 products of 3 to 64 rows, N = 720 to 49152 and K = 512 to 14336):
//   up to sixteen rows against 24 million of them, or 20 from five rows on: 16 x 11008 x 4096 11.9 / 12.5 (16 x 48), 16 x 3072 x 7872 10.2 / 11.0,
//   16 x 1984 x 12032 11.9 / 13.0 (3 x 1984 x 11008 1.02 times the rate);
//   up to 32 rows, tiles of 32 x 32 from K = 4096 on and of 32 x 64 from 1600: 32 x 6144 x 11008 23.3 / 26.0, 32 x 6144 x 4096 10.5 / 11.5,
//   24 x 12288 x 1920 9.0 / 9.7, 24 x 11136 x 2176 10.2 / 11.3 (K = 3072 level, 8192 1.0);
//   up to 48 rows tiles of 48 x 64 from 1600 on, up to 64 rows of 32 x 96 from 2048: 40 x 11008 x 4096 16.2 / 17.1, 56 x 11136 x 11008 37.3 / 40.5,
//   64 x 9216 x 12032 with zero points 41 / 45; up to 112 rows of 64 x 96 and more from 2048: 80 x 11008 x 4096 20.6 / 22.6; up to 96 of 64 x 96 whose results leave by
//   elements, or of a second slab that is mostly short (66 x 9866 x 304 5.5 / 6.8, 83 x 11894 x 1088 8.9 / 9.6, 77 x 10264 x 304 6.0 / 6.6; 108 rows 1.05);
//   with zero points, which every tile takes from its weights and the chunked kernel once a weight: up to sixteen rows tiles of sixteen
//   columns from K = 8192 on (16 x 1984 x 12032 12.7 / 13.8), up to 32 rows of 64 from 1600 (16 x 11136 x 2176 9.1 / 10.3, 24 x 5120 x 1920
//   7.2 / 7.8), up to 48 rows of 32 x 64 from 3072 (48 x 8192 x 11008 0.94); K = 2176 on tiles of 16 x 16 stays a twentieth behind
// -- unless there are more channels than that (40 x 14336 x 992 10.8 / 6.9, 16 x 14336 x 4096 16.9 / 15.0, 16 x 32000 x 5120 1.10, 32 x 32000 x 4096
// 38 / 32), but for up to sixteen rows where eight ninths and more of the CUs would have a tile of weights whose rows stand whole 4 KiB
// apart, which then come from the same channels: 8 x 24576 x 4096 21.7 / 25.8, 16 x 32768 x 4096 32.4 / 36.4, 6 x 22016 x 4096 20.5 / 23.0 (24576 x
// 5120 1.06, 40000 x 4096 1.05), and where three quarters and fewer would have one of 64 x 192 and K is past 3000 (14 x 36608 x 4128 34.8 / 46.7, 6 x
// 34731 x 5264 38 / 49, 3 x 33024 x 4192 32 / 37; 1.13 times the rate over 155, K to 3000 level, more channels 0.95 and less).
// Calls that the tiles of gemm.hip do not take (zero points, K off whole slabs of 64) would go in passes of 128 rows: they come
// here at any size, with the tile whose rounds cost least (weights: us per 3000 of K measured above; 511 x 10907 x 13056 1238 ->
// 180, 1000 x 14336 x 992 139 -> 53, 304 x 11008 x 4368 73 -> 60).
GemmFewTile plan_w8a16_few(int64_t M, int64_t N, int64_t K, bool tiles, bool zp) {
  const int64_t cus = hexmi_num_cus();
  if (cus <= 0 || M <= 2 || K > (1 << 22) || M > (1 << 30) || N > (1 << 30)) return {0, 0};
  const bool chunked = N <= 48 * cus, heavy = N * K >= (24 << 20) || (M > 4 && N * K > (20 << 20));    // the stream of
                                                                 // weights is most of the call
  struct Tile { GemmFewTile tile; int weight; };
  static constexpr Tile kShort[] = {{{16, 16}, 0}, {{16, 32}, 0}, {{16, 64}, 0}, {{32, 32}, 0}};
  static constexpr Tile kLong[] = {{{16, 16}, 0}, {{16, 32}, 0}, {{32, 32}, 0}, {{16, 64}, 0}};
  static constexpr Tile kLarge[] = {{{32, 64}, 20}, {{48, 64}, 0}, {{32, 96}, 0}, {{64, 64}, 30}, {{64, 96}, 0}, {{64, 128}, 50}, {{64, 192}, 65}};
  auto count = [&](const GemmFewTile& t) { return ((M + t.m - 1) / t.m) * ((N + t.n - 1) / t.n); };
  for (const Tile& t : K <= 2048 ? kShort : kLong) {
    if (count(t.tile) > cus) continue;
    if (chunked && heavy && (M <= 16 || (M <= 32 && t.tile.n == 64))) return {0, 0};
    if (chunked && M <= 32 && t.tile.m == 32 && K > 3072) return {0, 0};
    if (chunked && zp && ((M <= 16 && t.tile.n == 16 && K >= 8192) || (M <= 32 && t.tile.n == 64 && K > 1536))) return {0, 0};
    return t.tile;
  }
  GemmFewTile best = {0, 0};
  int64_t least = 0;
  for (const Tile& t : kLarge) {
    const int64_t rounds = (count(t.tile) + cus - 1) / cus;
    if (rounds == 1) {
      const int area = t.tile.m * t.tile.n;
      if (area == 64 * 96 && K > (M <= 192 ? 2048 : 4608)) continue;
      if (chunked && ((M <= 32 && K > 1536) || (M <= 48 && (area > 32 * 64 ? K > 1536 : zp && K >= 3072)) ||
                      (M <= 64 && t.tile.n == 96 && K >= 2048) || (M <= 112 && area >= 64 * 96 && K >= 2048))) return {0, 0};
      if (chunked && M <= 96 && area == 64 * 96 && (N % 8 != 0 || (K > 256 && K <= 384))) return {0, 0};
      if (M <= 16 && ((K % 4096 == 0 && 9 * count(t.tile) >= 8 * cus) || (t.tile.n == 192 && K > 3000 && 4 * count(t.tile) <= 3 * cus)))
        return {0, 0};
      return t.tile;
    }
    if (!t.weight || tiles || M <= 128 || count(t.tile) > 0x7fffffff) continue;
    if (!best.m || rounds * t.weight < least) best = t.tile, least = rounds * t.weight;
  }
  return best;
}

int launch_w8a16_few(const GemmFewTile& tile, int64_t M, int64_t N, int64_t K, const f16* A, const int8_t* W, const f16* scales,
                     const int8_t* zero_points, int per_tensor, f16* C, hipStream_t s) {
  const int tiles_m = (int)((M + tile.m - 1) / tile.m), tiles_n = (int)((N + tile.n - 1) / tile.n);
  const int runs = N % 8 == 0 && aligned_to(C, 16);
#define HEXMI_FEW_Z(BM, BN, ZP)                                                                                               \
  hipLaunchKernelGGL((w8a16_few_kernel<FewShape<BM, BN>::S, ZP>), dim3((unsigned)(tiles_m * tiles_n)),                        \
                     dim3(FewShape<BM, BN>::S::kThreads), 0, s, A, W, scales, zero_points, C, (int)M, (int)N, (int)K, tiles_m, \
                     tiles_n, per_tensor, runs)
#define HEXMI_FEW(BM, BN) \
  if (tile.m == BM && tile.n == BN) { if (zero_points) HEXMI_FEW_Z(BM, BN, true); else HEXMI_FEW_Z(BM, BN, false); return launch_status(); }
  HEXMI_FEW(16, 16) HEXMI_FEW(16, 32) HEXMI_FEW(16, 64) HEXMI_FEW(32, 32) HEXMI_FEW(32, 64) HEXMI_FEW(32, 96)
  HEXMI_FEW(48, 64) HEXMI_FEW(64, 64) HEXMI_FEW(64, 96) HEXMI_FEW(64, 128) HEXMI_FEW(64, 192)
#undef HEXMI_FEW
#undef HEXMI_FEW_Z
  return HEXMI_ENOTSUP;
}

}  // namespace hexmi
