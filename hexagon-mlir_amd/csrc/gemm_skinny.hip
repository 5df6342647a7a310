// C[M,N] = A[M,K] * B[N,K]^T for up to 64 rows of A (fp16 / bf16 in, fp32 sums): a stream of the weights B on the matrix
// cores. A workgroup takes 16, 32 or 64 output channels and all the rows; its waves split K in rounds of 64 (whole
// 128-byte lines), dealt out in turn, and their partial tiles meet in LDS.
//
// What bounds it: N = 4096, K = 11008 reads 90 MB of weights (15 us at 6 TB/s), and every workgroup pulls all the
// activations through L2, at 32 rows twice the bytes of its weights. Loading operands straight into the MFMA's register
// layout (lane -> row lane % 16) puts neighbouring lanes on different rows, so that every 16 bytes are a request of their
// own: a CU took in 29 GB/s that way whatever was in flight (4 to 16 waves, 2 to 8 steps: 36 to 38 us). Here a
// wave copies its rounds into LDS eight lanes to a 128-byte line (each wave its own two stages: no barrier in
// the K walk) and reads the operands from there, chunk c of row r at c ^ ((r / 2) % 8). Cold weights, us, before -> now:
//   N = 4096, K = 4096:   16 rows 11.8 -> 8.7, 32 rows 15.2 -> 10.3
//   N = 4096, K = 11008:  27.7 -> 19.7, 36 -> 24.6        N = 768, K = 3072: 9.3 -> 4.4, 12 -> 5.6
//   N = 11008, K = 4096 (on the 128 x 128 tiles before): 31.7 -> 19, 32.4 -> 24.2
// (Larger weights, and 33 rows and more, go to gemm_few.hip wherever one round of its tiles covers them.)
// Three and four stages, and counted waits in place of the loop's full ones, measured equal.
#include <algorithm>

#include "hexmi_common.h"

namespace hexmi {
namespace {

#define HEXMI_LDS(p) ((__attribute__((address_space(3))) void*)(p))
#define HEXMI_GLB(p) ((const __attribute__((address_space(1))) void*)(p))

constexpr int kRoundK = 64;             // k of a round: one 128-byte line of a row

__device__ __forceinline__ f32x4 mfma16(const f16x8& w, const f16x8& a, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(w, a, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mfma16(const bf16x8& w, const bf16x8& a, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, a, c, 0, 0, 0);
}
template <typename T> struct Frag8;
template <> struct Frag8<f16> { typedef f16x8 V; };
template <> struct Frag8<bf16> { typedef bf16x8 V; };

// MT, NT: 16-row tiles of activations and of channels; NWV waves. ONCE: the weights are too large to be in a cache at
// the next call, and are read non-temporally. K % 32 == 0, rows of both operands on 16-byte boundaries.
template <typename T, typename OutT, int MT, int NT, int NWV, bool ONCE>
__global__ __launch_bounds__(NWV * 64)
void gemm_nt_skinny_kernel(const T* __restrict__ A, const T* __restrict__ W, OutT* C, int M, int N, int K, int64_t lda,
                           int64_t ldb, int64_t ldc, const OutT* __restrict__ bias, const OutT* resid, int64_t ldr) {
  typedef typename Frag8<T>::V Frag;
  constexpr int kCopies = (NT + MT) * 2;                     // a copy instruction: eight rows of 128 bytes
  constexpr int kStage = (NT + MT) * 16 * kRoundK;           // elements of a wave's stage: channels, then rows
  // two objects: reads of one stage are told apart from copies into the other
  __shared__ __attribute__((aligned(16))) T stage0[NWV * kStage];
  __shared__ __attribute__((aligned(16))) T stage1[NWV * kStage];
  const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int r16 = lane % 16, kg = lane / 16;
  const int ch0 = blockIdx.x * (NT * 16);

  // past the last channel or row: the last one, not stored
  const T* src[kCopies];
#pragma unroll
  for (int j = 0; j < kCopies; ++j) {
    const int row = j * 8 + lane / 8, col = ((lane % 8) ^ ((row >> 1) & 7)) * 8;
    if (j < NT * 2) {
      const int n = ch0 + row;
      src[j] = W + (int64_t)(n < N ? n : N - 1) * ldb + col;
    } else {
      const int m = row - NT * 16;
      src[j] = A + (int64_t)(m < M ? m : M - 1) * lda + col;
    }
  }
  const int rounds = K / kRoundK;
  const int mine = rounds > wave ? (rounds - wave + NWV - 1) / NWV : 0;      // rounds wave, wave + NWV, ...
  auto load = [&](int i, T* stage) __attribute__((always_inline)) {
    const int64_t k0 = (int64_t)(wave + i * NWV) * kRoundK;
    T* dst = stage + wave * kStage;
#pragma unroll
    for (int j = 0; j < kCopies; ++j)
      if (ONCE && j < NT * 2)
        __builtin_amdgcn_global_load_lds(HEXMI_GLB(src[j] + k0), HEXMI_LDS(dst + j * 8 * kRoundK), 16, 0, 2);   // 2: nt
      else
        __builtin_amdgcn_global_load_lds(HEXMI_GLB(src[j] + k0), HEXMI_LDS(dst + j * 8 * kRoundK), 16, 0, 0);
  };

  f32x4 acc[NT][MT];
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[n][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](const T* stage) __attribute__((always_inline)) {
    const T* from = stage + wave * kStage + r16 * kRoundK;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int at = (((h * 4 + kg) ^ (r16 >> 1)) & 7) * 8;
      Frag w[NT], a[MT];
#pragma unroll
      for (int n = 0; n < NT; ++n) w[n] = *reinterpret_cast<const Frag*>(from + n * 16 * kRoundK + at);
#pragma unroll
      for (int t = 0; t < MT; ++t) a[t] = *reinterpret_cast<const Frag*>(from + (NT + t) * 16 * kRoundK + at);
#pragma unroll
      for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[n][t] = mfma16(w[n], a[t], acc[n][t]);
    }
    __builtin_amdgcn_sched_barrier(0);             // a stage is refilled when its reads have returned
  };
  if (0 < mine) load(0, stage0);
  if (1 < mine) load(1, stage1);
  // This thread's four-channel pieces of the result (the sums at the end): where they stand, and their bias and residual, asked
  // for here, under the K walk, and without a branch around each: read where they are added they were a chain of as many
  // latencies as a thread has values (40 rows x 14781 x 32 with both 7.5 us, 5.1 so). A residual that is the output itself
  // is read and written by the same thread.
  constexpr int kPieces = (NT * MT + NWV - 1) / NWV;
  OutT add_b[kPieces][4], add_r[kPieces][4];
  auto piece = [&](int p, int& gm, int& gn) __attribute__((always_inline)) {
    const int idx = threadIdx.x + p * NWV * 64, nt = idx / 64, l = idx % 64;
    gm = (nt % MT) * 16 + l % 16;
    gn = ch0 + (nt / MT) * 16 + (l / 16) * 4;
  };
  if (bias) {
#pragma unroll
    for (int p = 0; p < kPieces; ++p) {
      int gm, gn;
      piece(p, gm, gn);
#pragma unroll
      for (int e = 0; e < 4; ++e) add_b[p][e] = bias[gn + e < N ? gn + e : N - 1];
    }
  }
  if (resid) {
#pragma unroll
    for (int p = 0; p < kPieces; ++p) {
      int gm, gn;
      piece(p, gm, gn);
      const OutT* row = resid + (int64_t)(gm < M ? gm : M - 1) * ldr;
#pragma unroll
      for (int e = 0; e < 4; ++e) add_r[p][e] = row[gn + e < N ? gn + e : N - 1];
    }
  }
  int i = 0;
  for (; i + 3 < mine; i += 2) {
    multiply(stage0);
    load(i + 2, stage0);
    __builtin_amdgcn_sched_barrier(0);
    multiply(stage1);
    load(i + 3, stage1);
    __builtin_amdgcn_sched_barrier(0);
  }
  if (i < mine) {
    multiply(stage0);
    if (i + 2 < mine) load(i + 2, stage0);
  }
  if (i + 1 < mine) multiply(stage1);
  if (i + 2 < mine) multiply(stage0);
  if (K % kRoundK != 0 && wave == NWV - 1) {       // the last 32 of K, straight into registers
    const int k = rounds * kRoundK + kg * 8;
    Frag w[NT], a[MT];
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      const int r = ch0 + n * 16 + r16;
      w[n] = *reinterpret_cast<const Frag*>(W + (int64_t)(r < N ? r : N - 1) * ldb + k);
    }
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      const int r = t * 16 + r16;
      a[t] = *reinterpret_cast<const Frag*>(A + (int64_t)(r < M ? r : M - 1) * lda + k);
    }
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int t = 0; t < MT; ++t) acc[n][t] = mfma16(w[n], a[t], acc[n][t]);
  }

  // D[i = channel][j = row]: a lane holds row lane % 16, channels 4 * (lane / 16) + 0 .. 3
  static_assert(NT * MT * 256 * sizeof(float) <= kStage * sizeof(T), "the partial tiles fit into a stage");
  __syncthreads();
  float* red = reinterpret_cast<float*>(stage0);
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int t = 0; t < MT; ++t)
      *reinterpret_cast<f32x4*>(red + (((wave * NT + n) * MT + t) * 64 + lane) * 4) = acc[n][t];
  __syncthreads();
#pragma unroll
  for (int p = 0; p < kPieces; ++p) {
    const int idx = threadIdx.x + p * NWV * 64, nt = idx / 64, l = idx % 64;
    if (NT * MT % NWV != 0 && nt >= NT * MT) break;
    f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < NWV; ++w) sum += *reinterpret_cast<const f32x4*>(red + ((w * NT * MT + nt) * 64 + l) * 4);
    int gm, gn;
    piece(p, gm, gn);
    if (bias) {
#pragma unroll
      for (int e = 0; e < 4; ++e) sum[e] += to_f32<OutT>(add_b[p][e]);
    }
    if (resid) {
#pragma unroll
      for (int e = 0; e < 4; ++e) sum[e] += to_f32<OutT>(add_r[p][e]);
    }
    if (gm < M) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (gn + e < N) C[(int64_t)gm * ldc + gn + e] = from_f32<OutT>(sum[e]);
    }
  }
}

}  // namespace

// Channels and waves of a workgroup, or none of them (the 128 x 128 tiles). Few groups of 16 channels and a long K want many
// waves to a group, many groups or a short K few (a wave without a round costs its LDS and its part of the sum), rows the
// wider groups that read them less often. The lines are where both sides cross over 6 row counts x 19 N x 19 K on 256 CUs,
// cold weights; channels x waves in us:
//   16 rows: N = 4096: K = 256 16x8 3.3, 16x2 3.2; K = 4096 9.7, 15.0. N = 16384, K = 512: 16x8 7.5, 16x2 5.7. N = 40000,
//     K = 1024: 16x2 18.2, 32x4 16.5. N = 28672, K = 6144: 16x2 72, 16x8 66
//   32 rows: N = 8192: K = 512 16x2 4.6, 32x4 4.6. K = 2048: N = 11008 16x2 13.5, 32x2 14.7; N = 14336 17.1, 15.9. N = 50264,
//     K = 2048: 32x2 53, 32x4 48
//   64 rows (up to N = 16384 only where K is 128 or less, or rows of 2^21 elements and more): N = 32768: K = 512 64x4 16.5, tiles
//     12.0; K = 1024 24, 20. N = 30001 with a residual, where the tiles add it by elements: K = 256 32x2 12, tiles 22;
//     K = 1024 64x4 23, tiles 37
GemmSkinnyPlan plan_gemm_skinny(int64_t M, int64_t N, int64_t K, bool tiles) {
  const int64_t cus = std::max(1, hexmi_num_cus()), groups = (N + 15) / 16;
  if (M <= 16) {
    if (K <= 256) return {16, 2};
    if (groups <= 2 * cus) return {16, 8};
    if (groups > 8 * cus && K >= 768) return {32, 4};
    return {16, groups > 4 * cus && K >= 3072 ? 8 : 2};
  }
  if (M <= 32) {
    if (groups <= 5 * cus && K <= 256) return {16, 2};
    if (groups <= cus) return {16, 8};
    if (groups <= 2 * cus) return K < 768 ? GemmSkinnyPlan{16, 2} : GemmSkinnyPlan{32, 4};
    if (groups <= 3 * cus) return {16, 2};
    return {32, groups > 8 * cus && K >= 768 ? 4 : 2};
  }
  if (groups > 5 * cus || (groups > 4 * cus && K > 512)) {
    if (tiles) return {0, 0};
    return K <= 768 ? GemmSkinnyPlan{32, 2} : GemmSkinnyPlan{64, 4};
  }
  if (groups <= cus) return {16, 4};
  if (K <= 512) return groups <= 3 * cus ? GemmSkinnyPlan{16, 2} : GemmSkinnyPlan{32, 2};
  return {64, 4};
}

template <typename T, typename OutT>
int launch_gemm_skinny(const GemmSkinnyPlan& plan, const T* A, const T* B, OutT* C, int64_t M, int64_t N, int64_t K,
                       int64_t lda, int64_t ldb, int64_t ldc, hipStream_t s, const OutT* bias, const OutT* resid, int64_t ldr) {
  const dim3 grid((unsigned)((N + plan.channels - 1) / plan.channels));
  // Weights beyond 64 MB are gone from the 256 MB last-level cache when a program comes back to them. Non-temporal reads of
  // them gain 1 to 1.4 us of 21 to 36 (N = 4096, K = 11008) and cost as much where the weights stay (N = 768, K = 3072: 5.6 -> 7.8).
  const bool once = N * K > (int64_t)32 << 20;
#define HEXMI_SKINNY(MT, NT, NWV)                                                                                              \
  do {                                                                                                                         \
    if (once)                                                                                                                  \
      hipLaunchKernelGGL((gemm_nt_skinny_kernel<T, OutT, MT, NT, NWV, true>), grid, dim3(NWV * 64), 0, s, A, B, C, (int)M,    \
                         (int)N, (int)K, lda, ldb, ldc, bias, resid, ldr);                                                    \
    else                                                                                                                       \
      hipLaunchKernelGGL((gemm_nt_skinny_kernel<T, OutT, MT, NT, NWV, false>), grid, dim3(NWV * 64), 0, s, A, B, C, (int)M,   \
                         (int)N, (int)K, lda, ldb, ldc, bias, resid, ldr);                                                    \
  } while (0)
  if (M <= 16) {
    if (plan.channels == 32) HEXMI_SKINNY(1, 2, 4);
    else if (plan.waves == 8) HEXMI_SKINNY(1, 1, 8);
    else HEXMI_SKINNY(1, 1, 2);
  } else if (M <= 32) {
    if (plan.channels == 32 && plan.waves == 4) HEXMI_SKINNY(2, 2, 4);
    else if (plan.channels == 32) HEXMI_SKINNY(2, 2, 2);
    else if (plan.waves == 8) HEXMI_SKINNY(2, 1, 8);
    else HEXMI_SKINNY(2, 1, 2);
  } else {
    if (plan.channels == 64) HEXMI_SKINNY(4, 4, 4);
    else if (plan.channels == 32) HEXMI_SKINNY(4, 2, 2);
    else if (plan.waves == 4) HEXMI_SKINNY(4, 1, 4);
    else HEXMI_SKINNY(4, 1, 2);
  }
#undef HEXMI_SKINNY
  return launch_status();
}

#define HEXMI_INSTANCE(T, OutT)                                                                                              \
  template int launch_gemm_skinny<T, OutT>(const GemmSkinnyPlan&, const T*, const T*, OutT*, int64_t, int64_t, int64_t,   \
                                           int64_t, int64_t, int64_t, hipStream_t, const OutT*, const OutT*, int64_t);
HEXMI_INSTANCE(f16, f16)
HEXMI_INSTANCE(f16, float)
HEXMI_INSTANCE(bf16, bf16)
HEXMI_INSTANCE(bf16, float)
#undef HEXMI_INSTANCE

}  // namespace hexmi
