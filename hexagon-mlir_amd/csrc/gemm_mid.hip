// C[M,N] = A[M,K] * op(B) (+ bias + residual) on tiles of 128 x 128 to 256 x 192 (fp16 / bf16 in and out, fp32 sums), K a multiple of 8.
//
// What bounds a product of some hundred to some thousand rows and columns is how its tiles fill the rounds over the CUs, and under that
// what a CU takes in (92 GB/s through L2: a tile asks for BM + BN rows of each slab) and the power of the MFMAs. The schedule is
// gemm_kernel_k64's (gemm.hip: slabs of 64 of K, four waves of TM x TN tiles of 16 x 16, fragments of the next step read and copies of a later
// slab issued between the MFMAs of this one, one barrier a slab) for tiles that need not be square and two to four stages: what fits the
// LDS. A copy whose chunk or row lies past the end of K has its offset put past the end of its buffer descriptor, which the hardware
// answers with zeros: a short last slab and slabs past the last cost a comparison per copy, and no form of its own. Where K is whole
// slabs and the tile 128 x 128 that makes it 0 to 8 % slower than gemm_kernel_k64, which keeps those.
#include <algorithm>
#include <type_traits>

#include "hexmi_common.h"

namespace hexmi {
namespace {

constexpr int BK = 64;                 // K extent of a slab (elements)

template <typename T> struct Types;
template <> struct Types<f16> {
  typedef f16x8 Frag;
  typedef f16x4 Run;
  // tied accumulators: see gemm.hip
  static __device__ __forceinline__ void mfma(const f16x8& a, const f16x8& b, f32x4& c) {
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
  }
};
template <> struct Types<bf16> {
  typedef bf16x8 Frag;
  typedef bf16x4 Run;
  static __device__ __forceinline__ void mfma(const bf16x8& a, const bf16x8& b, f32x4& c) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
  }
};

__device__ __forceinline__ int swz_row(int row) { return (row >> 1) & 7; }
// a row of 192 columns is one and a half rows of banks: k & 1 already moves it by half of them
template <int BN> __device__ __forceinline__ int swz_col(int k) {
  return BN == 192 ? (((k >> 1) & 1) | (((k >> 3) & 1) << 1)) << 1 : ((k & 3) | (((k >> 3) & 1) << 2)) << 1;
}

constexpr int kPast = (int)0x80000000u;     // a copy's offset past the end of its descriptor: zeros

// ODD: output rows of any length at any place, with or without bias and residual: a wave's sums pass through LDS 16 rows at a time and
// leave, and take bias and residual, by elements, 64 columns of a row to an instruction; the residual of the next rows is on its way meanwhile.
// (us on 128 x 128 tiles of 32-k slabs, bias and residual one load after the other / here: 6177 x 869 x 1344 + residual 61 / 32, 896 x 35335 x 400 +
// residual 190 / 88, 1021 x 50257 x 768 + bias 239 / 159, 2942 x 3571 x 3984 163 / 118, 4524 x 3741 x 384 + both 133 / 53; 1.83 times the rate over 40.)
// PLAIN: the result leaves by plain stores. Those past the caches are for rows in whole lines or half of them; rows 16 or 32 bytes off share
// a line with the next tile, which memory then puts together twice.
template <typename T, int TM, int TN, int NS, bool TRANS_B, bool EPI, bool ODD = false, bool PLAIN = false>
__global__ __launch_bounds__(256)
void gemm_mid_kernel(const T* __restrict__ A, const T* __restrict__ B, T* C, int M, int N, int K, int64_t lda, int64_t ldb, int64_t ldc,
                     int tiles_m, int tiles_n, const T* __restrict__ bias, const T* resid, int64_t ldr) {
  typedef typename Types<T>::Frag Frag;
  typedef typename Types<T>::Run Run;
  constexpr int BM = 32 * TM, BN = 32 * TN;
  static_assert(!(EPI && ODD), "ODD takes bias and residual its own way");
  static_assert(NS >= 2 && NS <= 4 && TM % 2 == 0 && TN % 2 == 0 && TM >= 4 && TN >= 4, "shapes");
  __shared__ __attribute__((aligned(16))) T a_p0[BM * BK];
  __shared__ __attribute__((aligned(16))) T a_p1[BM * BK];
  __shared__ __attribute__((aligned(16))) T a_p2[NS >= 3 ? BM * BK : 8];
  __shared__ __attribute__((aligned(16))) T a_p3[NS >= 4 ? BM * BK : 8];
  __shared__ __attribute__((aligned(16))) T b_p0[BN * BK];
  __shared__ __attribute__((aligned(16))) T b_p1[BN * BK];
  __shared__ __attribute__((aligned(16))) T b_p2[NS >= 3 ? BN * BK : 8];
  __shared__ __attribute__((aligned(16))) T b_p3[NS >= 4 ? BN * BK : 8];

  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int wm = wave / 2, wn = wave % 2;
  int tm, tn;
  tile_of_block<4>(blockIdx.x, tiles_m, tiles_n, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;

  f32x4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  constexpr bool kResid = EPI && TM * TN <= 36;           // (256 x 192: no registers for a residual)
  Run resid_frag[kResid ? TM : 1][kResid ? TN : 1], bias_frag[EPI ? TN : 1];
  auto col_of = [&](int j) { const int col = n0 + (wn * TN + j) * 16 + 4 * (lane / 16); return col < N - 4 ? col : N - 4; };
  auto row_of = [&](int i) { const int row = m0 + (wm * TM + i) * 16 + lane % 16; return row < M ? row : M - 1; };
  if constexpr (EPI) {
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      if (bias) bias_frag[j] = *reinterpret_cast<const Run*>(bias + col_of(j));
      if constexpr (kResid) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
          if (resid) resid_frag[i][j] = *reinterpret_cast<const Run*>(resid + (int64_t)row_of(i) * ldr + col_of(j));
      }
    }
  }

  // copies: TM of A and TN of B a slab and wave, 1 KiB each
  constexpr int NL = TM + TN, CPRB = BN / 8;
  int voff[NL], kb[TRANS_B ? 1 : TN];
  const int kc = ((lane % 8) ^ swz_row(wave * 8 + lane / 8)) * 8;      // the chunk of K a lane copies of rows: the same in every copy
#pragma unroll
  for (int j = 0; j < TM; ++j) {
    const int row = (j * 4 + wave) * 8 + lane / 8, left = M - m0 - 1;
    voff[j] = (int)(((int64_t)(row < left ? row : left) * lda + kc) * 2);
  }
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    if constexpr (TRANS_B) {
      const int row = (j * 4 + wave) * 8 + lane / 8, left = N - n0 - 1;
      voff[TM + j] = (int)(((int64_t)(row < left ? row : left) * ldb + kc) * 2);
    } else {
      const int lin = (j * 4 + wave) * 64 + lane, k = lin / CPRB, c = (lin % CPRB) ^ swz_col<BN>(k), left = N - n0 - 8;
      voff[TM + j] = (int)(((int64_t)k * ldb + (c * 8 < left ? c * 8 : left)) * 2);
      kb[j] = k;
    }
  }
  const char* a_base = reinterpret_cast<const char*>(A + (int64_t)m0 * lda);
  const char* b_base = reinterpret_cast<const char*>(TRANS_B ? B + (int64_t)n0 * ldb : B + n0);
  const int64_t a_step = BK * 2, b_step = (TRANS_B ? BK : BK * ldb) * 2;
  const int KT = (K + BK - 1) / BK;
  // copy n of a slab: A's, then B's ([K,N]: B's first)
  auto copy_n = [&](int n, int slab, T* a_dst, T* b_dst) __attribute__((always_inline)) {
    const int i = TRANS_B ? n : (n < TN ? TM + n : n - TN);
    const int left = K - slab * BK;                                    // (negative in slabs past the last)
    const int at = i < TM || TRANS_B ? kc : kb[TRANS_B ? 0 : i - TM];
    const int off = at < left ? voff[i] : kPast;
    const int s = slab < KT ? slab : KT - 1;
    if (i < TM) copy_to_lds(a_base + s * a_step, off, a_dst + (i * 4 + wave) * 512);
    else copy_to_lds(b_base + s * b_step, off, b_dst + ((i - TM) * 4 + wave) * 512);
  };
  auto read_a = [&](const T* src, int ks, int i) __attribute__((always_inline)) {
    const int row = (wm * TM + i) * 16 + lane % 16;
    return *reinterpret_cast<const Frag*>(src + row * BK + (((ks * 4 + lane / 16) ^ swz_row(row)) * 8));
  };
  auto read_b = [&](const T* src, int ks, int j) __attribute__((always_inline)) {
    if constexpr (TRANS_B) {
      const int row = (wn * TN + j) * 16 + lane % 16;
      return *reinterpret_cast<const Frag*>(src + row * BK + (((ks * 4 + lane / 16) ^ swz_row(row)) * 8));
    } else {
      const int g = lane / 16, i = lane % 16;
      const int n = (wn * TN + j) * 16 + (i & 3) * 4, k = ks * 32 + g * 8 + (i >> 2);
      union { i16x4 h[2]; Frag f; } u;
#pragma unroll
      for (int p = 0; p < 2; ++p)
        u.h[p] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4*)(
            src + ((k + 4 * p) * CPRB + ((n / 8) ^ swz_col<BN>(k + 4 * p))) * 8 + n % 8));
      return u.f;
    }
  };
  Frag af[2][TM], bf[2][TN];
  auto read_n = [&](int n, const T* a_src, const T* b_src, int ks) __attribute__((always_inline)) {
    if (n < TN) bf[ks][n] = read_b(b_src, ks, n);
    else if (n < TM + TN) af[ks][n - TN] = read_a(a_src, ks, n - TN);
  };

  // A slab's copies go out in the window of 2 TM rounds between the barrier that frees their stage and the next one.
  constexpr int PER = (TM + TN + TM - 1) / TM;                         // reads, and with B as [N,K] copies, of a round: two or three
  static_assert(PER <= TN / 2, "a slot each");
  auto copies_before = [](int w) constexpr {
    int sum = 0;
    for (int r = 0; r < w; ++r) sum += TRANS_B ? PER : (r < std::max(TM / 2, NL - 2 * TM) ? 2 : 1);
    return sum < NL ? sum : NL;
  };
  constexpr int LATE = NL - copies_before(TM);
  static_assert(copies_before(2 * TM) == NL, "the window carries all of a slab's copies");
#pragma unroll
  for (int n = 0; n < NL; ++n) copy_n(n, 0, a_p0, b_p0);
  if constexpr (NS >= 3) {
#pragma unroll
    for (int n = 0; n < NL; ++n) copy_n(n, 1, a_p1, b_p1);
  }
  if constexpr (NS >= 4) {
#pragma unroll
    for (int n = 0; n < NL; ++n) copy_n(n, 2, a_p2, b_p2);
  }
#pragma unroll
  for (int n = 0; n < NL - LATE; ++n)
    copy_n(n, NS - 1, NS == 2 ? a_p1 : NS == 3 ? a_p2 : a_p3, NS == 2 ? b_p1 : NS == 3 ? b_p2 : b_p3);
  __builtin_amdgcn_s_waitcnt(waitcnt_imm((NS - 1) * NL - LATE));       // slab 0 landed
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int n = 0; n < TM + TN; ++n) read_n(n, a_p0, b_p0, 0);

#define HEXMI_FENCE __builtin_amdgcn_sched_barrier(0)
  auto slab = [&](T* acur, T* bcur, T* anxt, T* bnxt, T* aprv, T* bprv, int j) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < 2 * TM; ++q) {
      const int ks = q / TM, row = q % TM;
      if (q == TM) {
        HEXMI_FENCE;
        __builtin_amdgcn_s_waitcnt(waitcnt_imm((NS - 2) * NL));        // all but slabs j+2 .. j+NS-1 have landed
        __builtin_amdgcn_s_barrier();
        HEXMI_FENCE;
      }
#pragma unroll
      for (int jj = 0; jj < TN / 2; ++jj) {
        const int c0 = (row & 1) ? TN - 1 - 2 * jj : 2 * jj, c1 = (row & 1) ? c0 - 1 : c0 + 1;
        Types<T>::mfma(bf[ks][c0], af[ks][row], acc[row][c0]);
        Types<T>::mfma(bf[ks][c1], af[ks][row], acc[row][c1]);
        HEXMI_FENCE;
        if (jj < PER) {
          const int n = row * PER + jj;
          if (ks == 0) read_n(n, acur, bcur, 1);
          else read_n(n, anxt, bnxt, 0);
        }
        constexpr int CSLOT = (TN >= 8 && !TRANS_B) ? 2 : 0, CN = TRANS_B ? PER : 2;
        if (jj >= CSLOT && jj < CSLOT + CN) {
          const int c = jj - CSLOT, w = (q + TM) % (2 * TM);
          const int lo = copies_before(w), hi = copies_before(w + 1);
          if (lo + c < hi) {
            if (ks == 1) copy_n(lo + c, j + NS, acur, bcur);
            else copy_n(lo + c, j + NS - 1, aprv, bprv);
          }
        }
        HEXMI_FENCE;
      }
    }
  };
  for (int j = 0; j < KT; j += NS) {
    if constexpr (NS == 2) {
      slab(a_p0, b_p0, a_p1, b_p1, a_p1, b_p1, j);
      slab(a_p1, b_p1, a_p0, b_p0, a_p0, b_p0, j + 1);
    } else if constexpr (NS == 3) {
      slab(a_p0, b_p0, a_p1, b_p1, a_p2, b_p2, j);
      slab(a_p1, b_p1, a_p2, b_p2, a_p0, b_p0, j + 1);
      slab(a_p2, b_p2, a_p0, b_p0, a_p1, b_p1, j + 2);
    } else {
      slab(a_p0, b_p0, a_p1, b_p1, a_p3, b_p3, j);
      slab(a_p1, b_p1, a_p2, b_p2, a_p0, b_p0, j + 1);
      slab(a_p2, b_p2, a_p3, b_p3, a_p1, b_p1, j + 2);
      slab(a_p3, b_p3, a_p0, b_p0, a_p2, b_p2, j + 3);
    }
    if (j + NS >= KT) {                                // wait states between the last MFMA and the first read of a sum
      HEXMI_FENCE;
      asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
      HEXMI_FENCE;
    }
  }
#undef HEXMI_FENCE
  __builtin_amdgcn_s_waitcnt(waitcnt_imm(0));

  if constexpr (EPI) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if (bias) acc[i][j][r] += to_f32<T>(bias_frag[j][r]);
          if constexpr (kResid)
            if (resid) acc[i][j][r] += to_f32<T>(resid_frag[i][j][r]);
        }
      }
  }
  __syncthreads();
  if constexpr (ODD) {
    constexpr int W = TN * 16, PW = W + 4, EACH = W / 4;           // columns of the wave's tile, pitch, elements a lane takes of 16 rows
    float* st = reinterpret_cast<float*>(wave == 0 ? a_p0 : wave == 1 ? a_p1 : wave == 2 ? b_p0 : b_p1);
    static_assert(16 * PW * 4 <= BN * BK * 2 && 16 * PW * 4 <= BM * BK * 2, "16 rows of sums fit one stage");
    const int row0 = m0 + wm * TM * 16, col0 = n0 + wn * W;
    T add[EACH], res[2][EACH];
    auto ask = [&](int i, T* to) __attribute__((always_inline)) {
#pragma unroll
      for (int t = 0; t < EACH; ++t) {
        const int e = lane + 64 * t, row = row0 + i * 16 + e / W, col = col0 + e % W;
        to[t] = resid[(int64_t)(row < M ? row : M - 1) * ldr + (col < N ? col : N - 1)];
      }
    };
    if (bias) {
#pragma unroll
      for (int t = 0; t < EACH; ++t) {
        const int col = col0 + (lane + 64 * t) % W;
        add[t] = bias[col < N ? col : N - 1];
      }
    }
    if (resid) ask(0, res[0]);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
      for (int j = 0; j < TN; ++j) *reinterpret_cast<f32x4*>(st + (lane % 16) * PW + j * 16 + 4 * (lane / 16)) = acc[i][j];
      if (resid && i + 1 < TM) ask(i + 1, res[(i + 1) & 1]);
#pragma unroll
      for (int t = 0; t < EACH; ++t) {
        const int e = lane + 64 * t, row = row0 + i * 16 + e / W, col = col0 + e % W;
        float v = st[e / W * PW + e % W];
        if (bias) v += to_f32<T>(add[t]);
        if (resid) v += to_f32<T>(res[i & 1][t]);
        if (row < M && col < N) C[(int64_t)row * ldc + col] = from_f32<T>(v);
      }
    }
    return;
  }
  T* cs = wave == 0 ? a_p0 : wave == 1 ? a_p1 : wave == 2 ? b_p0 : b_p1;
  constexpr int CP = TN * 2, PITCH = TN * 16;          // 16-byte chunks and elements of a row of the wave's tile
  static_assert(TM * 16 * PITCH <= BM * BK && TM * 16 * PITCH <= BN * BK, "a wave's tile fits one stage");
  auto swz = [](int row) { return CP == 16 ? (row & 15) : CP == 8 ? ((row >> 1) & 7) : ((row >> 2) & 3); };
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int row = i * 16 + lane % 16;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int col = j * 16 + 4 * (lane / 16);
      store4<T>(cs + row * PITCH + (((col / 8) ^ swz(row)) * 8) + col % 8, acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]);
    }
  }
  constexpr int RPI = 64 / CP;
#pragma unroll
  for (int r0 = 0; r0 < TM * 16; r0 += RPI) {
    const int row = r0 + lane / CP, c = lane % CP;
    if (64 % CP && (lane >= RPI * CP || row >= TM * 16)) continue;
    const u32x4 v = *reinterpret_cast<const u32x4*>(cs + row * PITCH + ((c ^ swz(row)) * 8));
    const int grow = m0 + wm * TM * 16 + row, gcol = n0 + wn * TN * 16 + c * 8;
    u32x4* to = reinterpret_cast<u32x4*>(C + (int64_t)grow * ldc + gcol);
    if (grow < M && gcol < N) {
      if constexpr (PLAIN) *to = v; else __builtin_nontemporal_store(v, to);
    }
  }
}

}  // namespace

// What a launch takes, us: rounds of tiles over the CUs (two tiles to a CU where two fit), slabs of K in each. A round costs a part by its
// length and a part by how many of its tiles there are (they share L2 and the chip's power). Fitted to 370 random products of 65 to
// 8192 rows, K = 256 to 12288, on one card (mean error 7 to 10 %); of these tiles the one it names is 1.2 % off the best.
struct MidCost { int m, n, per_cu; double start, slab, slab_full, tile, tile_full, resid; };
static double mid_time(const MidCost& c, int64_t M, int64_t N, int64_t K, bool resid) {
  const int64_t tiles = ((M + c.m - 1) / c.m) * ((N + c.n - 1) / c.n), slots = std::max(1, hexmi_num_cus()) * c.per_cu;
  const double rounds = (double)((tiles + slots - 1) / slots), full = (double)tiles / slots, slabs = (double)((K + BK - 1) / BK);
  return c.start + slabs * (c.slab * rounds + c.slab_full * full) + c.tile * rounds + (c.tile_full + (resid ? c.resid : 0)) * full;
}
static constexpr MidCost kMidTiles[] = {
    {128, 128, 1, 2.3, 0.451, 0.047, 2.9, 0.8, 3.1}, {128, 128, 2, 2.7, 0.703, 0.199, 0.4, 4.3, 5.2}, {192, 128, 1, 2.1, 0.550, 0.080, 4.1, 1.2, 4.3},
    {256, 128, 1, 1.6, 0.692, 0.085, 5.0, 1.5, 5.6}, {192, 192, 1, 1.6, 0.718, 0.097, 6.1, 1.0, 7.2}, {256, 192, 1, 0.6, 1.020, 0.072, 6.7, 1.5, 0.0}};
// ... and the kernels of gemm.hip: 128 x 128 tiles, one and two to a CU, and 256 x 256
static constexpr MidCost kOne = {128, 128, 1, 4.0, 0.445, 0.073, 1.9, 0.0, 3.9}, kTwo = {128, 128, 2, 1.7, 0.626, 0.354, 3.1, 1.6, 4.9},
                         kLarge = {256, 256, 1, 5.0, 0.427, 1.151, 2.2, 6.6, 0.0};

// The tiles between 128 x 128 and 256 x 256 are for what those leave: products whose rounds of either are far from full, and products with
// bias or residual, for which the 256 x 256 tiles have no registers. K off whole 64s comes here always. us on 128 x 128 or 256 x 256 tiles /
// here: 1336 x 6400 x 1600 + bias 53 / 30 (192 x 192), 3787 x 1712 x 2920 + residual 77 / 49, 5712 x 3200 x 1576 + bias 127 / 65, 1291 x 3096 x 2552
// + bias 57 / 33, 862 x 11144 x 1216 + bias 35 / 29, 2206 x 3896 x 1344 36 / 27, 645 x 12456 x 6560 202 / 135; all 370: 1.11 times the rate,
// K off whole 64s 1.49. A twentieth's lead is asked for, since the fits are that good: without it one in ten is slower. With it, of 200 other
// products of whole 64s and of 8s 82 of whole 64s came here, at 1.13 times the rate, five of them 5 to 10 % slower than before (1636 x 21440 x
// 1408 + both 122 / 135, 4480 x 3840 x 320 + bias 26.2 / 27.5).
// The fits begin at K = 256 and say too little below for the tiles of 192 x 128: 339 x 28864 x 64 10.2 / 13.5, 285 x 31872 x 128 10.7 / 13.2, 192 x
// 12800 x 64 + residual 8.1 / 9.9, beside 256 x 256 tiles also 384 x 30464 x 384 18.3 / 21.2 (33 of 34 slower; up to 64 rows they are ahead
// of 256 x 256 tiles by a third, in the place of 128 x 128 ones two to a CU from 320 on).
// Odd rows of less than 1024 of K: the larger tiles' elements leave with nothing beside them, so two of 128 x 128 to a CU (or one), us on the
// 32-k slabs of gemm.hip / the tile of the fit / here: 8000 x 10001 x 456 151 / 205 / 143, 3000 x 15003 x 584 114 / 148 / 106, 6000 x 3333 x 584
// 61 / 66 / 55, 4000 x 2500 x 584 34.5 / 40 / 33.5 (3000 x 3001 x 776 42 / 34 / 39); from 1024 on the fit is ahead.
GemmMidTile plan_gemm_mid(int64_t M, int64_t N, int64_t K, int now, bool resid, bool odd) {
  const MidCost* best = nullptr;
  double least = now == 0 ? 1e30 : 0.95 * mid_time(now == 256 ? kLarge : now == 2 ? kTwo : kOne, M, N, K, resid);
  for (const MidCost& c : kMidTiles) {
    if (now != 0 && c.m == 128) continue;                    // (gemm.hip's own are the better ones of whole slabs)
    if (now != 0 && c.m * c.n == 192 * 128 && M > 64 && K <= (now == 256 ? 768 : 128)) continue;
    if ((resid && c.m * c.n > 192 * 192) || (odd && K < 1024 && c.m > 128)) continue;
    if (!grid_fits(((M + c.m - 1) / c.m) * ((N + c.n - 1) / c.n), 256)) continue;
    const double t = mid_time(c, M, N, K, resid);
    if (t < least) least = t, best = &c;
  }
  return best ? GemmMidTile{best->m, best->n, best->per_cu} : GemmMidTile{0, 0, 0};
}

template <typename T, bool TRANS_B>
int launch_gemm_mid(const GemmMidTile& tile, const T* A, const T* B, T* C, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb,
                    int64_t ldc, hipStream_t s, const T* bias, const T* resid, int64_t ldr, bool odd) {
  const int64_t tiles_m = (M + tile.m - 1) / tile.m, tiles_n = (N + tile.n - 1) / tile.n;
  if (!grid_fits(tiles_m * tiles_n, 256) || (resid && tile.m * tile.n > 192 * 192)) return HEXMI_ENOTSUP;
  // (us past the caches / plain: 4946 x 19608 x 32 + bias 94 / 62, 5925 x 6544 x 16 32 / 24, 1610 x 31888 x 32 45 / 32, 4108 x 8232 x 64 32 / 27, 5437 x 6200
  // x 256 39 / 34, 1400 x 23656 x 512 56 / 53; 1.20 times the rate over 400. Results of 8 to 32 MiB 0.96 to 1.04 times it, with a residual 0.98, rows
  // half a line off 0.95.)
  const bool plain = ldc % 32 != 0 && !resid && M * N >= (16 << 20);
#define HEXMI_MID_AS(TM, TN, NS, EPI, ODD, PLAIN)                                                                                    \
  hipLaunchKernelGGL((gemm_mid_kernel<T, TM, TN, NS, TRANS_B, EPI, ODD, PLAIN>), dim3((unsigned)(tiles_m * tiles_n)), dim3(256), 0, s, A, B, \
                     C, (int)M, (int)N, (int)K, lda, ldb, ldc, (int)tiles_m, (int)tiles_n, bias, resid, ldr)
#define HEXMI_MID(TM, TN, NS)                                                                                                  \
  do {                                                                                                                         \
    if (TRANS_B && odd) HEXMI_MID_AS(TM, TN, NS, false, TRANS_B, false);                                                        \
    else if (bias || resid) { if (plain) HEXMI_MID_AS(TM, TN, NS, true, false, true); else HEXMI_MID_AS(TM, TN, NS, true, false, false); } \
    else if (plain) HEXMI_MID_AS(TM, TN, NS, false, false, true);                                                              \
    else HEXMI_MID_AS(TM, TN, NS, false, false, false);                                                                         \
  } while (0)
  if (odd && !TRANS_B) return HEXMI_ENOTSUP;
  if (tile.m == 128 && tile.per_cu == 2) HEXMI_MID(4, 4, 2);
  else if (tile.m == 128) HEXMI_MID(4, 4, 4);
  else if (tile.m == 192 && tile.n == 128) HEXMI_MID(6, 4, 4);
  else if (tile.m == 256 && tile.n == 128) HEXMI_MID(8, 4, 3);
  else if (tile.m == 192) HEXMI_MID(6, 6, 3);
  else HEXMI_MID(8, 6, 2);
#undef HEXMI_MID
#undef HEXMI_MID_AS
  return launch_status();
}

#define HEXMI_INSTANCE(T, TB)                                                                                                  \
  template int launch_gemm_mid<T, TB>(const GemmMidTile&, const T*, const T*, T*, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, \
                                      hipStream_t, const T*, const T*, int64_t, bool);
HEXMI_INSTANCE(f16, false)
HEXMI_INSTANCE(f16, true)
HEXMI_INSTANCE(bf16, false)
HEXMI_INSTANCE(bf16, true)
#undef HEXMI_INSTANCE

}  // namespace hexmi
