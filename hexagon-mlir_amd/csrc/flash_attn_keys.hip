// Flash-attention forward for problems of few (head, query block) units: fp16 / bf16, head sizes up to 128 in multiples
// of 8, causal or with any key count and an optional additive mask.
//
// The kernels of flash_attn.hip give a (head, 128 or 256 queries) unit to a workgroup whose waves share the queries
// and walk all the keys; with fewer units than the chip holds workgroups, most SIMDs have one wave or none and the
// time is the chain of one unit's key blocks. Here a workgroup of eight waves takes 64 queries: two row tiles of 32
// times four key groups. Group g walks the 32-key tiles g, g + 4, g + 8, ... with its own K and V tiles in LDS (its
// two waves copy them, double buffered), so a unit's chain is a quarter as long and its waves fill two per SIMD. The
// four groups' sums meet in LDS at the end: every group adds up a quarter of the output columns. Where even that
// leaves compute units idle (a decode step: one query per head), the key range is cut over several workgroups whose
// fp32 sums go through a caller workspace (SPLIT, flash_merge_kernel).
//
// Per wave and 32-key tile the work is that of flash_attn.hip: S^T = K Q^T (a lane holds 16 scores of one query),
// online softmax in fp32 with a lagging maximum, O^T += V^T P^T with the probabilities taken from the score registers.
#include <type_traits>

#include "flash_attn_tiles.h"

namespace hexmi {
namespace {

constexpr int kTileKeys = 32;                    // keys of a tile
constexpr int kGroups = 4;                       // key groups of a workgroup
constexpr int kStepKeys = kTileKeys * kGroups;   // keys a workgroup takes per step
constexpr int kRows = 64;                        // queries of a workgroup: two tiles of 32

// global -> LDS copy of one [32 keys][D] tile by the two waves of a group, in the swizzled layout of the 64-key tiles.
// PADDED: the head is d < D columns wide (a multiple of 8); a lane whose chunk lies past them copies nothing, and its LDS
// positions, which no other lane writes, are zeroed once.
template <typename T, int D, bool IS_V, bool PADDED, bool PITCH>
struct GroupTileLoader {
  static constexpr int CPR = D / 8;                        // 16-byte chunks per row
  static constexpr int NI = kTileKeys * CPR / 128;         // instructions per wave
  static constexpr int kRowStep = 128 / CPR;               // rows between a wave's instructions
  int row0, col[NI], lds0;                                 // this lane's row of instruction 0, its columns, the wave's part
  int d, row_step;                                         // columns of the head; elements between rows in memory
  __device__ __forceinline__ void init(int rt, int lane, int head_dim, int pitch) {
    const int lin = rt * 64 + lane;
    d = PADDED ? head_dim : D;
    row_step = PITCH ? pitch : d;
    row0 = lin / CPR;
    lds0 = rt * 64 * 8;
#pragma unroll
    for (int j = 0; j < NI; ++j) {
      const int row = row0 + j * kRowStep;
      col[j] = ((lin % CPR) ^ (IS_V ? swz_vtile<D>(row) : swz_ktile<D>(row))) * 8;
    }
  }
  // instruction j of this wave; keys past the end of the sequence are clamped to the last one (their scores are dropped)
  __device__ __forceinline__ void issue_one(int j, const T* __restrict__ g, int key0, int Skv, T* lds) const {
    int key = key0 + row0 + j * kRowStep;
    key = key < Skv ? key : Skv - 1;
    if (!PADDED || col[j] < d)
      copy_to_lds(reinterpret_cast<const char*>(g), (key * row_step + col[j]) * (int)sizeof(T), lds + lds0 + j * (128 * 8));
  }
  __device__ __forceinline__ void zero_padding(T* lds, int lane) const {
#pragma unroll
    for (int j = 0; j < NI; ++j)
      if (col[j] >= d) *reinterpret_cast<u32x4*>(lds + lds0 + j * (128 * 8) + lane * 8) = u32x4{0u, 0u, 0u, 0u};
  }
};

// p[0..7] -= the eight packed values, exactly (they are the roundings of p). One instruction per value in fp16: left to
// itself the compiler converts every value a second time, to have it alone in a register.
__device__ __forceinline__ void take_part(const f16x8& part, float* p) {
  const u32x4 u = __builtin_bit_cast(u32x4, part);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    asm("v_fma_mix_f32 %0, %1, -1.0, %0 op_sel_hi:[1,0,0]" : "+v"(p[2 * i]) : "v"(u[i]));
    asm("v_fma_mix_f32 %0, %1, -1.0, %0 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "+v"(p[2 * i + 1]) : "v"(u[i]));
  }
}
__device__ __forceinline__ void take_part(const bf16x8& part, float* p) {
  const u32x4 u = __builtin_bit_cast(u32x4, part);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    p[2 * i] -= __builtin_bit_cast(float, u[i] << 16);
    p[2 * i + 1] -= __builtin_bit_cast(float, u[i] & 0xffff0000u);
  }
}

// FULL: the probabilities go into P V as two or three 16-bit parts, each the rounding of what the parts before it leave, and
// their sum is taken in fp32. Two parts hold 22 bits (fp16; the exponents are raised by 6 so that the second part of a
// small probability stays above 2^-24) or 16 (bf16, whose result is rounded to 8), three 24 (bf16 with an fp32 result). For
// an fp32 result the parts of a tile meet in registers of their own, so that the running sum is rounded once a tile.
// A part costs its share of MFMAs: 32 heads x 509 queries x 2555 keys of 128 with a mask 40 us in one part, 46 in two.
// PITCH: Q, K and V stand as `at` says (where they are not contiguous). COLS (with PADDED): as in flash_attn.hip.
template <typename T, typename OutT, int D, bool CAUSAL, bool MASKED, bool PADDED, bool FULL, bool PITCH, int COLS = D>
__global__ __launch_bounds__(512, D == 64 && !MASKED ? 4 : 2)
void flash_keys_kernel(const T* __restrict__ Q, const T* __restrict__ K, const T* __restrict__ V, OutT* __restrict__ O,
                       int ZH, int S, int Skv, float scale, const T* __restrict__ Mk, float* __restrict__ part,
                       int chunk, int splits, int head_dim, RowsArg<PITCH> at) {
  const int dh = PADDED ? head_dim : D;                 // elements between rows in memory
  static_assert(!(CAUSAL && MASKED), "the causal kernel has no mask");
  static_assert(!FULL || MASKED, "full probabilities: masked kernel");
  constexpr int kParts = !FULL ? 1 : (sizeof(OutT) == 4 && std::is_same<T, bf16>::value ? 3 : 2);
  constexpr bool kTileSums = FULL && sizeof(OutT) == 4;
  constexpr float kRaise = FULL && std::is_same<T, f16>::value ? 6.0f : 0.0f;
  // Without a mask `scale` carries log2 e and a score is scaled as its exponent is taken: one instruction. With one the
  // score is scaled and the mask added to it in natural units, and the difference to the maximum is taken before it
  // is multiplied by log2 e. That way a row whose keys all carry the same large finite value gives the average of V as any
  // other constant does: the value divided by the scale and added to the raw score overflowed from -3e37 on (bf16, heads
  // of 128), and a maximum that was multiplied and rounded was off by more than an exponent holds from about -2e9 on.
  constexpr float kUnit = MASKED ? kLog2e : 1.0f, kLag = kRescaleLag / kUnit;
  typedef typename MfmaT<T>::Frag Frag;
  constexpr int DS = (COLS + 15) / 16, DT = (COLS + 31) / 32, CPR = D / 8;
  constexpr int kTile = kTileKeys * D;
  __shared__ __attribute__((aligned(16))) T k_lds0[kGroups * kTile];
  __shared__ __attribute__((aligned(16))) T k_lds1[kGroups * kTile];
  __shared__ __attribute__((aligned(16))) T v_lds0[kGroups * kTile];
  __shared__ __attribute__((aligned(16))) T v_lds1[kGroups * kTile];
  // per wave: its mask tile, later its (m, l) for the merge
  constexpr int kWaveBytes = MASKED ? 32 * kTileKeys * (int)sizeof(T) : 64 * (int)sizeof(f32x2);
  __shared__ __attribute__((aligned(16))) char w_lds[8 * kWaveBytes];

  const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int rt = wave % 2, ks = wave / 2, half = lane / 32;

  // Workgroup -> (head, query block, key chunk). Workgroup ids go round robin to the 8 XCDs (one L2 each), and a head's
  // workgroups share one: an XCD takes an eighth of the list of all units, head by head. (Spread
  // over the XCDs, as head counts off the multiple of 8 were: 127 heads x 207 x 3967 of 64 76 us, 51 this way; 51 heads x
  // 1000 of 64 causal 21.2, 17.6.) Causal: the longest query blocks of all heads first, head h on XCD h % 8;
  // the last ZH % 8 heads wander.
  const int nqb = (S + kRows - 1) / kRows;
  int zh, qb, split;
  const unsigned b = blockIdx.x, xcd = b % 8;
  if (CAUSAL) {
    const int c = b % ZH;
    zh = c < ZH / 8 * 8 ? c / 8 * 8 + xcd : c;
    qb = nqb - 1 - b / ZH;
    split = 0;
  } else {
    const unsigned each = gridDim.x / 8, more = gridDim.x % 8;
    const unsigned u = xcd * each + (xcd < more ? xcd : more) + b / 8, r = u / splits;
    split = u % splits;
    zh = r / nqb;
    qb = nqb - 1 - r % nqb;
  }
  const int key_end = CAUSAL ? ((qb + 1) * kRows < S ? (qb + 1) * kRows : S) : Skv;
  const int unit_steps = (key_end + kStepKeys - 1) / kStepKeys;
  const int first = split * chunk;                      // causal units are never cut
  const int last = first + chunk < unit_steps ? first + chunk : unit_steps;

  const T *q_g = Q + (int64_t)zh * S * dh, *k_g = K + (int64_t)zh * Skv * dh, *v_g = V + (int64_t)zh * Skv * dh;
  int64_t q_row = dh;
  int k_row = dh, v_row = dh;
  if constexpr (PITCH) {
    q_g = Q + head_at(at.q, at.heads, zh);
    k_g = K + head_at(at.k, at.heads, zh);
    v_g = V + head_at(at.v, at.heads, zh);
    q_row = at.q.row;
    k_row = (int)at.k.row, v_row = (int)at.v.row;
  }
  const int q0 = qb * kRows + rt * 32;
  const int qrow = q0 + lane % 32;
  const int qr = qrow < S ? qrow : S - 1;

  GroupTileLoader<T, D, false, PADDED, PITCH> k_loader;
  GroupTileLoader<T, D, true, PADDED, PITCH> v_loader;
  k_loader.init(rt, lane, dh, k_row);
  v_loader.init(rt, lane, dh, v_row);
  const int lds_g = ks * kTile;
  if constexpr (PADDED) {                               // ahead of the first barrier of the key loop
    k_loader.zero_padding(k_lds0 + lds_g, lane);
    k_loader.zero_padding(k_lds1 + lds_g, lane);
    v_loader.zero_padding(v_lds0 + lds_g, lane);
    v_loader.zero_padding(v_lds1 + lds_g, lane);
  }
  constexpr int kCopies = 2 * GroupTileLoader<T, D, false, PADDED, PITCH>::NI;
  auto load_one = [&](int c, int n0, T* k_dst, T* v_dst) __attribute__((always_inline)) {
    if (c < kCopies / 2) k_loader.issue_one(c, k_g, n0, Skv, k_dst + lds_g);
    else v_loader.issue_one(c - kCopies / 2, v_g, n0, Skv, v_dst + lds_g);
  };
  auto load_kv = [&](int n0, T* k_dst, T* v_dst) __attribute__((always_inline)) {
    if (n0 < key_end) {
#pragma unroll
      for (int c = 0; c < kCopies; ++c) load_one(c, n0, k_dst, v_dst);
    }
  };
  load_kv(first * kStepKeys + ks * kTileKeys, k_lds0, v_lds0);

  // The mask tile of a wave, [32 queries][32 keys], comes as 16-byte pieces of its rows (four lanes a row, at element
  // alignment: any row length and base) two steps ahead into registers, and reaches the lanes that hold the scores
  // through a wave-private 2 KiB of LDS, its pieces XOR swizzled by row / 4. No branch around the loads: a merge of
  // loaded and unloaded registers would wait for them on the spot (63 us instead of 49 for 509 queries x 2555 keys x 32
  // heads). What a piece reads past the end of its row is dropped with the scores there; a piece that would
  // leave the mask itself is moved back to its end (`moved` elements) and put right on its way into LDS.
  typedef T MaskRun __attribute__((ext_vector_type(4)));
  typedef T MaskPiece __attribute__((ext_vector_type(8)));
  MaskPiece mk0[2] = {}, mk1[2] = {};
  const int64_t mask_end = (int64_t)ZH * S * Skv - 8;                // the last place a piece can be read at, >= 0
  auto mask_at = [&](int i, int n0) __attribute__((always_inline)) {
    int r = q0 + i * 16 + lane / 4;
    r = r < S ? r : S - 1;
    return ((int64_t)zh * S + r) * Skv + n0 + lane % 4 * 8;
  };
  auto load_mask = [&](int n0, MaskPiece* mk) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int64_t at = mask_at(i, n0);
      __builtin_memcpy(&mk[i], Mk + (at < mask_end ? at : mask_end), sizeof(MaskPiece));
    }
  };
  T* m_wave = reinterpret_cast<T*>(w_lds + wave * kWaveBytes);
  const int mask_n0 = first * kStepKeys + ks * kTileKeys;
  if constexpr (MASKED) {
    __builtin_amdgcn_sched_barrier(0);
    load_mask(mask_n0, mk0);
    load_mask(mask_n0 + kStepKeys, mk1);
  }

  Frag qf[DS];
#pragma unroll
  for (int ds = 0; ds < DS; ++ds) {
    if (!PADDED || ds * 16 + half * 8 < dh)
      qf[ds] = *reinterpret_cast<const Frag*>(q_g + qr * q_row + ds * 16 + half * 8);
    else
      qf[ds] = Frag{};
  }

  f32x16 o_acc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) o_acc[dt][r] = 0.0f;
  float m_i = -INFINITY, neg_m = 0.0f, l_i = 0.0f;

  auto process = [&](int step, const T* k_src, const T* v_src, T* k_dst, T* v_dst,
                     MaskPiece* mk_step) __attribute__((always_inline)) {
    const int n0 = step * kStepKeys + ks * kTileKeys;
    if constexpr (MASKED) {
      // the last piece of the tile would leave the mask (wave-uniform)
      const int last_row = q0 + 31 < S ? q0 + 31 : S - 1;
      const bool at_end = ((int64_t)zh * S + last_row) * Skv + n0 + 24 > mask_end;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int row = i * 16 + lane / 4;
        T* dst = m_wave + (row * 4 + (lane % 4 ^ (row / 4 % 4))) * 8;
        if (!at_end) {
          *reinterpret_cast<MaskPiece*>(dst) = mk_step[i];
        } else {
          const int64_t moved = mask_at(i, n0) - mask_end;
#pragma unroll
          for (int e = 0; e < 8; ++e)
            if (moved <= 0 || e >= moved) dst[moved > 0 ? e - (int)moved : e] = mk_step[i][e];
        }
      }
    }
    if (step + 1 < last) load_kv(n0 + kStepKeys, k_dst, v_dst);
    if constexpr (MASKED) {
      __builtin_amdgcn_sched_barrier(0);                // behind the copies: see wait_copies
      load_mask(n0 + 2 * kStepKeys, mk_step);
    }
    if (n0 >= key_end || (CAUSAL && n0 > q0 + 31)) return;      // wave-uniform; the barriers are outside
    const T* k_t = k_src + lds_g;
    const T* v_t = v_src + lds_g;
    f32x16 s;
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = 0.0f;
    {
      const int row = lane % 32;
      Frag kf[DS];
#pragma unroll
      for (int ds = 0; ds < DS; ++ds) {
        const int c = (ds * 2 + half) ^ swz_ktile<D>(row);
        kf[ds] = *reinterpret_cast<const Frag*>(k_t + (row * CPR + c) * 8);
      }
      __builtin_amdgcn_sched_barrier(0);                // all reads ahead of the first product
#pragma unroll
      for (int ds = 0; ds < DS; ++ds) s = MfmaT<T>::run(kf[ds], qf[ds], s);
    }
    Frag vf[2][DT];                                     // asked for before the softmax, which hides their latency
    {
      const int g = lane / 16, i16 = lane % 16;
#pragma unroll
      for (int hf = 0; hf < 2; ++hf)
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
          union { i16x4 h[2]; Frag f; } u;
#pragma unroll
          for (int pp = 0; pp < 2; ++pp) {
            const int row = hf * 16 + 8 * pp + 4 * (g >> 1) + (i16 >> 2);
            const int col = dt * 32 + (g & 1) * 16 + (i16 & 3) * 4;
            const int c = (col / 8) ^ swz_vtile<D>(row);
            const T* addr = v_t + (row * CPR + c) * 8 + (col % 8);
            u.h[pp] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4*)(addr));
          }
          vf[hf][dt] = u.f;
        }
    }
    if constexpr (MASKED) {
      MaskRun mk[4];
      const int row = lane % 32;
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4)
        mk[g4] = *reinterpret_cast<const MaskRun*>(m_wave + (row * 4 + (g4 ^ (row / 4 % 4))) * 8 + half * 4);
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = fmaf(s[r], scale, to_f32<T>(mk[r / 4][r % 4]));
    }
    if ((CAUSAL && n0 + kTileKeys - 1 > q0) || n0 + kTileKeys > Skv) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int key = n0 + 8 * (r / 4) + 4 * half + r % 4;
        if ((CAUSAL && key > qrow) || key >= Skv) s[r] = -INFINITY;
      }
    }
    float mx = -INFINITY;
#pragma unroll
    for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[r]);
    mx = fmaxf(mx, other_half(mx));
    const float m_blk = MASKED ? mx : mx * scale;
    const bool grow = m_blk > m_i + kLag;
    if (__builtin_amdgcn_ballot_w64(grow) != 0) {
      const float m_new = grow ? m_blk : m_i;
      const float alpha = grow ? __builtin_amdgcn_exp2f((m_i - m_new) * kUnit) : 1.0f;
      l_i *= alpha;
      m_i = m_new;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) o_acc[dt][r] *= alpha;
      neg_m = m_i == -INFINITY ? 0.0f : -m_i;           // every key so far masked out: exp2(-inf) = 0, not NaN
    }
    float p[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      if constexpr (FULL) p[r] = __builtin_amdgcn_exp2f(fmaf(s[r] + neg_m, kUnit, kRaise));
      else p[r] = __builtin_amdgcn_exp2f(MASKED ? (s[r] + neg_m) * kUnit : fmaf(s[r], scale, neg_m));
    }
    if constexpr (FULL) {
      float sum[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) sum[r] = (p[r] + p[r + 4]) + (p[r + 8] + p[r + 12]);
      l_i += (sum[0] + sum[1]) + (sum[2] + sum[3]);
    }
    Frag pf[kParts][2];
#pragma unroll
    for (int part = 0; part < kParts; ++part) {
      pf[part][0] = MfmaT<T>::pack(&p[0]);
      pf[part][1] = MfmaT<T>::pack(&p[8]);
      if constexpr (!FULL) l_i = MfmaT<T>::sum8(pf[part][1], MfmaT<T>::sum8(pf[part][0], l_i));
      if (part + 1 < kParts) {
        take_part(pf[part][0], &p[0]);
        take_part(pf[part][1], &p[8]);
      }
      if constexpr (!kTileSums) {
#pragma unroll
        for (int hf = 0; hf < 2; ++hf)
#pragma unroll
          for (int dt = 0; dt < DT; ++dt) o_acc[dt] = MfmaT<T>::run(vf[hf][dt], pf[part][hf], o_acc[dt]);
      }
    }
    if constexpr (kTileSums) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        f32x16 tile;
#pragma unroll
        for (int r = 0; r < 16; ++r) tile[r] = 0.0f;
#pragma unroll
        for (int part = kParts - 1; part >= 0; --part)
#pragma unroll
          for (int hf = 0; hf < 2; ++hf) tile = MfmaT<T>::run(vf[hf][dt], pf[part][hf], tile);
#pragma unroll
        for (int r = 0; r < 16; ++r) o_acc[dt][r] += tile[r];
      }
    }
  };

  // This wave's copies of the next tile are in LDS. The two mask loads behind them stay in flight (loads complete in
  // order). The builtin and not assembly: the compiler then knows the copies done and adds no waits of its own.
  auto wait_copies = [&]() __attribute__((always_inline)) {
    if constexpr (MASKED) __builtin_amdgcn_s_waitcnt(0x0f72);        // vmcnt(2)
    else __builtin_amdgcn_s_waitcnt(0x0f70);                         // vmcnt(0)
  };
  int step = first;
  for (; step + 1 < last; step += 2) {
    wait_copies();
    __syncthreads();
    process(step, k_lds0, v_lds0, k_lds1, v_lds1, mk0);
    wait_copies();
    __syncthreads();
    process(step + 1, k_lds1, v_lds1, k_lds0, v_lds0, mk1);
  }
  if (step < last) {
    wait_copies();
    __syncthreads();
    process(step, k_lds0, v_lds0, k_lds1, v_lds1, mk0);
  }

  // ---- the four groups' sums: scaled to the largest of their maxima, then group i adds up the i-th quarter of the
  // output registers (float4 units u = dt * 4 + q4). The pieces for group i go through the i-th tile array.
  constexpr int kUnits = D / 32 * 4 / kGroups;          // units of a group: of the whole tile, so that a column's sums meet in the
                                                        // same order at any COLS
  auto ml_of = [&](int g) __attribute__((always_inline)) {
    return reinterpret_cast<f32x2*>(w_lds + (g * 2 + rt) * kWaveBytes) + lane;
  };
  *ml_of(ks) = f32x2{m_i, l_i};
  __syncthreads();                                      // also: every wave is done with the tiles
  float m = -INFINITY, l = 0.0f;
#pragma unroll
  for (int g = 0; g < kGroups; ++g) m = fmaxf(m, (*ml_of(g))[0]);
  const float base = m == -INFINITY ? 0.0f : -m;
#pragma unroll
  for (int g = 0; g < kGroups; ++g) {
    const f32x2 v = *ml_of(g);
    l = fmaf(v[1], __builtin_amdgcn_exp2f((v[0] + base) * kUnit), l);
  }
  l += other_half(l);
  const float w = __builtin_amdgcn_exp2f((m_i + base) * kUnit);
  f32x4* pieces[kGroups] = {reinterpret_cast<f32x4*>(k_lds0), reinterpret_cast<f32x4*>(k_lds1),
                            reinterpret_cast<f32x4*>(v_lds0), reinterpret_cast<f32x4*>(v_lds1)};
#pragma unroll
  for (int i = 0; i < kGroups; ++i) {
    if (i == ks) continue;
    f32x4* dst = pieces[i] + ((ks < i ? ks : ks - 1) * 2 + rt) * (kUnits * 64) + lane;
#pragma unroll
    for (int j = 0; j < kUnits; ++j) {
      const int u = i * kUnits + j;
      if (u >= DT * 4) continue;
      dst[j * 64] = f32x4{o_acc[u / 4][u % 4 * 4 + 0] * w, o_acc[u / 4][u % 4 * 4 + 1] * w,
                          o_acc[u / 4][u % 4 * 4 + 2] * w, o_acc[u / 4][u % 4 * 4 + 3] * w};
    }
  }
  __syncthreads();
  const int64_t rows = (int64_t)ZH * S, row = (int64_t)zh * S + qrow;
  const bool whole = CAUSAL || splits == 1;
  const float inv_l = 1.0f / l;
#pragma unroll
  for (int i = 0; i < kGroups; ++i) {
    if (i != ks) continue;
#pragma unroll
    for (int j = 0; j < kUnits; ++j) {
      const int u = i * kUnits + j;
      if (u >= DT * 4) continue;
      f32x4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = o_acc[u / 4][u % 4 * 4 + e] * w;
#pragma unroll
      for (int g = 0; g < kGroups - 1; ++g) {
        const f32x4 x = pieces[i][(g * 2 + rt) * (kUnits * 64) + j * 64 + lane];
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] += x[e];
      }
      const int d = u / 4 * 32 + 8 * (u % 4) + 4 * half;
      if (qrow < S) {
        if (whole) {
          if (!PADDED || d < dh) store4o<OutT>(O + row * dh + d, o[0] * inv_l, o[1] * inv_l, o[2] * inv_l, o[3] * inv_l);
        } else *reinterpret_cast<f32x4*>(part + ((int64_t)split * rows + row) * D + d) = o;
      }
    }
  }
  // one of several chunks: (m, l) of its rows behind all the sums
  if (!whole && ks == 0 && half == 0 && qrow < S)
    *reinterpret_cast<f32x2*>(part + (int64_t)splits * rows * D + ((int64_t)split * rows + row) * 2) = f32x2{m, l};
}

// The chunks of a row added up: O = sum_s 2^(u (m_s - m)) o_s / sum_s 2^(u (m_s - m)) l_s with m the largest m_s and u the
// log2 units of an m_s (kUnit of the kernel that wrote them). A thread
// takes four columns. Bound by reading the sums, which have just been written and come from L2 / Infinity Cache.
template <typename OutT, int D>
__global__ __launch_bounds__(256)
void flash_merge_kernel(const float* __restrict__ part, OutT* __restrict__ O, int64_t rows, int splits, int head_dim,
                        float unit) {
  constexpr int TPR = D / 4;                               // threads per row
  const int64_t row = (int64_t)blockIdx.x * (256 / TPR) + threadIdx.x / TPR;
  if (row >= rows) return;
  const float* ml = part + (int64_t)splits * rows * D;
  float m = -INFINITY;
  for (int s = 0; s < splits; ++s) m = fmaxf(m, ml[((int64_t)s * rows + row) * 2]);
  const float base = m == -INFINITY ? 0.0f : -m;           // every key of the row masked out: l stays 0, the result NaN
  const int d = threadIdx.x % TPR * 4;
  if (d >= head_dim) return;                               // padded heads
  f32x4 o = {0.0f, 0.0f, 0.0f, 0.0f};
  float l = 0.0f;
#pragma unroll 4
  for (int s = 0; s < splits; ++s) {
    const f32x2 v = *reinterpret_cast<const f32x2*>(ml + ((int64_t)s * rows + row) * 2);
    const f32x4 x = *reinterpret_cast<const f32x4*>(part + ((int64_t)s * rows + row) * D + d);
    const float w = __builtin_amdgcn_exp2f((v[0] + base) * unit);
    l = fmaf(v[1], w, l);
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = fmaf(x[e], w, o[e]);
  }
  const float inv = 1.0f / l;
  store4o<OutT>(O + row * head_dim + d, o[0] * inv, o[1] * inv, o[2] * inv, o[3] * inv);
}

template <typename T, typename OutT, int D>
int launch_keys(const void* Q, const void* K, const void* V, const void* mask, void* O, int64_t ZH, int64_t S,
                int64_t Skv, int head_dim, float sm_scale, bool causal, const FlashKeysPlan& plan, float* part, const HeadRows& at,
                hipStream_t st) {
  const int64_t blocks = (S + kRows - 1) / kRows * ZH * plan.splits, rows = ZH * S;     // see plan_flash_keys
  const int64_t merge_blocks = (rows + 1024 / D - 1) / (1024 / D);
  const float unit = mask != nullptr ? kLog2e : 1.0f, scale = mask != nullptr ? sm_scale : sm_scale * kLog2e;
#define HEXMI_KEYS_AS(C, M, P, F, X, COLS)                                                                            \
  hipLaunchKernelGGL((flash_keys_kernel<T, OutT, D, C, M, P, F, X, COLS>), dim3((unsigned)blocks), dim3(512), 0, st,           \
                     static_cast<const T*>(Q), static_cast<const T*>(K), static_cast<const T*>(V),                    \
                     static_cast<OutT*>(O), (int)ZH, (int)S, (int)Skv, scale, static_cast<const T*>(mask), part,      \
                     plan.chunk, plan.splits, head_dim, rows_arg<X>(at))
#define HEXMI_KEYS(C, M, P, F, X) HEXMI_KEYS_AS(C, M, P, F, X, D)
  // heads of up to 80 and 96 columns without a mask
#define HEXMI_KEYS_NARROW(C, X)                                                                                       \
  do {                                                                                                                \
    if (D == 128 && head_dim <= 80) HEXMI_KEYS_AS(C, false, true, false, X, (D == 128 ? 80 : D));                      \
    else if (D == 128 && head_dim <= 96) HEXMI_KEYS_AS(C, false, true, false, X, (D == 128 ? 96 : D));                 \
    else HEXMI_KEYS(C, false, true, false, X);                                                                        \
  } while (0)
  const bool narrow = head_dim < D;
  if (!at.contiguous) {                                    // self-attention only: no mask
    if (narrow) { if (causal) HEXMI_KEYS_NARROW(true, true); else HEXMI_KEYS_NARROW(false, true); }
    else { if (causal) HEXMI_KEYS(true, false, false, false, true); else HEXMI_KEYS(false, false, false, false, true); }
  } else if (narrow) {
    if (causal) HEXMI_KEYS_NARROW(true, false);
    else if (plan.full) HEXMI_KEYS(false, true, true, true, false);
    else if (mask != nullptr) HEXMI_KEYS(false, true, true, false, false);
    else HEXMI_KEYS_NARROW(false, false);
  } else {
    if (causal) HEXMI_KEYS(true, false, false, false, false);
    else if (plan.full) HEXMI_KEYS(false, true, false, true, false);
    else if (mask != nullptr) HEXMI_KEYS(false, true, false, false, false);
    else HEXMI_KEYS(false, false, false, false, false);
  }
#undef HEXMI_KEYS_NARROW
#undef HEXMI_KEYS
#undef HEXMI_KEYS_AS
  if (plan.splits > 1)
    hipLaunchKernelGGL((flash_merge_kernel<OutT, D>), dim3((unsigned)merge_blocks), dim3(256), 0, st, part,
                       static_cast<OutT*>(O), rows, plan.splits, head_dim, unit);
  return launch_status();
}

}  // namespace

// Whether these kernels take a problem (splits > 0) and into how many key chunks its units are cut. units: workgroups of
// 64 queries. The lines are where the measured ratio to the kernels of flash_attn.hip crosses 1 (fp16, graph replay, 8 to
// 256 heads, 64 to 8192 keys; us there -> here):
//  - up to one workgroup per compute unit they win by 1.1 to 2.1 (one 64-key block excepted): 16 heads x 1024 queries and
//    keys of 128 25 -> 17, with a mask 38 -> 20; 12 heads x 1000 of 64 causal 16.5 -> 9.2; 8 heads x 2048 causal 38 -> 23;
//  - heads of 64: with up to 64 queries ahead at any count (512 heads x 16 x 2048 46 -> 41), else up to two per compute unit
//    from 512 keys on (84 heads x 317 x 635 14.0 -> 12.6; 128 heads x 192 x 200 would go 8.0 -> 8.5). With a mask only one
//    fits at a time (166 registers against 112), but so it is with the other kernel's larger tiles: from 512 keys on still
//    ahead (512 heads x 16 x 2048 69 -> 53, 226 heads x 78 x 1452 39 -> 34, 128 heads x 200 x 2000 56 -> 42);
//  - causal units differ in length and the longest start first, which balances more than one per unit where the units are
//    long: heads of 128 up to two from 768 keys on (16 heads x 2048: 40 -> 30; 48 heads x 512 would go 15 -> 16), heads of
//    64 up to two from 256 and four from 768 keys on (24 heads x 2048: 39 -> 26; 35 heads x 1839: 30 -> 28);
//  - causal heads of 4096 queries and more stay with those kernels whatever is faster: hexmi.h promises their callers the
//    same bits at any number of heads, which a choice by units cannot give (8 heads x 4095: 51 us here, x 4096: 73 there);
//  - beyond, the kernels whose waves share more queries do the same work with fewer copies and steps (128 heads x 1024 of
//    128: 80 -> 113).
// Chunks only where half the compute units would stay idle: a merge costs its launch (4 us, and 3 of the host's) and
// the fp32 sums (never worth it up to 768 keys), a step (128 keys) about 1.2 us with heads of 128 and 0.8 with heads of 64 (8 heads x 1 x 8192: 65 us in
// one chunk, 15 in 16; 32 heads x 200 x 2000 of 64: 20.5 and 17.5 in two).
FlashKeysPlan plan_flash_keys(int64_t ZH, int64_t S, int64_t Skv, int64_t D, bool causal, bool masked, bool any_mask,
                              bool may_split) {
  FlashKeysPlan p;
  const int64_t cus = hexmi_num_cus(), units = (S + kRows - 1) / kRows * ZH;
  if (D % 8 != 0 || D > 128 || cus <= 0 || !grid_fits(units, 512)) return p;
  if (!any_mask && (Skv <= 64 || (causal && S >= 4096))) return p;
  D = D <= 64 ? 64 : 128;                                  // narrower heads on tiles padded with zero columns
  bool take = units <= cus;
  if (causal)
    take = take || (D == 128 ? units <= 2 * cus && S >= 768 : (units <= 2 * cus && S >= 256) || (units <= 4 * cus && S >= 768));
  else if (D == 64)
    take = take || (S <= 64 && (!masked || Skv >= 512)) || (units <= 2 * cus && Skv >= 512);
  if (!take && !any_mask) return p;
  p.full = any_mask;
  const int64_t steps = (Skv + kStepKeys - 1) / kStepKeys;
  p.chunk = (int)steps;
  p.splits = 1;
  // self-attention without a mask is the entry point without a workspace, and gives its bits
  may_split = may_split && !causal && (masked || S != Skv) && Skv > HEXMI_ATTENTION_ONE_LAUNCH_KEYS;
  const double step_us = D == 128 ? 1.2 : 0.8, sums_us = 8.0 * (double)(ZH * S * D) / 4e6;
  double best = step_us * (double)steps;
  for (int64_t n = 2; may_split && n <= 32 && n <= steps && n * units <= cus; ++n) {
    const int64_t chunk = (steps + n - 1) / n;
    const double t = step_us * (double)chunk + 7.0 + sums_us * (double)n;
    if (t < best && (steps + chunk - 1) / chunk == n) {
      best = t;
      p.chunk = (int)chunk;
      p.splits = (int)n;
    }
  }
  return p;
}

int64_t flash_keys_workspace(const FlashKeysPlan& p, int64_t ZH, int64_t S, int64_t D) {
  return p.splits > 1 ? p.splits * ZH * S * ((D <= 64 ? 64 : 128) + 2) * (int64_t)sizeof(float) : 0;
}

int flash_keys(const void* Q, const void* K, const void* V, const void* mask, void* O, int64_t ZH, int64_t S,
               int64_t Skv, int64_t D, float sm_scale, bool causal, int in_dtype, int out_dtype,
               const FlashKeysPlan& plan, float* part, const HeadRows& at,
                hipStream_t st) {
#define HEXMI_KEYS_D(T, OutT)                                                                                          \
  return D > 64 ? launch_keys<T, OutT, 128>(Q, K, V, mask, O, ZH, S, Skv, (int)D, sm_scale, causal, plan, part, at, st) \
                : launch_keys<T, OutT, 64>(Q, K, V, mask, O, ZH, S, Skv, (int)D, sm_scale, causal, plan, part, at, st)
  if (in_dtype == HEXMI_F16 && out_dtype == HEXMI_F16) HEXMI_KEYS_D(f16, f16);
  if (in_dtype == HEXMI_F16 && out_dtype == HEXMI_F32) HEXMI_KEYS_D(f16, float);
  if (in_dtype == HEXMI_BF16 && out_dtype == HEXMI_BF16) HEXMI_KEYS_D(bf16, bf16);
  if (in_dtype == HEXMI_BF16 && out_dtype == HEXMI_F32) HEXMI_KEYS_D(bf16, float);
#undef HEXMI_KEYS_D
  return HEXMI_ENOTSUP;
}

}  // namespace hexmi
