// Attention of one query per head over many heads (a decode step of a batch): fp16 / bf16, heads of 64 or 128, any key
// count, an optional additive mask.
//
// Bound by streaming K and V, each read once. The matrix-core kernels give such a head a tile of 64 or 128 queries, of
// which one row is real: their key blocks go through LDS behind a barrier each and few bytes are in flight. Here a
// workgroup of eight waves takes a head without LDS or barriers in the key walk. A row of K or V is 16 bytes to each of
// D / 8 lanes, so a wave's load takes 64 * 8 / D rows; a wave asks for kU such loads of K and of V (16 KiB) before it
// uses the first, and two workgroups fit a compute unit. Lane group g of a wave takes kU consecutive keys of the wave's
// tile, whose mask values are then one 16-byte piece. Scores, probabilities and sums stay in fp32; every lane group has
// its own running (max, sum), and they meet once at the end. With a mask scores and maxima are in natural units (the reason
// is at kUnit in flash_attn_keys.hip), without one in log2 units.
// 512 heads x 2048 keys of 128 with a mask (537 MB): 99 us on the 128-query kernel, 79 here (6.8 TB/s); 256 x 8192 of 64
// with a mask 199 -> 80, 512 x 128 of 64 7.4 -> 4.5.
#include "flash_attn_tiles.h"

namespace hexmi {
namespace {

constexpr int kWaves = 8;
constexpr int kU = 8;                                  // keys of a lane group per tile

template <int LPR>
__device__ __forceinline__ float row_sum(float v) {    // over the D / 8 lanes that share a row; every lane has the sum
  v += dpp_move<0xB1>(v);
  v += dpp_move<0x4E>(v);
  v += dpp_move<0x141>(v);
  if constexpr (LPR == 16) v += dpp_move<0x140>(v);
  return v;
}

template <typename T, typename OutT, int D, bool MASKED>
__global__ __launch_bounds__(kWaves * kWave, 4)
void flash_decode_kernel(const T* __restrict__ Q, const T* __restrict__ K, const T* __restrict__ V,
                         const T* __restrict__ Mk, OutT* __restrict__ O, int Skv, float scale) {
  constexpr float kUnit = MASKED ? kLog2e : 1.0f;       // log2 units of a score's unit
  constexpr int LPR = D / 8, GROUPS = kWave / LPR, TILE = GROUPS * kU;
  typedef T Piece __attribute__((ext_vector_type(8)));
  __shared__ float o_lds[kWaves][D];
  __shared__ float m_lds[kWaves], l_lds[kWaves];
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const int group = lane / LPR, d0 = lane % LPR * 8;
  const int64_t head = blockIdx.x;
  const T* k_head = K + head * Skv * D + d0;
  const T* v_head = V + head * Skv * D + d0;
  const T* mask = MASKED ? Mk + head * Skv : nullptr;
  float q[8], o[8];
  {
    const Piece qp = *reinterpret_cast<const Piece*>(Q + head * D + d0);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      q[e] = to_f32<T>(qp[e]);
      o[e] = 0.0f;
    }
  }
  float m = -INFINITY, l = 0.0f;
  for (int n0 = wave * TILE; n0 < Skv; n0 += kWaves * TILE) {
    const int key0 = n0 + group * kU;
    const bool whole = n0 + TILE <= Skv;               // wave-uniform
    u32x4 kp[kU], vp[kU];
    Piece mk = {};
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int key = key0 + u < Skv ? key0 + u : Skv - 1;
      kp[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(k_head + (int64_t)key * D));
    }
    if constexpr (MASKED) {
      if (whole) {                                     // mask rows start at any element
        __builtin_memcpy(&mk, mask + key0, sizeof(mk));
      } else {
#pragma unroll
        for (int u = 0; u < kU; ++u) mk[u] = mask[key0 + u < Skv ? key0 + u : Skv - 1];
      }
    }
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int key = key0 + u < Skv ? key0 + u : Skv - 1;
      vp[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(v_head + (int64_t)key * D));
    }
    __builtin_amdgcn_sched_barrier(0);                 // all loads ahead of the first use
    float s[kU];
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const Piece k = __builtin_bit_cast(Piece, kp[u]);
      float dot = 0.0f;
#pragma unroll
      for (int e = 0; e < 8; ++e) dot = fmaf(to_f32<T>(k[e]), q[e], dot);
      if constexpr (MASKED) s[u] = fmaf(row_sum<LPR>(dot), scale, to_f32<T>(mk[u]));
      else s[u] = row_sum<LPR>(dot) * scale;
    }
    if (!whole) {                                      // keys past the end: no weight, and nothing of V
#pragma unroll
      for (int u = 0; u < kU; ++u)
        if (key0 + u >= Skv) {
          s[u] = -INFINITY;
          vp[u] = u32x4{0u, 0u, 0u, 0u};
        }
    }
    float m_new = m;
#pragma unroll
    for (int u = 0; u < kU; ++u) m_new = fmaxf(m_new, s[u]);
    const float base = m_new == -INFINITY ? 0.0f : m_new;        // every key so far masked out: exp2(-inf) = 0, not NaN
    const float alpha = __builtin_amdgcn_exp2f((m - base) * kUnit);
    m = m_new;
    l *= alpha;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] *= alpha;
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const float p = __builtin_amdgcn_exp2f((s[u] - base) * kUnit);
      const Piece v = __builtin_bit_cast(Piece, vp[u]);
      l += p;
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = fmaf(p, to_f32<T>(v[e]), o[e]);
    }
  }
  // the lane groups of the wave, then the waves
  float m_all = m;
#pragma unroll
  for (int x = LPR; x < kWave; x *= 2) m_all = fmaxf(m_all, __shfl_xor(m_all, x));
  const float base = m_all == -INFINITY ? 0.0f : m_all;
  const float w = __builtin_amdgcn_exp2f((m - base) * kUnit);
  l *= w;
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] *= w;
#pragma unroll
  for (int x = LPR; x < kWave; x *= 2) {
    l += __shfl_xor(l, x);
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] += __shfl_xor(o[e], x);
  }
  if (group == 0) {
#pragma unroll
    for (int e = 0; e < 8; ++e) o_lds[wave][d0 + e] = o[e];
    if (d0 == 0) {
      m_lds[wave] = m_all;
      l_lds[wave] = l;
    }
  }
  __syncthreads();
  const int d = threadIdx.x;
  if (d >= D) return;
  float top = -INFINITY, sum = 0.0f, out = 0.0f;
#pragma unroll
  for (int i = 0; i < kWaves; ++i) top = fmaxf(top, m_lds[i]);
  const float top_base = top == -INFINITY ? 0.0f : top;          // every key of the row masked out: 0 / 0, NaN
#pragma unroll
  for (int i = 0; i < kWaves; ++i) {
    const float f = __builtin_amdgcn_exp2f((m_lds[i] - top_base) * kUnit);
    sum = fmaf(l_lds[i], f, sum);
    out = fmaf(o_lds[i][d], f, out);
  }
  O[head * D + d] = from_f32<OutT>(out * (1.0f / sum));
}

template <typename T, typename OutT, int D>
int launch_decode(const void* Q, const void* K, const void* V, const void* mask, void* O, int64_t ZH, int64_t Skv,
                  float sm_scale, hipStream_t st) {
#define HEXMI_DECODE(M)                                                                                              \
  hipLaunchKernelGGL((flash_decode_kernel<T, OutT, D, M>), dim3((unsigned)ZH), dim3(kWaves * kWave), 0, st,            \
                     static_cast<const T*>(Q), static_cast<const T*>(K), static_cast<const T*>(V),                    \
                     static_cast<const T*>(mask), static_cast<OutT*>(O), (int)Skv, (M) ? sm_scale : sm_scale * kLog2e)
  if (mask != nullptr) HEXMI_DECODE(true);
  else HEXMI_DECODE(false);
#undef HEXMI_DECODE
  return launch_status();
}

}  // namespace

// One query per head and more heads than half the compute units (fewer leave the keys to be cut over workgroups,
// plan_flash_keys). Graph replay, fp16, without / with a mask, the 128-query kernel -> here in us: 129 heads x 128 keys of
// 64 5.2 / 5.6 -> 3.9 / 3.7, x 2048 29.5 / 42 -> 14.8 / 13.6; 256 x 2048 of 128 43 / 61 -> 41 / 40; 2048 x 512 of 128
// 103 / 107 -> 81 / 78. Up to 64 keys those kernels are one block and stay.
bool flash_decode_takes(int64_t ZH, int64_t S, int64_t Skv, int64_t D) {
  return S == 1 && (D == 64 || D == 128) && Skv > 64 && 2 * ZH > hexmi_num_cus() && grid_fits(ZH, kWaves * kWave);
}

int flash_decode(const void* Q, const void* K, const void* V, const void* mask, void* O, int64_t ZH, int64_t Skv,
                 int64_t D, float sm_scale, int in_dtype, int out_dtype, hipStream_t st) {
#define HEXMI_DECODE_D(T, OutT)                                                                      \
  return D == 128 ? launch_decode<T, OutT, 128>(Q, K, V, mask, O, ZH, Skv, sm_scale, st)          \
                  : launch_decode<T, OutT, 64>(Q, K, V, mask, O, ZH, Skv, sm_scale, st)
  if (in_dtype == HEXMI_F16 && out_dtype == HEXMI_F16) HEXMI_DECODE_D(f16, f16);
  if (in_dtype == HEXMI_F16 && out_dtype == HEXMI_F32) HEXMI_DECODE_D(f16, float);
  if (in_dtype == HEXMI_BF16 && out_dtype == HEXMI_BF16) HEXMI_DECODE_D(bf16, bf16);
  if (in_dtype == HEXMI_BF16 && out_dtype == HEXMI_F32) HEXMI_DECODE_D(bf16, float);
#undef HEXMI_DECODE_D
  return HEXMI_ENOTSUP;
}

}  // namespace hexmi
