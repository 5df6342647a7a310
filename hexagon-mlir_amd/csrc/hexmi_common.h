// Shared device/host helpers for the hexmi kernels (gfx950 only).
#pragma once
#include <type_traits>
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "hexmi.h"

namespace hexmi {

constexpr int kWave = 64;  // CDNA wavefront width

typedef _Float16 f16;
typedef __bf16 bf16;

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef short i16x4 __attribute__((ext_vector_type(4)));

// ---- scalar conversions -------------------------------------------------
template <typename T> __device__ __forceinline__ float to_f32(T v);
template <> __device__ __forceinline__ float to_f32<float>(float v) { return v; }
template <> __device__ __forceinline__ float to_f32<f16>(f16 v) { return (float)v; }
template <> __device__ __forceinline__ float to_f32<bf16>(bf16 v) { return (float)v; }

template <typename T> __device__ __forceinline__ T from_f32(float v);
template <> __device__ __forceinline__ float from_f32<float>(float v) { return v; }
template <> __device__ __forceinline__ f16 from_f32<f16>(float v) { return (f16)v; }   // round-to-nearest-even
template <> __device__ __forceinline__ bf16 from_f32<bf16>(float v) { return (bf16)v; }  // round-to-nearest-even

// four consecutive elements, rounded once to the output type, in one store (p aligned to 4 elements)
template <typename OutT>
__device__ __forceinline__ void store4(OutT* p, float a, float b, float c, float d);
template <> __device__ __forceinline__ void store4<float>(float* p, float a, float b, float c, float d) {
  f32x4 v = {a, b, c, d};
  *reinterpret_cast<f32x4*>(p) = v;
}
template <> __device__ __forceinline__ void store4<f16>(f16* p, float a, float b, float c, float d) {
  f16x4 v = {(f16)a, (f16)b, (f16)c, (f16)d};
  *reinterpret_cast<f16x4*>(p) = v;
}
template <> __device__ __forceinline__ void store4<bf16>(bf16* p, float a, float b, float c, float d) {
  bf16x4 v = {(bf16)a, (bf16)b, (bf16)c, (bf16)d};
  *reinterpret_cast<bf16x4*>(p) = v;
}

// ---- wavefront reductions -----------------------------------------------
// Butterfly over the 64 lanes on the vector ALU (no LDS round trips): DPP exchanges inside a row of 16 lanes
// (quad permutes for lane^1 and lane^2; the half-row and row mirrors stand in for lane^4 and lane^8 because the
// partial results are already uniform inside groups of 4 and 8), then v_permlane16_swap / v_permlane32_swap
// for the exchanges between rows. Every lane ends with the full result.
// (Every lane has a valid source under these permutations, so the value for lanes without one is never used; it is
// given as 0 with the bound-control bit set, the form the compiler folds into the add or max that consumes the
// exchange - v_add_f32_dpp, one instruction per step - where "keep the own value" leaves a copy, the exchange and
// the add: three.)
template <int CTRL>
__device__ __forceinline__ float dpp_move(float v) {
  const int i = __builtin_bit_cast(int, v);
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, i, CTRL, 0xF, 0xF, true));
}
// {a, b} with a = value of the partner row (16 lanes) / half (32 lanes) and b = own, in some order that is the
// same for both partners up to exchange: callers combine them with a commutative operation.
__device__ __forceinline__ void swap16(float v, float& a, float& b) {
  const unsigned u = __builtin_bit_cast(unsigned, v);
  auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  a = __builtin_bit_cast(float, (unsigned)r[0]);
  b = __builtin_bit_cast(float, (unsigned)r[1]);
}
__device__ __forceinline__ void swap32(float v, float& a, float& b) {
  const unsigned u = __builtin_bit_cast(unsigned, v);
  auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  a = __builtin_bit_cast(float, (unsigned)r[0]);
  b = __builtin_bit_cast(float, (unsigned)r[1]);
}
__device__ __forceinline__ float wave_sum(float v) {
  v += dpp_move<0xB1>(v);      // quad_perm [1,0,3,2]
  v += dpp_move<0x4E>(v);      // quad_perm [2,3,0,1]
  v += dpp_move<0x141>(v);     // row_half_mirror
  v += dpp_move<0x140>(v);     // row_mirror
  float a, b;
  swap16(v, a, b);
  v = a + b;
  swap32(v, a, b);
  return a + b;
}
__device__ __forceinline__ float wave_max(float v) {
  v = fmaxf(v, dpp_move<0xB1>(v));
  v = fmaxf(v, dpp_move<0x4E>(v));
  v = fmaxf(v, dpp_move<0x141>(v));
  v = fmaxf(v, dpp_move<0x140>(v));
  float a, b;
  swap16(v, a, b);
  v = fmaxf(a, b);
  swap32(v, a, b);
  return fmaxf(a, b);
}

// ---- int8 -> fp16 (weight-only quantisation) --------------------------------
// 4 int8 (one dword) -> 4 fp16 in two dwords, exact (|w| <= 128 has at most eight significant bits): one
// v_cvt_f16_i16 per weight, its source the sign-extended byte picked by the instruction's operand selector and its
// destination one half of the result register. (One instruction fewer per dword than building 1024 + (w ^ 0x80) with
// byte permutes and subtracting 1152 in packed fp16: 0.157 -> 0.164 of the HBM figure at M = 256, +1 % at M = 1.)
__device__ __forceinline__ void cvt4(uint32_t w, uint32_t& lo, uint32_t& hi) {
  asm("v_cvt_f16_i16_sdwa %0, sext(%2) dst_sel:WORD_0 dst_unused:UNUSED_PAD src0_sel:BYTE_0\n\t"
      "v_cvt_f16_i16_sdwa %0, sext(%2) dst_sel:WORD_1 dst_unused:UNUSED_PRESERVE src0_sel:BYTE_1\n\t"
      "v_cvt_f16_i16_sdwa %1, sext(%2) dst_sel:WORD_0 dst_unused:UNUSED_PAD src0_sel:BYTE_2\n\t"
      "v_cvt_f16_i16_sdwa %1, sext(%2) dst_sel:WORD_1 dst_unused:UNUSED_PRESERVE src0_sel:BYTE_3"
      : "=&v"(lo), "=&v"(hi)
      : "v"(w));
}

// 16 int8 -> two 8-element fp16 fragments (bytes 0..7 and 8..15), as ONE statement that ends in two idle issue
// slots. A matrix instruction must not read a register in the two slots after a vector instruction wrote it, and
// the compiler, which keeps that distance for its own instructions, cannot see the writes inside an asm statement:
// with a conversion one slot ahead of its MFMA, and the matrix pipe still busy with the MFMA before, the MFMA read
// the register without the last converted byte (k = 11 mod 16 lost in every product; one slot was enough wherever
// the pipe was idle). Callers of cvt4 keep the distance themselves.
__device__ __forceinline__ void cvt16(const u32x4& w, f16x8& f0, f16x8& f1) {
  union { uint32_t u[4]; f16x8 f; } a, b;
#define HEXMI_CVT4(LO, HI, SRC) \
      "v_cvt_f16_i16_sdwa " LO ", sext(" SRC ") dst_sel:WORD_0 dst_unused:UNUSED_PAD src0_sel:BYTE_0\n\t" \
      "v_cvt_f16_i16_sdwa " LO ", sext(" SRC ") dst_sel:WORD_1 dst_unused:UNUSED_PRESERVE src0_sel:BYTE_1\n\t" \
      "v_cvt_f16_i16_sdwa " HI ", sext(" SRC ") dst_sel:WORD_0 dst_unused:UNUSED_PAD src0_sel:BYTE_2\n\t" \
      "v_cvt_f16_i16_sdwa " HI ", sext(" SRC ") dst_sel:WORD_1 dst_unused:UNUSED_PRESERVE src0_sel:BYTE_3\n\t"
  asm(HEXMI_CVT4("%0", "%1", "%8") HEXMI_CVT4("%2", "%3", "%9") HEXMI_CVT4("%4", "%5", "%10")
      HEXMI_CVT4("%6", "%7", "%11") "s_nop 1"
      : "=&v"(a.u[0]), "=&v"(a.u[1]), "=&v"(a.u[2]), "=&v"(a.u[3]), "=&v"(b.u[0]), "=&v"(b.u[1]), "=&v"(b.u[2]),
        "=&v"(b.u[3])
      : "v"(w[0]), "v"(w[1]), "v"(w[2]), "v"(w[3]));
#undef HEXMI_CVT4
  f0 = a.f;
  f1 = b.f;
}

// ---- host helpers ---------------------------------------------------------
inline hipStream_t as_stream(hexmi_stream_t s) { return reinterpret_cast<hipStream_t>(s); }

// Every entry point calls begin_call() once its arguments are accepted and before its first launch: HIP keeps one
// pending error per host thread, and one left there by unrelated code would otherwise be reported (and cleared) by
// the launch_status() of the next launch here.
inline void begin_call() { (void)hipGetLastError(); }

// A launch holds at most 2^32 - 1 threads per dimension.
inline bool grid_fits(int64_t blocks, int threads) { return blocks <= 0xffffffffll / threads; }

inline int launch_status() {
  return hipGetLastError() == hipSuccess ? HEXMI_OK : HEXMI_ELAUNCH;
}

// C[rows, cols] = 0 with leading dimension ld (elements of elem_size bytes): what a product over an empty inner
// dimension is (gemm.hip).
int fill_zero_2d(void* C, int64_t rows, int64_t cols, int64_t ld, int elem_size, hipStream_t stream);

// 16 bytes per lane, global -> LDS, as a buffer load: the address is a uniform base (a buffer descriptor in scalar
// registers, built by scalar arithmetic) plus a per-lane 32-bit byte offset, and the LDS destination (lds + lane*16
// bytes) is a scalar, so a copy costs no vector arithmetic. voff must stay below 2^31; the descriptor's own range
// check is left wide open, callers clamp what must not be read.
// POLICY: the cache-policy bits of the load (0 = default, 2 = non-temporal: data that is read once).
template <typename T, int POLICY = 0>
__device__ __forceinline__ void copy_to_lds(const char* base, int voff, T* lds) {
#if defined(__HIP_DEVICE_COMPILE__)        // the descriptor type exists in the device pass only
  const __amdgpu_buffer_rsrc_t rsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(base), 0, 0x7fffffff, 0x00020000);
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void*)(lds), 16, voff, 0, 0, POLICY);
#endif
}

// copy_to_lds written as asm, for kernels whose LDS destination the compiler cannot name (a stage picked at run
// time, a wave-private region at a run-time base): a copy into LDS with an unknown target makes the compiler wait
// for ALL copies in flight (vmcnt(0)) before every later LDS read that might alias it. A kernel that uses this for
// its copies does its own waiting (s_waitcnt vmcnt) before reading what they fill: the compiler does not know the
// copies exist. Its own vmcnt waits for other loads only get stronger (the counter counts these copies too, and
// loads complete in issue order). M0 (the LDS destination of such a copy) is saved and restored because the
// compiler tracks its own uses of it. lds must be wave-uniform.
template <typename T>
__device__ __forceinline__ void copy_to_lds_asm(const char* base, int voff, T* lds) {
#if defined(__HIP_DEVICE_COMPILE__)
  typedef int i32x4_rsrc __attribute__((ext_vector_type(4)));
  const uint64_t b = reinterpret_cast<uint64_t>(base);
  i32x4_rsrc rsrc;
  rsrc[0] = __builtin_amdgcn_readfirstlane((int)(uint32_t)b);
  rsrc[1] = __builtin_amdgcn_readfirstlane((int)((uint32_t)(b >> 32) & 0xffffu));
  rsrc[2] = 0x7fffffff;
  rsrc[3] = 0x00020000;
  const uint32_t dst = __builtin_amdgcn_readfirstlane(
      (uint32_t)(uintptr_t)((__attribute__((address_space(3))) void*)(lds)));
  uint32_t saved;
  asm volatile(
      "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\t"
      "buffer_load_dwordx4 %2, %3, 0 offen lds\n\ts_mov_b32 m0, %0"
      : "=&s"(saved)
      : "s"(dst), "v"(voff), "s"(rsrc)
      : "memory");
#endif
}

// The same from an address of each lane's own.
__device__ __forceinline__ void copy_ptr_to_lds_asm(const char* src, char* lds) {
#if defined(__HIP_DEVICE_COMPILE__)
  const uint32_t dst = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)((__attribute__((address_space(3))) void*)(lds)));
  uint32_t saved;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, off\n\ts_mov_b32 m0, %0"
               : "=&s"(saved) : "s"(dst), "v"(src) : "memory");
#endif
}

// sixteen 16-bit columns in two chunks, from column `by` (0 .. 7) on: eight of them
__device__ __forceinline__ u32x4 shift_columns(const u32x4& lo, const u32x4& hi, int by) {
  auto pick = [](bool second, uint32_t v0, uint32_t v1) { return second ? v1 : v0; };    // (values, not places: no scratch)
  const bool by4 = by & 4, by2 = by & 2;
  const uint32_t x0 = pick(by4, lo[0], lo[2]), x1 = pick(by4, lo[1], lo[3]), x2 = pick(by4, lo[2], hi[0]),
                 x3 = pick(by4, lo[3], hi[1]), x4 = pick(by4, hi[0], hi[2]), x5 = pick(by4, hi[1], hi[3]);
  const uint32_t y0 = pick(by2, x0, x1), y1 = pick(by2, x1, x2), y2 = pick(by2, x2, x3), y3 = pick(by2, x3, x4),
                 y4 = pick(by2, x4, x5);
  const int bits = (by & 1) * 16;
  const u32x4 o = {__builtin_amdgcn_alignbit(y1, y0, bits), __builtin_amdgcn_alignbit(y2, y1, bits),
                   __builtin_amdgcn_alignbit(y3, y2, bits), __builtin_amdgcn_alignbit(y4, y3, bits)};
  return o;
}
// s_waitcnt immediate (gfx9 encoding): at most `vm` vector-memory operations outstanding, all LDS reads returned.
constexpr int waitcnt_imm(int vm) { return (vm & 0xF) | ((vm >> 4) << 14) | (7 << 4) | (0 << 8); }

// Map the linear workgroup id to a C tile: consecutive ids go to different XCDs (each with its own L2), so
// first give every XCD a contiguous run of logical ids, then walk tiles in bands of GROUP_M tile-rows so the
// tiles resident on one XCD share A and B panels.
template <int GROUP_M>
__device__ __forceinline__ void tile_of_block(int pid, int tiles_m, int tiles_n, int& tm, int& tn) {
  const int total = tiles_m * tiles_n;
  // XCD x runs ids x, x + 8, ...: total/8 of them, one more on the first total%8 XCDs
  const int xcd = pid % 8, per = total / 8, extra = total % 8;
  const int logical = xcd * per + (xcd < extra ? xcd : extra) + pid / 8;
  const int group_size = GROUP_M * tiles_n;
  const int group = logical / group_size;
  const int first_m = group * GROUP_M;
  const int gm = (tiles_m - first_m) < GROUP_M ? (tiles_m - first_m) : GROUP_M;
  const int in_group = logical % group_size;
  tm = first_m + in_group % gm;
  tn = in_group / gm;
}

inline bool aligned_to(const void* p, size_t a) { return (reinterpret_cast<uintptr_t>(p) % a) == 0; }

inline int dtype_size(int dtype) {
  switch (dtype) {
    case HEXMI_F32: return 4;
    case HEXMI_F16: case HEXMI_BF16: return 2;
    case HEXMI_I8: return 1;
    default: return 0;
  }
}

// Block sums (elementwise.hip). A program of kTwoPassMinBlock elements and more is summed in two passes when a
// scratch buffer for fp32 partial sums of runs of kSumRun elements is at hand (ceil(n / kSumRun) floats): the runs of
// a program must be whole, which they are when block % kSumRun == 0 or there is a single program.
constexpr int64_t kSumRun = 4096;
constexpr int64_t kTwoPassMinBlock = 1 << 16;
inline bool two_pass_sum(int64_t n, int64_t block) {
  const int64_t programs = (n + block - 1) / block;
  return block >= kTwoPassMinBlock && (programs == 1 || block % kSumRun == 0);
}
// partials == nullptr: one pass; otherwise two_pass_sum(n, block) holds and partials has room for every run.
int block_sum_any(const void* x, void* out, int64_t n, int64_t block, int dtype, float* partials, hipStream_t s);

// Up to 64 rows against [N,K] weights (gemm_skinny.hip): output channels and waves of a workgroup (0: leave it to the tiles),
// and the launch. K % 32 == 0, operand rows on 16-byte boundaries; bias and residual may be null. tiles: whether the tiles
// are a choice (with bias or residual off whole runs of four columns they take twice to three times as long).
struct GemmSkinnyPlan { int channels, waves; };
GemmSkinnyPlan plan_gemm_skinny(int64_t M, int64_t N, int64_t K, bool tiles);
template <typename T, typename OutT>
int launch_gemm_skinny(const GemmSkinnyPlan& plan, const T* A, const T* B, OutT* C, int64_t M, int64_t N, int64_t K,
                       int64_t lda, int64_t ldb, int64_t ldc, hipStream_t s, const OutT* bias, const OutT* resid, int64_t ldr);

// Products of few 128 x 128 tiles (gemm_few.hip): the tile, m == 0 for none, and the launch. K % 8 == 0, operand rows on 16-byte
// boundaries, leading dimensions below 2^21 (per-lane copy offsets), B as [K,N]: N % 8 == 0; any output side.
struct GemmFewTile { int m, n; };
GemmFewTile plan_gemm_few(bool trans_b, int64_t M, int64_t N, int64_t K);
// ... and in parts of K whose fp32 sums go through a caller workspace: rows of gemm_parts_pitch(N) floats, M of them for each part
struct GemmParts { GemmFewTile tile; int parts, part; };           // parts: 0 where the product goes as a whole
// any: operand rows off the boundaries, [K,N] weights
GemmParts plan_gemm_parts(bool trans_b, int64_t M, int64_t N, int64_t K, bool any);
inline int64_t gemm_parts_pitch(int64_t N) { return (N + 7) / 8 * 8; }
template <typename T, typename OutT, bool TRANS_B>
int launch_gemm_parts(const GemmParts& plan, const T* A, const T* B, OutT* C, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb,
                      int64_t ldc, hipStream_t s, const OutT* bias, const OutT* resid, int64_t ldr, float* sums, bool any);
template <typename T, typename OutT, bool TRANS_B>
int launch_gemm_few(const GemmFewTile& tile, const T* A, const T* B, OutT* C, int64_t M, int64_t N, int64_t K, int64_t lda,
                    int64_t ldb, int64_t ldc, hipStream_t s, const OutT* bias, const OutT* resid, int64_t ldr);
// ... and products on operand rows at any alignment, any K, any strides.
template <typename T, typename OutT, bool TRANS_B>
int launch_gemm_any(const T* A, const T* B, OutT* C, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t ldc, hipStream_t s,
                    const OutT* bias, const OutT* resid, int64_t ldr);

// Tiles of 128 x 128 to 256 x 192 for products of 16-bit results (gemm_mid.hip): the tile, m == 0 for none, and the launch. K % 8 == 0,
// operand rows on 16-byte boundaries, leading dimensions below 2^21 (per-lane copy offsets), B as [K,N]: N % 8 == 0; the output on 16-byte
// boundaries too, in whole runs of eight columns, bias and residual on 8-byte ones, or, odd (B as [N,K]), any of them anywhere. now: what takes the call otherwise, 256 x 256 tiles
// (256), 128 x 128 two (2) or one (1) to a CU, or nothing of that rate (0).
struct GemmMidTile { int m, n, per_cu; };
GemmMidTile plan_gemm_mid(int64_t M, int64_t N, int64_t K, int now, bool resid, bool odd);
template <typename T, bool TRANS_B>
int launch_gemm_mid(const GemmMidTile& tile, const T* A, const T* B, T* C, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb,
                    int64_t ldc, hipStream_t s, const T* bias, const T* resid, int64_t ldr, bool odd);

// Tiled W8A16 GEMM for many activation rows (gemm.hip): C[M,N] = (A[M,K] * W[N,K]^T) * scales[N].
int gemm_w8a16_tiled(int64_t M, int64_t N, int64_t K, const f16* A, const int8_t* W, const f16* scales, f16* C,
                     hipStream_t stream);
int gemm_w8a16_any_shape(int64_t M, int64_t N, int64_t K, const f16* A, const int8_t* W, const f16* scales,
                         const int8_t* zero_points, int per_tensor, f16* C, hipStream_t stream);

// W8A16 of 33 rows and more in one round of tiles over the CUs (w8a16_few.hip): the tile, m == 0 for none, and the launch. K % 16 == 0,
// A and W on 16-byte boundaries; zero_points may be null. tiles: whether the tiles of gemm.hip are a choice.
GemmFewTile plan_w8a16_few(int64_t M, int64_t N, int64_t K, bool tiles, bool zero_points);
int launch_w8a16_few(const GemmFewTile& tile, int64_t M, int64_t N, int64_t K, const f16* A, const int8_t* W, const f16* scales,
                     const int8_t* zero_points, int per_tensor, f16* C, hipStream_t s);

// W8A16 on a (channel range x K part) decomposition with the K parts summed through a caller workspace
// (w8a16_split.hip). w8a16_split_workspace: bytes the shape needs (0: one K part, or a shape the kernel does not
// take). w8a16_split returns false when it does not take the call (shape, alignment, workspace too small).
int64_t w8a16_split_workspace(int64_t M, int64_t N, int64_t K, int cus);
int64_t w8a16_split_header(int64_t M, int64_t N, int64_t K, int cus);   // leading bytes that must be zero at launch
bool w8a16_split(int64_t M, int64_t N, int64_t K, const f16* A, const int8_t* W, const f16* scales, f16* C,
                 void* workspace, int64_t workspace_bytes, int cus, hipStream_t stream, int* status);
// zeroes the first `bytes` of a workspace (a kernel, not a memset: callers may be under graph capture)
int w8a16_split_clear(void* workspace, int64_t bytes, hipStream_t stream);

// fp32 GEMM on the matrix cores (gemm_f32.hip): launches and returns true when the shapes fit (K % 32 == 0, aligned
// operands), with the launch status in *status; false leaves the product to the vector-ALU kernel.
bool gemm_f32_mfma(bool trans_b, const float* A, const float* B, float* C, int64_t M, int64_t N, int64_t K,
                   int64_t lda, int64_t ldb, int64_t ldc, hipStream_t stream, int* status);

// fp32 flash attention on the fp32 matrix cores (flash_attn_f32.hip): launches and returns true when the shapes fit
// (head size 64 or 128, aligned operands), with the launch status in *status.
bool flash_attn_f32_mfma(const float* Q, const float* K, const float* V, const float* mask, float* O, int64_t ZH,
                         int64_t S, int64_t Skv, int64_t D, float scale_log2e, bool causal, hipStream_t stream,
                         int* status);

// Where the rows of Q, K and V stand, in elements: head h of batch z starts at z * batch + h * head, its rows row apart. Contiguous
// [Z,H,S,D] is what the attention kernels are compiled for; other strides (the slices of one projection) they take as arguments.
struct RowStrides { int64_t batch, head, row; };
struct HeadRows {
  RowStrides q, k, v;
  int heads;
  bool contiguous;
};
inline HeadRows contiguous_heads(int64_t S, int64_t Skv, int64_t D) {
  return {{S * D, S * D, D}, {Skv * D, Skv * D, D}, {Skv * D, Skv * D, D}, 1, true};
}
#if defined(__HIPCC__)
__device__ __forceinline__ int64_t head_at(const RowStrides& r, int heads, int zh) {
  const int z = zh / heads;
  return z * r.batch + (zh - z * heads) * r.head;
}
// the kernel argument: heads that are contiguous need none
struct NoRows {};
template <bool PITCH> using RowsArg = std::conditional_t<PITCH, HeadRows, NoRows>;
template <bool PITCH> inline RowsArg<PITCH> rows_arg(const HeadRows& at) {
  if constexpr (PITCH) return at; else return {};
}
#endif

// 16-bit flash attention of few (head, query block) units, the keys of a unit divided inside and over workgroups
// (flash_attn_keys.hip). plan: splits == 0, leave it to the other kernels; > 1, the fp32 sums of that many chunks of
// the key range go through a workspace; full, the probabilities keep fp32 precision into the second product. any_mask: a
// mask that is not whole aligned runs of four keys, which no other kernel of that speed reads (taken at any size, full).
struct FlashKeysPlan {
  int chunk = 0, splits = 0;
  bool full = false;
};
FlashKeysPlan plan_flash_keys(int64_t ZH, int64_t S, int64_t Skv, int64_t D, bool causal, bool masked, bool any_mask,
                              bool may_split);
int64_t flash_keys_workspace(const FlashKeysPlan& plan, int64_t ZH, int64_t S, int64_t D);
int flash_keys(const void* Q, const void* K, const void* V, const void* mask, void* O, int64_t ZH, int64_t S,
               int64_t Skv, int64_t D, float sm_scale, bool causal, int in_dtype, int out_dtype,
               const FlashKeysPlan& plan, float* part, const HeadRows& at, hipStream_t st);

// 16-bit attention of one query per head over many heads (flash_decode.hip): whether it takes a problem, and the launch.
bool flash_decode_takes(int64_t ZH, int64_t S, int64_t Skv, int64_t D);
int flash_decode(const void* Q, const void* K, const void* V, const void* mask, void* O, int64_t ZH, int64_t Skv,
                 int64_t D, float sm_scale, int in_dtype, int out_dtype, hipStream_t st);

}  // namespace hexmi
