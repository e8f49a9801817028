// Shared device/host helpers for libquik_hip.so (gfx950 only).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "quik_hip.h"

namespace quik {

// Last HIP error text, for quik_last_hip_error().
void set_last_hip_error(hipError_t e);
int check_launch();  // QUIK_OK or QUIK_ERR_LAUNCH after a kernel launch
constexpr int kLdsBytes = 160 * 1024;  // per CU, and the most one workgroup may ask for
// Raises the kernel's dynamic LDS limit to `smem` bytes: once per kernel and device, with one size per kernel (the most that
// any of its launches asks for).  Nothing to do up to 48 KB.
int prepare_lds(const void *kern, int smem);
template <typename K>
int prepare(K kern, int smem) {
  return smem > 48 * 1024 ? prepare_lds(reinterpret_cast<const void *>(kern), smem) : QUIK_OK;
}
int num_cus();       // compute units of the GPU (asked once per process; 256 when no device answers)

inline hipStream_t as_stream(void *s) { return reinterpret_cast<hipStream_t>(s); }

// runtime.hip: flags word of a column map (colmap.h: bit 0 = streams, bit 1 = in-place order), copied from the
// device once per (address, shape) and remembered; colmap_forget drops what is known about an address.
// QUIK_ERR_COLMAP when the word is not known yet and `st` is being captured (no synchronisation possible there).
constexpr uint32_t kColmapStreams = 1u, kColmapInPlace = 2u;
int colmap_flags(const void *colmap, int64_t cols, int64_t num_int, int64_t num_fp, hipStream_t st, uint32_t *flags);
// all four flag words of the map (flags, number of dirty groups, number of holes, reserved), same look-up
int colmap_words(const void *colmap, int64_t cols, int64_t num_int, int64_t num_fp, hipStream_t st, uint32_t (&out)[4]);
void colmap_forget(const void *colmap);
// QUIK_OK when the column map has all bits of `need` set, QUIK_ERR_COLMAP when not (or an error of colmap_flags)
inline int colmap_require(const void *colmap, int64_t cols, int64_t num_int, int64_t num_fp, hipStream_t st,
                          uint32_t need) {
  uint32_t flags = 0;
  if (int rc = colmap_flags(colmap, cols, num_int, num_fp, st, &flags)) return rc;
  return (flags & need) == need ? QUIK_OK : QUIK_ERR_COLMAP;
}

// gemm.hip: MixedQLinear forward for one or two token rows in ONE launch, the quantize inside the kernel
// (w_red == NULL: symmetric activations with scale = max |x| / sym_divisor, fp16 only).  Returns kChainNotHandled
// (below) for shapes it leaves to the two-launch path.
bool gemv_one_launch_pays(int64_t rows, int64_t cols, int64_t N);
int gemv_forward_one_launch(const void *x, int dtype, int64_t rows, int64_t cols, const void *colmap, int64_t num_int,
                            int64_t num_fp, int bits, const void *qw, const void *s_col, const void *w_red,
                            const void *fp_w, const void *bias, int64_t N, void *out, float sym_divisor,
                            hipStream_t st);

// The tile-ordered steps of a layer forward, for any number of integer columns that fills whole fragments (4 bits: a
// multiple of kLayerK4, 8 bits: of kLayerK8).  The exported functions of the same steps (quik_asym_quantize_fp6, ...) ask
// for whole pairs of k-steps, 128 / 64 columns, and pass that as `k_multiple`.
constexpr int64_t kLayerK4 = 32, kLayerK8 = 16;
int64_t fp6_operand_bytes(int64_t rows, int64_t K, int64_t F, int64_t k_multiple);
int64_t tile8_operand_bytes(int64_t rows, int64_t K, int64_t F, int64_t k_multiple);
int64_t tile4_operand_bytes(int64_t rows, int64_t K, int64_t F);
int asym_quantize_fp6(const void *x, int dtype, int64_t rows, int64_t cols, const void *colmap, int64_t num_int,
                      int64_t num_fp, void *out6, void *meta, void *stream, int64_t k_multiple, bool four = false);
int asym_quantize_few(const void *x, int dtype, int64_t rows, int64_t cols, const void *colmap, int64_t num_int, int64_t num_fp, int bits,
                      void *dst, void *meta, void *fp_x, void *stream);
int asym_quantize_tile8(const void *x, int dtype, int64_t rows, int64_t cols, const void *colmap, int64_t num_int,
                        int64_t num_fp, void *out8, void *meta, void *stream, int64_t k_multiple);
int sym_quantize_mapped(const void *x, int64_t rows, int64_t cols, const void *colmap, int64_t num_int, int64_t num_fp,
                        int bits, float divisor, int tiled, void *dst, void *scale, void *fp_x, void *stream,
                        int64_t k_multiple);
int mixed_linear_fp6(const void *x6, const void *w6, const void *meta, const void *s_col, const void *w_reduced,
                     const void *bias, int dtype, int64_t M, int64_t N, int64_t K, int64_t F, void *out,
                     void *workspace, int64_t workspace_bytes, void *stream, int64_t k_multiple);
// 4-bit weights: the format (4 or 6 bits) in which the GEMM of this shape takes its activation, and the GEMM (either format)
int tile4_activation_bits(int64_t M, int64_t N, int64_t K, int64_t F);
int mixed_linear_tile4(const void *x, int x_bits, const void *w4, const void *meta, const void *s_col, const void *w_reduced,
                       const void *bias, int dtype, int64_t M, int64_t N, int64_t K, int64_t F, void *out, void *workspace,
                       int64_t workspace_bytes, void *stream);
int mixed_linear_tile8(const void *x8, const void *w8, const void *meta, const void *s_col, const void *w_reduced,
                       const void *bias, int dtype, int64_t M, int64_t N, int64_t K, int64_t F, void *out,
                       void *workspace, int64_t workspace_bytes, void *stream, int64_t k_multiple);

// gemm.hip: integer GEMM + the fp16-arithmetic epilogue of the reference's fused ops in one launch (zero_row ==
// NULL: symmetric form).  Returns kChainNotHandled for calls it leaves to the two-launch path; two_launches: the caller has
// the workspace for that one (without it the tiles take what they can).
constexpr int kChainNotHandled = 1;
int int_gemm_chain(const void *A, const void *B, const void *s_row, const void *s_col, const void *zero_row,
                   const void *w_red, uint16_t shift_bits, const void *y, int64_t M, int64_t N, int64_t K, int bits,
                   void *out, bool two_launches, hipStream_t st);

// ---- storage types as 16-bit patterns --------------------------------------------------
// Half values are handled with the native _Float16 type; bfloat16 with explicit bit math
// so that every rounding is a visible round-to-nearest-even.

template <bool BF16>
__device__ __forceinline__ float to_f32(uint16_t v) {
  if constexpr (BF16) {
    return __uint_as_float(static_cast<uint32_t>(v) << 16);
  } else {
    return static_cast<float>(__builtin_bit_cast(_Float16, v));
  }
}

// Two fp32 values -> bf16, round to nearest even (subnormals included), first value in the low half: one v_cvt_pk_bf16_f32.
// A NaN keeps its sign and the upper bits of its payload: what is stored goes through canonical_nans.
__device__ __forceinline__ uint32_t pack2_bf16(float a, float b) {
  typedef __bf16 bf2_t __attribute__((ext_vector_type(2)));
  typedef float float2_t __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(float2_t{a, b}, bf2_t));
}
// (every NaN becomes 0x7FC0)
__device__ __forceinline__ uint16_t f32_to_bf16_bits(float f) {
  return f != f ? uint16_t{0x7FC0u} : __builtin_bit_cast(uint16_t, static_cast<__bf16>(f));
}

template <bool BF16>
__device__ __forceinline__ uint16_t from_f32(float f) {
  if constexpr (BF16) {
    return f32_to_bf16_bits(f);
  } else {
    return __builtin_bit_cast(uint16_t, static_cast<_Float16>(f));
  }
}

// Two fp32 values -> two storage values in one dword (first value in the low half).  fp16: the packed
// convert instruction of gfx950, same round-to-nearest-even as the scalar one.
template <bool BF16>
__device__ __forceinline__ uint32_t pack2_from_f32(float a, float b) {
  if constexpr (BF16) {
    return pack2_bf16(a, b);
  } else {
    typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
    typedef float float2_t __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(float2_t{a, b}, half2_t));
  }
}

// Where pairs of pack2_from_f32 are stored, every NaN becomes the one that from_f32 makes of it for bf16 (0x7FC0), so that a
// result's bits do not depend on the kernel that a call takes.  A wave looks for NaNs in the packed words while it stores them,
// one product with zero per word, and where it found one (or an infinity) it replaces the NaNs in what it has staged and stores
// that again.  us per forward, without the watch and with it: 777 x 4096 -> 22016 65.4 / 65.4, 2048 x 4096 -> 4096 36.7 / 36.6, 777 x
// 4096 -> 4096 23.0 / 23.5, int8 2048 x 28672 -> 8192 423 / 429.  (Looking at the accumulators instead costs registers that the
// large tiles do not have: replacing NaNs there spilled up to 322 of them and took 777 x 4096 -> 22016 from 69 to 81 us, comparing
// them alone spilled 34, 61.9 -> 66.5.)
template <bool BF16>
struct NanWatch {
  float seen = 0.0f;  // NaN once one was seen
  template <class V4>
  __device__ __forceinline__ void add(const V4 &words) {
    if constexpr (BF16) {
      typedef __bf16 bf2_t __attribute__((ext_vector_type(2)));
      const bf2_t zero = {static_cast<__bf16>(0.0f), static_cast<__bf16>(0.0f)};
#pragma unroll
      for (int k = 0; k < 4; ++k) seen = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf2_t, static_cast<uint32_t>(words[k])), zero, seen, false);
    }
  }
  // (wave-uniform)
  __device__ __forceinline__ bool any() const {
    if constexpr (BF16) return __builtin_amdgcn_ballot_w64(seen != seen) != 0;
    return false;
  }
};
__device__ __forceinline__ uint32_t canonical_bf16_pair(uint32_t w) {
  const uint32_t lo = (w & 0x7FFFu) > 0x7F80u ? 0x7FC0u : w & 0xFFFFu, hi = (w & 0x7FFF0000u) > 0x7F800000u ? 0x7FC00000u : w & 0xFFFF0000u;
  return lo | hi;
}
// stage: `bytes` (a multiple of 16) of LDS that this wave has staged and stored; afterwards it can be stored again
__device__ __forceinline__ void canonical_nans(uint8_t *stage, int bytes) {
#pragma unroll 1
  for (int i = (threadIdx.x & 63) * 16; i < bytes; i += 1024) {
    uint4 *at = reinterpret_cast<uint4 *>(stage + i);
    const uint4 w = *at;
    *at = make_uint4(canonical_bf16_pair(w.x), canonical_bf16_pair(w.y), canonical_bf16_pair(w.z), canonical_bf16_pair(w.w));
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (a wait only: no hazard; the first stores are done)
}

// Round an fp32 value to the storage type and return it as fp32 again.
template <bool BF16>
__device__ __forceinline__ float round_storage(float f) {
  return to_f32<BF16>(from_f32<BF16>(f));
}

// Lane exchange inside a row of 16 lanes through the DPP path of the vector ALU (no LDS traffic).
template <int CTRL>
__device__ __forceinline__ float dpp_move(float v) {
  return __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, false));
}
constexpr int kDppSwap1 = 0xB1;        // quad_perm [1,0,3,2]
constexpr int kDppSwap2 = 0x4E;        // quad_perm [2,3,0,1]
constexpr int kDppHalfMirror = 0x141;  // lane i <-> 7 - i inside each group of 8
constexpr int kDppMirror = 0x140;      // lane i <-> 15 - i inside each row of 16

// Wave-wide reductions; every lane of the wave must be active.  Four DPP steps make each row of 16
// uniform, the four rows are then combined through scalar registers.
__device__ __forceinline__ float wave_max(float v) {
  v = fmaxf(v, dpp_move<kDppSwap1>(v));
  v = fmaxf(v, dpp_move<kDppSwap2>(v));
  v = fmaxf(v, dpp_move<kDppHalfMirror>(v));
  v = fmaxf(v, dpp_move<kDppMirror>(v));
  const int b = __builtin_bit_cast(int, v);
  const float r0 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 0));
  const float r1 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 16));
  const float r2 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 32));
  const float r3 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 48));
  return fmaxf(fmaxf(r0, r1), fmaxf(r2, r3));
}
__device__ __forceinline__ float wave_min(float v) {
  v = fminf(v, dpp_move<kDppSwap1>(v));
  v = fminf(v, dpp_move<kDppSwap2>(v));
  v = fminf(v, dpp_move<kDppHalfMirror>(v));
  v = fminf(v, dpp_move<kDppMirror>(v));
  const int b = __builtin_bit_cast(int, v);
  const float r0 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 0));
  const float r1 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 16));
  const float r2 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 32));
  const float r3 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 48));
  return fminf(fminf(r0, r1), fminf(r2, r3));
}

// integer sum over the wave (every lane active), same scheme
template <int CTRL>
__device__ __forceinline__ int dpp_move_i(int v) {
  return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xF, 0xF, false);
}
__device__ __forceinline__ int wave_sum(int v) {
  v += dpp_move_i<kDppSwap1>(v);
  v += dpp_move_i<kDppSwap2>(v);
  v += dpp_move_i<kDppHalfMirror>(v);
  v += dpp_move_i<kDppMirror>(v);
  return __builtin_amdgcn_readlane(v, 0) + __builtin_amdgcn_readlane(v, 16) + __builtin_amdgcn_readlane(v, 32) +
         __builtin_amdgcn_readlane(v, 48);
}

// ---- direct global -> LDS copies ---------------------------------------------------------
// One wave-wide 64 x 16-byte copy global -> LDS: lane i reads 16 bytes at sbase + voff_i and
// they land at LDS address m0 + 16 i.  sbase (scalar) and m0 are wave-uniform, so advancing K
// costs scalar adds only and a load is two instructions (s_mov m0, global_load_lds).  Written
// as inline assembly so that the outstanding-load count stays under this file's control: the
// loop waits with vmcnt(loads per stage), leaving the newest stage in flight across the barrier.
// (s_nop 0: one wait state between the scalar write of m0 and the copy that reads it, which the compiler
// keeps for its own LDS copies on this generation and cannot see inside an asm statement.  m0 is declared
// clobbered; the "memory" clobber orders the statement against the compiler's own LDS and global accesses.)
__device__ __forceinline__ void dma_load16(const uint8_t *sbase, uint32_t voff, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(lds_addr), "v"(voff), "s"(sbase) : "memory", "m0");
}

// The same with 2 and 4 bytes per lane, any 2- and 4-byte aligned addresses: lane i's value lands in the four bytes at LDS
// address m0 + 4 i (2 bytes: in the low half; the high half is not to be read).
__device__ __forceinline__ void dma_load_u16(const void *sbase, uint32_t voff, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_ushort %1, %2" : : "s"(lds_addr), "v"(voff), "s"(sbase) : "memory", "m0");
}
__device__ __forceinline__ void dma_load_u32(const void *sbase, uint32_t voff, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" : : "s"(lds_addr), "v"(voff), "s"(sbase) : "memory", "m0");
}

__device__ __forceinline__ uint32_t lds_address(const void *p) {
  return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((const __attribute__((address_space(3))) void *)p));
}

// s_waitcnt immediate for "vmcnt <= n", every other counter unconstrained (gfx9 encoding)
constexpr int vmcnt_imm(int n) { return (n & 0xF) | ((n >> 4) << 14) | 0x0F70; }

}  // namespace quik
