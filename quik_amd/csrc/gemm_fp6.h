// int4 x int4 GEMM on the 6-bit matrix-core path of CDNA4 (gfx950), exact.
//
// v_mfma_f32_32x32x64_f8f6f4 with 6-bit E2M3 operands runs at twice the rate of the int8 MFMA.
// The E2M3 bit patterns 0 .. 15 (sign 0, exponent 00 / 01) are the uniformly spaced values
// L / 8, so a 4-bit level L = code + 8 IS an E2M3 number, zero-extended to 6 bits.  Products
// La Lw / 64 are multiples of 1/64 and their sum over K stays below 2^24 / 64 for K <= 74496 (225 K <
// 2^24), so the fp32 accumulation is exact in any order, and
//     sum_k a_k w_k = 64 S - 8 sum_k La_k - 8 sum_k Lw_k + 64 K,      S = sum_k (La_k / 8)(Lw_k / 8)
// recovers the integer accumulator exactly (every term is an integer below 2^24).  The accumulators
// start at K - sum_k La_k / 8 - sum_k Lw_k / 8 (between -176 K and 64 K 64ths, from where they only rise, to the result:
// still exact) and end at a 64th of the integer; the 64 goes into the row's scale where that is exact (scales_take_64), else onto
// the sum.  From there the epilogue is the one of gemm_kernels.h, so the output is bit-identical to the int8-MFMA path.
//
// Operand format: fp6_format.h.  Both operand buffers are stored as the sequence of LDS images the
// tiles need, so a copy instruction moves one contiguous kilobyte and every cache line is requested
// once per tile (with row-major operands a 32-byte piece per row and step asks for each line four
// times, and the 64 KB a tile touches in four steps do not survive in the 32 KB vector cache: the
// loop was bound by the cache-to-CU path at a quarter of its rate).  One MFMA k-step (64 elements)
// of a lane is a 16-byte head read plus an 8-byte tail read, both free of bank conflicts.
//
// Pipeline: a ring of NS LDS slots (six to twelve), one per k-step, filled by global_load_lds_dwordx4.  While step j
// feeds the MFMAs, the fragments of step j + 1 are read into registers and steps j + 2 .. j + NS - 1 are
// landing (the slot of step j was handed to step j + NS when step j's reads were done); the outlier
// GEMM's fp16/bf16 steps (16 elements each, 32 bytes per row like a head) run through the same ring
// after the integer steps.
#pragma once
#include "fp6_format.h"
#include "gemm_kernels.h"

namespace quik {

typedef int v2i __attribute__((ext_vector_type(2)));
typedef int v8i __attribute__((ext_vector_type(8)));

// One wave-wide copy global -> LDS (see dma_load16) whose instruction offset moves both addresses: the three
// kilobytes of a block unit are copied with one source pointer and one LDS base.
// (Hazards: one wait state between the scalar write of m0 and the copy that reads it, the s_nop 0; m0 is in the
// clobber list, so the compiler does not keep a value of its own in it across the statement; the "memory" clobber
// keeps LDS accesses of the compiler on their side of the copy, and completion is awaited through vmcnt.)
template <int OFFSET>
__device__ __forceinline__ void dma_load16k(const uint8_t *sbase, uint32_t voff, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 offset:%3"
               : : "s"(lds_addr), "v"(voff), "s"(sbase), "n"(OFFSET) : "memory", "m0");
}

// The same for all lanes or none (`lanes`: all bits set or none): a copy that only some waves make, in a stream whose outstanding copies all
// waves count alike (with no lane active the copy moves nothing and is counted as any other).  exec holds all lanes outside.
template <int OFFSET>
__device__ __forceinline__ void dma_load16k_if(uint32_t lanes, const uint8_t *sbase, uint32_t voff, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_mov_b32 exec_lo, %4\n\ts_mov_b32 exec_hi, %4\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 offset:%3\n\ts_mov_b64 exec, -1"
               : : "s"(lds_addr), "v"(voff), "s"(sbase), "n"(OFFSET), "s"(lanes) : "memory", "m0", "exec");
}

// LDS slots of the tile-ordered rings, `stage` bytes each: six, or with one workgroup per CU (DMA_STAGES > 4) as many as
// fit 144 KB, an even number, at most twelve.
template <class C>
constexpr int ring_slots(int stage) {
  const int most = 144 * 1024 / stage / 2 * 2;
  return C::DMA_STAGES <= 4 ? 6 : most < 12 ? most : 12;
}

// a fragment of the 4-bit format -> its 6 operand dwords (fp6_format.h)
typedef int v6i __attribute__((ext_vector_type(6)));
__device__ __forceinline__ v6i nib_expand(const v4i q) {
  constexpr int kU = static_cast<int>(kNibUpper), kL = static_cast<int>(kNibLower);
  return v6i{q.x & ~kU, q.y & ~kL, (q.x & kU) | (q.y & kL), q.z & ~kU, q.w & ~kL, (q.z & kU) | (q.w & kL)};
}
// acc += w_frag x x_frag, 64 levels (block scales 0, 0: the unscaled instruction, see gemm_fp6.h)
__device__ __forceinline__ void nib_mma(const v6i &x, const v6i &w, v16f &acc) {
  const v8i w8 = {w[0], w[1], w[2], w[3], w[4], w[5], 0, 0}, x8 = {x[0], x[1], x[2], x[3], x[4], x[5], 0, 0};
  acc = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(w8, x8, acc, 2, 2, 0, 0, 0, 0);
}
// the value is there at this point (empty statement: no hazard): a fragment is expanded where the source says, not later, in
// front of the products that read it, where nothing covers it
__device__ __forceinline__ void pin(v6i &x) { asm volatile("" : "+v"(x)); }

// W4: the weights are in the 4-bit format
template <class C, bool W4 = false>
struct Fp6Pipe {
  static constexpr int MI = C::MI, NI = C::NI, NF = MI + NI;
  static constexpr int NT = W4 ? MI : NF;  // fragments that have a tail
  static constexpr int WU = W4 ? 2048 : 3072;  // bytes of a weight unit
  static constexpr int NS = ring_slots<C>(C::BM * 48 + C::BN * (WU / 64));  // LDS slots; one step is multiplied, NS - 1 are landed or in flight
  // a wave's fragments start at a 64-row block of the operand, or the wave has a single 32-row fragment (then it may
  // be the second half of a block)
  static_assert(C::WM % 64 == 0 || C::MI == 1, "a wave's token rows");
  static_assert(C::WN % 64 == 0 || C::NI == 1, "a wave's weight rows");
  static_assert(C::WAVES == 4 || C::WAVES == 8, "copy assignment below");
  // LDS slot of one step: the 3 KB units of the tile's X blocks, then of its W blocks, as they are in memory
  static constexpr int W_OFF = C::BM * 48;
  static constexpr int STAGE = C::BM * 48 + C::BN * (WU / 64);
  static constexpr int SMEM = NS * STAGE;
  // Copies per step: 3 per 64-row block, 2 per weight block in the 4-bit format (head image of rows 0..31, of rows 32..63, tail image), XB + WB blocks.
  // Every wave copies one whole block from its source A (X block w, or W block w - XB when the tile has
  // fewer than 4 X blocks), and NB further kilobytes from its source B:
  //   256x256: W block w (3);  256x128: W block w % 2, pieces w / 2 and w / 2 + 1 (piece 1 is copied twice);
  //   128x128: none;  128x64: none (two waves copy the one W block: the same bytes to the same place).
  // (W4: a wave whose source A is a W block makes its third copy with no lane; 256x128: one further kilobyte, none twice)
  static constexpr int XB = C::BM / 64, WB = C::BN / 64;
  // (eight waves, 256x256: one block per wave, no source B)
  static constexpr int NB = C::WAVES == 8 ? 0 : XB + WB == 8 ? WU / 1024 : XB + WB == 6 ? (W4 ? 1 : 2) : 0;
  static_assert((XB == 4 && (WB == 4 || WB == 2)) || (XB == 2 && (WB == 2 || WB == 1)), "supported tile shapes");
  static_assert(C::WAVES == 4 || XB + WB == 8, "eight waves copy eight blocks");
  static constexpr int P = 3 + NB;  // copies per wave and step
  static_assert((NS - 3) * P <= 63, "the steps in flight must fit the vmcnt counter");

  uint8_t *smem;
  uint32_t lds0;
  const uint8_t *pa, *pb;   // wave-uniform: sources of the next step to be copied
  uint32_t da, db;          // wave-uniform: destinations inside a slot
  int adv_a;                // W4: bytes of source A's units
  uint32_t third;           // W4: lanes of source A's third copy: none where it is a W block
  uint32_t fill;            // wave-uniform: LDS address of the slot the next copy fills
  int left;                 // steps whose copy has not been issued yet
  uint32_t lane16;
  uint32_t rd;              // byte offset of the slot the next fragment read looks at
  int steps0, steps;        // integer steps, all steps
  uint32_t x_head, w_head;  // this lane's head offsets inside a slot (fragment j: + 1024 j)
  uint32_t x_head3[NS / 2], w_head3[NS / 2], tail3[NS / 2][NT];  // the same inside slots 0, 2, 4, .. (for steps whose slot is
                                                  // known at compile time: the odd slot is an immediate offset away)
  uint32_t tail[NT];        // this lane's tail offsets inside a slot, one register per fragment: reads that share
                            // a base register are paired into one 4-register read by the compiler, and the halves
                            // then have to be copied into the operand tuples behind an exposed LDS round trip

  // xb0 / wb0: first 64-row block of the tile in each operand buffer
  // unit0: first unit (step) of every block to copy; n_int / n_f: integer and outlier steps from there on
  // (-1: all of the block's, from its first unit)
  template <class LayoutW>
  __device__ __forceinline__ void init(uint8_t *smem_, const uint8_t *xbuf, const Fp6Layout &lx, int64_t xb0,
                                       const uint8_t *wbuf, const LayoutW &lw, int64_t wb0, int unit0 = 0,
                                       int n_int = -1, int n_f = -1) {
    smem = smem_;
    lds0 = lds_address(smem_);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave / C::WAVES_N, wn = wave % C::WAVES_N;
    auto block_ptr = [&](bool is_x, int blk) {
      const int64_t blocks = is_x ? lx.blocks : lw.blocks, bytes = is_x ? lx.block_bytes : lw.block_bytes;
      int64_t B = (is_x ? xb0 : wb0) + blk;
      B = B < blocks ? B : blocks - 1;  // blocks past the matrix: any valid block, results never stored
      return (is_x ? xbuf : wbuf) + B * bytes + int64_t(unit0) * (is_x ? 3072 : WU);
    };
    {
      const bool is_x = wave < XB;
      const int blk = is_x ? wave : (wave - XB) % WB;
      pa = block_ptr(is_x, blk);
      da = is_x ? blk * 3072 : W_OFF + blk * WU;
      adv_a = is_x ? 3072 : WU;
      third = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(is_x ? -1 : 0));
    }
    pb = pa;
    db = da;
    if constexpr (XB + WB == 8 && C::WAVES == 4) {
      pb = block_ptr(false, wave);
      db = W_OFF + wave * WU;
    } else if constexpr (W4 && NB == 1) {
      pb = block_ptr(false, wave & 1) + (wave >> 1) * 1024;
      db = W_OFF + (wave & 1) * WU + (wave >> 1) * 1024;
    } else if constexpr (NB == 2) {
      pb = block_ptr(false, wave & 1) + (wave >> 1) * 1024;
      db = W_OFF + (wave & 1) * 3072 + (wave >> 1) * 1024;
    }
    lane16 = lane * 16;
    fill = lds0;
    rd = 0;
    steps0 = n_int < 0 ? static_cast<int>(lx.steps) : n_int;
    steps = steps0 + (n_f < 0 ? static_cast<int>(lx.fsteps) : n_f);
    left = steps;
    const int r = lane & 31, h = lane >> 5;
    const int slot16 = (h ^ ((r >> 3) & 1)) << 4;
    // first 32-row fragment of the wave in each operand: block fx0 / 2 (fw0 / 2), half fx0 % 2 (odd only for waves of
    // a single fragment)
    const int fx0 = wm * C::WM / 32, fw0 = wn * C::WN / 32;
    x_head = (fx0 >> 1) * 3072 + (fx0 & 1) * 1024 + r * 32 + slot16;
    w_head = W_OFF + (fw0 >> 1) * WU + (fw0 & 1) * 1024 + r * 32 + slot16;
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const int jj = j < MI ? j : j - MI;
      const int f0 = j < MI ? fx0 : fw0;
      tail[j] = (j < MI ? 0 : W_OFF) + (f0 >> 1) * 3072 + (jj >> 1) * 3072 + 2048 + h * 512 +
                ((((f0 & 1) + jj) & 1) * 32 + r) * 8;
      asm volatile("" : "+v"(tail[j]));  // unrelated values as far as the compiler can tell (empty statement: no hazard)
    }
#pragma unroll
    for (int q = 0; q < NS / 2; ++q) {
      x_head3[q] = x_head + q * 2 * STAGE;
      w_head3[q] = w_head + q * 2 * STAGE;
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        tail3[q][j] = tail[j] + q * 2 * STAGE;
        asm volatile("" : "+v"(tail3[q][j]));
      }
    }
  }

  // Copy G (0 .. P-1) of the step being copied; after the last one the scalar bookkeeping: two pointer
  // bumps and one slot bump.  Past the last step the pointers stop and the last step is copied again into
  // a slot nobody reads.
  // FS: slot being filled when known at compile time (the caller keeps `fill` consistent), -1: `fill`
  template <int G, int FS = -1>
  __device__ __forceinline__ void issue_one() {
    const uint32_t slot = FS < 0 ? fill : lds0 + (FS < 0 ? 0 : FS) * STAGE;
    if constexpr (G < 3) {
      if constexpr (W4 && G == 2 && !(XB == 4 && C::WAVES == 4)) {  // (some waves' source A is a W block)
        dma_load16k_if<2048>(third, pa, lane16, slot + da);
      } else {
        dma_load16k<G * 1024>(pa, lane16, slot + da);
      }
    } else {
      dma_load16k<(G - 3) * 1024>(pb, lane16, slot + db);
    }
    if constexpr (G == P - 1) {
      const bool more = left > 1;
      left -= 1;
      pa += more ? (W4 ? adv_a : 3072) : 0;
      pb += more ? WU : 0;
      if constexpr (FS < 0) {
        fill += STAGE;
        fill = fill == lds0 + NS * STAGE ? lds0 : fill;
      }
    }
  }
  template <int G = 0>
  __device__ __forceinline__ void issue() {
    if constexpr (G < P) {
      issue_one<G>();
      issue<G + 1>();
    }
  }

  // Fill the ring: afterwards steps 0 and 1 are visible and steps 2 .. NS - 2 are in flight; the copies of step
  // NS - 1 are made during the MFMAs of step 0.
  // In two parts: landed() is what this wave does with what it requested before the ring, behind the first part the others have
  // done so too, and what needs that goes in front of the second, under the first steps' way here.
  template <class Landed>
  __device__ __forceinline__ void start_vectors(Landed landed) {
    static_for<NS - 1>([&](auto) { issue(); });
    static_assert((NS - 1) * P <= 63, "the vmcnt counter");
    __builtin_amdgcn_s_waitcnt(vmcnt_imm((NS - 1) * P));
    asm volatile("" ::: "memory");  // (empty: LDS reads of what has landed stay behind the wait)
    landed();
    __syncthreads();
  }
  __device__ __forceinline__ void start_steps() {
    __builtin_amdgcn_s_waitcnt(vmcnt_imm((NS - 3) * P));
    asm volatile("" ::: "memory");  // (empty, as above)
    __syncthreads();
  }
  __device__ __forceinline__ void start() {
    static_for<NS - 1>([&](auto) { issue(); });
    start_steps();
  }

  __device__ __forceinline__ void next_read_slot() {
    rd += STAGE;
    rd = rd == NS * STAGE ? 0 : rd;
  }

  // fragment j (32 rows) of this wave: head image j, tail image j / 2 at row offset 32 (j % 2)
  // RS: slot being read when known at compile time, -1: `rd`
  template <int J, int RS = -1>
  __device__ __forceinline__ void read6_one(v4i (&fh)[NF], v2i (&ft)[NF]) const {
    constexpr int jj = J < MI ? J : J - MI;
    if constexpr (J >= NT) {  // 4-bit format: no tail
      if constexpr (RS < 0) {
        fh[J] = *reinterpret_cast<const v4i *>(smem + rd + w_head + (jj >> 1) * WU + (jj & 1) * 1024);
      } else {
        constexpr int q = (RS < 0 ? 0 : RS) / 2, odd = ((RS < 0 ? 0 : RS) % 2) * STAGE;
        fh[J] = *reinterpret_cast<const v4i *>(smem + w_head3[q] + odd + (jj >> 1) * WU + (jj & 1) * 1024);
      }
    } else if constexpr (RS < 0) {
      const uint8_t *s = smem + rd;
      fh[J] = *reinterpret_cast<const v4i *>(s + (J < MI ? x_head : w_head) + (jj >> 1) * 3072 + (jj & 1) * 1024);
      ft[J] = *reinterpret_cast<const v2i *>(s + tail[J]);
    } else {
      constexpr int q = (RS < 0 ? 0 : RS) / 2, odd = ((RS < 0 ? 0 : RS) % 2) * STAGE;
      fh[J] = *reinterpret_cast<const v4i *>(smem + (J < MI ? x_head3[q] : w_head3[q]) + odd + (jj >> 1) * 3072 +
                                             (jj & 1) * 1024);
      ft[J] = *reinterpret_cast<const v2i *>(smem + tail3[q][J] + odd);
    }
  }
  template <int J>
  __device__ __forceinline__ void read16_one(v4i (&f)[NF]) const {
    constexpr int jj = J < MI ? J : J - MI;
    f[J] = *reinterpret_cast<const v4i *>(smem + rd + (J < MI ? x_head : w_head) + (jj >> 1) * (J < MI ? 3072 : WU) + (jj & 1) * 1024);
  }
  template <int J = 0>
  __device__ __forceinline__ void read6(v4i (&fh)[NF], v2i (&ft)[NF]) {
    if constexpr (J < NF) {
      read6_one<J>(fh, ft);
      read6<J + 1>(fh, ft);
    } else {
      next_read_slot();
    }
  }
  template <int J = 0>
  __device__ __forceinline__ void read16(v4i (&f)[NF]) {
    if constexpr (J < NF) {
      read16_one<J>(f);
      read16<J + 1>(f);
    } else {
      next_read_slot();
    }
  }

  // MFMA I (0 .. MI NI - 1) of a step: block (mi, ni) = (I % MI, I / MI)
  template <int I>
  static __device__ __forceinline__ void mfma6_one(const v4i (&fh)[NF], const v2i (&ft)[NF], v16f (&acc)[MI][NI]) {
    constexpr int mi = I % MI, ni = I / MI;
    const v8i w = v8i{fh[MI + ni].x, fh[MI + ni].y, fh[MI + ni].z, fh[MI + ni].w, ft[MI + ni].x, ft[MI + ni].y, 0, 0};
    const v8i x = v8i{fh[mi].x, fh[mi].y, fh[mi].z, fh[mi].w, ft[mi].x, ft[mi].y, 0, 0};
    // Block scales of 2^0.  Written as scale operands 0, 0 the compiler emits the plain v_mfma_f32_32x32x64_f8f6f4,
    // whose scales are 1.0 by definition; with the equivalent E8M0 value 127 spelled out it emits the scaled form,
    // a scale-load instruction in front of every MFMA, which costs an issue slot each (measured on chains of
    // dependent MFMAs: identical results, 21 % more time).  Were a compiler to keep the scaled form WITH operands 0,
    // every product would be scaled by 2^-127: the Makefile's check-mfma target reads the mnemonics of the built
    // object and fails the build on a scaled f8f6f4 MFMA.
    acc[mi][ni] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(w, x, acc[mi][ni], 2, 2, 0, 0, 0, 0);
  }
  template <bool BF16, int I>
  static __device__ __forceinline__ void mfma16_one(const v4i (&f)[NF], v16f (&acc)[MI][NI]) {
    constexpr int mi = I % MI, ni = I / MI;
    FragOps<BF16 ? kBF16 : kF16>::mma(f[mi], f[MI + ni], acc[mi][ni]);
  }

  // One step, cut into P chunks: chunk G holds its share of the step's MFMAs (on the fragments in `cur`),
  // of the next step's fragment reads (into `nxt`) and one of the P copies of the step NS - 1 ahead of
  // the one in the MFMAs.  A copy instruction occupies the wave until the memory pipeline has taken its 64
  // addresses; six of them in a row at the start of a step stall the MFMA issue for as long as the copies
  // take, so they go one by one between groups of MFMAs.  Then: wait until the step after next has
  // landed (the NS - 3 newer ones stay in flight) and a barrier makes it visible; behind it every wave has
  // issued the MFMAs of this step, which waited for their fragments, so this step's slot may be overwritten
  // by the copies issued during the next step.
  // RS / FS: the slots read and filled during this step when they are known at compile time (NS steps in a
  // row return to the same slots, so `rd` and `fill` stay valid without being touched), -1: `rd` / `fill`
  template <int RS = -1, int FS = -1, int G = 0>
  __device__ __forceinline__ void step6(const v4i (&ch)[NF], const v2i (&ct)[NF], v4i (&nh)[NF], v2i (&nt)[NF],
                                        v16f (&acc)[MI][NI]) {
    constexpr int MM = MI * NI;
    if constexpr (G < P) {
      constexpr int r_lo = G * NF / P, r_hi = (G + 1) * NF / P, m_lo = G * MM / P, m_hi = (G + 1) * MM / P;
      chunk_reads6<RS, r_lo, r_hi>(nh, nt);
      chunk_mfmas6<m_lo, m_hi>(ch, ct, acc);
      if constexpr (m_hi > m_lo) {
#pragma unroll
        for (int i = m_lo; i < m_hi; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, (2 * (r_hi - r_lo) + (m_hi - m_lo) - 1) / (m_hi - m_lo), 0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      issue_one<G, FS>();
      __builtin_amdgcn_sched_barrier(0);
      step6<RS, FS, G + 1>(ch, ct, nh, nt, acc);
    } else {
      if constexpr (RS < 0) next_read_slot();
      __builtin_amdgcn_s_waitcnt(vmcnt_imm((NS - 3) * P));
      __builtin_amdgcn_s_barrier();
    }
  }
  // W4: the same step.  The weight fragments are read first, as they are in memory, and expanded behind the reads of the
  // activation's, in the last chunks of the step, in front of the one that multiplies them.
  template <int LO, int HI>
  static __device__ __forceinline__ void chunk_expand(const v4i (&h)[NF], v6i (&w)[NI]) {
    if constexpr (LO < HI) {
      w[LO] = nib_expand(h[MI + LO]);
      chunk_expand<LO + 1, HI>(h, w);
    }
  }
  template <int LO, int HI>
  static __device__ __forceinline__ void chunk_mfmas64(const v4i (&ch)[NF], const v2i (&ct)[NF], const v6i (&cw)[NI], v16f (&acc)[MI][NI]) {
    if constexpr (LO < HI) {
      constexpr int mi = LO % MI, ni = LO / MI;
      nib_mma(v6i{ch[mi].x, ch[mi].y, ch[mi].z, ch[mi].w, ct[mi].x, ct[mi].y}, cw[ni], acc[mi][ni]);
      chunk_mfmas64<LO + 1, HI>(ch, ct, cw, acc);
    }
  }
  template <int RS, int LO, int HI>  // in the order W, X
  __device__ __forceinline__ void chunk_reads64(v4i (&nh)[NF], v2i (&nt)[NF]) const {
    if constexpr (LO < HI) {
      read6_one<(LO < NI ? MI + LO : LO - NI), RS>(nh, nt);
      chunk_reads64<RS, LO + 1, HI>(nh, nt);
    }
  }
  template <int RS = -1, int FS = -1, int G = 0>
  __device__ __forceinline__ void step64(const v4i (&ch)[NF], const v2i (&ct)[NF], const v6i (&cw)[NI], v4i (&nh)[NF], v2i (&nt)[NF],
                                         v6i (&nw)[NI], v16f (&acc)[MI][NI]) {
    constexpr int MM = MI * NI, E0 = (P - 1) / 2 + 1;  // reads in chunks 0 .. E0 - 1, expansion in E0 .. P - 1
    if constexpr (G < P) {
      constexpr int m_lo = G * MM / P, m_hi = (G + 1) * MM / P;
      constexpr int r_lo = G < E0 ? G * NF / E0 : NF, r_hi = G < E0 ? (G + 1) * NF / E0 : NF;
      constexpr int e_lo = G < E0 ? 0 : (G - E0) * NI / (P - E0), e_hi = G < E0 ? 0 : (G - E0 + 1) * NI / (P - E0);
      chunk_reads64<RS, r_lo, r_hi>(nh, nt);
      chunk_expand<e_lo, e_hi>(nh, nw);
      chunk_mfmas64<m_lo, m_hi>(ch, ct, cw, acc);
      if constexpr (m_hi > m_lo) {
#pragma unroll
        for (int i = m_lo; i < m_hi; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, (2 * (r_hi - r_lo) + (m_hi - m_lo) - 1) / (m_hi - m_lo), 0);
          __builtin_amdgcn_sched_group_barrier(0x002, (8 * (e_hi - e_lo) + (m_hi - m_lo) - 1) / (m_hi - m_lo), 0);
        }
      }
      static_for<e_hi - e_lo>([&](auto J) __attribute__((always_inline)) { pin(nw[e_lo + J]); });
      __builtin_amdgcn_sched_barrier(0);
      issue_one<G, FS>();
      __builtin_amdgcn_sched_barrier(0);
      step64<RS, FS, G + 1>(ch, ct, cw, nh, nt, nw, acc);
    } else {
      if constexpr (RS < 0) next_read_slot();
      __builtin_amdgcn_s_waitcnt(vmcnt_imm((NS - 3) * P));
      __builtin_amdgcn_s_barrier();
    }
  }
  __device__ __forceinline__ void run_fp64(v16f (&acc)[MI][NI], v4i (&h0)[NF]) {
    v4i h1[NF];
    v2i t0[NF], t1[NF];
    v6i w0[NI], w1[NI];
    read6(h0, t0);
    chunk_expand<0, NI>(h0, w0);
    int j = 0;
    for (; j + NS <= steps0; j += NS) {
      static_for<NS / 2>([&](auto I) __attribute__((always_inline)) {
        constexpr int i = 2 * I;
        step64<i + 1, (i + NS - 1) % NS>(h0, t0, w0, h1, t1, w1, acc);
        step64<(i + 2) % NS, i>(h1, t1, w1, h0, t0, w0, acc);
      });
    }
    for (; j < steps0; j += 2) {
      step64(h0, t0, w0, h1, t1, w1, acc);
      step64(h1, t1, w1, h0, t0, w0, acc);
    }
  }
  template <int RS, int LO, int HI>
  __device__ __forceinline__ void chunk_reads6(v4i (&nh)[NF], v2i (&nt)[NF]) const {
    if constexpr (LO < HI) {
      read6_one<LO, RS>(nh, nt);
      chunk_reads6<RS, LO + 1, HI>(nh, nt);
    }
  }
  template <int LO, int HI>
  static __device__ __forceinline__ void chunk_mfmas6(const v4i (&ch)[NF], const v2i (&ct)[NF], v16f (&acc)[MI][NI]) {
    if constexpr (LO < HI) {
      mfma6_one<LO>(ch, ct, acc);
      chunk_mfmas6<LO + 1, HI>(ch, ct, acc);
    }
  }
  // The next step's fragments are read in the first chunks, the weights' first, as the MFMAs take them: read over the whole
  // step, the last one was on its way when the next step began with it.
  template <bool BF16, int G = 0>
  __device__ __forceinline__ void step16(const v4i (&cf)[NF], v4i (&nf)[NF], v16f (&acc)[MI][NI]) {
    constexpr int MM = MI * NI, E0 = (P - 1) / 2 + 1;
    if constexpr (G < P) {
      constexpr int r_lo = G < E0 ? G * NF / E0 : NF, r_hi = G < E0 ? (G + 1) * NF / E0 : NF, m_lo = G * MM / P, m_hi = (G + 1) * MM / P;
      chunk_reads16<r_lo, r_hi>(nf);
      chunk_mfmas16<BF16, m_lo, m_hi>(cf, acc);
      if constexpr (m_hi > m_lo) {
#pragma unroll
        for (int i = m_lo; i < m_hi; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, ((r_hi - r_lo) + (m_hi - m_lo) - 1) / (m_hi - m_lo), 0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      issue_one<G>();
      __builtin_amdgcn_sched_barrier(0);
      step16<BF16, G + 1>(cf, nf, acc);
    } else {
      next_read_slot();
      __builtin_amdgcn_s_waitcnt(vmcnt_imm((NS - 3) * P));
      __builtin_amdgcn_s_barrier();
    }
  }
  template <int LO, int HI>
  __device__ __forceinline__ void chunk_reads16(v4i (&nf)[NF]) const {
    if constexpr (LO < HI) {  // in the order W, X
      read16_one<(LO < NI ? MI + LO : LO - NI)>(nf);
      chunk_reads16<LO + 1, HI>(nf);
    }
  }
  template <bool BF16, int LO, int HI>
  static __device__ __forceinline__ void chunk_mfmas16(const v4i (&cf)[NF], v16f (&acc)[MI][NI]) {
    if constexpr (LO < HI) {
      mfma16_one<BF16, LO>(cf, acc);
      chunk_mfmas16<BF16, LO + 1, HI>(cf, acc);
    }
  }

  // Integer steps [0, steps0): acc += (Lw / 8)(Lx / 8) summed over 64 elements per MFMA.  h0: afterwards the heads of the
  // step behind them, the fragments of the first outlier step.
  __device__ __forceinline__ void run_fp6(v16f (&acc)[MI][NI], v4i (&h0)[NF]) {
    if constexpr (W4) return run_fp64(acc, h0);
    v4i h1[NF];
    v2i t0[NF], t1[NF];
    read6(h0, t0);
    // here: step 0 in h0 / t0, `rd` at slot 1, `fill` at slot NS - 1.  NS steps at a time with the slots as
    // immediates (no address arithmetic in the loop), then the remaining pairs with `rd` / `fill`
    int j = 0;
    for (; j + NS <= steps0; j += NS) {
      static_for<NS / 2>([&](auto I) __attribute__((always_inline)) {
        constexpr int i = 2 * I;
        step6<i + 1, (i + NS - 1) % NS>(h0, t0, h1, t1, acc);
        step6<(i + 2) % NS, i>(h1, t1, h0, t0, acc);
      });
    }
    for (; j < steps0; j += 2) {
      step6(h0, t0, h1, t1, acc);
      step6(h1, t1, h0, t0, acc);
    }
  }

  // Outlier steps [steps0, steps): acc += fp_w fp_x^T, 16 elements per MFMA.  f0: the first one's fragments
  template <bool BF16>
  __device__ __forceinline__ void run_f16(v16f (&acc)[MI][NI], v4i (&f0)[NF]) {
    v4i f1[NF];
    for (int j = steps0; j < steps; j += 2) {
      step16<BF16>(f0, f1, acc);
      step16<BF16>(f1, f0, acc);
    }
  }

  // All steps of a wave whose rows or columns lie past the matrix: its copies, waits and barriers, no products.
  __device__ __forceinline__ void run_idle() {
    for (int j = 0; j < steps; ++j) {
      issue();
      __builtin_amdgcn_s_waitcnt(vmcnt_imm((NS - 3) * P));
      __builtin_amdgcn_s_barrier();
    }
  }

  __device__ __forceinline__ void drain() const {
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
    __syncthreads();
  }
};

struct Fused6Args {
  const uint8_t *xbuf, *wbuf;  // operand buffers (activations, weights), outlier columns included
  const uint16_t *meta, *s_col, *w_red, *bias;
  uint16_t *out;
  int M, N, ldo, K, F;  // N: columns of this launch (wbuf, s_col, ... start at its first column)
  int n_first;          // first column of this launch inside the weight buffer's row numbering
  int N_total;          // rows of the weight buffer
};

// Per-tile vectors in LDS behind the ring: the five of TileVectors plus the two integer corrections
//   rowc[m] = K - sum_k Lx / 8,  colc[n] = -sum_k Lw / 8: the accumulators start at their sum (exact in fp32).
template <class C>
struct TileVectors6 {
  static constexpr int kBytes = (4 * C::BN + 3 * C::BM) * 4;
  float *scol, *wred, *bias, *colc, *srow, *zs, *rowc;
  __device__ __forceinline__ explicit TileVectors6(uint8_t *base) {
    scol = reinterpret_cast<float *>(base);
    wred = scol + C::BN;
    bias = wred + C::BN;
    colc = bias + C::BN;
    srow = colc + C::BN;
    zs = srow + C::BM;
    rowc = zs + C::BM;
  }
};

// The scales, zero points, reduced weights and bias of a tile, requested in front of the ring's copies (a thread per row and
// column, 16 bits each into the low half of its slot) and widened in place, by the same thread, when they have landed.  Read
// into registers and written to the LDS they cost two trips to memory, one for the columns and one for the rows, before
// the first copy left: 128 x 5120 -> 13824 19.1 -> 18.3 us per forward, 300 x 4544 -> 4544 18.1 -> 17.4, 512 x 4096 -> 4096
// 18.2 -> 17.7, bf16 777 x 4096 -> 22016 70.1 -> 68.8; where a tile takes long, no difference beyond the noise (2048 x 8192 -> 28672,
// 2048 x 8192 -> 1024, int8 365 x 28672 -> 8192).
template <class C, class Vectors, class Args>
__device__ __forceinline__ void tile_vector_request(const Vectors &tv, const Args &p, int m0, int n0, int wave) {
  const int i = threadIdx.x;
  if (wave * 64 < C::BN) {
    const uint32_t off = static_cast<uint32_t>(n0 + i < p.N ? n0 + i : p.N - 1) * 2, at = wave * 256;
    dma_load_u16(p.s_col, off, lds_address(tv.scol) + at);
    if (p.w_red) dma_load_u16(p.w_red, off, lds_address(tv.wred) + at);
    if (p.bias) dma_load_u16(p.bias, off, lds_address(tv.bias) + at);
  }
  if (wave * 64 < C::BM) {
    const uint32_t m = static_cast<uint32_t>(m0 + i < p.M ? m0 + i : p.M - 1), at = wave * 256;
    dma_load_u16(p.meta, p.w_red ? 4 * m : 2 * m, lds_address(tv.srow) + at);
    if (p.w_red) dma_load_u16(p.meta, 4 * m + 2, lds_address(tv.zs) + at);
  }
}
template <class C, bool BF16, class Vectors>
__device__ __forceinline__ void tile_vector_widen(const Vectors &tv, bool bias, bool asym, float shift) {
  const int i = threadIdx.x;
  auto wide = [&](const float *v) { return to_f32<BF16>(static_cast<uint16_t>(__float_as_uint(v[i]))); };
  if (i < C::BN) {
    tv.scol[i] = wide(tv.scol);
    tv.wred[i] = asym ? wide(tv.wred) : 0.0f;
    tv.bias[i] = bias ? wide(tv.bias) : 0.0f;
  }
  if (i < C::BM) {
    const float s = wide(tv.srow);
    tv.srow[i] = s;
    tv.zs[i] = asym ? wide(tv.zs) + shift * s : 0.0f;
  }
}

// The level sums behind the operand blocks of a 4- or 6-bit buffer, in the same way.
template <class C, class Vectors, class Args>
__device__ __forceinline__ void tile_sums_request(const Vectors &tv, const Args &p, int64_t x_sums, int64_t w_sums, int m0, int n0,
                                                  int wave) {
  const int i = threadIdx.x;
  if (wave * 64 < C::BN) {
    const int n = n0 + i < p.N ? n0 + i : p.N - 1;
    dma_load_u32(p.wbuf + w_sums + static_cast<int64_t>(p.n_first) * 4, static_cast<uint32_t>(n) * 4, lds_address(tv.colc) + wave * 256);
  }
  if (wave * 64 < C::BM) {
    const int m = m0 + i < p.M ? m0 + i : p.M - 1;
    dma_load_u32(p.xbuf + x_sums, static_cast<uint32_t>(m) * 4, lds_address(tv.rowc) + wave * 256);
  }
}
template <class C, class Vectors>
__device__ __forceinline__ void tile_sums_widen(const Vectors &tv, int K) {
  const int i = threadIdx.x;
  if (i < C::BN) tv.colc[i] = static_cast<float>(__float_as_int(tv.colc[i])) * -0.125f;
  if (i < C::BM) tv.rowc[i] = static_cast<float>(8 * K - __float_as_int(tv.rowc[i])) * 0.125f;
}

template <class C, bool W4 = false>
constexpr int fused6_vectors_offset() {
  constexpr int staging = BlockStore<C, uint16_t>::kBytes * C::MI * C::WAVES;
  return staging > Fp6Pipe<C, W4>::SMEM ? staging : Fp6Pipe<C, W4>::SMEM;
}
template <class C, bool W4 = false>
constexpr int fused6_smem() {
  return fused6_vectors_offset<C, W4>() + TileVectors6<C>::kBytes;
}

// Split over K (few tiles, long K): `splits` workgroups per tile take `per` integer steps each and add their raw
// accumulators (int32, or the exact fp32 sums of the 6-bit path) through `partials`; the one that arrives last (counted in `counters`, which are zero between
// launches) sums them, exactly, and goes on with the outlier steps and the epilogue as a whole-K tile would: the
// result has the same bits.  partials: [tile][split][register][thread], 4 bytes each.
struct SplitK {
  int splits, per, grid_tiles;
  uint32_t *counters;
  int32_t *partials;
};
// The partial sums cross from one XCD's L2 to another's.  A device-wide fence would do that by writing back and
// invalidating the whole L2 of the XCD, once per wave, under the operand streams of the other tiles (measured: the
// launch takes three times as long), and device-scope atomic loads are issued one at a time.  Instead the partial
// sums are moved by ordinary 16-byte stores and loads that carry the device-scope cache policy (sc1: past the L2,
// one access at a time); the stores are complete (vmcnt) before the workgroup's barrier and the arrival count
// behind it, and the loads are issued only after the count has been seen.
// partials: [tile][split][group of 4 registers][thread][4].
// (the wait states: a store of more than 8 bytes reads its data registers over several cycles, and the instruction
// after this statement may be one that overwrites them; between the compiler's own instructions the compiler
// keeps that distance, around inline assembly it does not)
__device__ __forceinline__ void splitk_store4(int32_t *p, v4i v) {
  asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 2" : : "v"(p), "v"(v) : "memory");
}
// (a wait only: no register or wait-state hazard; "memory" keeps the compiler from moving stores across it)
__device__ __forceinline__ void splitk_stores_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
// eight 16-byte loads, STRIDE int32 apart, and the wait for them in one statement: the compiler sees the
// registers only once they hold the data (hazards: the outputs are early-clobber, so no load's destination
// overlaps an address register that a later load of the statement still reads; the statement ends with
// vmcnt(0), so nothing it started is in flight when the compiler's instructions resume)
template <int STRIDE>
__device__ __forceinline__ void splitk_load8(const int32_t *p, v4i *r) {
  asm volatile(
      "global_load_dwordx4 %0, %8, off sc1\n\tglobal_load_dwordx4 %1, %9, off sc1\n\t"
      "global_load_dwordx4 %2, %10, off sc1\n\tglobal_load_dwordx4 %3, %11, off sc1\n\t"
      "global_load_dwordx4 %4, %12, off sc1\n\tglobal_load_dwordx4 %5, %13, off sc1\n\t"
      "global_load_dwordx4 %6, %14, off sc1\n\tglobal_load_dwordx4 %7, %15, off sc1\n\t"
      "s_waitcnt vmcnt(0)"
      : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3]), "=&v"(r[4]), "=&v"(r[5]), "=&v"(r[6]), "=&v"(r[7])
      : "v"(p), "v"(p + STRIDE), "v"(p + 2 * STRIDE), "v"(p + 3 * STRIDE), "v"(p + 4 * STRIDE), "v"(p + 5 * STRIDE),
        "v"(p + 6 * STRIDE), "v"(p + 7 * STRIDE)
      : "memory");
}

template <int STRIDE>
__device__ __forceinline__ void splitk_load4(const int32_t *p, v4i *r) {
  asm volatile(
      "global_load_dwordx4 %0, %4, off sc1\n\tglobal_load_dwordx4 %1, %5, off sc1\n\t"
      "global_load_dwordx4 %2, %6, off sc1\n\tglobal_load_dwordx4 %3, %7, off sc1\n\t"
      "s_waitcnt vmcnt(0)"
      : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3])
      : "v"(p), "v"(p + STRIDE), "v"(p + 2 * STRIDE), "v"(p + 3 * STRIDE)
      : "memory");
}

// Adds a tile's raw accumulators over the splits (see SplitK).  Returns false in every workgroup but the one that
// arrived last; there `acc` holds the whole-K sums (INT: int32 bit patterns, else fp32) and the ring is idle.
template <class C, bool INT>
__device__ __forceinline__ bool splitk_combine(v16f (&acc)[C::MI][C::NI], const SplitK &sk, int tile_id, int split,
                                               uint8_t *smem) {
  static_assert(C::MI * C::NI == 4, "16 groups of 4 registers");
  constexpr int STRIDE = C::kThreads * 4;
  asm volatile("s_nop 15\n\ts_nop 15");  // the last MFMA results are architecturally visible
  int32_t *mine = sk.partials + (int64_t(tile_id) * sk.splits + split) * 16 * STRIDE + threadIdx.x * 4;
#pragma unroll
  for (int b = 0; b < C::MI * C::NI; ++b)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const v16f &a = acc[b / C::NI][b % C::NI];
      splitk_store4(mine + (b * 4 + g) * STRIDE,
                    v4i{__float_as_int(agpr_read(a[4 * g])), __float_as_int(agpr_read(a[4 * g + 1])),
                        __float_as_int(agpr_read(a[4 * g + 2])), __float_as_int(agpr_read(a[4 * g + 3]))});
    }
  splitk_stores_done();
  __syncthreads();
  int *last_s = reinterpret_cast<int *>(smem);
  if (threadIdx.x == 0) {
    const uint32_t before = __hip_atomic_fetch_add(sk.counters + tile_id, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *last_s = before == static_cast<uint32_t>(sk.splits - 1);
  }
  __syncthreads();
  const bool last = *last_s != 0;
  __syncthreads();
  if (!last) return false;
  for (int q = 0; q < sk.splits; ++q) {  // exact sums: the order does not matter
    if (q == split) continue;
    const int32_t *theirs = sk.partials + (int64_t(tile_id) * sk.splits + q) * 16 * STRIDE + threadIdx.x * 4;
    v4i t[16];
    splitk_load8<STRIDE>(theirs, t);
    splitk_load8<STRIDE>(theirs + 8 * STRIDE, t + 8);
#pragma unroll
    for (int b = 0; b < C::MI * C::NI; ++b)
#pragma unroll
      for (int g = 0; g < 4; ++g)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v16f &a = acc[b / C::NI][b % C::NI];
          const float mine_v = agpr_read(a[4 * g + e]);
          a[4 * g + e] = agpr_write(INT ? __int_as_float(__float_as_int(mine_v) + t[b * 4 + g][e])
                                        : mine_v + __int_as_float(t[b * 4 + g][e]));
        }
  }
  if (threadIdx.x == 0) __hip_atomic_store(sk.counters + tile_id, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return true;
}

// A wave of a tile at (m0, n0) that has no row or no column of the result: the tiles of the last row and column are padding
// in part, and a large GEMM takes what its power and LDS traffic take, not what its last round takes.  Without the MFMAs and
// LDS reads of such waves (us per forward): bf16 777 x 4096 -> 22016 71.5 -> 68.6, 552 x 5120 -> 13824 38.5 -> 36.3,
// 300 x 5120 -> 13824 30.7 -> 29.4, int8 600 x 28672 -> 8192 185 -> 175; full tiles unchanged within 0.5 %.
template <class C, class Args>
__device__ __forceinline__ bool wave_is_idle(const Args &p, int m0, int n0) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  return m0 + wave / C::WAVES_N * C::WM >= p.M || n0 + wave % C::WAVES_N * C::WN >= p.N;
}

// Whether the factor 64 may go into this wave's row scales: neither does 64 s_row s_col overflow nor is s_row s_col subnormal.
template <class C, class Vectors>
__device__ __forceinline__ bool scales_take_64(const Vectors &tv, int wm, int wn, int lane) {
  bool all = true;
  auto look = [&](float s) {
    const float a = __builtin_fabsf(s);
    all &= (a >= 0x1p-60f && a <= 0x1p60f) || a == 0.0f;
  };
#pragma unroll
  for (int mi = 0; mi < C::MI; ++mi) look(tv.srow[wm * C::WM + mi * 32 + (lane & 31)]);
#pragma unroll
  for (int ni = 0; ni < C::NI; ++ni) look(tv.scol[wn * C::WN + ni * 32 + (lane & 31)]);
  return __all(all);
}

// The accumulators of a tile between its two MFMA phases, 64ths of the integers -> f32(integer) * (s_row * s_col) + (zs * w_red + bias),
// 32x32 block by block.  What bounds it is the issue of its instructions: a wave issues one in four cycles, one that needs the result of
// the one before in eight.  So four values go side by side, and the 64 goes into the row's scale wherever the wave's scales allow it (any
// trained layer's do; the same bits), onto each value only elsewhere.  us per forward against a 64 in the scale whatever the scales are:
// always onto each value bf16 777 x 4096 -> 22016 60.9 -> 61.7, 2048 x 8192 -> 28672 245.3 -> 247.4, by this rule 62.05 -> 62.3, 250.4 -> 251.8
// (another card).  AGPR: the accumulators are in accumulation registers, which the VALU cannot address; where a wave holds at most 128 of
// them they are ordinary registers (two instructions less per value).
template <class C, bool AGPR, class Vectors>
__device__ __forceinline__ void convert_tile(v16f (&acc)[C::MI][C::NI], const Vectors &tv, int wm, int wn, int lane, bool scaled) {
  float srow[C::MI], zsr[C::MI];
  const float factor = scaled ? 64.0f : 1.0f;
#pragma unroll
  for (int mi = 0; mi < C::MI; ++mi) {
    srow[mi] = tv.srow[wm * C::WM + mi * 32 + (lane & 31)] * factor;
    zsr[mi] = tv.zs[wm * C::WM + mi * 32 + (lane & 31)];
  }
  if constexpr (AGPR) asm volatile("s_nop 15\n\ts_nop 15");  // the last MFMA results are architecturally visible to the reads below
  if (!scaled) {
#pragma unroll
    for (int ni = 0; ni < C::NI; ++ni)
#pragma unroll
      for (int mi = 0; mi < C::MI; ++mi)
#pragma unroll
        for (int v = 0; v < 16; ++v)
          acc[mi][ni][v] = AGPR ? agpr_write(agpr_read(acc[mi][ni][v]) * 64.0f) : acc[mi][ni][v] * 64.0f;
  }
#pragma unroll
  for (int ni = 0; ni < C::NI; ++ni) {
    float scv[16], wrv[16], bsv[16];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int c = wn * C::WN + ni * 32 + acc_col(g, lane);
      const float4 sc = *reinterpret_cast<const float4 *>(tv.scol + c);
      const float4 wr = *reinterpret_cast<const float4 *>(tv.wred + c);
      const float4 bs = *reinterpret_cast<const float4 *>(tv.bias + c);
      scv[4 * g] = sc.x, scv[4 * g + 1] = sc.y, scv[4 * g + 2] = sc.z, scv[4 * g + 3] = sc.w;
      wrv[4 * g] = wr.x, wrv[4 * g + 1] = wr.y, wrv[4 * g + 2] = wr.z, wrv[4 * g + 3] = wr.w;
      bsv[4 * g] = bs.x, bsv[4 * g + 1] = bs.y, bsv[4 * g + 2] = bs.z, bsv[4 * g + 3] = bs.w;
    }
#pragma unroll
    for (int mi = 0; mi < C::MI; ++mi)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        float a[4], t[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) a[e] = AGPR ? agpr_read(acc[mi][ni][4 * g + e]) : acc[mi][ni][4 * g + e];
#pragma unroll
        for (int e = 0; e < 4; ++e) t[e] = __builtin_fmaf(zsr[mi], wrv[4 * g + e], bsv[4 * g + e]);
#pragma unroll
        for (int e = 0; e < 4; ++e) a[e] = __builtin_fmaf(a[e], srow[mi] * scv[4 * g + e], t[e]);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[mi][ni][4 * g + e] = AGPR ? agpr_write(a[e]) : a[e];
      }
  }
}

// AGPR: see convert_tile
template <class C>
constexpr bool acc_in_agpr() { return C::MI * C::NI > 8; }

template <class C, bool BF16, bool SPLITK = false, bool W4 = false, bool AGPR = acc_in_agpr<C>()>
__device__ __forceinline__ void fused6_tile(const Fused6Args &p, int tm, int tn, uint8_t *smem, int split = 0,
                                            int tile_id = 0, const SplitK *sk = nullptr) {
  using Pipe = Fp6Pipe<C, W4>;
  const int m0 = tm * C::BM, n0 = tn * C::BN;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave / C::WAVES_N, wn = wave % C::WAVES_N;
  const Fp6Layout lx = fp6_layout(p.M, p.K, p.F);
  const auto layout_w = [&] {
    if constexpr (W4) {
      return tile4_layout(p.N_total, p.K, p.F);
    } else {
      return fp6_layout(p.N_total, p.K, p.F);
    }
  };
  const auto lw = layout_w();
  const TileVectors6<C> tv(smem + fused6_vectors_offset<C, W4>());
  // thread i requests column i and row i of the vectors, raw, and widens them in place when they have landed
  static_assert(C::BM <= C::kThreads && C::BN <= C::kThreads && C::BM % 64 == 0 && C::BN % 64 == 0, "a thread per row and column");
  const int swave = __builtin_amdgcn_readfirstlane(wave);
  const bool asym = p.w_red != nullptr;  // asymmetric: meta holds (scale, zero) pairs; symmetric: one scale per row, no zero term
  tile_vector_request<C>(tv, p, m0, n0, swave);
  tile_sums_request<C>(tv, p, lx.sums_off, lw.sums_off, m0, n0, swave);
  auto widen = [&] {
    tile_vector_widen<C, BF16>(tv, p.bias != nullptr, asym, 8.0f);
    tile_sums_widen<C>(tv, p.K);
  };

  Pipe pipe;
  const int total = static_cast<int>(lx.steps);
  int k0 = 0, k1 = total;
  if constexpr (SPLITK) {
    k0 = split * sk->per;
    k1 = k0 + sk->per < total ? k0 + sk->per : total;
    pipe.init(smem, p.xbuf, lx, m0 / 64, p.wbuf, lw, (p.n_first + n0) / 64, k0, k1 - k0, 0);
  } else {
    pipe.init(smem, p.xbuf, lx, m0 / 64, p.wbuf, lw, (p.n_first + n0) / 64);
  }
  pipe.start_vectors(widen);
  if constexpr (!SPLITK) {
    // (nothing behind the drain meets another wave)
    if (wave_is_idle<C>(p, m0, n0)) {
      pipe.start_steps();
      pipe.run_idle();
      pipe.drain();
      return;
    }
  }
  const bool scaled = scales_take_64<C>(tv, wm, wn, lane);  // (here, while the first steps are on their way)
  v16f acc[C::MI][C::NI];
  // The start values are an outer sum, K = 2 of the fp32 MFMA: column term times 1 plus 1 times row term, both exact.
  {
    const bool upper = lane >= 32;
    const float once = !SPLITK || split == 0 ? 1.0f : 0.0f;  // (both terms enter once)
    float rc[C::MI], cc[C::NI];
#pragma unroll
    for (int mi = 0; mi < C::MI; ++mi) rc[mi] = upper ? tv.rowc[wm * C::WM + mi * 32 + (lane & 31)] : once;
#pragma unroll
    for (int ni = 0; ni < C::NI; ++ni) cc[ni] = upper ? once : tv.colc[wn * C::WN + ni * 32 + (lane & 31)];
#pragma unroll
    for (int ni = 0; ni < C::NI; ++ni)
#pragma unroll
      for (int mi = 0; mi < C::MI; ++mi) acc[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x2f32(cc[ni], rc[mi], v16f{}, 0, 0, 0);
  }
  pipe.start_steps();

  v4i frag[Pipe::NF];
  pipe.run_fp6(acc, frag);
  if constexpr (SPLITK) {
    pipe.drain();  // the copies past the last step have landed too: the ring is free
    if (!splitk_combine<C, false>(acc, *sk, tile_id, split, smem)) return;
    if (lx.fsteps > 0) {
      pipe.init(smem, p.xbuf, lx, m0 / 64, p.wbuf, lw, (p.n_first + n0) / 64, total, 0, static_cast<int>(lx.fsteps));
      pipe.start();
      pipe.read16(frag);
    } else {
      pipe.steps0 = pipe.steps = 0;
    }
  }

  convert_tile<C, AGPR>(acc, tv, wm, wn, lane, scaled);
  pipe.template run_f16<BF16>(acc, frag);
  pipe.drain();

  // out = storage(acc), written through a staging area in the (now idle) ring: all MI row
  // blocks of the wave are staged, then read back as whole row segments, then stored, so the LDS round trip and
  // the store issue are paid once per tile and not once per row block.  The per-column vectors are read once;
  // the fragment registers are free by now.
  using Store = BlockStore<C, uint16_t>;
  static_assert(Store::kBytes * C::MI * C::WAVES <= fused6_vectors_offset<C, W4>(), "staging ends before the vectors");
  uint8_t *stage = smem + wave * (Store::kBytes * C::MI);
  const bool vec = (p.ldo & 7) == 0 && (reinterpret_cast<uintptr_t>(p.out) & 15) == 0;
  const int nw = n0 + wn * C::WN, mw = m0 + wm * C::WM;
#pragma unroll
  for (int mi = 0; mi < C::MI; ++mi)
#pragma unroll
    for (int ni = 0; ni < C::NI; ++ni)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        Store::put_pairs(stage + mi * Store::kBytes, lane, ni, g,
                         pack2_from_f32<BF16>(acc[mi][ni][4 * g], acc[mi][ni][4 * g + 1]),
                         pack2_from_f32<BF16>(acc[mi][ni][4 * g + 2], acc[mi][ni][4 * g + 3]));
  NanWatch<BF16> nans;
  if (vec && p.M - mw >= C::WM && p.N - nw >= C::WN) {  // interior (wave-uniform): straight-line code
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    v4i piece[C::MI][Store::kIters];
#pragma unroll
    for (int mi = 0; mi < C::MI; ++mi) Store::read_block(stage + mi * Store::kBytes, lane, piece[mi]);
#pragma unroll
    for (int mi = 0; mi < C::MI; ++mi)
      Store::write_block(piece[mi], lane, p.out + int64_t(mw + mi * 32) * p.ldo + nw, p.ldo, nans);
  } else {
#pragma unroll
    for (int mi = 0; mi < C::MI; ++mi) {
      const int mb = mw + mi * 32;
      if (mb < p.M && nw < p.N)
        Store::flush(stage + mi * Store::kBytes, lane, p.out + int64_t(mb) * p.ldo + nw, p.ldo, p.M - mb, p.N - nw, vec, nans);
    }
  }
  if (nans.any()) {
    canonical_nans(stage, C::MI * Store::kBytes);
#pragma unroll 1
    for (int mi = 0; mi < C::MI; ++mi) {
      const int mb = mw + mi * 32;
      if (mb < p.M && nw < p.N)
        Store::flush(stage + mi * Store::kBytes, lane, p.out + int64_t(mb) * p.ldo + nw, p.ldo, p.M - mb, p.N - nw, vec, nans);
    }
  }
}

template <class C, bool BF16, bool W4 = false>
__global__ __launch_bounds__(C::kThreads, acc_in_agpr<C>() ? 1 : 2) void gemm_fused6_kernel(Fused6Args p, int tiles_m, int tiles_n) {
  extern __shared__ __align__(16) uint8_t smem[];
  int tm, tn;
  if (!tile_of_block<C::BM>(blockIdx.x, tiles_m, tiles_n, tm, tn)) return;
  fused6_tile<C, BF16, false, W4>(p, tm, tn, smem);
}

// K split over sk.splits workgroups per tile: block b works on tile b % grid_tiles, split b / grid_tiles.
template <class C, bool BF16>
__global__ __launch_bounds__(C::kThreads, 2) void gemm_fused6_splitk_kernel(Fused6Args p, int tiles_m, int tiles_n,
                                                                          SplitK sk) {
  extern __shared__ __align__(16) uint8_t smem[];
  int tm, tn;
  const int split = blockIdx.x / sk.grid_tiles;
  if (!tile_of_block<C::BM>(blockIdx.x - split * sk.grid_tiles, tiles_m, tiles_n, tm, tn)) return;
  fused6_tile<C, BF16, true>(p, tm, tn, smem, split, tm * tiles_n + tn, &sk);
}

// One launch, two tile shapes (see gemm_i32_split_kernel).
template <class CW, class CT, bool BF16, bool W4 = false>
__global__ __launch_bounds__(CW::kThreads) void gemm_fused6_split_kernel(Fused6Args wide, Fused6Args tail,
                                                                         SplitGrid grid) {
  static_assert(CW::kThreads == CT::kThreads && CW::BM == CT::BM, "one block size, one tile height");
  extern __shared__ __align__(16) uint8_t smem[];
  int tm, tn;
  const int kind = grid.template locate<CW::BM>(blockIdx.x, tm, tn);
  if (kind == 1) {
    fused6_tile<CW, BF16, false, W4, true>(wide, tm, tn, smem);
  } else if (kind == 2) {
    fused6_tile<CT, BF16, false, W4, true>(tail, tm, tn, smem);
  }
}

// One launch of whole rounds of 256x256 tiles and, for the columns that are left (from `first` on, in 128-column tiles), 128x128
// tiles: at most one per CU.  Both regions start at multiples of 8 workgroups.
struct RestGrid {
  int tiles_m_wide, tiles_n_wide, wide_blocks, tiles_m, tiles_n, first;
};
template <class CW, class CT, bool BF16, bool W4 = false>
__global__ __launch_bounds__(CW::kThreads) void gemm_fused6_rest_kernel(Fused6Args p, RestGrid g) {
  static_assert(CW::kThreads == CT::kThreads, "one block size");
  extern __shared__ __align__(16) uint8_t smem[];
  int tm, tn;
  const int bid = blockIdx.x;
  if (bid < g.wide_blocks) {
    if (tile_of_block<CW::BM>(bid, g.tiles_m_wide, g.tiles_n_wide, tm, tn)) fused6_tile<CW, BF16, false, W4, true>(p, tm, tn, smem);
  } else if (tile_of_block<CT::BM>(bid - g.wide_blocks, g.tiles_m, g.tiles_n, tm, tn)) {
    fused6_tile<CT, BF16, false, W4, true>(p, tm, g.first + tn, smem);
  }
}

}  // namespace quik
