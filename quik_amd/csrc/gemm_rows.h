// Stand-alone integer GEMMs on row-major operands for problems of few tiles: every wave streams its own share of K
// through a private LDS ring.
//
// What bounds the shared rings of gemm_kernels.h on few and narrow tiles is the step: 64 bytes of K per row between two
// barriers, two to eight MFMAs per wave, a wait for copies issued two steps before (256 rows, 4096 columns, over K: 312 ns a
// step at 4 bits, 233 at 8).  Here the four waves of a workgroup split K: each computes the WHOLE 64x64 (128x64) tile
// over every fourth 128-byte stage, copies only what it multiplies itself and never meets a barrier in the main loop.  A
// copy instruction takes 8 rows of a whole cache line: with 64-byte pieces of 16 rows a CU took in 23 bytes per cycle
// instead of about 45 (int8 256 x 4096 x 4096: 13.8 .. 14.9 us against 9.9).  Two stages are in flight or in LDS and one in
// registers; 128x64 tiles have room for one and one, enough for the longer multiplication of a stage.  Afterwards the
// waves add their sums through LDS (integers: in any order), each ending up with the blocks it stores.
//
// Measured (launch in a graph, us): int4 256 x 4096 x 4096 13.7 -> 8.6 (fused dequantize 15.2 -> 9.2), 40 x 4096 x 3968
// 12.6 -> 7.4; int8 256 x 4096 x 4096 18.2 -> 9.9, 128 x 13824 x 4864 30.7 -> 22.6.  What is left (256 rows, 4096
// columns, over K): 4 .. 5 us of launch, first copies, exchange and stores, then per stage of 16 KB 174 ns at 8 bits (94
// bytes per ns and CU) and 220 .. 260 at 4 bits, where a stage is twice the products and has to be unpacked.
#pragma once
#include "gemm_kernels.h"

#define QUIK_INLINE __attribute__((always_inline))

namespace quik {

// MI: 32-row blocks of X per tile (a tile has two of W)
template <int MI_>
struct RowsCfg {
  static constexpr int MI = MI_, WAVES = 4, kThreads = 64 * WAVES, BM = 32 * MI, BN = 64;
  using Tile = Cfg<BM, BN, 2, 2, 2>;  // (wave, blocks it ends up with) and the epilogues' staging
  static constexpr int BKB = 128;     // K bytes per row and stage: a whole cache line
  static constexpr int STAGE = (BM + BN) * BKB;
  static constexpr int NS = MI == 2 ? 2 : 1, RING = NS * STAGE;  // per wave; a further stage is in registers
  static constexpr int kLoads = STAGE / 1024;                    // copies per stage
  static constexpr int OWN = MI / 2;                             // blocks a wave ends up with
  static constexpr int RED_BYTES = WAVES * OWN * (WAVES - 1) * 4096;
  static constexpr int STAGING = 32 * (32 * 4 + 16);             // per wave, behind the exchange area
  static constexpr int kExchange = RED_BYTES + WAVES * STAGING;
  static constexpr int SMEM = WAVES * RING > kExchange ? WAVES * RING : kExchange;
  static_assert(MI == 2 || MI == 4, "supported tiles");
};

template <int N>
__device__ __forceinline__ void wait_copies() {
  asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory");
}

// own: this wave's blocks (Tile: rows wave / 2, columns wave % 2) of X W^T over all of K, of the tile at X, W
template <class R, int MODE>
__device__ __forceinline__ void rows_mainloop(const uint8_t *__restrict__ X, int rows_x, const uint8_t *__restrict__ W,
                                              int rows_w, int kbytes, uint8_t *smem, v16i (&own)[R::OWN][1]) {
  using Ops = FragOps<MODE>;
  constexpr int H = Ops::H, WAVES = R::WAVES, KS = R::BKB / 32, MI = R::MI, NF = MI + 2, NS = R::NS, P1 = NS - 1;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  uint8_t *const ring = smem + wave * R::RING;
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_address(ring));
  // A copy takes 8 rows: lane -> (row, chunk of 16 bytes), chunk c of row r stored at place c ^ (r % 8), so that the
  // reads of eight consecutive rows of one chunk column fall into distinct bank groups.
  const int lrow = lane >> 3, gchunk = (lane & 7) ^ lrow;
  uint32_t voff[R::kLoads];
#pragma unroll
  for (int j = 0; j < R::kLoads; ++j) {
    const int row = (j < 4 * MI ? j : j - 4 * MI) * 8 + lrow, rows = j < 4 * MI ? rows_x : rows_w;
    voff[j] = static_cast<uint32_t>(row < rows ? row : rows - 1) * static_cast<uint32_t>(kbytes) + gchunk * 16;
  }
  // stages wave, wave + WAVES, ...; the last one may be half a stage, whose second half is never multiplied: its
  // copies take the first half twice, to stay inside the rows
  const int stages = (kbytes + R::BKB - 1) / R::BKB;
  const int mine = stages > wave ? (stages - wave + WAVES - 1) / WAVES : 0;
  const uint32_t half_off = gchunk >= 4 ? 64u : 0u;
  auto issue = [&](int i) QUIK_INLINE {
    const int kb = (i * WAVES + wave) * R::BKB;
    const uint32_t back = kb + R::BKB > kbytes ? half_off : 0u;
    const uint32_t slot = lds0 + (i & (NS - 1)) * R::STAGE;
    static_for<R::kLoads>([&](auto J) QUIK_INLINE {
      constexpr int j = J;
      dma_load16((j < 4 * MI ? X : W) + kb, voff[j] - back, slot + j * 1024);
    });
  };
  v4i raw[NS][KS][NF];  // [parity][sub-step][row blocks of X, of W]
  const int r_off = (lane & 31) * R::BKB, swz = lane & 7, h = lane >> 5;
  auto read = [&](auto P, int i) QUIK_INLINE {
    const uint8_t *slot = ring + (i & (NS - 1)) * R::STAGE + r_off;
    static_for<KS>([&](auto S) QUIK_INLINE {
      const int place = ((2 * S + h) ^ swz) << 4;
      static_for<NF>([&](auto J) QUIK_INLINE {
        raw[P][S][J] = *reinterpret_cast<const v4i *>(slot + place + J * 32 * R::BKB);
      });
    });
  };
  v16i acc[MI][2];
#pragma unroll
  for (int mi = 0; mi < MI; ++mi)
#pragma unroll
    for (int ni = 0; ni < 2; ++ni)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[mi][ni][v] = 0;
  auto multiply = [&](auto P, int i) QUIK_INLINE {
    const int live = kbytes - (i * WAVES + wave) * R::BKB;
    static_for<KS>([&](auto S) QUIK_INLINE {
      if (S >= KS / 2 && live < R::BKB) return;
      v4i ux[MI][H], uw[2][H];
#pragma unroll
      for (int j = 0; j < MI; ++j) Ops::unpack(raw[P][S][j], ux[j]);
#pragma unroll
      for (int j = 0; j < 2; ++j) Ops::unpack(raw[P][S][MI + j], uw[j]);
#pragma unroll
      for (int hh = 0; hh < H; ++hh)
#pragma unroll
        for (int ni = 0; ni < 2; ++ni)
#pragma unroll
          for (int mi = 0; mi < MI; ++mi) Ops::mma(ux[mi][hh], uw[ni][hh], acc[mi][ni]);
    });
  };

  if (mine > 0) issue(0);
  if (NS > 1 && mine > 1) {
    issue(1);
    wait_copies<R::kLoads>();
  } else {
    wait_copies<0>();
  }
  if (mine > 0) read(std::integral_constant<int, 0>{}, 0);
  auto step = [&](auto P, int i) QUIK_INLINE {
    asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");  // stage i is in registers: its slot is free
    if constexpr (NS == 1) {
      if (i + 1 < mine) issue(i + 1);
      multiply(P, i);
      __builtin_amdgcn_sched_barrier(0);  // (the wait stays behind the products)
      if (i + 1 < mine) {
        wait_copies<0>();
        read(P, i + 1);
      }
    } else {
      if (i + 1 < mine) {
        if (i + 2 < mine) {
          issue(i + 2);
          wait_copies<R::kLoads>();
        } else {
          wait_copies<0>();
        }
        read(std::integral_constant<int, 1 - P>{}, i + 1);
      }
      multiply(P, i);
    }
  };
  for (int i = 0; i < mine; i += NS) {
    step(std::integral_constant<int, 0>{}, i);
    if (NS > 1 && i + 1 < mine) step(std::integral_constant<int, P1>{}, i + 1);
  }

  // exchange: wave w leaves its sums of the blocks that wave o owns in slots (o, block, w), o adds the three it finds
  __syncthreads();
  static_for<WAVES>([&](auto O) QUIK_INLINE {
    static_for<R::OWN>([&](auto B) QUIK_INLINE {
      constexpr int o = O, q = B;
      const v16i &b = acc[(o >> 1) * R::OWN + q][o & 1];
      if (o == wave) {
        own[q][0] = b;
      } else {
        uint8_t *slot = smem + ((o * R::OWN + q) * (WAVES - 1) + (wave < o ? wave : wave - 1)) * 4096 + lane * 16;
#pragma unroll
        for (int g = 0; g < 4; ++g)
          *reinterpret_cast<v4i *>(slot + g * 1024) = v4i{b[4 * g], b[4 * g + 1], b[4 * g + 2], b[4 * g + 3]};
      }
    });
  });
  __syncthreads();
#pragma unroll
  for (int q = 0; q < R::OWN; ++q)
#pragma unroll
    for (int s = 0; s < WAVES - 1; ++s) {
      const uint8_t *slot = smem + ((wave * R::OWN + q) * (WAVES - 1) + s) * 4096 + lane * 16;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const v4i t = *reinterpret_cast<const v4i *>(slot + g * 1024);
#pragma unroll
        for (int e = 0; e < 4; ++e) own[q][0][4 * g + e] += t[e];
      }
    }
}

template <class R, int MODE>
__global__ __launch_bounds__(R::kThreads) void gemm_i32_rows_kernel(I32Args a, int tiles_m, int tiles_n) {
  extern __shared__ __align__(16) uint8_t smem[];
  int tm, tn;
  if (!tile_of_block<R::BM>(blockIdx.x, tiles_m, tiles_n, tm, tn)) return;
  const int m0 = tm * R::BM, n0 = tn * R::BN;
  v16i own[R::OWN][1];
  rows_mainloop<R, MODE>(a.X + int64_t(m0) * a.kbytes, a.M - m0, a.W + int64_t(n0) * a.kbytes, a.N - n0, a.kbytes, smem, own);
  i32_store<typename R::Tile, MODE>(a, m0, n0, smem + R::RED_BYTES, own);
}

template <class R, int MODE, bool ASYM>
__global__ __launch_bounds__(R::kThreads) void gemm_chain_rows_kernel(I32Args a, ChainArgs e, int tiles_m, int tiles_n) {
  extern __shared__ __align__(16) uint8_t smem[];
  int tm, tn;
  if (!tile_of_block<R::BM>(blockIdx.x, tiles_m, tiles_n, tm, tn)) return;
  const int m0 = tm * R::BM, n0 = tn * R::BN;
  v16i own[R::OWN][1];
  rows_mainloop<R, MODE>(a.X + int64_t(m0) * a.kbytes, a.M - m0, a.W + int64_t(n0) * a.kbytes, a.N - n0, a.kbytes, smem, own);
  chain_store<typename R::Tile, MODE, ASYM>(a, e, m0, n0, smem + R::RED_BYTES, own);
}

}  // namespace quik
