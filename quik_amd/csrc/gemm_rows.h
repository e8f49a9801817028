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
// One wave per SIMD: whatever else it issues stands between its MFMAs.  A copy holds the wave until the memory pipeline has
// taken its addresses, so the copies go one by one between MFMAs (128x64 tiles: of the first half, so that the next stage
// has landed when it is read), the unpacking of int4 and the LDS reads of the next stage too.  Launch in a graph, us: int4 256 x
// 4096 x 4096 13.7 (ring) -> 8.6 (copies in a burst) -> 8.3, 40 x 4096 x 3968 12.6 -> 7.6 -> 7.0, 128x64 tiles 256 x 8192 x 7936 24.1 (ring)
// -> 24.8 -> 18.9.  What is left, 128x64 tiles at 4 bits over K: 28 ns per MFMA, the sum of its 32 cycles and of six vector
// instructions and half a copy (at 8 bits 24 KB of operands in 290 ns, 83 bytes per ns and CU).  One ring shared by the four
// waves, six stages deep, each wave taking 32 bytes of every stage behind a barrier, was slower (256 x 4096 x 4096 10.2 us).
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
  // whole stages wave, wave + WAVES, ...; what is left behind the last whole stage goes straight into registers, 32 bytes
  // per wave and zeros past the end, and is multiplied last
  const int stages = kbytes / R::BKB, rest = kbytes - stages * R::BKB;
  const int mine = stages > wave ? (stages - wave + WAVES - 1) / WAVES : 0;
  const int h = lane >> 5;
  v4i rest_f[NF];
#pragma unroll
  for (int j = 0; j < NF; ++j) rest_f[j] = v4i{0, 0, 0, 0};
  if (rest > 32 * wave + 16 * h) {
#pragma unroll
    for (int j = 0; j < NF; ++j) {
      const int row = (j < MI ? j : j - MI) * 32 + (lane & 31), rows = j < MI ? rows_x : rows_w;
      rest_f[j] = *reinterpret_cast<const v4i *>((j < MI ? X : W) + static_cast<uint32_t>(row < rows ? row : rows - 1) * static_cast<uint32_t>(kbytes) +
                                                 stages * R::BKB + 32 * wave + 16 * h);
    }
  }
  auto issue_one = [&](int i, auto J) QUIK_INLINE {
    constexpr int j = J;
    dma_load16((j < 4 * MI ? X : W) + (i * WAVES + wave) * R::BKB, voff[j], lds0 + (i & (NS - 1)) * R::STAGE + j * 1024);
  };
  auto issue = [&](int i) QUIK_INLINE { static_for<R::kLoads>([&](auto J) QUIK_INLINE { issue_one(i, J); }); };
  v4i raw[NS][KS][NF];  // [parity][sub-step][row blocks of X, of W]
  const int r_off = (lane & 31) * R::BKB, swz = lane & 7;
  auto read_one = [&](auto P, int i, auto S, auto J) QUIK_INLINE {
    const uint8_t *slot = ring + (i & (NS - 1)) * R::STAGE + r_off;
    raw[P][S][J] = *reinterpret_cast<const v4i *>(slot + (((2 * S + h) ^ swz) << 4) + J * 32 * R::BKB);
  };
  auto read = [&](auto P, int i) QUIK_INLINE {
    static_for<KS>([&](auto S) QUIK_INLINE { static_for<NF>([&](auto J) QUIK_INLINE { read_one(P, i, S, J); }); });
  };
  v16i acc[MI][2];
#pragma unroll
  for (int mi = 0; mi < MI; ++mi)
#pragma unroll
    for (int ni = 0; ni < 2; ++ni)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[mi][ni][v] = 0;
  // The products of stage i (in raw[P]), one MFMA at a time with what else the wave has to issue between them: a share of the
  // next sub-step's unpacking, one copy of stage i + NS (COPY; its slot is free: the caller has waited for the reads of
  // stage i) and, in the last sub-step, the reads of stage i + 1 (READ).  A copy holds the wave until the memory pipeline
  // has taken its addresses: in one burst in front of the products they cost a stage as much as its products.
  v4i u[2][NF][H];
  auto unpack = [&](const v4i (&f)[NF], auto S, auto Q) QUIK_INLINE {  // piece Q of sub-step S
    v4i &to = u[S & 1][Q / H][Q % H];
    Ops::template unpack_part<Q % H>(f[Q / H], to);
    if constexpr (H > 1) asm volatile("" : "+v"(to));  // (stays between its MFMAs; empty statement: no hazard)
  };
  constexpr int MM = H * 2 * MI, PIECES = NF * H;
  auto mma = [&](auto S, auto T) QUIK_INLINE {
    constexpr int s = S, t = T, hh = t / (2 * MI), ni = t / MI % 2, mi = t % MI;
    Ops::mma(u[s & 1][mi][hh], u[s & 1][MI + ni][hh], acc[mi][ni]);
  };
  constexpr std::integral_constant<int, 0> kZero{};
  auto multiply = [&](auto P, int i, auto COPY, auto READ) QUIK_INLINE {
    // the copies share the MFMAs of the sub-steps in front of the reads; with one slot, where the next stage is awaited right
    // behind the products, those of the first half
    constexpr int SLOTS = (NS > 1 ? KS - 1 : KS / 2) * MM;
    static_for<PIECES>([&](auto Q) QUIK_INLINE { unpack(raw[P][0], kZero, Q); });
    __builtin_amdgcn_sched_barrier(0);
    static_for<KS>([&](auto S) QUIK_INLINE {
      if constexpr (READ && S == KS - 1) wait_copies<(COPY && NS > 1 ? R::kLoads : 0)>();
      static_for<MM>([&](auto T) QUIK_INLINE {
        constexpr int s = S, t = T, at = s * MM + t;
        mma(S, T);
        if constexpr (s + 1 < KS)
          static_for<(t + 1) * PIECES / MM - t * PIECES / MM>([&](auto Q) QUIK_INLINE {
            unpack(raw[P][s + 1], std::integral_constant<int, s + 1>{}, std::integral_constant<int, t * PIECES / MM + Q>{});
          });
        if constexpr (COPY && at < SLOTS)
          static_for<(at + 1) * R::kLoads / SLOTS - at * R::kLoads / SLOTS>(
              [&](auto J) QUIK_INLINE { issue_one(i + NS, std::integral_constant<int, at * R::kLoads / SLOTS + J>{}); });
        if constexpr (READ && s == KS - 1)
          static_for<(t + 1) * KS * NF / MM - t * KS * NF / MM>([&](auto J) QUIK_INLINE {
            constexpr int k = t * KS * NF / MM + J;
            read_one(std::integral_constant<int, (NS > 1 ? 1 - P : 0)>{}, i + 1, std::integral_constant<int, k / NF>{},
                     std::integral_constant<int, k % NF>{});
          });
        __builtin_amdgcn_sched_barrier(0);
      });
    });
  };

  // (a wait only: no hazard)
  auto in_registers = [&]() QUIK_INLINE { asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory"); };
  constexpr std::true_type kYes{};
  constexpr std::false_type kNo{};
  if (mine > 0) issue(0);
  if (NS > 1 && mine > 1) {
    issue(1);
    wait_copies<R::kLoads>();
  } else {
    wait_copies<0>();
  }
  if (mine > 0) read(kZero, 0);
  int i = 0;
  auto step = [&](auto P, auto COPY, auto READ) QUIK_INLINE {
    in_registers();
    multiply(P, i, COPY, READ);
    ++i;
  };
  constexpr std::integral_constant<int, P1> kOne{};
  if constexpr (NS == 1) {
    while (i + 1 < mine) step(kZero, kYes, kYes);
    if (i < mine) step(kZero, kNo, kNo);
  } else {
    while (i + 3 < mine) {
      step(kZero, kYes, kYes);
      step(kOne, kYes, kYes);
    }
    if (i + 2 < mine) {  // three left
      step(kZero, kYes, kYes);
      step(kOne, kNo, kYes);
      step(kZero, kNo, kNo);
    } else if (i + 1 < mine) {
      step(kZero, kNo, kYes);
      step(kOne, kNo, kNo);
    } else if (i < mine) {
      step(kZero, kNo, kNo);
    }
  }
  if (rest > 0) {
    static_for<PIECES>([&](auto Q) QUIK_INLINE { unpack(rest_f, kZero, Q); });
    static_for<MM>([&](auto T) QUIK_INLINE { mma(kZero, T); });
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

// The inputs of chain_store for a tile, copied to the LDS behind the rings in front of the main loop: scales, zero points and
// reduced weights as 16 bits in slots of four bytes, y as rows of 128 bytes whose 16-byte pieces are swapped as in the rings.
// (y only where its pieces are aligned and whole: has.)  Read at the end instead, they were a chain of trips to memory
// behind the products: us per call 256 x 4096 x 4096 int4 8.86 -> 8.24, 512 x 4096 x 4096 15.3 -> 13.7, 32 x 4096 x 11008 8.43 ->
// 7.75, int8 64 x 8192 x 1024 14.15 -> 13.53; with y unaligned (130 x 4096 x 4100) 10.78 -> 10.76.
template <class R>
struct ChainStaged {
  static constexpr int kBytes = (2 * R::BN + 2 * R::BM) * 4 + R::BM * R::BN * 2;
  uint8_t *base;
  int m0, n0;
  bool has;
  __device__ __forceinline__ uint16_t u16(int slot) const {
    return static_cast<uint16_t>(*reinterpret_cast<const uint32_t *>(base + slot * 4));
  }
  __device__ __forceinline__ uint16_t s_col(int col) const { return u16(col - n0); }
  __device__ __forceinline__ uint16_t w_red(int col) const { return u16(R::BN + col - n0); }
  __device__ __forceinline__ uint16_t s_row(int row) const { return u16(2 * R::BN + row - m0); }
  __device__ __forceinline__ uint16_t zero_row(int row) const { return u16(2 * R::BN + R::BM + row - m0); }
  __device__ __forceinline__ bool has_y() const { return has; }
  __device__ __forceinline__ uint8_t *y_rows() const { return base + (2 * R::BN + 2 * R::BM) * 4; }
  __device__ __forceinline__ void y(int row, int col, uint16_t (&v)[4]) const {
    const int r = row - m0, c = col - n0;
    const uint2 w = *reinterpret_cast<const uint2 *>(y_rows() + r * 128 + (((c >> 3) ^ (r & 7)) << 4) + (c & 4) * 2);
    v[0] = static_cast<uint16_t>(w.x), v[1] = static_cast<uint16_t>(w.x >> 16);
    v[2] = static_cast<uint16_t>(w.y), v[3] = static_cast<uint16_t>(w.y >> 16);
  }
  // (visible to the other waves behind the barriers of the main loop's exchange; every wave waits for its own copies there)
  template <bool ASYM>
  __device__ __forceinline__ void request(const ChainArgs &e, int M, int N) const {
    static_assert(R::BN == 64 && R::BM <= 64 * R::WAVES, "a wave per vector piece");
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t lds = __builtin_amdgcn_readfirstlane(lds_address(base));
    if (wave == R::WAVES - 1) {
      const uint32_t n = n0 + lane < N ? n0 + lane : N - 1;
      dma_load_u16(e.s_col, 2 * n, lds);
      if constexpr (ASYM) dma_load_u16(e.w_red, 2 * n, lds + R::BN * 4);
    }
    if (wave * 64 < R::BM) {
      const uint32_t i = wave * 64 + lane, m = m0 + static_cast<int>(i) < M ? m0 + i : M - 1;
      dma_load_u16(e.s_row, 2 * m, lds + (2 * R::BN + wave * 64) * 4);
      if constexpr (ASYM) dma_load_u16(e.zero_row, 2 * m, lds + (2 * R::BN + R::BM + wave * 64) * 4);
    }
    if (has) {
      const uint8_t *y0 = reinterpret_cast<const uint8_t *>(e.y + int64_t(m0) * e.ldy + n0);
#pragma unroll
      for (int j = 0; j < R::BM / 8 / R::WAVES; ++j) {
        const int at = (j * R::WAVES + wave) * 8, row = at + (lane >> 3);
        dma_load16(y0, static_cast<uint32_t>(m0 + row < M ? row : M - 1 - m0) * static_cast<uint32_t>(e.ldy) * 2u + (((lane & 7) ^ (lane >> 3)) << 4),
                   lds + (2 * R::BN + 2 * R::BM) * 4 + at * 128);
      }
    }
  }
};
template <class R>
constexpr int chain_rows_smem() {
  return R::SMEM + ChainStaged<R>::kBytes;
}

template <class R, int MODE, bool ASYM>
__global__ __launch_bounds__(R::kThreads) void gemm_chain_rows_kernel(I32Args a, ChainArgs e, int tiles_m, int tiles_n) {
  extern __shared__ __align__(16) uint8_t smem[];
  int tm, tn;
  if (!tile_of_block<R::BM>(blockIdx.x, tiles_m, tiles_n, tm, tn)) return;
  const int m0 = tm * R::BM, n0 = tn * R::BN;
  const ChainStaged<R> in{smem + R::SMEM, m0, n0,
                          n0 + R::BN <= a.N && (e.ldy & 7) == 0 && e.ldy < (1 << 23) && (reinterpret_cast<uintptr_t>(e.y) & 15) == 0};
  in.template request<ASYM>(e, a.M, a.N);
  v16i own[R::OWN][1];
  rows_mainloop<R, MODE>(a.X + int64_t(m0) * a.kbytes, a.M - m0, a.W + int64_t(n0) * a.kbytes, a.N - n0, a.kbytes, smem, own);
  chain_store<typename R::Tile, MODE, ASYM>(a, e, m0, n0, smem + R::RED_BYTES, own, in);
}

}  // namespace quik
