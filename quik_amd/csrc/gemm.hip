// Host side of the GEMM entry points: argument checks, tile planning, launches.
// The kernels live in gemm_kernels.h.
#include <cstdint>

#include "colmap.h"
#include "gemm_gemv.h"
#ifndef GEMV_MAX_ROWS
#define GEMV_MAX_ROWS 2
#endif
#include "gemm_rows.h"
#include "gemm_kernels.h"
#include "gemm_skinny.h"
#include "gemm_plan.h"

namespace quik {
namespace {

template <class C, int MODE>
int launch_i32(const I32Args &a, hipStream_t st) {
  if (a.N <= 0) return QUIK_OK;
  int tiles_m, tiles_n;
  const int grid = grid_of<C>(a.M, a.N, tiles_m, tiles_n);
  auto kern = gemm_i32_kernel<C, MODE>;
  if (int rc = prepare(kern, C::SMEM)) return rc;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(C::kThreads), C::SMEM, st, a, tiles_m, tiles_n);
  return check_launch();
}

template <class CW, class CT, int MODE>
int launch_i32_split(const I32Args &wide, const I32Args &tail, hipStream_t st) {
  if (wide.N <= 0) return launch_i32<CT, MODE>(tail, st);
  if (tail.N <= 0) return launch_i32<CW, MODE>(wide, st);
  int tail_blocks;
  const SplitGrid grid = split_grid<CW, CT>(wide.M, wide.N, tail.N, tail_blocks);
  auto kern = gemm_i32_split_kernel<CW, CT, MODE>;
  constexpr int smem = CW::SMEM > CT::SMEM ? CW::SMEM : CT::SMEM;
  if (int rc = prepare(kern, smem)) return rc;
  hipLaunchKernelGGL(kern, dim3(grid.wide_blocks + tail_blocks), dim3(CW::kThreads), smem, st, wide, tail, grid);
  return check_launch();
}

template <class C, int MODE, bool BF16>
int launch_fused(const FusedArgs &p, hipStream_t st) {
  if (p.N <= 0) return QUIK_OK;
  int tiles_m, tiles_n;
  const int grid = grid_of<C>(p.M, p.N, tiles_m, tiles_n);
  auto kern = gemm_fused_kernel<C, MODE, BF16>;
  constexpr int smem = fused_smem<C>();
  if (int rc = prepare(kern, smem)) return rc;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(C::kThreads), smem, st, p, tiles_m, tiles_n);
  return check_launch();
}

template <class CW, class CT, int MODE, bool BF16>
int launch_fused_split(const FusedArgs &wide, const FusedArgs &tail, hipStream_t st) {
  if (wide.N <= 0) return launch_fused<CT, MODE, BF16>(tail, st);
  if (tail.N <= 0) return launch_fused<CW, MODE, BF16>(wide, st);
  int tail_blocks;
  const SplitGrid grid = split_grid<CW, CT>(wide.M, wide.N, tail.N, tail_blocks);
  auto kern = gemm_fused_split_kernel<CW, CT, MODE, BF16>;
  constexpr int smem = fused_smem<CW>() > fused_smem<CT>() ? fused_smem<CW>() : fused_smem<CT>();
  if (int rc = prepare(kern, smem)) return rc;
  hipLaunchKernelGGL(kern, dim3(grid.wide_blocks + tail_blocks), dim3(CW::kThreads), smem, st, wide, tail, grid);
  return check_launch();
}

// M <= 32: the weight-streaming kernel of gemm_skinny.h.  The columns go to the CUs in equal shares, in as few rounds as the
// registers allow: seven blocks of 16 columns with one block of token rows, four with two.  (28672 columns in rounds of 56
// instead of one of 112: int4 8192 -> 28672, 4 rows, 22.7 against 22.0 us; 20480 in two of 40, 7168 deep, 17.5 against 15.7.)
template <class C, int MODE, bool BF16, bool FUSED>
int launch_skinny_cfg(const FusedArgs &p, int bn, int32_t *C_, int ldc, hipStream_t st) {
  auto kern = gemm_skinny_kernel<C, MODE, BF16, FUSED>;
  if (int rc = prepare(kern, C::smem(16 * C::MT, FUSED))) return rc;
  hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>((p.N + bn - 1) / bn)), dim3(C::kThreads), C::smem(p.M, FUSED), st, p, bn, C_, ldc);
  return check_launch();
}
// Register turns in flight: three of one block are as fast as two or faster (int4 11008 -> 4096, 4 rows, 5.5 against 5.8 us),
// three of two blocks slower (int8 13824 -> 5120, 16 rows, 14.2 against 13.8), two of four blocks slower than one (int4 8192 ->
// 28672, 32 rows, 29.2 against 26.4).
template <int MT, int MODE, bool BF16, bool FUSED>
int launch_skinny_rows(const FusedArgs &p, int32_t *C, int ldc, hipStream_t st) {
  constexpr int64_t kMost = MT == 1 ? 112 : 64;
  const int64_t cus = num_cus(), longest = p.kbytes > int64_t(p.F) * 2 ? p.kbytes : int64_t(p.F) * 2;
  int64_t most = (int64_t(1) << 32) / longest / 4 * 4 - 4;  // (32-bit offsets inside a workgroup)
  most = most < 4 ? 4 : most > kMost ? kMost : most;
  const int64_t rounds = (p.N + most * cus - 1) / (most * cus), share = (p.N + rounds * cus - 1) / (rounds * cus);
  const int bn = static_cast<int>((share + 3) / 4 * 4);  // (whole 8-byte pieces of the output rows)
  if constexpr (MT == 1 && !FUSED) {
    // Integer products, whose waves request nothing else: many columns of few rows in two rounds of at most 64 instead of one, and
    // longer rows with three turns of two blocks in flight.  us, weights from memory / in the Infinity Cache, otherwise and so:
    // int4 2 x 8192 -> 28672 27.0 / 19.2, 24.9 / 18.7; 8 x 8192 -> 20480 20.8 / 15.0, 19.1 / 15.2; int8 8 x 8192 -> 28672 46.3 / 37.6, 44.6 /
    // 36.5 (16 rows: int4 8192 -> 28672 27.7 / 19.4, 28.0 / 20.7); int8 2 x 28672 -> 8192 47.7 / 34.1, 43.1 / 34.1, 16 x 20480 -> 6144 27.8 /
    // 20.4, 26.3 / 20.3, 8 x 16384 -> 8192 32.3 / 27.1, 31.2 / 25.5 (but 8 x 14336 -> 8192 21.6 / 18.1, 22.0 / 18.3).
    if (rounds == 1 && bn > 64 && p.M <= 8)
      return launch_skinny_cfg<SkinnyCfg<4, MT, 1>, MODE, BF16, FUSED>(p, (bn / 2 + 3) / 4 * 4, C, ldc, st);
    if (bn > 16 && bn <= 32 && p.kbytes >= 16384) return launch_skinny_cfg<SkinnyCfg<2, MT, 3>, MODE, BF16, FUSED>(p, bn, C, ldc, st);
  }
  if (bn <= 16) return launch_skinny_cfg<SkinnyCfg<1, MT, 3>, MODE, BF16, FUSED>(p, bn, C, ldc, st);
  if (bn <= 32) return launch_skinny_cfg<SkinnyCfg<2, MT, 2>, MODE, BF16, FUSED>(p, bn, C, ldc, st);
  if (bn <= 48) return launch_skinny_cfg<SkinnyCfg<3, MT, 2>, MODE, BF16, FUSED>(p, bn, C, ldc, st);
  if (bn <= 64) return launch_skinny_cfg<SkinnyCfg<4, MT, 1>, MODE, BF16, FUSED>(p, bn, C, ldc, st);
  if constexpr (MT == 1) {
    if (bn <= 96) return launch_skinny_cfg<SkinnyCfg<6, MT, 1>, MODE, BF16, FUSED>(p, bn, C, ldc, st);
    return launch_skinny_cfg<SkinnyCfg<7, MT, 1>, MODE, BF16, FUSED>(p, bn, C, ldc, st);
  }
  return QUIK_ERR_SHAPE;  // (not reached: bn is at most kMost)
}
template <int MODE, bool BF16, bool FUSED>
int launch_skinny(const FusedArgs &p, int32_t *C, int ldc, hipStream_t st) {
  const int64_t longest = p.kbytes > int64_t(p.F) * 2 ? p.kbytes : int64_t(p.F) * 2;
  if (p.M * longest > 0xffffffffll) {  // (32-bit offsets of the token rows: as many of them per launch as these reach)
    const int some = static_cast<int>(0xffffffffll / longest);
    for (int m = 0; m < p.M; m += some) {
      FusedArgs q = p;
      q.M = p.M - m < some ? p.M - m : some;
      q.qx += int64_t(m) * p.kbytes;
      if constexpr (FUSED) {
        q.meta += int64_t(m) * p.meta_stride;
        q.fp_x = p.F > 0 ? q.fp_x + int64_t(m) * p.F : nullptr;
        q.out += int64_t(m) * p.ldo;
      }
      const int rc = launch_skinny<MODE, BF16, FUSED>(q, FUSED ? nullptr : C + int64_t(m) * ldc, ldc, st);
      if (rc != QUIK_OK) return rc;
    }
    return QUIK_OK;
  }
  return p.M <= 16 ? launch_skinny_rows<1, MODE, BF16, FUSED>(p, C, ldc, st) : launch_skinny_rows<2, MODE, BF16, FUSED>(p, C, ldc, st);
}

// At most kGemvMaxRows token rows (fused form): one wave per output column, gemm_gemv.h.  Needs 16-byte aligned rows
// of both weight arrays and room in LDS for the token rows.
constexpr int kGemvMaxRows = GEMV_MAX_ROWS;
bool gemv_ok(const FusedArgs &p, bool quant = false) {
  const auto aligned = [](const void *q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
  const int mt = p.M <= 1 ? 1 : p.M <= 2 ? 2 : 4;
  return p.M >= 1 && p.M <= kGemvMaxRows && p.kbytes >= 16 && p.kbytes % 16 == 0 && p.F % 8 == 0 &&
         (quant || aligned(p.qx)) && aligned(p.qw) && (p.F == 0 || ((quant || aligned(p.fp_x)) && aligned(p.fp_w))) &&
         gemv_smem(mt, p.kbytes, p.F) + gemv_table_bytes((p.N + kGemvWaves * num_cus() - 1) / (kGemvWaves * num_cus())) <=
             kLdsBytes;
}
template <int MODE, bool BF16, int MT, int QUANT>
int launch_gemv_mt(const FusedArgs &p, const GemvQuant &q, hipStream_t st) {
  // persistent waves, one column at a time each: two workgroups per CU when their LDS fits twice.  But one where each wave then has
  // at most two columns of rows that are quantised here: two workgroups quantise them twice on their CU.  us per forward, two / one:
  // one row, int4 2048 -> 4096 6.8 / 5.8, 4096 -> 4096 7.4 / 6.6, 11008 -> 4096 10.2 / 9.3, 16384 -> 4096 12.3 / 11.3, int8 4096 -> 4096 8.2 /
  // 7.5, 6144 -> 4096 8.9 / 8.5, but with longer int8 rows the stream counts for more, from memory 8192 -> 4096 11.3 / 11.3, 11008 -> 4096
  // 13.5 / 14.2, 13824 -> 4096 13.8 / 14.7; two rows 1472 -> 3200 8.6 / 7.2, 1024 -> 4096 8.4 / 7.2, int8 1536 -> 4096 8.7 / 7.8.  (One
  // workgroup for up to four columns of a wave: 8192 -> 8192 10.5 / 10.4, but 13824 -> 5120 11.2 / 11.8.)
  const int64_t fixed = gemv_smem(MT, p.kbytes, p.F) + (QUANT != kGemvNoQuant ? gemv_quant_lds(q.cols, q.num_int).bytes : 0);
  const bool short_rows = MODE == kInt4 || p.kbytes <= 6400;
  const bool quantise_bound = QUANT != kGemvNoQuant && (MT == 2 || short_rows) && p.N <= 2 * kGemvWaves * num_cus();
  const int64_t per_cu = 2 * (fixed + 4096) <= kLdsBytes && !quantise_bound ? 2 : 1;
  int64_t grid = (p.N + kGemvWaves - 1) / kGemvWaves;
  if (grid > per_cu * num_cus()) grid = per_cu * num_cus();
  const int64_t smem = fixed + gemv_table_bytes((p.N + kGemvWaves * grid - 1) / (kGemvWaves * grid));
  if (smem > kLdsBytes) return kChainNotHandled;
  auto launch = [&](auto kern) {
    if (int rc = prepare(kern, kLdsBytes)) return rc;  // (the size varies with the layer: set once to the most)
    hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(grid)), dim3(kGemvWaves * 64), static_cast<size_t>(smem), st, p, q);
    return check_launch();
  };
  if constexpr (QUANT != kGemvNoQuant) {
    if (quantise_bound) return launch(gemv_decode_kernel<MODE, BF16, MT, QUANT, true>);
  }
  return launch(gemv_decode_kernel<MODE, BF16, MT, QUANT>);
}
template <int MODE, bool BF16, int QUANT = kGemvNoQuant>
int launch_gemv(const FusedArgs &p, const GemvQuant &q, hipStream_t st) {
  if (p.M <= 1) return launch_gemv_mt<MODE, BF16, 1, QUANT>(p, q, st);
  if constexpr (kGemvMaxRows > 2) {  // (only built when the row limit is raised: gemv_ok() admits no such call otherwise)
    if (p.M > 2) return launch_gemv_mt<MODE, BF16, 4, QUANT>(p, q, st);
  }
  return launch_gemv_mt<MODE, BF16, 2, QUANT>(p, q, st);
}

template <int MODE, bool BF16, bool FUSED>
int launch_decode(const FusedArgs &p, int32_t *C, int ldc, hipStream_t st) {
  if constexpr (FUSED) {
    // One row.  Two are faster on the kernel below, 4096 -> 11008 int4 11.4 -> 9.7 us per forward, 2176 -> 15032 int8 13.2 -> 10.9,
    // 13824 -> 5120 int8 19.4 -> 18.0, unless the rows are long int4 ones: 11008 -> 4096 10.6 -> 9.7, 13824 -> 5120 13.2 -> 13.4,
    // 14272 -> 9816 18.6 -> 19.6.  (The same bits on either.)
    const bool two_here = MODE == kInt4 && p.kbytes > 6400;
    if ((p.M <= 1 || two_here) && gemv_ok(p)) {
      const int rc = launch_gemv<MODE, BF16>(p, GemvQuant{}, st);
      if (rc != kChainNotHandled) return rc;
    }
  }
  return launch_skinny<MODE, BF16, FUSED>(p, C, ldc, st);
}

Plan make_plan(int64_t M, int64_t N, bool dma_ok) {
  if (M <= 32) return {Plan::kSmall, 0};
  const int64_t tiles_m = (M + 255) / 256;
  auto rounds = [](int64_t tiles) { return (tiles + num_cus() - 1) / num_cus(); };
  if (!dma_ok) {
    // a round of 128x128 tiles, two per CU, takes 0.64 of a round of 256x256 ones (int4 2048 x 4096 x 3904, one round each:
    // 45 against 66 us; 4096 x 4096 x 10720, two against one: 190 / 168)
    const int64_t large = rounds(tiles_m * ((N + 255) / 256)) * 100, pairs = (((M + 127) / 128) * ((N + 127) / 128) + 1) / 2;
    return {M <= 128 || rounds(pairs) * 64 < large ? Plan::kMidPlain : Plan::kLargePlain, 0};
  }
  const int64_t mid = rounds(((M + 127) / 128) * ((N + 127) / 128)) * kCostMid;
  int64_t best = INT64_MAX, best_n = 0;
  for (int64_t n_wide = 0; n_wide <= N; n_wide += 256) {
    const int64_t c = makespan(tiles_m * (n_wide / 256), tiles_m * ((N - n_wide + 127) / 128));
    if (c <= best) {
      best = c;
      best_n = n_wide;
    }
  }
  if (M <= 128 || mid < best) {
    // with few 128x128 tiles most CUs would idle: 128x64 tiles put twice as many to work
    // (measured: 15-20 % less time up to about 130 tiles, no gain at 224)
    const int64_t mid_tiles = ((M + 127) / 128) * ((N + 127) / 128);
    return {mid_tiles <= 160 ? Plan::kNarrow : Plan::kMid, 0};
  }
  return {Plan::kSplit, best_n};
}

int check_gemm_args(const void *A, const void *B, const void *C, int64_t M, int64_t N, int64_t K, int bits) {
  if (M < 0 || N < 0 || K <= 0) return QUIK_ERR_SHAPE;
  if (M == 0 || N == 0) return QUIK_OK;
  if (!A || !B || !C) return QUIK_ERR_NULL;
  if (bits == 4 ? (K % 32 != 0) : (K % 16 != 0)) return QUIK_ERR_ALIGN;
  auto misaligned = [](const void *p) { return reinterpret_cast<uintptr_t>(p) % 16 != 0; };
  if (misaligned(A) || misaligned(B)) return QUIK_ERR_ALIGN;
  if (M > (1 << 30) || N > (1 << 30) || K > (int64_t(1) << 30)) return QUIK_ERR_RANGE;
  if (bits == 4 && K >= 131072) return QUIK_ERR_RANGE;
  return QUIK_OK;
}

// Which row-streaming tile (gemm_rows.h) serves a product, as its number of 32-row blocks; 0: the ring or plain kernels.
//   one round of 64x64 tiles: always (256 x 4096 x 4096 13.7 -> 8.3 us int4, 18.2 -> 9.9 int8; 122 x 2312 x 1344 int4 11.6 -> 5.0);
//   one round of 128x64 tiles, K long enough for their exchange, 2 us more than the ring kernels' epilogue (512 x 4096 x 3968
//   int4 14.7 -> 13.5, int8 16.9 -> 14.9; 2048 x 1024 x 7936 24.8 -> 19.7 and 29.7 -> 24.7; 300 x 4544 x 4352 14.8 -> 12.9; 128 x
//   13824 x 4864 16.4 -> 13.6; but 512 x 4096 x 1024 int4 6.9 -> 7.2, 512 x 4096 x 2048 int8 10.9 -> 11.6);
//   two rounds of 64x64 tiles, few rows and long K, where the weights come from memory and the ring kernels wait for them
//   (64 x 28672 x 7936 int4 41.1 -> 31.8, int8 61.4 -> 51.5; 64 x 28672 x 2048 int4 12.2 -> 11.5, int8 13.6 -> 16.0);
//   rows that are no multiple of 64 bytes, which leave only the plain kernels otherwise: up to four rounds (155 x 5120 x 13792
//   int4 75 -> 18, int8 178 -> 37; 680 x 4096 x 10944 int4 61.6 -> 43.7; 300 x 11008 x 3904 34 -> 27; 2048 x 4096 x 3904, eight
//   rounds, 53.6 against 45 of the plain 128x128 tiles).
int rows_blocks(int64_t M, int64_t N, int64_t kbytes, int mode) {
  if (M <= 32 || kbytes > (1 << 24)) return 0;  // (32-bit offsets inside a tile)
  const int64_t tiles_n = (N + 63) / 64, tiles2 = (M + 63) / 64 * tiles_n, tiles4 = (M + 127) / 128 * tiles_n, cus = num_cus();
  const bool ragged = kbytes % 64 != 0, long_k = kbytes >= (mode == kInt4 ? 1024 : 3072);
  if (tiles2 <= cus) return 2;
  if (tiles4 <= cus && (long_k || ragged)) return 4;
  if (ragged) return tiles2 <= 4 * cus ? 2 : 0;
  return M <= 256 && long_k && tiles2 <= 2 * cus ? 2 : 0;
}
// 128x64 tiles on the ring kernels: int8 with one tile per CU takes the ring of eight stages, which covers the memory's
// latency (512 x 4096 x 3968 19.4 -> 16.5 us, 2048 x 1024 x 7936 33.9 -> 28.6); int4 steps are bound by their unpacking
// (14.6 against 14.2), and a second workgroup per CU is worth more than the depth (int8 1024 x 4096 x 3840 27.7 / 29.8).
bool deep_ring(int64_t M, int64_t N, int mode) {
  return mode == kInt8 && (M + 127) / 128 * ((N + 63) / 64) <= num_cus();
}

template <class R, int MODE>
int launch_i32_rows(const I32Args &a, hipStream_t st) {
  int tiles_m, tiles_n;
  const int grid = grid_of<R>(a.M, a.N, tiles_m, tiles_n);
  auto kern = gemm_i32_rows_kernel<R, MODE>;
  if (int rc = prepare(kern, R::SMEM)) return rc;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(R::kThreads), R::SMEM, st, a, tiles_m, tiles_n);
  return check_launch();
}
template <class R, int MODE, bool ASYM>
int launch_chain_rows(const I32Args &a, const ChainArgs &e, hipStream_t st) {
  int tiles_m, tiles_n;
  const int grid = grid_of<R>(a.M, a.N, tiles_m, tiles_n);
  auto kern = gemm_chain_rows_kernel<R, MODE, ASYM>;
  if (int rc = prepare(kern, chain_rows_smem<R>())) return rc;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(R::kThreads), chain_rows_smem<R>(), st, a, e, tiles_m, tiles_n);
  return check_launch();
}

template <int MODE>
int run_i32(const uint8_t *X, const uint8_t *W, int32_t *C, int64_t M, int64_t N, int64_t kbytes, hipStream_t st) {
  I32Args a{X, W, C, static_cast<int>(M), static_cast<int>(N), static_cast<int>(N), static_cast<int>(kbytes)};
  const Plan plan = make_plan(M, N, kbytes % 64 == 0);
  switch (rows_blocks(M, N, kbytes, MODE)) {
    case 2: return launch_i32_rows<RowsCfg<2>, MODE>(a, st);
    case 4: return launch_i32_rows<RowsCfg<4>, MODE>(a, st);
    default: break;
  }
  switch (plan.kind) {
    case Plan::kSmall: {
      FusedArgs p{};
      p.qx = X;
      p.qw = W;
      p.M = a.M;
      p.N = a.N;
      p.kbytes = a.kbytes;
      return launch_decode<MODE, false, false>(p, C, a.ldc, st);
    }
    case Plan::kMid: return launch_i32<CfgM, MODE>(a, st);
    case Plan::kNarrow:
      if constexpr (MODE == kInt8) {
        if (deep_ring(M, N, MODE)) return launch_i32<CfgDN, MODE>(a, st);
      }
      return launch_i32<CfgN, MODE>(a, st);
    case Plan::kMidPlain: return launch_i32<CfgMp, MODE>(a, st);
    case Plan::kLargePlain: return launch_i32<CfgLp, MODE>(a, st);
    default: break;
  }
  I32Args wide = a, tail = a;
  wide.N = static_cast<int>(plan.n_wide);
  tail.N = static_cast<int>(N - plan.n_wide);
  tail.W = W + plan.n_wide * kbytes;
  tail.C = C + plan.n_wide;
  return launch_i32_split<CfgL, CfgH, MODE>(wide, tail, st);
}

template <class C, int MODE, bool ASYM>
int launch_chain(const I32Args &a, const ChainArgs &e, hipStream_t st) {
  int tiles_m, tiles_n;
  const int grid = grid_of<C>(a.M, a.N, tiles_m, tiles_n);
  auto kern = gemm_chain_kernel<C, MODE, ASYM>;
  if (int rc = prepare(kern, C::SMEM)) return rc;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(C::kThreads), C::SMEM, st, a, e, tiles_m, tiles_n);
  return check_launch();
}

template <class CW, class CT, int MODE, bool ASYM>
int launch_chain_split(const I32Args &a, const ChainArgs &e, int64_t n_wide, hipStream_t st) {
  if (n_wide <= 0) return launch_chain<CT, MODE, ASYM>(a, e, st);
  if (n_wide >= a.N) return launch_chain<CW, MODE, ASYM>(a, e, st);
  I32Args wide = a, tail = a;
  ChainArgs etail = e;
  wide.N = static_cast<int>(n_wide);
  tail.N = static_cast<int>(a.N - n_wide);
  tail.W = a.W + n_wide * a.kbytes;
  etail.s_col = e.s_col + n_wide;
  etail.w_red = e.w_red ? e.w_red + n_wide : nullptr;
  etail.y = e.y + n_wide;
  etail.out = e.out + n_wide;
  int tail_blocks;
  const SplitGrid grid = split_grid<CW, CT>(a.M, wide.N, tail.N, tail_blocks);
  auto kern = gemm_chain_split_kernel<CW, CT, MODE, ASYM>;
  constexpr int smem = CW::SMEM > CT::SMEM ? CW::SMEM : CT::SMEM;
  if (int rc = prepare(kern, smem)) return rc;
  hipLaunchKernelGGL(kern, dim3(grid.wide_blocks + tail_blocks), dim3(CW::kThreads), smem, st, wide, tail, e, etail, grid);
  return check_launch();
}

// Fused dequantize of at most 32 rows: one round of row-streaming tiles can take the call.  Rows of more than 11 KB leave a
// tile's waves too long a chain (two launches / tiles, us in a graph: int8 16 x 13824 -> 5120 14.8 / 18.1, 16 x 28672 -> 8192 35.9 / 36.5),
// up to four tiles are too few for long rows (int4 16 x 8192 -> 256 6.0 / 9.4).
bool few_rows_on_tiles(int64_t M, int64_t N, int64_t kbytes) {
  return M <= 32 && N > 256 && (N + 63) / 64 <= num_cus() && kbytes <= 11 * 1024;
}
// .. but product (gemm_skinny.h) and epilogue in two launches are faster.  The tiles multiply 64 rows whatever M is and keep N / 64
// CUs busy, so their time grows with K alone; the product has every CU stream its share of the columns.  us per call in a graph /
// launched one by one (the second launch starts later then: no call of two takes less than 8.3 us), two launches, tiles:
//   int4, K = 8192   1024 columns, 16 rows 6.4 / 8.7, 9.4 / 9.7; 32 rows 7.7 / 8.6, 9.4 / 9.7; 8192 columns, 16 rows 8.3 / 8.6, 10.0 / 9.8,
//                    32 rows 10.2 / 10.3, 10.1 / 9.8; 11008 columns, 8 rows 11.6 / 11.7, 10.9 / 10.7
//   int4, K = 22016  1024 columns, 32 rows 11.8 / 12.1, 18.2 / 18.7; 4096 columns, 32 rows 14.3 / 14.2, 18.8 / 18.7
//   int4, K = 16384  4096 columns, 16 rows 8.6 / 8.7, 15.1 / 14.9; 8192 columns, 16 rows 17.9 / 17.6, 15.6 / 15.2
//   int8, K = 8192   1024 columns, 16 rows 6.8 / 9.1, 11.0 / 11.1; 4096 columns, 32 rows 9.8 / 10.0, 12.3 / 11.6
//   int8, K = 5632   4096 columns, 8 rows 5.9 / 8.9, 9.1 / 9.2; 2048 columns, 16 rows 6.1 / 9.5, 9.0 / 9.2
// Shorter rows are faster in two launches only where they are replayed (int4, K = 4096, 16 rows, 1024 columns 5.2 / 8.7, 6.9 / 7.0): they
// stay on the tiles, as do calls of more than 4096 columns, whose shares outgrow one turn of registers, but for int4 rows of 4 to 5 KB.
bool few_rows_two_launches(int64_t M, int64_t N, int64_t kbytes, int mode) {
  if (N <= 16 * num_cus()) return kbytes >= (mode == kInt4 ? 4096 : M <= 8 ? 5120 : 7168);
  return mode == kInt4 && kbytes >= 4096 && kbytes < 5120 && N <= 32 * num_cus() && M <= 16;
}

// two_launches: the caller has a workspace for the product
template <int MODE, bool ASYM>
int run_chain(const I32Args &a, const ChainArgs &e, bool two_launches, hipStream_t st) {
  if (few_rows_on_tiles(a.M, a.N, a.kbytes) && !(two_launches && few_rows_two_launches(a.M, a.N, a.kbytes, MODE)))
    return launch_chain_rows<RowsCfg<2>, MODE, ASYM>(a, e, st);
  switch (rows_blocks(a.M, a.N, a.kbytes, MODE)) {
    case 2: return launch_chain_rows<RowsCfg<2>, MODE, ASYM>(a, e, st);
    case 4: return launch_chain_rows<RowsCfg<4>, MODE, ASYM>(a, e, st);
    default: break;
  }
  const Plan plan = make_plan(a.M, a.N, a.kbytes % 64 == 0);
  switch (plan.kind) {
    case Plan::kSmall: return kChainNotHandled;  // at most 32 rows: the weight-streaming kernel has no such epilogue
    case Plan::kMid: return launch_chain<CfgM, MODE, ASYM>(a, e, st);
    case Plan::kNarrow:
      if constexpr (MODE == kInt8) {
        if (deep_ring(a.M, a.N, MODE)) return launch_chain<CfgDN, MODE, ASYM>(a, e, st);
      }
      return launch_chain<CfgN, MODE, ASYM>(a, e, st);
    case Plan::kMidPlain:
    case Plan::kLargePlain: return launch_chain<CfgMp, MODE, ASYM>(a, e, st);
    default: break;
  }
  // The epilogue is exposed where one workgroup has the CU to itself: with few int4 k-steps two 128x128 tiles per CU hide
  // more of it than the large tiles gain (777 x 5120 x 4864 33.5 against 36.6 us, 2048 x 11008 x 3840 92.7 / 97.1; at
  // 2048 x 8192 x 7936 119 against 110).  (256x256 tiles alone: 65.5, 121 and 110 us.)
  if (MODE == kInt4 && a.kbytes <= 2560) return launch_chain<CfgM, MODE, ASYM>(a, e, st);
  return launch_chain_split<CfgL, CfgH, MODE, ASYM>(a, e, plan.n_wide, st);
}

template <int MODE, bool BF16>
int run_fused(const FusedArgs &p, hipStream_t st) {
  const Plan plan = make_plan(p.M, p.N, p.kbytes % 64 == 0 && (p.F * 2) % 64 == 0);
  switch (plan.kind) {
    case Plan::kSmall: return launch_decode<MODE, BF16, true>(p, nullptr, 0, st);
    case Plan::kMid: return launch_fused<CfgM, MODE, BF16>(p, st);
    case Plan::kNarrow: return launch_fused<CfgN, MODE, BF16>(p, st);
    case Plan::kMidPlain: return launch_fused<CfgMp, MODE, BF16>(p, st);
    case Plan::kLargePlain: return launch_fused<CfgLp, MODE, BF16>(p, st);
    default: break;
  }
  FusedArgs wide = p, tail = p;
  const int64_t nw = plan.n_wide;
  wide.N = static_cast<int>(nw);
  tail.N = static_cast<int>(p.N - nw);
  tail.qw = p.qw + nw * p.kbytes;
  tail.s_col = p.s_col + nw;
  tail.w_red = p.w_red ? p.w_red + nw : nullptr;
  tail.bias = p.bias ? p.bias + nw : nullptr;
  tail.fp_w = p.fp_w ? p.fp_w + nw * p.F : nullptr;
  tail.out = p.out + nw;
  return launch_fused_split<CfgL, CfgH, MODE, BF16>(wide, tail, st);
}

}  // namespace

// Integer GEMM with the fp16-arithmetic epilogue of the reference's fused ops in one launch (see ChainArgs in
// gemm_kernels.h); kChainNotHandled when the call belongs to the weight-streaming kernel (at most 32 rows), which
// has no such epilogue: the caller then runs the product and the epilogue as two launches.
int int_gemm_chain(const void *A, const void *B, const void *s_row, const void *s_col, const void *zero_row,
                   const void *w_red, uint16_t shift_bits, const void *y, int64_t M, int64_t N, int64_t K, int bits,
                   void *out, bool two_launches, hipStream_t st) {
  if (int rc = check_gemm_args(A, B, out, M, N, K, bits)) return rc;
  I32Args a{static_cast<const uint8_t *>(A), static_cast<const uint8_t *>(B), nullptr, static_cast<int>(M),
            static_cast<int>(N), static_cast<int>(N), static_cast<int>(bits == 4 ? K / 2 : K)};
  ChainArgs e{static_cast<const uint16_t *>(s_row), static_cast<const uint16_t *>(s_col),
              static_cast<const uint16_t *>(zero_row), static_cast<const uint16_t *>(w_red),
              static_cast<const uint16_t *>(y), static_cast<uint16_t *>(out), static_cast<int>(N), shift_bits};
  const bool asym = zero_row != nullptr;
  if (bits == 4) return asym ? run_chain<kInt4, true>(a, e, two_launches, st) : run_chain<kInt4, false>(a, e, two_launches, st);
  return asym ? run_chain<kInt8, true>(a, e, two_launches, st) : run_chain<kInt8, false>(a, e, two_launches, st);
}
}  // namespace quik

using namespace quik;

extern "C" int64_t quik_fused_dequantize_acc_bytes(int64_t M, int64_t N, int64_t K, int bits) {
  if (M <= 0 || M > 32 || N <= 0 || K <= 0 || (bits != 4 && bits != 8)) return 0;
  const int64_t kbytes = bits == 4 ? K / 2 : K;
  return few_rows_on_tiles(M, N, kbytes) && !few_rows_two_launches(M, N, kbytes, bits == 4 ? kInt4 : kInt8) ? 0 : M * N * 4;
}

extern "C" int quik_int4_matmul(const uint8_t *A, const uint8_t *B, int32_t *C, int64_t M, int64_t N, int64_t K,
                                void *stream) {
  if (int rc = check_gemm_args(A, B, C, M, N, K, 4)) return rc;
  if (M == 0 || N == 0) return QUIK_OK;
  return run_i32<kInt4>(A, B, C, M, N, K / 2, as_stream(stream));
}

extern "C" int quik_int8_matmul(const int8_t *A, const int8_t *B, int32_t *C, int64_t M, int64_t N, int64_t K,
                                void *stream) {
  if (int rc = check_gemm_args(A, B, C, M, N, K, 8)) return rc;
  if (M == 0 || N == 0) return QUIK_OK;
  return run_i32<kInt8>(reinterpret_cast<const uint8_t *>(A), reinterpret_cast<const uint8_t *>(B), C, M, N, K,
                        as_stream(stream));
}

// One launch or two.  One row: one.  Two rows: every workgroup quantises both, one after the other in front of its products, and
// multiplies them without matrix instructions; the other kernels' second launch is cheaper (us per forward, one after the other on a
// stream, two launches / one: int4 4096 -> 4096 8.5 / 9.5, 4096 -> 11008 9.7 / 12.0, 11008 -> 4096 9.7 / 14.4, int8 13824 -> 5120
// 18.0 / 20.6, 1024 -> 16384 8.4 / 10.5), but for
//   few columns, at most one per wave of a workgroup on each CU, or twice as many of short rows, where the second launch is all
//   there is (2048 -> 2048 7.6 / 6.8, 1280 -> 1664 7.8 / 6.6, 4096 -> 1024 8.2 / 7.5, int8 2048 -> 2048 8.4 / 6.9; 1024 -> 4096
//   7.6 / 7.1, 1472 -> 3200 with 448 outlier columns 7.6 / 7.0; replayed from a graph two are as fast, 1472 -> 3200 with none 6.0 / 6.5;
//   rows too long: 2048 -> 4096 7.7 / 8.4, 8192 -> 512 8.6 / 8.8, 14272 -> 1024 9.7 / 11.0);
//   very many columns, whose stream hides the rest (8192 -> 22016 21.6 / 21.1, 8192 -> 28672 25.5 / 24.9, int8 42.8 / 40.6; but
//   14272 -> 9816 19.6 / 19.5).
bool quik::gemv_one_launch_pays(int64_t rows, int64_t cols, int64_t N) {
  const int64_t each = kGemvWaves * num_cus();
  return rows <= 1 || (N <= each && cols <= 6144) || (N <= 2 * each && cols <= 1536) || N > 10 * each;
}

// MixedQLinear forward for at most kGemvMaxRows token rows in ONE launch: the kernel of gemm_gemv.h quantises the
// rows itself (asymmetric activations, or symmetric ones when w_red is NULL: fp16 only, scale = max |x| /
// sym_divisor).  kChainNotHandled: the shape is left to the two-launch path.
int quik::gemv_forward_one_launch(const void *x, int dtype, int64_t rows, int64_t cols, const void *colmap,
                                  int64_t num_int, int64_t num_fp, int bits, const void *qw, const void *s_col,
                                  const void *w_red, const void *fp_w, const void *bias, int64_t N, void *out,
                                  float sym_divisor, hipStream_t st) {
  const bool sym = w_red == nullptr;
  // (cols % 8: rows of whole 16-byte pieces; num_int % 16: whole units.  us in a graph, two launches / here, 1 row: int4 1280 ->
  // 1664 6.6 / 5.1, 3648 -> 7144 8.7 / 8.1, 14272 -> 9816 18.6 / 15.9, int8 11200 -> 512 9.9 / 8.2)
  if (rows < 1 || rows > kGemvMaxRows || (sym && dtype != QUIK_F16) || cols % 8 != 0 || cols > kStreamMaxCols || num_int % 16 != 0 ||
      num_fp > kGemvWaves * 64 ||
      (reinterpret_cast<uintptr_t>(x) & 15) != 0 || N > (1 << 30))
    return kChainNotHandled;
  uint32_t words[4];
  if (int rc = colmap_words(colmap, cols, num_int, num_fp, st, words)) return rc == QUIK_ERR_COLMAP ? kChainNotHandled : rc;
  if (!(words[0] & kColmapStreams)) return kChainNotHandled;
  const ColmapLayout l = colmap_layout(cols, num_int, num_fp);
  const uint8_t *cm = static_cast<const uint8_t *>(colmap);
  FusedArgs p{};
  p.qw = static_cast<const uint8_t *>(qw);
  p.s_col = static_cast<const uint16_t *>(s_col);
  p.w_red = static_cast<const uint16_t *>(w_red);
  p.fp_w = static_cast<const uint16_t *>(fp_w);
  p.bias = static_cast<const uint16_t *>(bias);
  p.out = static_cast<uint16_t *>(out);
  p.M = static_cast<int>(rows);
  p.N = static_cast<int>(N);
  p.ldo = static_cast<int>(N);
  p.kbytes = static_cast<int>(bits == 4 ? num_int / 2 : num_int);
  p.F = static_cast<int>(num_fp);
  p.meta_stride = sym ? 1 : 2;
  p.shift = bits == 4 ? 8.0f : 128.0f;
  if (!gemv_ok(p, true)) return kChainNotHandled;
  GemvQuant q{};
  q.x = static_cast<const uint16_t *>(x);
  q.fp_col = reinterpret_cast<const uint16_t *>(cm + l.off_fp);
  q.grp = reinterpret_cast<const uint32_t *>(cm + l.off_grp);
  q.unit = reinterpret_cast<const uint16_t *>(cm + l.off_unit);
  q.gather_unit = reinterpret_cast<const uint16_t *>(cm + l.off_gunit);
  q.gather_cols = reinterpret_cast<const uint16_t *>(cm + l.off_gcols);
  q.cols = static_cast<int>(cols), q.num_int = static_cast<int>(num_int), q.num_fp = static_cast<int>(num_fp);
  q.ngather = static_cast<int>(words[3]);
  q.sym_divisor = sym_divisor;
  if (q.ngather > kGemvWaves * 64) return kChainNotHandled;  // (one gathered unit per thread)
  if (sym) return bits == 4 ? launch_gemv<kInt4, false, kGemvSym>(p, q, st) : launch_gemv<kInt8, false, kGemvSym>(p, q, st);
  if (bits == 4)
    return dtype == QUIK_F16 ? launch_gemv<kInt4, false, kGemvAsym>(p, q, st) : launch_gemv<kInt4, true, kGemvAsym>(p, q, st);
  return dtype == QUIK_F16 ? launch_gemv<kInt8, false, kGemvAsym>(p, q, st) : launch_gemv<kInt8, true, kGemvAsym>(p, q, st);
}

extern "C" int quik_mixed_linear_fwd(const void *qx, const void *qw, const void *meta, const void *s_col,
                                     const void *w_reduced, const void *fp_x, const void *fp_w, const void *bias,
                                     int dtype, int64_t M, int64_t N, int64_t K, int64_t F, int bits, void *out,
                                     void *stream) {
  if (bits != 4 && bits != 8) return QUIK_ERR_BITS;
  if (dtype != QUIK_F16 && dtype != QUIK_BF16) return QUIK_ERR_DTYPE;
  if (F < 0) return QUIK_ERR_SHAPE;
  if (int rc = check_gemm_args(qx, qw, out, M, N, K, bits)) return rc;
  if (M == 0 || N == 0) return QUIK_OK;
  if (!meta || !s_col) return QUIK_ERR_NULL;
  if (F > 0 && (!fp_x || !fp_w)) return QUIK_ERR_NULL;
  if (F % 8 != 0) return QUIK_ERR_ALIGN;
  if (F > 0 && (reinterpret_cast<uintptr_t>(fp_x) % 16 != 0 || reinterpret_cast<uintptr_t>(fp_w) % 16 != 0))
    return QUIK_ERR_ALIGN;
  FusedArgs p;
  p.qx = static_cast<const uint8_t *>(qx);
  p.qw = static_cast<const uint8_t *>(qw);
  p.meta = static_cast<const uint16_t *>(meta);
  p.s_col = static_cast<const uint16_t *>(s_col);
  p.w_red = static_cast<const uint16_t *>(w_reduced);
  p.fp_x = static_cast<const uint16_t *>(fp_x);
  p.fp_w = static_cast<const uint16_t *>(fp_w);
  p.bias = static_cast<const uint16_t *>(bias);
  p.out = static_cast<uint16_t *>(out);
  p.M = static_cast<int>(M);
  p.N = static_cast<int>(N);
  p.ldo = static_cast<int>(N);
  p.kbytes = static_cast<int>(bits == 4 ? K / 2 : K);
  p.F = static_cast<int>(F);
  p.meta_stride = w_reduced ? 2 : 1;
  p.shift = bits == 4 ? 8.0f : 128.0f;
  hipStream_t st = as_stream(stream);
  if (bits == 4)
    return dtype == QUIK_F16 ? run_fused<kInt4, false>(p, st) : run_fused<kInt4, true>(p, st);
  return dtype == QUIK_F16 ? run_fused<kInt8, false>(p, st) : run_fused<kInt8, true>(p, st);
}
