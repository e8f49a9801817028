// Host side of the int4 layer GEMM on 4-bit weights in tile order (fp6_format.h): which kernel, and with it which format the
// activation comes in.
//
// A weight takes 4 bits in memory and in the caches and becomes a field of the 6-bit MFMA operand in registers, by eight VALU
// instructions per 32 x 64 fragment.  Where a fragment meets many others that is free; where it meets few, the instructions
// are what a wave waits for.  So:
//   few and narrow tiles (gemm_direct.h): both operands in 4 bits.  The waves of a workgroup split K, each multiplies whole
//     tiles, and what a CU takes in from its L2 bounds it: two thirds of the bytes of the 6-bit format.
//   tiles of 128 x 128 and more (gemm_fp6.h, W4): the weights in 4 bits, the activation in 6.  The waves of a workgroup share
//     a tile through the LDS and each expands what it reads: the activation's fragments would cost as many instructions again
//     (2048 x 8192 -> 28672, GEMM, us: 257 with both in 4 bits, 238 with the activation in 6, 237 with both).
// GEMM launch in a graph, us, against the 6-bit weights (one copy of them / 700 MB of copies in turn): 64 x 8192 -> 10240 14.5 /
// 21.4 -> 11.3 / 15.9, 128 x 5120 -> 13824 14.8 / 19.8 -> 13.1 / 16.9, 300 x 4544 -> 4544 14.4 / 15.1 -> 10.5 / 12.8, 2048 x 8192 ->
// 1024 19.9 / 24.3 -> 16.6 / 16.4, 40 x 8192 -> 28672 30.9 / 38.6 -> 22.3 / 30.7, 256 x 13824 -> 5120 26.2 / 37.3 -> 20.5 / 26.7,
// 1024 x 8192 -> 8192 39.8 / 49.6 -> 38.3 / 44.9, 2048 x 8192 -> 28672 237 / 253 -> 238 / 245.
#include <cstdint>

#include "gemm_direct.h"
#include "gemm_plan.h"

namespace quik {
namespace {

// Steps in flight: what bounds the stream is what a CU takes in, not its latency, so no more than cover it.  us per forward with more
// and with these: 64x32 tiles, eight and four, 64 x 5120 -> 5120 10.65 / 9.95, 40 x 4096 -> 4096 9.7 / 9.35, 64 x 14336 -> 4096 15.55 / 15.1;
// 64x64 tiles, four and two, where two of them share a CU, 300 x 4096 -> 4096 14.55 / 14.15, 64 x 5120 -> 20480 19.2 / 18.35, 777 x 4096 ->
// 1280 16.2 / 15.5, and where one has it alone 64 x 8192 -> 10240 15.3 / 16.1; 128x64 tiles, four and two, of at most two rows of tiles,
// whose weights each come from beyond the L2, 128 x 5120 -> 13824 17.05 / 16.75 (22.5 / 22.1 from memory), 200 x 5120 -> 5120 15.35 / 15.3
// (19.3 / 19.15), and of more 500 x 4096 -> 2048 12.65 / 12.95, 300 x 4544 -> 4544 15.4 / 15.35 (17.7 / 18.05).
using Direct64x32 = DirectCfg<kDirect4, 2, 1, 4>;
using Direct64x64 = DirectCfg<kDirect4, 2, 2, 4>;
using Direct64x64Pairs = DirectCfg<kDirect4, 2, 2, 2>;
using Direct128x64 = DirectCfg<kDirect4, 4, 2, 4>;
using Direct128x64Few = DirectCfg<kDirect4, 4, 2, 2>;

enum class Tiles4 { k64x32, k64x64, k128x64, kRing };

// The register-streaming kernels against the ring of 128x128 tiles, below the 256-row tiles.  Picoseconds; r: tiles of the
// busiest CU, s: k-steps, outlier steps included, w: kilobytes of weights,
//   t = a + r (b s + c) + d w
// fitted to 16 row counts of 40 .. 3072 on each of 12 layer shapes (2048 -> 2048 to 13824 -> 5120), warm weights; the ring of one
// tile per CU to 130 calls, warm and cold alike; all with eight (64x32) and four steps in flight and loaded empty steps, 0.02 % behind
// the fastest of the four over 150 calls of 100 .. 1024 rows.  With the tiles above, which are up to 7 % faster, 64x32 and 64x64 ones most, the pick
// is 0.6 % behind over 145 calls (40 .. 1024 rows, 13 layer shapes, warm), more than 1 % in 14 of them, eight of those on 128x64
// tiles where 64x64 are faster: 300 x 5120 -> 5120 16.55 / 15.6 us, 200 x 4544 -> 4544 14.7 / 13.95, 300 x 4544 -> 4544 15.4 / 14.7.  Two 128x128 tiles
// share a CU: 1.9 of a single one's time.
int64_t direct_cost(Tiles4 t, int64_t M, int64_t N, int64_t s, int64_t w) {
  const int64_t cus = num_cus();
  auto tiles = [&](int64_t bm, int64_t bn) { return (M + bm - 1) / bm * ((N + bn - 1) / bn); };
  auto rounds = [](int64_t n, int64_t per) { return (n + per - 1) / per; };
  switch (t) {
    case Tiles4::k64x32: return 3620000 + rounds(tiles(64, 32), cus) * (24600 * s + 970000) + 40 * w;
    case Tiles4::k64x64: return 3420000 + rounds(tiles(64, 64), cus) * (33700 * s + 880000) + 52 * w;
    case Tiles4::k128x64: return 700000 + rounds(tiles(128, 64), cus) * (53600 * s + 5800000) + 25 * w;
    default: {
      const int64_t n = tiles(128, 128);
      if (n <= cus) return 3750000 + 106000 * s + 670000 + 20 * w;  // (the deep ring)
      return 4070000 + 19 * rounds(n, 2 * cus) * (116200 * s + 670000) / 10 + 34 * w;
    }
  }
}
Tiles4 plan_tile4(int64_t M, int64_t N, int64_t K, int64_t F) {
  if (make_plan6(M, N, 1).kind != Plan::kMid) return Tiles4::kRing;
  const Tile4Layout l = tile4_layout(N, K, F);
  Tiles4 best = Tiles4::kRing;
  int64_t least = INT64_MAX;
  for (const Tiles4 t : {Tiles4::k64x32, Tiles4::k64x64, Tiles4::k128x64, Tiles4::kRing}) {
    const int64_t c = direct_cost(t, M, N, l.steps + l.fsteps, N * (l.block_bytes / 64) / 1000);
    if (c < least) least = c, best = t;
  }
  return best;
}

// K split over `splits` workgroups per 64x32 tile (SplitK): few tiles of a long K leave most CUs idle, and with them what the
// chip can have open towards memory.  The exchange through memory costs 1.5 us and 0.3 per workgroup, against 24.6 ns for each step
// that a workgroup has less (same fit, of the tiles before), so it is taken from some 150 k-steps on.  us per forward, warm / cold weights, without and
// with the split: 64 x 14336 -> 512 15.0 / 17.8, 13.4 / 14.8 (4); 128 x 14336 -> 1024 15.5 / 20.2, 15.0 / 16.7 (4); 64 x 12288 -> 1024
// 14.0 / 18.4, 13.4 / 15.1 (3); 40 x 14336 -> 4096 15.3 / 20.9, 15.0 / 19.1 (2).  At 8192 columns it costs warm what it gives cold (64 ->
// 1024 12.0 / 14.3, 12.3 / 13.6); eight workgroups per tile, or 64x64 tiles, were nowhere the faster form.
constexpr int kMostSplits4 = 4;
int plan_splits4(int64_t M, int64_t N, int64_t K, int64_t F) {
  const int64_t steps = tile4_layout(N, K, F).steps, tiles = (M + 63) / 64 * ((N + 31) / 32);
  if (2 * tiles > num_cus() || tiles * 4 > kSplitCounterBytes || plan_tile4(M, N, K, F) != Tiles4::k64x32) return 1;
  int best = 1;
  int64_t least = steps * 24600;
  for (int splits = 2; splits <= kMostSplits4 && splits * tiles <= num_cus(); ++splits) {
    const int64_t per = (steps + splits - 1) / splits, c = 1500000 + 300000 * splits + per * 24600;
    if ((splits - 1) * per < steps && c < least) least = c, best = splits;
  }
  return best;
}
int64_t split_bytes4(int64_t M, int64_t N, int64_t K, int64_t F) {
  const int splits = plan_splits4(M, N, K, F);
  return splits == 1 ? 0 : kSplitCounterBytes + (M + 63) / 64 * ((N + 31) / 32) * splits * Direct64x32::PARTIAL_BYTES;
}

template <bool BF16>
int launch_split4(const Fused8Args &p, int splits, void *workspace, hipStream_t st) {
  using D = Direct64x32;
  int tiles_m, tiles_n;
  const int grid = grid_of<D>(p.M, p.N, tiles_m, tiles_n);
  const int steps = static_cast<int>(tile4_layout(p.M, p.K, p.F).steps);
  SplitK sk{splits, (steps + splits - 1) / splits, grid, static_cast<uint32_t *>(workspace),
            reinterpret_cast<int32_t *>(static_cast<uint8_t *>(workspace) + kSplitCounterBytes)};
  auto kern = gemm_direct_splitk_kernel<D, BF16, Fused8Args>;
  if (int rc = prepare(kern, D::SMEM)) return rc;
  hipLaunchKernelGGL(kern, dim3(grid * splits), dim3(D::kThreads), D::SMEM, st, p, tiles_m, tiles_n, sk);
  return splitk_launch_status(workspace, st);
}

template <class D, bool BF16>
int launch_direct4(const Fused8Args &p, hipStream_t st) {
  int tiles_m, tiles_n;
  const int grid = grid_of<D>(p.M, p.N, tiles_m, tiles_n);
  auto kern = gemm_direct_kernel<D, BF16, Fused8Args>;
  if (int rc = prepare(kern, D::SMEM)) return rc;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(D::kThreads), D::SMEM, st, p, tiles_m, tiles_n);
  return check_launch();
}

// the activation in 4 bits; any size (where the plan is the ring, the widest tiles: a caller that did not ask)
template <bool BF16>
int run_direct4(const Fused8Args &p, void *workspace, int64_t workspace_bytes, hipStream_t st) {
  if (workspace) {
    const int splits = plan_splits4(p.M, p.N, p.K, p.F);
    if (splits > 1 && workspace_bytes >= split_bytes4(p.M, p.N, p.K, p.F)) return launch_split4<BF16>(p, splits, workspace, st);
  }
  switch (plan_tile4(p.M, p.N, p.K, p.F)) {
    case Tiles4::k64x32: return launch_direct4<Direct64x32, BF16>(p, st);
    case Tiles4::k64x64:
      if ((p.M + 63) / 64 * ((p.N + 63) / 64) > num_cus()) return launch_direct4<Direct64x64Pairs, BF16>(p, st);
      return launch_direct4<Direct64x64, BF16>(p, st);
    default:
      if (p.M <= 256) return launch_direct4<Direct128x64Few, BF16>(p, st);
      return launch_direct4<Direct128x64, BF16>(p, st);
  }
}

template <class C, bool BF16>
int launch_ring4(const Fused6Args &p, hipStream_t st) {
  if (p.N <= 0) return QUIK_OK;
  int tiles_m, tiles_n;
  const int grid = grid_of<C>(p.M, p.N, tiles_m, tiles_n);
  auto kern = gemm_fused6_kernel<C, BF16, true>;
  constexpr int smem = fused6_smem<C, true>();
  if (int rc = prepare(kern, smem)) return rc;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(C::kThreads), smem, st, p, tiles_m, tiles_n);
  return check_launch();
}

template <class CW, class CT, bool BF16>
int launch_ring4_split(const Fused6Args &p, int64_t n_wide, hipStream_t st) {
  if (n_wide <= 0) return launch_ring4<CT, BF16>(p, st);
  Fused6Args wide = p, tail = p;
  wide.N = static_cast<int>(n_wide);
  tail.N = static_cast<int>(p.N - n_wide);
  tail.n_first = static_cast<int>(n_wide);
  tail.s_col = p.s_col + n_wide;
  tail.w_red = p.w_red ? p.w_red + n_wide : nullptr;
  tail.bias = p.bias ? p.bias + n_wide : nullptr;
  tail.out = p.out + n_wide;
  int tail_blocks;
  SplitGrid grid = split_grid<CW, CT>(wide.M, wide.N, tail.N, tail_blocks);
  grid.lead = 0;  // tiles of an XCD that share operand rows stay in step (L2 hits)
  auto kern = gemm_fused6_split_kernel<CW, CT, BF16, true>;
  constexpr int sw = fused6_smem<CW, true>(), stail = fused6_smem<CT, true>(), smem = sw > stail ? sw : stail;
  if (int rc = prepare(kern, smem)) return rc;
  hipLaunchKernelGGL(kern, dim3(grid.wide_blocks + tail_blocks), dim3(CW::kThreads), smem, st, wide, tail, grid);
  return check_launch();
}

// the activation in 6 bits; any size.  The plan is the 6-bit path's, whose tiles these are.
template <bool BF16>
int run_ring4(const Fused6Args &p, hipStream_t st) {
  const Plan plan = make_plan6(p.M, p.N, 1);
  if (const int64_t n_wide = plan_rest(p.M, p.N, plan); n_wide > 0)
    return launch_rest<CfgL, CfgM>(gemm_fused6_rest_kernel<CfgL, CfgM, BF16, true>, fused6_smem<CfgL, true>(), p, n_wide, st);
  if (plan.kind != Plan::kSplit) {
    // One tile per CU: twelve slots, 90 KB in flight instead of 30.  us per forward, warm / cold weights: 300 x 8192 -> 8192 26.8 /
    // 33.6 -> 26.7 / 30.8, 777 x 11008 -> 4096 38.9 / 44.0 -> 38.2 / 40.5, 400 x 5120 -> 5120 21.6 / 25.9 -> 21.7 / 24.2.  (128x64 tiles in
    // that ring are behind it and the register-streaming tiles everywhere: 300 x 4096 -> 4096 17.6 against 14.5.)
    if ((p.M + 127) / 128 * ((p.N + 127) / 128) <= num_cus()) return launch_ring4<CfgDM, BF16>(p, st);
    return launch_ring4<CfgM, BF16>(p, st);
  }
  if (plan.n_wide >= p.N) return launch_ring4<CfgL8, BF16>(p, st);
  return launch_ring4_split<CfgL, CfgDH, BF16>(p, plan.n_wide, st);
}

template <class Args>
Args args_of(const void *x, const void *w4, const void *meta, const void *s_col, const void *w_reduced, const void *bias, int64_t M,
             int64_t N, int64_t K, int64_t F, void *out) {
  Args p;
  p.xbuf = static_cast<const uint8_t *>(x);
  p.wbuf = static_cast<const uint8_t *>(w4);
  p.meta = static_cast<const uint16_t *>(meta);
  p.s_col = static_cast<const uint16_t *>(s_col);
  p.w_red = static_cast<const uint16_t *>(w_reduced);
  p.bias = static_cast<const uint16_t *>(bias);
  p.out = static_cast<uint16_t *>(out);
  p.M = static_cast<int>(M);
  p.N = static_cast<int>(N);
  p.ldo = static_cast<int>(N);
  p.K = static_cast<int>(K);
  p.F = static_cast<int>(F);
  p.n_first = 0;
  p.N_total = static_cast<int>(N);
  return p;
}

}  // namespace

int tile4_activation_bits(int64_t M, int64_t N, int64_t K, int64_t F) {
  return plan_tile4(M, N, K, F) == Tiles4::kRing ? 6 : 4;
}

// checks as mixed_linear_fp6; without a workspace (16-byte aligned) no K split
int mixed_linear_tile4(const void *x, int x_bits, const void *w4, const void *meta, const void *s_col, const void *w_reduced,
                       const void *bias, int dtype, int64_t M, int64_t N, int64_t K, int64_t F, void *out, void *workspace,
                       int64_t workspace_bytes, void *stream) {
  if (dtype != QUIK_F16 && dtype != QUIK_BF16) return QUIK_ERR_DTYPE;
  if (x_bits != 4 && x_bits != 6) return QUIK_ERR_BITS;
  if (M < 0 || N < 0 || K <= 0 || F < 0) return QUIK_ERR_SHAPE;
  if (M == 0 || N == 0) return QUIK_OK;
  if (!x || !w4 || !meta || !s_col || !out) return QUIK_ERR_NULL;  // w_reduced == NULL: symmetric activations
  if (K % kLayerK4 != 0 || F % 32 != 0) return QUIK_ERR_ALIGN;
  auto misaligned = [](const void *p) { return reinterpret_cast<uintptr_t>(p) % 256 != 0; };
  if (misaligned(x) || misaligned(w4)) return QUIK_ERR_ALIGN;
  if (M > (1 << 30) || N > (1 << 30) || K > 74496) return QUIK_ERR_RANGE;  // 225 K < 2^24: the fp32 sums stay exact
  if (reinterpret_cast<uintptr_t>(workspace) % 16 != 0) workspace = nullptr;
  hipStream_t st = as_stream(stream);
  if (x_bits == 4) {
    const Fused8Args p = args_of<Fused8Args>(x, w4, meta, s_col, w_reduced, bias, M, N, K, F, out);
    return dtype == QUIK_F16 ? run_direct4<false>(p, workspace, workspace_bytes, st)
                             : run_direct4<true>(p, workspace, workspace_bytes, st);
  }
  const Fused6Args p = args_of<Fused6Args>(x, w4, meta, s_col, w_reduced, bias, M, N, K, F, out);
  return dtype == QUIK_F16 ? run_ring4<false>(p, st) : run_ring4<true>(p, st);
}
}  // namespace quik

using namespace quik;

extern "C" int quik_tile4_activation_bits(int64_t M, int64_t N, int64_t K, int64_t F) {
  if (M <= 0 || N <= 0 || K <= 0 || F < 0) return 0;
  return tile4_activation_bits(M, N, K, F);
}

extern "C" int quik_tile4_tile(int64_t M, int64_t N, int64_t K, int64_t F) {
  if (M <= 0 || N <= 0 || K <= 0 || F < 0) return 0;
  switch (plan_tile4(M, N, K, F)) {
    case Tiles4::k64x32: return Direct64x32::BM << 16 | Direct64x32::BN;
    case Tiles4::k64x64: return Direct64x64::BM << 16 | Direct64x64::BN;
    case Tiles4::k128x64: return Direct128x64::BM << 16 | Direct128x64::BN;
    default: return 0;
  }
}

extern "C" int64_t quik_tile4_splitk_bytes(int64_t M, int64_t N, int64_t K, int64_t F) {
  if (M <= 0 || N <= 0 || K <= 0 || F < 0) return 0;
  return split_bytes4(M, N, K, F);
}

extern "C" int quik_mixed_linear_fwd_tile4(const void *x, int x_bits, const void *w4, const void *meta, const void *s_col,
                                           const void *w_reduced, const void *bias, int dtype, int64_t M, int64_t N,
                                           int64_t K, int64_t F, void *out, void *stream) {
  return mixed_linear_tile4(x, x_bits, w4, meta, s_col, w_reduced, bias, dtype, M, N, K, F, out, nullptr, 0, stream);
}

extern "C" int quik_mixed_linear_fwd_tile4_ws(const void *x, int x_bits, const void *w4, const void *meta, const void *s_col,
                                           const void *w_reduced, const void *bias, int dtype, int64_t M, int64_t N,
                                           int64_t K, int64_t F, void *out, void *workspace, int64_t workspace_bytes,
                                           void *stream) {
  return mixed_linear_tile4(x, x_bits, w4, meta, s_col, w_reduced, bias, dtype, M, N, K, F, out, workspace, workspace_bytes, stream);
}
