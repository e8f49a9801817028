// Tile configurations, plans and launch grids that the translation units of the GEMMs share (host side).
#pragma once
#include <cstdint>

#include "gemm_fp6.h"

namespace quik {
namespace {

// Tile configurations.  "dma" ones use the direct-to-LDS pipelined main loop and need K bytes
// (and outlier bytes) per row to be a multiple of 64; the plain ones accept anything.
using CfgL = Cfg<256, 256, 2, 2, 2>;   // prefill: 128x128 per wave, 256 accumulator registers
using CfgH = Cfg<256, 128, 2, 2, 2>;   // half-width tile that evens out the last round
using CfgM = Cfg<128, 128, 2, 2, 2>;   // mid-size problems, two workgroups per CU
using CfgN = Cfg<128, 64, 2, 2, 2>;    // few tiles: narrower ones put more CUs to work, three workgroups per CU
// with one workgroup per CU, the LDS of a CU full of copies in flight: eight stages here, up to twelve slots in the tile-ordered
// rings (ring_slots)
using CfgDN = Cfg<128, 64, 2, 2, 2, 8>;
using CfgDM = Cfg<128, 128, 2, 2, 2, 8>;
using CfgDH = Cfg<256, 128, 2, 2, 2, 8>;
using CfgL8 = Cfg<256, 256, 2, 4, 2>;  // 6-bit path, launches of 256x256 tiles only: two waves per SIMD (1-5 % faster than CfgL)
using CfgLp = Cfg<256, 256, 2, 2, 0>;  // plain fallbacks
using CfgMp = Cfg<128, 128, 2, 2, 0>;

constexpr int kMaxCUs = 256;  // MI355X; sizes the static K-split scratch array

template <class C>
int grid_of(int64_t M, int64_t N, int &tiles_m, int &tiles_n) {
  tiles_m = static_cast<int>((M + C::BM - 1) / C::BM);
  tiles_n = static_cast<int>((N + C::BN - 1) / C::BN);
  return static_cast<int>(((int64_t(tiles_m) * tiles_n + 7) / 8) * 8);
}

// Workgroup id layout of a two-shape launch: half of the narrow tiles (at most half a round) lead.
template <class CW, class CT>
SplitGrid split_grid(int64_t M, int64_t n_wide, int64_t n_tail, int &tail_blocks) {
  SplitGrid g;
  g.wide_blocks = grid_of<CW>(M, n_wide, g.tiles_m, g.tiles_n_wide);
  tail_blocks = grid_of<CT>(M, n_tail, g.tiles_m, g.tiles_n_tail);
  int lead = (tail_blocks / 2) & ~7;
  if (lead > num_cus() / 2) lead = num_cus() / 2;
  g.lead = lead;
  return g;
}

// How a problem is cut into tiles.  Columns [0, n_wide) go to 256x256 tiles, [n_wide, N) to
// 256x128 tiles, all in one launch with the wide tiles first.  One workgroup fits per CU and the
// hardware hands the next workgroup to whichever CU frees up, so the run time is the makespan of
// that list schedule; the narrow tiles even out its end.
struct Plan {
  enum Kind { kSmall, kMid, kNarrow, kMidPlain, kLargePlain, kSplit } kind;
  int64_t n_wide;
};

// relative tile costs in percent of a 256x256 tile (measured)
constexpr int kCostWide = 100, kCostHalf = 55, kCostMid = 28;

// Makespan of `wide` tiles followed by `half` tiles on the GPU's CUs under greedy list scheduling.
int64_t makespan(int64_t wide, int64_t half, int cost_half = kCostHalf) {
  // after the wide tiles: `rem` CUs carry one tile more than the others
  const int64_t full = wide / num_cus(), rem = wide % num_cus();
  int64_t lo_level = full * kCostWide, lo_count = num_cus() - rem;  // less loaded CUs
  int64_t hi_level = lo_level + kCostWide, hi_count = rem;
  // the half tiles go to the least loaded CUs, a whole level at a time
  while (half > 0) {
    if (hi_count == 0 || lo_level + cost_half <= hi_level) {
      if (half >= lo_count && lo_level + cost_half < hi_level && hi_count > 0) {
        lo_level += cost_half;
        half -= lo_count;
      } else if (hi_count == 0) {
        const int64_t rounds = half / lo_count, left = half % lo_count;
        return lo_level + rounds * cost_half + (left ? cost_half : 0);
      } else if (half >= lo_count) {  // lo reaches hi's level exactly
        lo_level += cost_half;
        half -= lo_count;
        if (lo_level == hi_level) {
          lo_count += hi_count;
          hi_count = 0;
        }
      } else {
        const int64_t top = lo_level + cost_half;
        return top > hi_level ? top : hi_level;
      }
    } else {
      // adding a half tile to the lower level overtakes the higher one: swap roles afterwards
      if (half >= lo_count) {
        half -= lo_count;
        const int64_t new_hi = lo_level + cost_half, new_hi_count = lo_count;
        lo_level = hi_level;
        lo_count = hi_count;
        hi_level = new_hi;
        hi_count = new_hi_count;
      } else {
        return lo_level + cost_half;
      }
    }
  }
  return hi_count > 0 ? hi_level : lo_level;
}

// Tile plan of the 6-bit path (gemm_fp6.h).  Costs in percent of a 256x256 tile, measured at K = 7936, F = 256:
// a 256x128 tile 59; 128x128 tiles run two to a CU, 66 for a pair, 36 for one that has the CU to itself.  (With 4-bit weights and the
// conversion as it is now, kernel us of one round each, 256x256 72.6, 256x128 43.3, a pair of 128x128 48.75: 60 and 67; int8 115.5, 66.0, 69.7: 57
// and 60.)
Plan make_plan6(int64_t M, int64_t N, int64_t min_rows) {
  if (M < min_rows) return {Plan::kSmall, 0};
  const int64_t tiles_m = (M + 255) / 256;
  const int64_t mid_tiles = ((M + 127) / 128) * ((N + 127) / 128);
  const int64_t pairs = mid_tiles / (2 * num_cus()), left = mid_tiles % (2 * num_cus());
  const int64_t mid = pairs * 66 + (left == 0 ? 0 : left <= num_cus() ? 36 : 66);
  int64_t best = INT64_MAX, best_n = 0;
  for (int64_t n_wide = 0; n_wide <= N + 255; n_wide += 256) {
    const int64_t nw = n_wide < N ? n_wide : N;   // the last candidate: wide tiles only, the last one ragged
    const int64_t c = makespan(tiles_m * ((nw + 255) / 256), tiles_m * ((N - nw + 127) / 128), 59);
    if (c <= best) {
      best = c;
      best_n = nw;
    }
  }
  if (mid < best) return {Plan::kMid, 0};
  return {Plan::kSplit, best_n};
}

// The 6-bit matrix-core path (gemm_fp6.h): 256x256 tiles alone (eight waves), 256x256 + 256x128 tiles in one
// launch (four waves), or 128x128 tiles.
// Whole rounds of 256x256 tiles with little left over: a last round of 256x128 tiles costs 59, on part of the CUs; the same
// columns in 128x128 tiles are one per CU at 36 (percent of a wide tile).  2048 x 8192 -> 10240: 111.5 -> 102.6 us per
// forward (with the bands of tile_of_block), int8 179 -> 168.
// Only behind whole rounds: narrow tiles that run beside wide ones are slower than the costs say (777 x 4096 -> 22016 by
// the same costs 159 -> 136, measured 72.2 -> 73.8 us), and two of them per CU cost more than a 256x128 tile.
// Returns the columns of the wide part, 0: the plan of make_plan6 stands.
int64_t plan_rest(int64_t M, int64_t N, const Plan &plan) {
  if (plan.kind != Plan::kSplit) return 0;
  const int64_t cus = num_cus(), tiles_m = (M + 255) / 256, rounds = tiles_m * (N / 256) / cus, wide_n = rounds * cus / tiles_m;
  if (rounds < 1 || rounds * cus - tiles_m * wide_n > cus / 16) return 0;
  const int64_t rest = (M + 127) / 128 * ((N + 127) / 128 - 2 * wide_n), nw = plan.n_wide;
  const int64_t now = makespan(tiles_m * ((nw + 255) / 256), tiles_m * ((N - nw + 127) / 128), 59);
  return rest > 0 && rest <= cus && rounds * kCostWide + 36 < now ? wide_n * 256 : 0;
}
template <class CW, class CT, class Args, class Kernel>
int launch_rest(Kernel kern, int smem, const Args &p, int64_t n_wide, hipStream_t st) {
  RestGrid g{};
  g.wide_blocks = grid_of<CW>(p.M, n_wide, g.tiles_m_wide, g.tiles_n_wide);
  const int rest_blocks = grid_of<CT>(p.M, p.N - n_wide, g.tiles_m, g.tiles_n);
  g.first = static_cast<int>(n_wide / CT::BN);
  if (int rc = prepare(kern, smem)) return rc;
  hipLaunchKernelGGL(kern, dim3(g.wide_blocks + rest_blocks), dim3(CW::kThreads), smem, st, p, g);
  return check_launch();
}

// Zero-fill of a few words by a kernel: the arrival counters of the K split are cleared with it, not with
// hipMemsetAsync, because the caller's stream may be under capture and a memset node in a captured graph is not
// reliable on replays.
__global__ __launch_bounds__(256) void clear_words_kernel(uint32_t *p, int words) {
  for (int i = blockIdx.x * 256 + threadIdx.x; i < words; i += gridDim.x * 256) p[i] = 0u;
}
constexpr int64_t kSplitCounterBytes = 4096;  // arrival counters of a K split, one per tile, in front of the partial sums
// The arrival counters are zero between launches because every launch that completes returns them there.  After a
// launch that was refused nothing ran, but the caller may not know how far an earlier one got: clear the counters
// behind a failed launch so that the next one on this workspace starts clean.
int splitk_launch_status(void *workspace, hipStream_t st) {
  const int rc = check_launch();
  if (rc != QUIK_OK) {
    hipLaunchKernelGGL(clear_words_kernel, dim3(static_cast<unsigned>(kSplitCounterBytes / 4 / 256)), dim3(256), 0, st,
                       static_cast<uint32_t *>(workspace), static_cast<int>(kSplitCounterBytes / 4));
    (void)hipGetLastError();  // the status reported is that of the launch that failed
  }
  return rc;
}

}  // namespace
}  // namespace quik
