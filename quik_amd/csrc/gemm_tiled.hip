// Host side of the GEMMs on tile-ordered operands of 6 bits (gemm_fp6.h) and int8 (gemm_tile8.h, gemm_direct.h): plans, launches,
// entry points.
#include <atomic>
#include <cstdint>
#include <mutex>

#include "gemm_direct.h"
#include "gemm_plan.h"

namespace quik {
namespace {

// Split over K for the tile-ordered kernels: few 128x128 tiles (at most half the CUs) and a long K.  Each of
// `splits` workgroups per tile takes `per` steps (even); workspace = counters (one per tile, zero between launches)
// followed by the partial accumulators.
constexpr int64_t kSplitMinSteps = 32;  // at least 1024 (int8) / 2048 (6-bit) elements of K per workgroup
enum Operands { kOperands6, kOperands8 };
// integer k-steps of an operand buffer and bytes of a 64-row unit (fp6_layout, tile8_layout)
int64_t tile_steps(int64_t K, Operands ops) { return ops == kOperands8 ? (K + 63) / 64 * 2 : (K + 127) / 128 * 2; }
constexpr int64_t unit_bytes(Operands ops) { return ops == kOperands6 ? 3072 : 2048; }
struct SplitPlan {
  int splits, per;
  int64_t bytes;
};
// min_splits: with two workgroups per tile the exchange and the restart for the outlier steps cost the 6-bit path
// (K <= 8192 in every Llama layer it serves) what the halved K loop saves; measured gains start at three.
SplitPlan plan_splitk(int64_t M, int64_t N, int64_t K, Operands ops) {
  const int64_t steps = tile_steps(K, ops), min_steps = kSplitMinSteps, min_splits = ops == kOperands8 ? 2 : 3;
  SplitPlan none{1, 0, 0};
  if (make_plan6(M, N, 1).kind != Plan::kMid) return none;
  const int64_t tiles = ((M + 127) / 128) * ((N + 127) / 128);
  if (tiles > num_cus() / 2 || tiles * 4 > kSplitCounterBytes) return none;
  for (int64_t splits = num_cus() / tiles < 8 ? num_cus() / tiles : 8; splits >= min_splits; --splits) {
    const int64_t per = ((steps + splits - 1) / splits + 1) / 2 * 2;
    if (per >= min_steps && (splits - 1) * per < steps)
      return {static_cast<int>(splits), static_cast<int>(per), kSplitCounterBytes + tiles * splits * 128 * 128 * 4};
  }
  return none;
}

template <bool BF16>
int launch_fused6_splitk(const Fused6Args &p, const SplitPlan &sp, void *workspace, hipStream_t st) {
  int tiles_m, tiles_n;
  const int grid_tiles = grid_of<CfgM>(p.M, p.N, tiles_m, tiles_n);
  SplitK sk{sp.splits, sp.per, grid_tiles, static_cast<uint32_t *>(workspace),
            reinterpret_cast<int32_t *>(static_cast<uint8_t *>(workspace) + kSplitCounterBytes)};
  auto kern = gemm_fused6_splitk_kernel<CfgM, BF16>;
  constexpr int smem = fused6_smem<CfgM>();
  if (int rc = prepare(kern, smem)) return rc;
  hipLaunchKernelGGL(kern, dim3(grid_tiles * sp.splits), dim3(CfgM::kThreads), smem, st, p, tiles_m, tiles_n, sk);
  return splitk_launch_status(workspace, st);
}

template <bool BF16>
int launch_fused8t_splitk(const Fused8Args &p, const SplitPlan &sp, void *workspace, hipStream_t st) {
  int tiles_m, tiles_n;
  const int grid_tiles = grid_of<CfgM>(p.M, p.N, tiles_m, tiles_n);
  SplitK sk{sp.splits, sp.per, grid_tiles, static_cast<uint32_t *>(workspace),
            reinterpret_cast<int32_t *>(static_cast<uint8_t *>(workspace) + kSplitCounterBytes)};
  auto kern = gemm_fused8t_splitk_kernel<CfgM, BF16>;
  constexpr int smem = fused8t_smem<CfgM>();
  if (int rc = prepare(kern, smem)) return rc;
  hipLaunchKernelGGL(kern, dim3(grid_tiles * sp.splits), dim3(CfgM::kThreads), smem, st, p, tiles_m, tiles_n, sk);
  return splitk_launch_status(workspace, st);
}

template <class C, bool BF16>
int launch_fused6(const Fused6Args &p, hipStream_t st) {
  if (p.N <= 0) return QUIK_OK;
  int tiles_m, tiles_n;
  const int grid = grid_of<C>(p.M, p.N, tiles_m, tiles_n);
  auto kern = gemm_fused6_kernel<C, BF16>;
  constexpr int smem = fused6_smem<C>();
  if (int rc = prepare(kern, smem)) return rc;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(C::kThreads), smem, st, p, tiles_m, tiles_n);
  return check_launch();
}

template <class CW, class CT, bool BF16>
int launch_fused6_split(const Fused6Args &wide, const Fused6Args &tail, hipStream_t st) {
  if (wide.N <= 0) return launch_fused6<CT, BF16>(tail, st);
  if (tail.N <= 0) return launch_fused6<CW, BF16>(wide, st);
  int tail_blocks;
  SplitGrid grid = split_grid<CW, CT>(wide.M, wide.N, tail.N, tail_blocks);
  grid.lead = 0;  // this kernel lives on L2 hits between the tiles of an XCD that share operand rows: keep them in step
  auto kern = gemm_fused6_split_kernel<CW, CT, BF16>;
  constexpr int smem = fused6_smem<CW>() > fused6_smem<CT>() ? fused6_smem<CW>() : fused6_smem<CT>();
  if (int rc = prepare(kern, smem)) return rc;
  hipLaunchKernelGGL(kern, dim3(grid.wide_blocks + tail_blocks), dim3(CW::kThreads), smem, st, wide, tail, grid);
  return check_launch();
}

// Register-streaming kernel (gemm_direct.h), ring kernel or ring kernel with a K split, for problems below the 256-row
// tiles.  All are priced in ns: a fixed part, the operand bytes the busiest CU takes in at 103 bytes per ns (87 in the ring
// of 128x64 tiles), never less than the weights take: up to 128 MB at 8 TB/s, more at what each kernel reaches from memory,
// and at most 24 bytes per ns for each CU that works.  The 8 TB/s is not where such weights come from, a model's are cold; it is
// what ranks the kernels as they were measured, warm and cold alike (layers over 700 MB in turn): over 23 layer shapes of 6 ..
// 222 MB at 40 .. 192 rows, both widths, the pick is 0.6 % behind the fastest kernel warm and 1.7 % cold.  (Fitted with ten and six int8 steps
// in flight; with six and four, over 35 int8 calls of 40 .. 200 rows, it is 1.5 % behind warm, most where the ring is the faster one: 200 x 13824
// -> 5120 42.2 / 37.2 us with its K split, 200 x 8192 -> 8192 34.3 / 31.1 without.)  us per forward, warm /
// cold, as picked and as the memory's rates would pick: 64 x 4096 -> 11008 13.6 / 18.2 (64x64 tiles) and 15.3 / 19.9 (ring),
// 64 x 8192 -> 10240 18.4 / 27.2 and 20.8 / 29.9, 128 x 8192 -> 20480 28.8 / 46.5 (ring) and 36.5 / 54.2; int8 64 x 13824 -> 5120 23.4 /
// 34.7 (64x64, two splits) and 27.9 / 35.8, but 64 x 14336 -> 8192 26.4 / 40.5 (64x32) and 29.0 / 36.4.  Beyond, the memory's rates
// are the better ones cold: 64 x 28672 -> 8192 37.0 / 46.6 and 35.6 / 54.5 at 8 TB/s, int8 46.7 / 65.9 and 44.0 / 77.5.  A K split
// adds the exchange: its partial sums cross memory, 16 KB per workgroup in the register-streaming kernel, 64 KB in the ring
// kernel (measured 13 us with its start for two workgroups per tile, 22 .. 24 for three to eight).
struct DirectPlan {
  int bn, splits;   // tile width (64 or 32; 0: ring kernel), workgroups per tile
  int64_t bytes;    // workspace of the split
  bool ring_split;  // the ring kernel splits K (plan_splitk)
};
DirectPlan plan_direct(int64_t M, int64_t N, int64_t K, Operands ops, int64_t workspace_bytes) {
  DirectPlan plan{0, 1, 0, false};
  if (make_plan6(M, N, 1).kind != Plan::kMid) return plan;
  const int64_t steps = tile_steps(K, ops), unit = unit_bytes(ops), cus = num_cus();
  const int64_t weights = N * steps * unit / 64;
  auto up = [](int64_t a, int64_t b) { return (a + b - 1) / b; };
  auto busiest = [&](int64_t groups, int64_t per, int64_t step_bytes, int64_t rate, int64_t memory) {
    const int64_t ns = up(groups, cus) * per * step_bytes / rate, by_cus = 24 * (groups < cus ? groups : cus);
    const int64_t stream = weights / (weights <= (128 << 20) ? 8000 : by_cus < memory ? by_cus : memory);
    return ns > stream ? ns : stream;
  };
  const int64_t tiles128 = up(M, 128) * up(N, 128), tiles64 = up(M, 128) * up(N, 64);
  int64_t best = 5300 + (ops != kOperands8 && tiles64 <= cus ? busiest(tiles64, steps, 3 * unit, 87, 5500)
                                                     : busiest(tiles128, steps, 4 * unit, 103, 5500));
  const SplitPlan sp = plan_splitk(M, N, K, ops);
  if (sp.splits > 1 && workspace_bytes >= sp.bytes) {
    const int64_t ns = (sp.splits == 2 ? 13500 : 23500) + busiest(tiles128 * sp.splits, sp.per, 4 * unit, 103, 5500);
    if (ns < best) best = ns, plan.ring_split = true;
  }
  for (const int bn : {64, 32}) {
    const int64_t tiles = up(M, 64) * up(N, bn);
    for (const int splits : {1, 2, 4}) {
      const int64_t bytes = splits > 1 ? kSplitCounterBytes + tiles * splits * DirectCfg<kDirect6, 2, 2, 4>::PARTIAL_BYTES : 0;
      if (splits > 1 && (tiles * 4 > kSplitCounterBytes || bytes > workspace_bytes || up(steps, splits) * (splits - 1) >= steps))
        continue;
      const int64_t ns = 6300 + (splits > 1 ? 1500 + 500 * splits : 0) +
                         busiest(tiles * splits, up(steps, splits), unit + unit * bn / 64, 103, bn == 64 ? 4300 : 3400);
      if (ns < best) best = ns, plan = {bn, splits, bytes, false};
    }
  }
  return plan;
}

template <class D, bool BF16, class Args>
int launch_direct(const Args &p, int splits, void *workspace, hipStream_t st) {
  int tiles_m, tiles_n;
  const int grid = grid_of<D>(p.M, p.N, tiles_m, tiles_n);
  if (splits > 1) {
    const int steps = static_cast<int>(tile_steps(p.K, D::SIX ? kOperands6 : kOperands8));
    SplitK sk{splits, (steps + splits - 1) / splits, grid, static_cast<uint32_t *>(workspace),
              reinterpret_cast<int32_t *>(static_cast<uint8_t *>(workspace) + kSplitCounterBytes)};
    auto kern = gemm_direct_splitk_kernel<D, BF16, Args>;
    if (int rc = prepare(kern, D::SMEM)) return rc;
    hipLaunchKernelGGL(kern, dim3(grid * splits), dim3(D::kThreads), D::SMEM, st, p, tiles_m, tiles_n, sk);
    return splitk_launch_status(workspace, st);
  }
  auto kern = gemm_direct_kernel<D, BF16, Args>;
  if (int rc = prepare(kern, D::SMEM)) return rc;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(D::kThreads), D::SMEM, st, p, tiles_m, tiles_n);
  return check_launch();
}
// Steps in flight: what bounds the stream is what a CU takes in, not its latency.  int8, six of 64x64 and ten of 64x32 tiles with the
// remainder behind the loop / six and ten / four and six / two and four, us per forward: 96 x 8192 -> 8192 21.9 / 21.7 / 21.05 / 22.5, 256 x
// 4096 -> 4096 14.2 / 14.0 / 13.75 / 14.4, 136 x 13824 -> 5120 29.5 / 29.15 / 28.85 / 31.5, 64 x 1024 -> 4096 8.75 / 8.55 / 8.3 / 8.2, 64 x
// 4096 -> 4096 from memory 15.55 / 15.1 / 15.1 / 15.15, but 128 x 11008 -> 4096 20.75 / 20.6 / 20.85 / 21.6.
template <int KIND, bool BF16, class Args>
int run_direct(const Args &p, const DirectPlan &d, void *workspace, hipStream_t st) {
  if (d.bn == 64) return launch_direct<DirectCfg<KIND, 2, 2, 4>, BF16>(p, d.splits, workspace, st);
  return launch_direct<DirectCfg<KIND, 2, 1, KIND == kDirect6 ? 8 : 6>, BF16>(p, d.splits, workspace, st);
}

template <bool BF16>
int run_fused6(const Fused6Args &p, hipStream_t st, void *workspace, int64_t workspace_bytes) {
  // any row count: up to 32 rows the weight-streaming kernel on the packed nibbles reads a third fewer bytes, and
  // callers that keep both weight copies route such calls there
  const DirectPlan d = plan_direct(p.M, p.N, p.K, kOperands6, workspace ? workspace_bytes : 0);
  if (d.bn) return run_direct<kDirect6, BF16>(p, d, workspace, st);
  if (d.ring_split) return launch_fused6_splitk<BF16>(p, plan_splitk(p.M, p.N, p.K, kOperands6), workspace, st);
  const Plan plan = make_plan6(p.M, p.N, 1);
  if (const int64_t n_wide = plan_rest(p.M, p.N, plan); n_wide > 0)
    return launch_rest<CfgL, CfgM>(gemm_fused6_rest_kernel<CfgL, CfgM, BF16>, fused6_smem<CfgL>(), p, n_wide, st);
  if (plan.kind == Plan::kSplit && plan.n_wide >= p.N) return launch_fused6<CfgL8, BF16>(p, st);
  if (plan.kind != Plan::kSplit) {
    // One 128x64 tile per CU: a ring of twelve slots (110 KB of LDS) instead of six, nine steps in flight instead of three.
    // Layer forward 300 x 4544 -> 4544 19.1 -> 18.6 us, 2048 x 8192 -> 1024 31.3 -> 30.7, 128 x 5120 -> 13824 20.3 -> 20.0, 256 x
    // 8192 -> 8192 26.5 -> 25.9: a step takes 106 ns, some 210 cycles, for 64 of MFMA, against 111 ns with six slots (two
    // steps between barriers, or no second copy of the W block, changed nothing on top).
    // More of them than CUs, two on some, take longer than the half as many 128x128 tiles, one per CU: 512 x 4096 -> 5120
    // 25.6 -> 20.8, 236 x 13824 -> 10240 80 -> 59.5.
    if ((p.M + 127) / 128 * ((p.N + 63) / 64) <= num_cus()) return launch_fused6<CfgDN, BF16>(p, st);
    if ((p.M + 127) / 128 * ((p.N + 127) / 128) <= num_cus()) return launch_fused6<CfgDM, BF16>(p, st);
    return launch_fused6<CfgM, BF16>(p, st);
  }
  Fused6Args wide = p, tail = p;
  const int64_t nw = plan.n_wide;
  wide.N = static_cast<int>(nw);
  tail.N = static_cast<int>(p.N - nw);
  tail.n_first = static_cast<int>(nw);
  tail.s_col = p.s_col + nw;
  tail.w_red = p.w_red ? p.w_red + nw : nullptr;
  tail.bias = p.bias ? p.bias + nw : nullptr;
  tail.out = p.out + nw;
  // (the 256x128 tiles have the LDS of a CU to themselves as well: eight slots, int8 twelve; 946 x 13824 -> 5120 74.5 -> 73.1 us,
  // int8 2048 x 11008 -> 4096 102.3 -> 101.0)
  return launch_fused6_split<CfgL, CfgDH, BF16>(wide, tail, st);
}

template <class C, bool BF16>
int launch_fused8t(const Fused8Args &p, hipStream_t st) {
  if (p.N <= 0) return QUIK_OK;
  int tiles_m, tiles_n;
  const int grid = grid_of<C>(p.M, p.N, tiles_m, tiles_n);
  auto kern = gemm_fused8t_kernel<C, BF16>;
  constexpr int smem = fused8t_smem<C>();
  if (int rc = prepare(kern, smem)) return rc;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(C::kThreads), smem, st, p, tiles_m, tiles_n);
  return check_launch();
}

template <class CW, class CT, bool BF16>
int launch_fused8t_split(const Fused8Args &wide, const Fused8Args &tail, hipStream_t st) {
  if (wide.N <= 0) return launch_fused8t<CT, BF16>(tail, st);
  if (tail.N <= 0) return launch_fused8t<CW, BF16>(wide, st);
  int tail_blocks;
  SplitGrid grid = split_grid<CW, CT>(wide.M, wide.N, tail.N, tail_blocks);
  grid.lead = 0;  // tiles of an XCD that share operand rows stay in step (L2 hits)
  auto kern = gemm_fused8t_split_kernel<CW, CT, BF16>;
  constexpr int smem = fused8t_smem<CW>() > fused8t_smem<CT>() ? fused8t_smem<CW>() : fused8t_smem<CT>();
  if (int rc = prepare(kern, smem)) return rc;
  hipLaunchKernelGGL(kern, dim3(grid.wide_blocks + tail_blocks), dim3(CW::kThreads), smem, st, wide, tail, grid);
  return check_launch();
}

// W8A8 on tile-ordered operands (gemm_tile8.h): same plan and tile shapes as the 6-bit path.
template <bool BF16>
int run_fused8t(const Fused8Args &p, hipStream_t st, void *workspace, int64_t workspace_bytes) {
  const DirectPlan d = plan_direct(p.M, p.N, p.K, kOperands8, workspace ? workspace_bytes : 0);
  if (d.bn) return run_direct<kDirect8, BF16>(p, d, workspace, st);
  if (d.ring_split) return launch_fused8t_splitk<BF16>(p, plan_splitk(p.M, p.N, p.K, kOperands8), workspace, st);
  const Plan plan = make_plan6(p.M, p.N, 1);  // any row count: with few rows this path competes with the weight-streaming kernel
  if (plan.kind != Plan::kSplit) {
    // one tile per CU: twelve slots, 72 KB in flight instead of 24 (365 x 28672 -> 8192 157 -> 144 us, 652 x 11008 -> 4096
    // 48.6 -> 46.3)
    if ((p.M + 127) / 128 * ((p.N + 127) / 128) <= num_cus()) return launch_fused8t<CfgDM, BF16>(p, st);
    return launch_fused8t<CfgM, BF16>(p, st);
  }
  if (const int64_t n_wide = plan_rest(p.M, p.N, plan); n_wide > 0)
    return launch_rest<CfgL, CfgM>(gemm_fused8t_rest_kernel<CfgL, CfgM, BF16>, fused8t_smem<CfgL>(), p, n_wide, st);
  if (plan.n_wide >= p.N) return launch_fused8t<CfgL8, BF16>(p, st);
  Fused8Args wide = p, tail = p;
  const int64_t nw = plan.n_wide;
  wide.N = static_cast<int>(nw);
  tail.N = static_cast<int>(p.N - nw);
  tail.n_first = static_cast<int>(nw);
  tail.s_col = p.s_col + nw;
  tail.w_red = p.w_red ? p.w_red + nw : nullptr;
  tail.bias = p.bias ? p.bias + nw : nullptr;
  tail.out = p.out + nw;
  return launch_fused8t_split<CfgL, CfgDH, BF16>(wide, tail, st);
}

}  // namespace
}  // namespace quik

using namespace quik;

extern "C" int64_t quik_splitk_workspace_bytes(int64_t M, int64_t N, int64_t K, int bits) {
  if (M <= 0 || N <= 0 || K <= 0 || (bits != 4 && bits != 8)) return 0;
  if (bits == 4 ? K % kLayerK4 != 0 : K % kLayerK8 != 0) return 0;
  // whichever kernel a call with that much workspace takes; a shape the ring kernels would split keeps its workspace
  // even where the register-streaming kernel then does without
  const Operands ops = bits == 4 ? kOperands6 : kOperands8;
  const int64_t ring = plan_splitk(M, N, K, ops).bytes;
  const int64_t direct = plan_direct(M, N, K, ops, kSplitCounterBytes + int64_t(kMaxCUs) * 128 * 128 * 4).bytes;
  return ring > direct ? ring : direct;
}

extern "C" int quik_mixed_linear_fwd_fp6(const void *x6, const void *w6, const void *meta, const void *s_col,
                                         const void *w_reduced, const void *bias, int dtype, int64_t M, int64_t N,
                                         int64_t K, int64_t F, void *out, void *stream) {
  return quik_mixed_linear_fwd_fp6_ws(x6, w6, meta, s_col, w_reduced, bias, dtype, M, N, K, F, out, nullptr, 0, stream);
}

int quik::mixed_linear_fp6(const void *x6, const void *w6, const void *meta, const void *s_col, const void *w_reduced,
                           const void *bias, int dtype, int64_t M, int64_t N, int64_t K, int64_t F, void *out,
                           void *workspace, int64_t workspace_bytes, void *stream, int64_t k_multiple) {
  if (dtype != QUIK_F16 && dtype != QUIK_BF16) return QUIK_ERR_DTYPE;
  if (M < 0 || N < 0 || K <= 0 || F < 0) return QUIK_ERR_SHAPE;
  if (M == 0 || N == 0) return QUIK_OK;
  if (!x6 || !w6 || !meta || !s_col || !out) return QUIK_ERR_NULL;  // w_reduced == NULL: symmetric activations
  if (K % k_multiple != 0 || F % 32 != 0) return QUIK_ERR_ALIGN;
  auto misaligned = [](const void *p) { return reinterpret_cast<uintptr_t>(p) % 256 != 0; };
  if (misaligned(x6) || misaligned(w6)) return QUIK_ERR_ALIGN;
  if (M > (1 << 30) || N > (1 << 30) || K > 74496) return QUIK_ERR_RANGE;  // 225 K < 2^24: the fp32 sums stay exact
  Fused6Args p;
  p.xbuf = static_cast<const uint8_t *>(x6);
  p.wbuf = static_cast<const uint8_t *>(w6);
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
  hipStream_t st = as_stream(stream);
  if (workspace && reinterpret_cast<uintptr_t>(workspace) % 16 != 0) return QUIK_ERR_ALIGN;
  return dtype == QUIK_F16 ? run_fused6<false>(p, st, workspace, workspace_bytes)
                           : run_fused6<true>(p, st, workspace, workspace_bytes);
}

extern "C" int quik_mixed_linear_fwd_fp6_ws(const void *x6, const void *w6, const void *meta, const void *s_col,
                                            const void *w_reduced, const void *bias, int dtype, int64_t M, int64_t N,
                                            int64_t K, int64_t F, void *out, void *workspace,
                                            int64_t workspace_bytes, void *stream) {
  return mixed_linear_fp6(x6, w6, meta, s_col, w_reduced, bias, dtype, M, N, K, F, out, workspace, workspace_bytes, stream, 128);
}

extern "C" int quik_mixed_linear_fwd_tile8(const void *x8, const void *w8, const void *meta, const void *s_col,
                                           const void *w_reduced, const void *bias, int dtype, int64_t M, int64_t N,
                                           int64_t K, int64_t F, void *out, void *stream) {
  return quik_mixed_linear_fwd_tile8_ws(x8, w8, meta, s_col, w_reduced, bias, dtype, M, N, K, F, out, nullptr, 0, stream);
}

int quik::mixed_linear_tile8(const void *x8, const void *w8, const void *meta, const void *s_col, const void *w_reduced,
                             const void *bias, int dtype, int64_t M, int64_t N, int64_t K, int64_t F, void *out,
                             void *workspace, int64_t workspace_bytes, void *stream, int64_t k_multiple) {
  if (dtype != QUIK_F16 && dtype != QUIK_BF16) return QUIK_ERR_DTYPE;
  if (M < 0 || N < 0 || K <= 0 || F < 0) return QUIK_ERR_SHAPE;
  if (M == 0 || N == 0) return QUIK_OK;
  if (!x8 || !w8 || !meta || !s_col || !out) return QUIK_ERR_NULL;  // w_reduced == NULL: symmetric activations
  if (K % k_multiple != 0 || F % 32 != 0) return QUIK_ERR_ALIGN;
  auto misaligned = [](const void *p) { return reinterpret_cast<uintptr_t>(p) % 256 != 0; };
  if (misaligned(x8) || misaligned(w8)) return QUIK_ERR_ALIGN;
  if (M > (1 << 30) || N > (1 << 30) || K > (1 << 24)) return QUIK_ERR_RANGE;
  Fused8Args p;
  p.xbuf = static_cast<const uint8_t *>(x8);
  p.wbuf = static_cast<const uint8_t *>(w8);
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
  hipStream_t st = as_stream(stream);
  if (workspace && reinterpret_cast<uintptr_t>(workspace) % 16 != 0) return QUIK_ERR_ALIGN;
  return dtype == QUIK_F16 ? run_fused8t<false>(p, st, workspace, workspace_bytes)
                           : run_fused8t<true>(p, st, workspace, workspace_bytes);
}

extern "C" int quik_mixed_linear_fwd_tile8_ws(const void *x8, const void *w8, const void *meta, const void *s_col,
                                              const void *w_reduced, const void *bias, int dtype, int64_t M, int64_t N,
                                              int64_t K, int64_t F, void *out, void *workspace,
                                              int64_t workspace_bytes, void *stream) {
  return mixed_linear_tile8(x8, w8, meta, s_col, w_reduced, bias, dtype, M, N, K, F, out, workspace, workspace_bytes, stream, 64);
}

// ---- the entry point that allocates nothing ------------------------------------------------------------------
// quik_mixed_linear_fwd_tile8_ws with the K-split workspace in a file-scope device array instead of a caller
// buffer: counters (kSplitCounterBytes) followed by the partial accumulators, the size of the largest plan
// plan_splitk makes (tiles x splits <= kMaxCUs workgroups of one 128x128 int32 tile each).  Every GPU that loads this
// library holds its own copy of the array until the process ends.
constexpr int64_t kStaticScratchBytes = kSplitCounterBytes + int64_t(kMaxCUs) * 128 * 128 * 4;
static __device__ __align__(256) uint8_t scratch[kStaticScratchBytes];

namespace quik {
namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
std::atomic<uint8_t *> g_scratch_ptr[kMaxDevices];

// Device address of `scratch` on the current device.  In host code the array's name is only a handle for
// hipGetSymbolAddress: the address is looked up once per device, with that device current, and kept.
int scratch_of_current_device(uint8_t **out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) {
    set_last_hip_error(e);
    return QUIK_ERR_LAUNCH;
  }
  if (dev < 0 || dev >= kMaxDevices) return QUIK_ERR_RANGE;
  uint8_t *p = g_scratch_ptr[dev].load(std::memory_order_acquire);
  if (!p) {
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    p = g_scratch_ptr[dev].load(std::memory_order_relaxed);
    if (!p) {
      void *sym = nullptr;
      e = hipGetSymbolAddress(&sym, HIP_SYMBOL(scratch));
      if (e != hipSuccess || !sym) {
        set_last_hip_error(e != hipSuccess ? e : hipErrorInvalidSymbol);
        return QUIK_ERR_LAUNCH;
      }
      p = static_cast<uint8_t *>(sym);
      g_scratch_ptr[dev].store(p, std::memory_order_release);
    }
  }
  *out = p;
  return QUIK_OK;
}

// (the counters of `scratch` are cleared with clear_words_kernel in front of each launch that uses them: launches
// leave them at zero, but a launch that failed half way would not, and this array outlives every caller)
}  // namespace
}  // namespace quik

extern "C" int quik_mixed_linear_fwd_tile8_noalloc(const void *x8, const void *w8, const void *meta, const void *s_col,
                                                   const void *w_reduced, const void *bias, int dtype, int64_t M,
                                                   int64_t N, int64_t K, int64_t F, void *out, void *stream) {
  if (dtype != QUIK_F16 && dtype != QUIK_BF16) return QUIK_ERR_DTYPE;
  if (M < 0 || N < 0 || K <= 0 || F < 0) return QUIK_ERR_SHAPE;
  if (K % 64 != 0 || F % 32 != 0) return QUIK_ERR_ALIGN;
  const int64_t need = quik_splitk_workspace_bytes(M, N, K, 8);
  if (need > kStaticScratchBytes) return QUIK_ERR_RANGE;  // a K split larger than the static array holds
  if (need == 0 || M == 0 || N == 0)                      // no K split for this shape: no scratch memory involved
    return quik_mixed_linear_fwd_tile8_ws(x8, w8, meta, s_col, w_reduced, bias, dtype, M, N, K, F, out, nullptr, 0, stream);
  if (!x8 || !w8 || !meta || !s_col || !out) return QUIK_ERR_NULL;
  uint8_t *ws = nullptr;
  if (int rc = scratch_of_current_device(&ws)) return rc;
  hipLaunchKernelGGL(clear_words_kernel, dim3(static_cast<unsigned>(kSplitCounterBytes / 4 / 256)), dim3(256), 0,
                     as_stream(stream), reinterpret_cast<uint32_t *>(ws), static_cast<int>(kSplitCounterBytes / 4));
  if (int rc = check_launch()) return rc;
  return quik_mixed_linear_fwd_tile8_ws(x8, w8, meta, s_col, w_reduced, bias, dtype, M, N, K, F, out, ws,
                                        kStaticScratchBytes, stream);
}
