// Fused layer GEMM on tile-ordered operands for problems of few tiles: every wave streams its own share of K straight
// from memory into the MFMA operand registers.
//
// What bounds the ring kernels (gemm_fp6.h, gemm_tile8.h) on few and narrow tiles is the step itself: a 128x64 tile has
// two MFMAs per wave and k-step, 64 cycles of work between two barriers, an LDS round trip and a wait for copies
// (measured over K: 106 .. 112 ns a step, some 210 cycles).  The operand buffers hold
// each fragment as one contiguous kilobyte (fp6_format.h), so a wave can load fragments directly, and nothing has to be
// shared inside the workgroup if the waves split K instead of the tile: each of the four waves computes the WHOLE tile
// (64x64 or 64x32, at 4 bits also 128x64) over every fourth k-step, without a barrier or an LDS access in the main loop, with SETS steps of
// loads in flight.  What bounds it is the rate at which a CU takes in operands: over K, 70 ns per step of 6 KB (88 bytes
// per ns) for 64x64 tiles at 6 bits, 33 ns per 3 KB (94) for 64x32 tiles at 8.  Afterwards the waves add their
// integer sums through LDS (exact, so in any order), each ending up with the blocks it owns, convert them, run the
// outlier steps on them in the same order as the ring kernels and store: the same output bits.
//
// Beside the stream (what a CU takes in, 80 to 85 bytes per ns with 128x64 tiles at 4 bits, or 34 MB of weights in 5 us), a
// launch of 128x64 tiles spends 12 us like this (128 x 5120 -> 13824; clock of the chip, per workgroup, before / now): arguments and
// first addresses 1.2 / 1.0, stream and last steps 6.6 / 6.7, exchange 1.8 / 1.4, conversion and outlier steps 1.6 / 1.4, output 1.0.
// The exchange reads a block's twelve pieces in one burst, not pair by pair; the outlier steps are requested in front of the last
// integer steps and in place of what those and the exchange leave; a usual count of them has no loads between its products.
// us per forward: 128 x 5120 -> 13824 17.6 -> 16.8, 300 x 4544 -> 4544 16.2 -> 15.3, 64 x 8192 -> 10240 15.4 -> 14.9, 40 x 4096 -> 4096
// 10.2 -> 9.6, 523 x 7616 -> 1808 23.7 -> 22.6, int8 136 x 13824 -> 5120 31.4 -> 30.5, 64 x 28672 -> 8192 46.8 -> 46.9.
//
// Workgroups may share a tile's K further (SplitK, as in gemm_fp6.h): when the tiles are fewer than the CUs.
//
// Measured against the ring kernels (GEMM launch in a graph, us): W4A4 64 x 8192 x 7936 22.3 -> 13.7, 64 x 10240 x 7936
// 22.5 -> 14.3, 128 x 8192 x 7936 22.8 -> 13.8, 40 x 4096 x 3840 10.5 -> 7.1, 256 x 4096 x 3840 10.8 -> 8.6,
// 512 x 1024 x 3840 10.5 -> 7.3; W8A8 64 x 5120 x 13568 26.7 -> 18.1, 64 x 4096 x 10752 26.2 -> 15.1.
#pragma once
#include <type_traits>

#include "gemm_tile8.h"

#define QUIK_INLINE __attribute__((always_inline))

namespace quik {

// 6-bit operands (Fused6Args), int8 or 4-bit ones (Fused8Args: the same fields)
enum DirectKind { kDirect6, kDirect8, kDirect4 };
template <int KIND_, int MI_, int NI_, int SETS_>
struct DirectCfg {
  static constexpr int KIND = KIND_;
  static constexpr bool SIX = KIND != kDirect8;  // multiplied on the 6-bit instructions: fp32 sums and their corrections
  static constexpr int MI = MI_, NI = NI_, SETS = SETS_, NF = MI + NI;
  static constexpr int WAVES = 4, kThreads = 64 * WAVES;
  static constexpr int BM = 32 * MI, BN = 32 * NI;
  static constexpr int UNIT = KIND == kDirect6 ? 3072 : 2048;
  static_assert((MI == 2 || MI == 4) && (NI == 1 || NI == 2 || NI == 4), "supported tiles");
  // 32x32 blocks that a wave owns after the exchange: OM x ON, at (OM * (w & 1), ON * (w >> 1)); tiles of 32 columns: waves 2
  // and 3 own none
  static constexpr int OM = MI / 2, ON = NI == 1 ? 1 : NI / 2, OWN = OM * ON;
  static constexpr int kOutlierSets = OWN <= 2 ? 16 : 8;  // outlier steps in flight (16: all of them for 256 columns)
  static constexpr int kEarlySets = KIND == kDirect6 ? 0 : OWN <= 2 ? 8 : 0;  // .. requested in front of the last integer steps
  static constexpr int kSetsInExchange = OWN <= 2 ? 12 : kOutlierSets;        // .. in front of the exchange (its reads take the registers of the others)
  // exchange: one owned block per round, in two areas by turns
  static constexpr int ROUND_BYTES = WAVES * (WAVES - 1) * 4096;
  static constexpr int RED_BYTES = (OWN > 1 ? 2 : 1) * ROUND_BYTES;
  static constexpr int PARTIAL_BYTES = WAVES * OWN * 4096;  // a workgroup's partial sums (SplitK)
  static constexpr int OUT_STRIDE = BN * 2 + 16;
  static constexpr int VEC_OFF = RED_BYTES > BM * OUT_STRIDE ? RED_BYTES : BM * OUT_STRIDE;
  static constexpr int SMEM = VEC_OFF + (4 * BN + 3 * BM) * 4;
  static constexpr int own_mi(int w) { return OM * (w & 1); }
  static constexpr int own_ni(int w) { return ON * (w >> 1); }
  static constexpr bool owns(int w) { return own_ni(w) < NI; }
};

// One step's fragments of a wave.  6-bit: head in dwords 0 .. 3, tail in 4 and 5, as the MFMA takes it; 4-bit: as in memory,
// expanded in front of its products.  (Kept as whole
// operand vectors: with heads and tails in arrays of their own the compiler merges neighbouring elements into one
// wider access, cannot split the arrays into registers any more and puts them into scratch memory.)
template <class D>
struct DirectFrag {
  std::conditional_t<D::KIND == kDirect6, v8i, v4i> f[D::NF];
};

template <class D, bool BF16, bool SPLITK, class Args>
__device__ __forceinline__ void direct_tile(const Args &p, int tm, int tn, uint8_t *smem, int split, int tile_id,
                                            const SplitK *sk) {
  constexpr int MI = D::MI, NI = D::NI, SETS = D::SETS, NF = D::NF, WAVES = D::WAVES, UNIT = D::UNIT;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int m0 = tm * D::BM, n0 = tn * D::BN;
  int64_t x_blocks, w_blocks, block_bytes, x_sums = 0, w_sums = 0;
  int steps, fsteps;
  if constexpr (D::KIND == kDirect4) {
    const Tile4Layout lx = tile4_layout(p.M, p.K, p.F), lw = tile4_layout(p.N_total, p.K, p.F);
    x_blocks = lx.blocks, w_blocks = lw.blocks, block_bytes = lx.block_bytes;
    x_sums = lx.sums_off, w_sums = lw.sums_off;
    steps = static_cast<int>(lx.steps), fsteps = static_cast<int>(lx.fsteps);
  } else if constexpr (D::KIND == kDirect6) {
    const Fp6Layout lx = fp6_layout(p.M, p.K, p.F), lw = fp6_layout(p.N_total, p.K, p.F);
    x_blocks = lx.blocks, w_blocks = lw.blocks, block_bytes = lx.block_bytes;
    x_sums = lx.sums_off, w_sums = lw.sums_off;
    steps = static_cast<int>(lx.steps), fsteps = static_cast<int>(lx.fsteps);
  } else {
    const Tile8Layout lx = tile8_layout(p.M, p.K, p.F), lw = tile8_layout(p.N_total, p.K, p.F);
    x_blocks = lx.blocks, w_blocks = lw.blocks, block_bytes = lx.block_bytes;
    steps = static_cast<int>(lx.steps), fsteps = static_cast<int>(lx.fsteps);
  }

  // sources: one scalar base per 64-row block; a 32-row fragment is half a block (blocks past the matrix: any valid
  // one, results never stored)
  const int r = lane & 31, h = lane >> 5;
  const uint32_t head_off = r * 32 + ((h ^ ((r >> 3) & 1)) << 4), tail_off = 2048 + h * 512 + r * 8;
  const int wrow = p.n_first + n0, whalf = (wrow >> 5) & 1;  // (whalf: single-fragment tiles may start inside a block)
  auto block = [&](int64_t b, int64_t blocks) { return (b < blocks ? b : blocks - 1) * block_bytes; };
  const uint8_t *base[MI / 2 + (NI + 1) / 2];
#pragma unroll
  for (int b = 0; b < MI / 2; ++b) base[b] = p.xbuf + block(m0 / 64 + b, x_blocks);
#pragma unroll
  for (int b = 0; b < (NI + 1) / 2; ++b) base[MI / 2 + b] = p.wbuf + block(wrow / 64 + b, w_blocks);
  // nothing: the registers only have to be written (the compiler's waits count loads), all lanes read the block's first bytes
  auto load_step = [&](DirectFrag<D> &f, int64_t step, bool nothing) QUIK_INLINE {
    // (opaque per step: the lane offsets stay 32-bit offsets to a scalar base, instead of being folded into a 64-bit
    // vector address per fragment that every step then has to advance)
    uint32_t ho = nothing ? 0 : head_off, to = nothing ? 0 : tail_off;
    asm volatile("" : "+v"(ho), "+v"(to));
    const int64_t at = nothing ? 0 : step * UNIT;
    static_for<NF>([&](auto J) QUIK_INLINE {
      constexpr int j = J, jj = j < MI ? j : j - MI, b = j < MI ? j / 2 : MI / 2 + jj / 2;
      const int half = j < MI || NI > 1 ? jj & 1 : whalf;
      const v4i head = *reinterpret_cast<const v4i *>(base[b] + at + half * 1024 + ho);
      if constexpr (D::KIND == kDirect6) {
        const v2i tail = *reinterpret_cast<const v2i *>(base[b] + at + half * 256 + to);
        f.f[j] = v8i{head.x, head.y, head.z, head.w, tail.x, tail.y, 0, 0};
      } else {
        f.f[j] = head;
      }
    });
  };

  int k0 = 0, k1 = steps;
  if constexpr (SPLITK) {
    k0 = split * sk->per;
    k1 = k0 + sk->per < steps ? k0 + sk->per : steps;
  }
  // This wave's steps: k0 + wave, k0 + wave + WAVES, ...  4 and 8 bits: the loop's rounds are whole and what is left behind the loop is
  // always the same code, with loads and waits that do not depend on the remainder; the first round begins in its middle, `empty`
  // steps late, with code of its own for each number of them.  (With the remainder behind the loop, each of its up to 2 SETS steps
  // with its loads under a condition, the compiler's waits there were waits for every load.  With empty steps loaded like the others, from
  // the block's first bytes, each took its share of what a CU takes in: us per forward 64 x 4096 -> 8192 9.8 -> 9.6, 90 x 5120 -> 5120 11.5 ->
  // 11.3, 300 x 4544 -> 4544 15.6 -> 15.4.)  Where a wave has no whole round, empty steps are loaded so.
  const int mine = k1 - k0 > wave ? (k1 - k0 - wave + WAVES - 1) / WAVES : 0;
  auto at = [&](int i) { return k0 + wave + i * WAVES; };
  constexpr bool kWhole = D::KIND != kDirect6;                             // the rounds are whole
  constexpr int kAhead = SETS + (D::KIND == kDirect4 ? 1 : 0);             // steps in registers: loaded, at 4 bits one more expanded
  const int more = mine > kAhead ? (mine - kAhead + SETS - 1) / SETS : 0;  // rounds of the loop
  const int empty = kWhole ? kAhead + more * SETS - mine : 0;
  const int last_step = k1 > 0 ? k1 - 1 : 0;
  // per-row and per-column scalars of this thread: requested first, unconditionally (a load under a branch would make
  // the waits of everything around it waits for all loads), used after the main loop
  const int vi = threadIdx.x;
  const int64_t vn = n0 + vi % D::BN < p.N ? n0 + vi % D::BN : p.N - 1, vm = m0 + vi % D::BM < p.M ? m0 + vi % D::BM : p.M - 1;
  const bool asym = p.w_red != nullptr;  // asymmetric: meta holds (scale, zero) pairs; symmetric: one scale per row, no zero term
  const uint16_t v_sc = p.s_col[vn], v_wr = (asym ? p.w_red : p.s_col)[vn], v_bs = (p.bias ? p.bias : p.s_col)[vn];
  const uint16_t v_sr = p.meta[asym ? 2 * vm : vm], v_zr = p.meta[asym ? 2 * vm + 1 : vm];
  int v_cs = 0, v_rs = 0;
  if constexpr (D::SIX) {
    v_cs = reinterpret_cast<const int32_t *>(p.wbuf + w_sums)[p.n_first + vn];
    v_rs = reinterpret_cast<const int32_t *>(p.xbuf + x_sums)[vm];
  }

  // 4 and 8 bits: the wave's next step to load, as the lane's offset to the (scalar) addresses of the blocks: one addition per
  // step.  The instructions of a step are what bounds it, not the bytes.
  uint32_t pos = head_off + static_cast<uint32_t>(at(kAhead - empty)) * UNIT;
  const uint8_t *const wbase = base[MI / 2] + (NI == 1 ? whalf * 1024 : 0);
  auto load_next = [&](auto &f) QUIK_INLINE {
    static_for<NF>([&](auto J) QUIK_INLINE {
      constexpr int j = J, jj = j < MI ? j : j - MI, b = j < MI ? j / 2 : MI / 2 + jj / 2;
      f.f[j] = *reinterpret_cast<const v4i *>((j < MI || NI > 1 ? base[b] : wbase) + pos + (jj & 1) * 1024);
    });
    pos += WAVES * UNIT;
  };

  DirectFrag<D> set[SETS];
  // step i of this wave, empty ones included (unconditional, as every load in front of the loop: the compiler's waits in it
  // count on them)
  auto load_one = [&](DirectFrag<D> &f, int i) QUIK_INLINE {
    const int step = at(i - empty);
    load_step(f, step < last_step ? step : last_step, i < empty);
  };
  if constexpr (!kWhole) static_for<SETS>([&](auto S) QUIK_INLINE { load_one(set[S], S); });

  v16f acc[MI][NI];  // fp32 sums (SIX) or int32 bit patterns
#pragma unroll
  for (int mi = 0; mi < MI; ++mi)
#pragma unroll
    for (int ni = 0; ni < NI; ++ni)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[mi][ni][v] = 0.0f;
  // outlier steps of the blocks that this wave will own; the first ones are requested in front of the exchange, some of them in
  // front of the last integer steps
  constexpr int OS = D::kOutlierSets, OM = D::OM, ON = D::ON, OWN = D::OWN;
  v4i ox[OS][OM], ow[OS][ON];
  const int omi = D::own_mi(wave), oni = D::owns(wave) ? D::own_ni(wave) : 0;
  const uint8_t *ox_base[OM], *ow_base[ON];
#pragma unroll
  for (int i = 0; i < OM; ++i) ox_base[i] = p.xbuf + block((m0 + 32 * (omi + i)) / 64, x_blocks) + ((omi + i) & 1) * 1024;
#pragma unroll
  for (int j = 0; j < ON; ++j) {
    const int row = wrow + 32 * (oni + j);
    ow_base[j] = p.wbuf + block(row / 64, w_blocks) + ((row >> 5) & 1) * 1024;
  }
  // (a step behind the last one: not used, the block's first bytes to all lanes)
  auto load_outlier = [&](auto S, int t) QUIK_INLINE {
    const bool real = t < fsteps;
    const int64_t at_step = real ? int64_t(steps + t) * UNIT : 0;
    const uint32_t off = real ? head_off : 0;
    auto from = [&](const uint8_t *b) QUIK_INLINE { return *reinterpret_cast<const v4i *>(b + at_step + off); };
    static_for<OM>([&](auto I) QUIK_INLINE { ox[S][I] = from(ox_base[I]); });
    static_for<ON>([&](auto J) QUIK_INLINE { ow[S][J] = from(ow_base[J]); });
  };
  // sets [LO, HI) of a round
  auto load_outliers = [&](auto LO, auto HI, int t0) QUIK_INLINE {
    static_for<HI - LO>([&](auto I) QUIK_INLINE {
      constexpr int S = LO + I;
      load_outlier(std::integral_constant<int, S>{}, t0 + S);
    });
  };
  using std::integral_constant;
  constexpr integral_constant<int, 0> kNone{};
  constexpr integral_constant<int, D::kEarlySets> kEarly{};
  constexpr integral_constant<int, OS> kAll{};
  if constexpr (kWhole) {
    constexpr bool FOUR = D::KIND == kDirect4;
    // 4 bits: a step's fragments are expanded (eight VALU instructions each) while the step before is multiplied: a wave has its SIMD
    // to itself, nothing else would run under its products.  Step i is expanded in u[i & 1], steps i + 1 .. i + SETS are in the sets
    // (i + k in set (i + k) % SETS); 8 bits: steps i .. i + SETS - 1 are.
    v6i u[2][NF];
    auto expand = [&](v6i (&to)[NF], const DirectFrag<D> &f) QUIK_INLINE {
      static_for<NF>([&](auto J) QUIK_INLINE { to[J] = nib_expand(f.f[J]); });
    };
    auto multiply = [&](const auto &v) QUIK_INLINE {
      static_for<MI * NI>([&](auto I) QUIK_INLINE {
        constexpr int mi = I % MI, ni = I / MI;
        if constexpr (FOUR) {
          nib_mma(v[mi], v[MI + ni], acc[mi][ni]);
        } else {
          FragOps<kInt8>::mma(v[mi], v[MI + ni], acc[mi][ni]);
        }
      });
    };
    static_assert(SETS % 2 == 0, "operand sets alternate");
    auto interleave = [&]() QUIK_INLINE {
      static_for<MI * NI>([&](auto) QUIK_INLINE {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, (8 * NF + MI * NI - 1) / (MI * NI), 0);
      });
    };
    // steps in front of the first real one are skipped; skip: how many
    auto step = [&](auto S, auto skip) QUIK_INLINE {
      if constexpr (FOUR) {
        constexpr int next = (S + 1) % SETS;
        if (S >= skip) {
          expand(u[(S + 1) & 1], set[next]);
          multiply(u[S & 1]);
          interleave();
          static_for<NF>([&](auto J) QUIK_INLINE { pin(u[(S + 1) & 1][J]); });
        } else if (S + 1 == skip) {
          expand(u[(S + 1) & 1], set[next]);
        }
      } else {
        if (S >= skip) multiply(set[S].f);
      }
    };
    auto round = [&](auto skip) QUIK_INLINE {
      static_for<SETS>([&](auto S) QUIK_INLINE {
        __builtin_amdgcn_s_waitcnt(vmcnt_imm((SETS - 1) * NF));  // (one wait for the set, not one per fragment)
        __builtin_amdgcn_sched_barrier(0);
        step(S, skip);
        load_next(set[FOUR ? (S + 1) % SETS : S]);
        __builtin_amdgcn_sched_barrier(0);  // (left alone the scheduler delays the loads behind later steps' MFMAs)
      });
    };
    // The first steps and the first round, a copy for every number of empty steps in front of them.
    if (more > 0) {
      static_for<SETS>([&](auto E) QUIK_INLINE {
        if (empty == E) {
          static_for<SETS - E>([&](auto S) QUIK_INLINE { load_one(set[E + S], E + S); });
          if constexpr (FOUR) {
            if constexpr (E == 0) expand(u[0], set[0]);
            load_one(set[0], SETS);
          }
          round(E);
        }
      });
    } else {
      static_for<SETS>([&](auto S) QUIK_INLINE { load_one(set[S], S); });
      if constexpr (FOUR) {
        expand(u[0], set[0]);
        load_one(set[0], SETS);
      }
    }
    for (int i = 1; i < more; ++i) round(integral_constant<int, 0>{});
    // the last steps: outlier steps are requested in front of them and in place of the sets they leave
    if constexpr (!SPLITK) load_outliers(kNone, kEarly, 0);
    const int skip = more > 0 ? 0 : empty;
    static_for<SETS>([&](auto S) QUIK_INLINE {
      constexpr int late = D::kSetsInExchange - D::kEarlySets;
      constexpr int sets = D::kEarlySets + late * S / SETS, sets_then = D::kEarlySets + late * (S + 1) / SETS;
      constexpr int behind = SPLITK ? 0 : sets * (OM + ON);
      __builtin_amdgcn_s_waitcnt(vmcnt_imm((SETS - 1 - S) * NF + behind));
      __builtin_amdgcn_sched_barrier(0);
      step(S, skip);
      if constexpr (!SPLITK)
        load_outliers(integral_constant<int, sets>{}, integral_constant<int, sets_then>{}, 0);
      __builtin_amdgcn_sched_barrier(0);
    });
    if constexpr (FOUR) {
      if (mine > 0) multiply(u[SETS & 1]);
    }
  } else {
    auto multiply = [&](const DirectFrag<D> &f) QUIK_INLINE {
      static_for<MI * NI>([&](auto I) QUIK_INLINE {
        constexpr int mi = I % MI, ni = I / MI;
        acc[mi][ni] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(f.f[MI + ni], f.f[mi], acc[mi][ni], 2, 2, 0, 0, 0, 0);
      });
    };
    int it = 0;
    for (; it + 2 * SETS <= mine; it += SETS) {
      static_for<SETS>([&](auto S) QUIK_INLINE {
        multiply(set[S]);
        load_step(set[S], at(it + SETS + S), false);
        __builtin_amdgcn_sched_barrier(0);  // (left alone the scheduler delays the loads behind later steps' MFMAs)
      });
    }
    static_for<SETS>([&](auto S) QUIK_INLINE {
      if (it + S < mine) multiply(set[S]);
      if (it + SETS + S < mine) load_step(set[S], at(it + SETS + S), false);
    });
    static_for<SETS>([&](auto S) QUIK_INLINE {
      if (it + SETS + S < mine) multiply(set[S]);
    });
  }

  float *const scol = reinterpret_cast<float *>(smem + D::VEC_OFF), *const wred = scol + D::BN, *const bias = wred + D::BN,
               *const colc = bias + D::BN, *const srow = colc + D::BN, *const zs = srow + D::BM, *const rowc = zs + D::BM;
  if (vi < D::BN) {
    scol[vi] = to_f32<BF16>(v_sc);
    wred[vi] = asym ? to_f32<BF16>(v_wr) : 0.0f;
    bias[vi] = p.bias ? to_f32<BF16>(v_bs) : 0.0f;
    colc[vi] = static_cast<float>(v_cs) * -0.125f;
  }
  if (vi < D::BM) {
    const float s = to_f32<BF16>(v_sr);
    srow[vi] = s;
    zs[vi] = asym ? to_f32<BF16>(v_zr) + (D::SIX ? 8.0f : 128.0f) * s : 0.0f;
    rowc[vi] = D::SIX ? static_cast<float>(8 * v_rs - 64 * p.K) : 0.0f;
  }  // (visible behind the exchange's barrier)

  constexpr integral_constant<int, D::kSetsInExchange> kExchanged{};
  if constexpr (!SPLITK && !kWhole) load_outliers(kNone, kExchanged, 0);

  // exchange, owned block by owned block: wave w leaves its sums of the block that wave o owns in slot (o, w), o adds the
  // three it finds
  v16f own[OWN];
  auto add = [](float a, int b) QUIK_INLINE {
    return D::SIX ? a + __int_as_float(b) : __int_as_float(__float_as_int(a) + b);
  };
  constexpr int AREAS = OWN > 1 ? 2 : 1;
  static_for<OWN / AREAS>([&](auto G) QUIK_INLINE {
    if constexpr (G > 0) __syncthreads();  // every wave has read the areas
    static_for<AREAS>([&](auto Q) QUIK_INLINE {
      constexpr int B = G * AREAS + Q, bm = B % OM, bn = B / OM;
      own[B] = v16f{};
      static_for<WAVES>([&](auto O) QUIK_INLINE {
        constexpr int o = O;
        if constexpr (D::owns(o)) {
          const v16f &b = acc[D::own_mi(o) + bm][D::own_ni(o) + bn];
          if (o == wave) {
            own[B] = b;
          } else {
            uint8_t *slot = smem + Q * D::ROUND_BYTES + (o * (WAVES - 1) + (wave < o ? wave : wave - 1)) * 4096 + lane * 16;
#pragma unroll
            for (int g = 0; g < 4; ++g)
              *reinterpret_cast<float4 *>(slot + g * 1024) = make_float4(b[4 * g], b[4 * g + 1], b[4 * g + 2], b[4 * g + 3]);
          }
        }
      });
    });
    if constexpr (!SPLITK && G == OWN / AREAS - 1) load_outliers(kExchanged, kAll, 0);  // (in place of the sums just written)
    __syncthreads();
    if (D::owns(wave)) {
      // (a block's reads in one burst: left alone the compiler waits for every pair)
      static_for<AREAS>([&](auto Q) QUIK_INLINE {
        v4i t[WAVES - 1][4];
#pragma unroll
        for (int s = 0; s < WAVES - 1; ++s)
#pragma unroll
          for (int g = 0; g < 4; ++g)
            t[s][g] = *reinterpret_cast<const v4i *>(smem + Q * D::ROUND_BYTES + (wave * (WAVES - 1) + s) * 4096 + lane * 16 + g * 1024);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < WAVES - 1; ++s)
#pragma unroll
          for (int g = 0; g < 4; ++g)
#pragma unroll
            for (int e = 0; e < 4; ++e) own[G * AREAS + Q][4 * g + e] = add(own[G * AREAS + Q][4 * g + e], t[s][g][e]);
        __builtin_amdgcn_sched_barrier(0);
      });
    }
  });

  if constexpr (SPLITK) {
    // the same between the workgroups of a tile, through memory (see splitk_combine in gemm_fp6.h): partial sums
    // [tile][split][owned block][wave][group of 4][lane][4]
    constexpr int kPer = D::PARTIAL_BYTES / 4;
    int32_t *part = sk->partials + int64_t(tile_id) * sk->splits * kPer + wave * 1024 + lane * 4;
    if (D::owns(wave)) {
      static_for<OWN>([&](auto B) QUIK_INLINE {
#pragma unroll
        for (int g = 0; g < 4; ++g)
          splitk_store4(part + int64_t(split) * kPer + B * (WAVES * 1024) + g * 256,
                        v4i{__float_as_int(own[B][4 * g]), __float_as_int(own[B][4 * g + 1]), __float_as_int(own[B][4 * g + 2]),
                            __float_as_int(own[B][4 * g + 3])});
      });
    }
    splitk_stores_done();
    __syncthreads();
    int *last_s = reinterpret_cast<int *>(smem);
    if (threadIdx.x == 0) {
      const uint32_t before = __hip_atomic_fetch_add(sk->counters + tile_id, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      *last_s = before == static_cast<uint32_t>(sk->splits - 1);
    }
    __syncthreads();
    if (*last_s == 0) return;
    load_outliers(kNone, kAll, 0);
    if (D::owns(wave)) {
      for (int o = 0; o < sk->splits; ++o) {
        if (o == split) continue;
        static_for<OWN>([&](auto B) QUIK_INLINE {
          v4i t[4];
          splitk_load4<256>(part + int64_t(o) * kPer + B * (WAVES * 1024), t);
#pragma unroll
          for (int g = 0; g < 4; ++g)
#pragma unroll
            for (int e = 0; e < 4; ++e) own[B][4 * g + e] = add(own[B][4 * g + e], t[g][e]);
        });
      }
    }
    if (threadIdx.x == 0) __hip_atomic_store(sk->counters + tile_id, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }

  // conversion, outlier steps, storage type: the arithmetic of fused6_tile / fused8t_tile on the owned blocks
  if (D::owns(wave)) {
    struct Columns {
      float4 sc, wr, bs, cc;
    };
    Columns columns[ON][4];
#pragma unroll
    for (int j = 0; j < ON; ++j)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int c = (oni + j) * 32 + acc_col(g, lane);
        columns[j][g] = {*reinterpret_cast<const float4 *>(scol + c), *reinterpret_cast<const float4 *>(wred + c),
                         *reinterpret_cast<const float4 *>(bias + c), *reinterpret_cast<const float4 *>(colc + c)};
      }
    static_for<OWN>([&](auto B) QUIK_INLINE {
      constexpr int bm = B % OM, bn = B / OM;
      const float rs = srow[32 * (omi + bm) + r], rz = zs[32 * (omi + bm) + r], rc = rowc[32 * (omi + bm) + r];
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const float4 sc = columns[bn][g].sc, wr = columns[bn][g].wr, bs = columns[bn][g].bs, cc = columns[bn][g].cc;
        const float scv[4] = {sc.x, sc.y, sc.z, sc.w}, wrv[4] = {wr.x, wr.y, wr.z, wr.w}, bsv[4] = {bs.x, bs.y, bs.z, bs.w},
                    ccv[4] = {cc.x, cc.y, cc.z, cc.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float raw = own[B][4 * g + e];
          const float iacc = D::SIX ? __builtin_fmaf(raw + ccv[e], 64.0f, -rc)  // exact: integers below 2^24
                                    : static_cast<float>(__float_as_int(raw));
          own[B][4 * g + e] = __builtin_fmaf(iacc, rs * scv[e], __builtin_fmaf(rz, wrv[e], bsv[e]));
        }
      }
    });
    auto outlier_step = [&](auto S) QUIK_INLINE {
      static_for<OWN>([&](auto B) QUIK_INLINE { FragOps<BF16 ? kBF16 : kF16>::mma(ox[S][B % OM], ow[S][B / OM], own[B]); });
    };
    auto outlier_round = [&](int t0) QUIK_INLINE {
      const bool again = t0 + OS < fsteps;
      static_for<OS / 4>([&](auto G) QUIK_INLINE {
        constexpr int S = 4 * G;
        if (t0 + S < fsteps) {  // (an even number of steps: outlier columns are a multiple of 32)
          outlier_step(integral_constant<int, S>{}), outlier_step(integral_constant<int, S + 1>{});
          if (t0 + S + 2 < fsteps) outlier_step(integral_constant<int, S + 2>{}), outlier_step(integral_constant<int, S + 3>{});
          int next = t0 + OS;
          asm volatile("" : "+s"(next));  // (opaque: else the addresses of all steps advance together, in registers)
          if (again) load_outliers(integral_constant<int, S>{}, integral_constant<int, S + 4>{}, next);
        }
      });
    };
    if (fsteps > 0) outlier_round(0);  // (usually the only one, with waits of its own)
    for (int t0 = OS; t0 < fsteps; t0 += OS) outlier_round(t0);
  }
  __syncthreads();  // every wave has read its slots: the area becomes the output tile
  if (D::owns(wave)) {
    static_for<OWN>([&](auto B) QUIK_INLINE {
      constexpr int bm = B % OM, bn = B / OM;
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<uint2 *>(smem + (32 * (omi + bm) + r) * D::OUT_STRIDE + ((oni + bn) * 32 + acc_col(g, lane)) * 2) =
            make_uint2(pack2_from_f32<BF16>(own[B][4 * g], own[B][4 * g + 1]), pack2_from_f32<BF16>(own[B][4 * g + 2], own[B][4 * g + 3]));
    });
  }
  __syncthreads();
  const bool vec = (p.ldo & 7) == 0 && (reinterpret_cast<uintptr_t>(p.out) & 15) == 0;
  constexpr int kPieces = D::BN / 8;  // 16-byte pieces of a row
  NanWatch<BF16> nans;
  auto store = [&](auto again) QUIK_INLINE {
#pragma unroll
    for (int i = threadIdx.x; i < D::BM * kPieces; i += D::kThreads) {
      const int row = i / kPieces, col = (i % kPieces) * 8;
      if (m0 + row >= p.M || n0 + col >= p.N) continue;
      v4i piece = *reinterpret_cast<const v4i *>(smem + row * D::OUT_STRIDE + col * 2);
      if constexpr (again) {
#pragma unroll
        for (int k = 0; k < 4; ++k) piece[k] = static_cast<int>(canonical_bf16_pair(static_cast<uint32_t>(piece[k])));
      }
      uint16_t *dst = p.out + int64_t(m0 + row) * p.ldo + n0 + col;
      if (vec && n0 + col + 8 <= p.N) {
        __builtin_nontemporal_store(piece, reinterpret_cast<v4i *>(dst));
      } else {
        uint16_t tmp[8];
        __builtin_memcpy(tmp, &piece, 16);
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (n0 + col + e < p.N) dst[e] = tmp[e];
      }
      if constexpr (!again) nans.add(piece);
    }
  };
  store(std::false_type{});
  if (nans.any()) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (a wait only: no hazard; the first stores are done)
    store(std::true_type{});
  }
}

template <class D, bool BF16, class Args>
__global__ __launch_bounds__(D::kThreads, D::OWN == 1 ? 2 : 1) void gemm_direct_kernel(Args p, int tiles_m, int tiles_n) {
  extern __shared__ __align__(16) uint8_t smem[];
  int tm, tn;
  asm volatile("" : : "s"(p.xbuf), "s"(p.wbuf), "s"(p.M), "s"(p.N), "s"(p.K), "s"(p.F), "s"(p.n_first), "s"(p.N_total), "s"(p.meta), "s"(p.s_col),
               "s"(p.w_red), "s"(p.bias));  // (all arguments in one trip, not those behind the branch in a second one; no instruction)
  if (!tile_of_block<D::BM>(blockIdx.x, tiles_m, tiles_n, tm, tn)) return;
  direct_tile<D, BF16, false>(p, tm, tn, smem, 0, 0, nullptr);
}
template <class D, bool BF16, class Args>
__global__ __launch_bounds__(D::kThreads, D::OWN == 1 ? 2 : 1) void gemm_direct_splitk_kernel(Args p, int tiles_m, int tiles_n, SplitK sk) {
  extern __shared__ __align__(16) uint8_t smem[];
  int tm, tn;
  const int split = blockIdx.x / sk.grid_tiles;
  if (!tile_of_block<D::BM>(blockIdx.x - split * sk.grid_tiles, tiles_m, tiles_n, tm, tn)) return;
  direct_tile<D, BF16, true>(p, tm, tn, smem, split, tm * tiles_n + tn, &sk);
}

}  // namespace quik
