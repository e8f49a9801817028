// Skinny GEMM for at most 32 token rows (decode) on row-major operands: the weights are read exactly once, straight from memory
// into registers, and the problem is bound by that stream.
//
// A workgroup has `bn` output columns, at most 16 NT, and all token rows (MT blocks of 16); its eight waves split K, 128 bytes
// per row and turn, and meet once, at the end.  What a CU takes in from beyond its L2 is bound by the requests that it may have
// open, some 30 bytes per ns: the columns are dealt evenly to all CUs (5120 columns: 256 workgroups of 20, where 160 of 32 left
// 96 CUs idle), in one round as far as the registers reach (a second one begins with empty queues).
// A request costs by the lines that neighbouring lanes touch.  Both operands are read as whole 128-byte lines of eight rows per
// instruction and turned into the order of v_mfma_i32_16x16x64_i8 (16 K bytes of row l % 16, K quarter l / 16, in lane l) in LDS;
// read in that order from memory, 64 bytes of sixteen rows per instruction, a W8A8 28672 -> 8192 layer with 32 rows took 52 us,
// now 47, and every token row of a 4096 x 10752 int4 call added 0.1 us, now 0.04.  The weights go through SETS turns of registers
// and a tile of the wave's own in LDS; the token rows are copied straight to LDS, `ring` turns ahead and before the weights of
// that turn: loads return in order, so a wave that has its weights has its token rows.
// The fp16 / bf16 outlier columns are split over the waves too, 32 columns per step (v_mfma_f32_16x16x32).  At the end the waves'
// int32 sums (exact in any order) and fp32 outlier sums (added in wave order) meet in LDS, and wave w finalises block w with the
// epilogue formula of the large tiles.
//
// Time of the fused product, weights in the Infinity Cache / from HBM, before (slabs of 32 columns, eight waves, registers) and
// now, us: int4 4096 -> 4096, 16 rows 6.7 / 8.2, 4.3 / 5.6; 5120 -> 13824 11.7 / 13.6, 8.9 / 11.0; 8192 -> 28672 26.8 / 30.0,
// 22.7 / 26.2; int8 13824 -> 5120, 16 rows 15.6 / 20.2, 13.8 / 16.5 (70 MB: 10.5 us at 6.6 TB/s).
#pragma once
#include "gemm_kernels.h"

namespace quik {

constexpr int kSkinnyWaves = 8;
template <int NT_, int MT_, int SETS_>
struct SkinnyCfg {
  static constexpr int NT = NT_, MT = MT_, SETS = SETS_;
  static constexpr int BLOCKS = NT * MT, kThreads = 64 * kSkinnyWaves;
  // turns of token rows in LDS per wave: at least SETS, and two, so that a turn's copies are not waited for at once
  static constexpr int kRing = SETS > 2 ? SETS : 2;
  static int smem(int rows, bool fused) {
    const int stream = kSkinnyWaves * (kRing * ((rows + 7) / 8) * 1024 + NT * 2048);  // token rows and the waves' tiles
    const int sums = kSkinnyWaves * BLOCKS * 1024 * (fused ? 2 : 1);                  // .. and what takes their place
    return stream > sums ? stream : sums;
  }
};

// FUSED: p.out receives the MixedQLinear output.  !FUSED: Cm receives the int32 product.
// bn * K bytes, bn * outlier bytes and the same of the token rows fit 32 bits.
template <class C, int MODE, bool BF16, bool FUSED>
__global__ __launch_bounds__(C::kThreads, 2) void gemm_skinny_kernel(FusedArgs p, int bn, int32_t *__restrict__ Cm, int ldc) {
  constexpr int NT = C::NT, MT = C::MT, SETS = C::SETS, WAVES = kSkinnyWaves;
  extern __shared__ __align__(16) uint8_t smem[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, q = lane >> 4;
  // (columns past the workgroup's: its last one again, the same lines, never stored; token rows likewise)
  const int n0 = blockIdx.x * bn, n_end = n0 + bn < p.N ? n0 + bn : p.N;
  auto column = [&](int n) { return n < n_end ? n : n_end - 1; };
  auto token = [&](int m) { return m < p.M ? m : p.M - 1; };
  const int kbytes = p.kbytes, chunks = kbytes >> 7;  // wave w: chunks w, w + WAVES, ... of 128 bytes
  const int mine = chunks > wave ? (chunks - wave + WAVES - 1) / WAVES : 0;
  constexpr uint32_t kTurn = WAVES * 128;
  uint32_t w_turn = 0, x_turn = 0;  // the next ones to request

  // the blocks that this wave finalises: scalars of their columns and rows, requested first, used last
  constexpr int PW = (C::BLOCKS + WAVES - 1) / WAVES;
  uint16_t e_sc[PW][4], e_wr[PW][4], e_bs[PW][4], e_sr[PW], e_zr[PW];
  const bool asym = p.w_red != nullptr;
  if constexpr (FUSED) {
    const uint16_t *wr = asym ? p.w_red : p.s_col, *bs = p.bias ? p.bias : p.s_col;
#pragma unroll
    for (int i = 0; i < PW; ++i) {
      const int b = wave + i * WAVES;
      const int64_t mm = token(16 * (b % MT) + r);
      e_sr[i] = p.meta[mm * p.meta_stride];
      e_zr[i] = p.meta[asym ? 2 * mm + 1 : mm];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int nn = column(n0 + 16 * (b / MT) + 4 * q + v);
        e_sc[i][v] = p.s_col[nn], e_wr[i][v] = wr[nn], e_bs[i][v] = bs[nn];
      }
    }
  }
  // The wave's first outlier step (all of them up to 256 columns).  Unconditional, from valid addresses: what must not count is
  // masked when it is used (loads under a branch would make every wait behind them a wait for all loads)
  const int fbytes = FUSED ? p.F * 2 : 0, fsteps = (fbytes + 63) >> 6;
  const uint8_t *fw0 = p.qw, *fx0 = p.qx;  // (without outlier columns: any 16 bytes)
  uint32_t fwv[NT], fxv[MT];
  v4i fw[NT], fx[MT];
  auto load_outlier = [&](int t) __attribute__((always_inline)) {
    const uint32_t at = t * 64 + q * 16, off = at < static_cast<uint32_t>(fbytes) ? at : 0;
#pragma unroll
    for (int g = 0; g < NT; ++g) fw[g] = *reinterpret_cast<const v4i *>(fw0 + fwv[g] + off);
#pragma unroll
    for (int g = 0; g < MT; ++g) fx[g] = *reinterpret_cast<const v4i *>(fx0 + fxv[g] + off);
  };
  if constexpr (FUSED) {
    if (fbytes > 0) {
      fw0 = reinterpret_cast<const uint8_t *>(p.fp_w) + int64_t(n0) * fbytes;
      fx0 = reinterpret_cast<const uint8_t *>(p.fp_x);
    }
#pragma unroll
    for (int g = 0; g < NT; ++g) fwv[g] = static_cast<uint32_t>(column(n0 + 16 * g + r) - n0) * fbytes;
#pragma unroll
    for (int g = 0; g < MT; ++g) fxv[g] = static_cast<uint32_t>(token(16 * g + r)) * fbytes;
    load_outlier(wave);
  }

  // the token rows of a turn: 128 bytes each, eight rows per copy; 16-byte piece c of row r stands in slot c ^ (r & 7)
  const int xrows = (p.M + 7) & ~7, xturn = xrows * 128;
  uint8_t *const x_ring = smem + wave * C::kRing * xturn;
  const uint32_t x_lds = lds_address(x_ring);
  uint32_t xv[2 * MT], xo[MT];
#pragma unroll
  for (int g = 0; g < 2 * MT; ++g) xv[g] = static_cast<uint32_t>(token(8 * g + (lane >> 3))) * kbytes + (((lane & 7) ^ (lane >> 3)) << 4);
#pragma unroll
  for (int g = 0; g < MT; ++g) xo[g] = (16 * g + r < xrows ? 16 * g + r : xrows - 1) * 128 + ((q ^ (r & 7)) << 4);
  auto copy_x = [&](uint32_t to) __attribute__((always_inline)) {
    const uint8_t *const from = p.qx + __builtin_amdgcn_readfirstlane(wave * 128u + x_turn * kTurn);
    const uint32_t lds = __builtin_amdgcn_readfirstlane(to);
    static_for<2 * MT>([&](auto G) __attribute__((always_inline)) {
      if (8 * G < xrows) dma_load16(from, xv[G], lds + G * 1024);
    });
    ++x_turn;
  };
  for (int t = 0; t < mine && t < C::kRing; ++t) copy_x(x_lds + t * xturn);

  struct Set {
    v4i w[NT][2];
  };
  uint32_t wv[NT][2];  // this lane's columns, relative to the wave-uniform address of the stream
#pragma unroll
  for (int g = 0; g < 2 * NT; ++g) wv[g >> 1][g & 1] = static_cast<uint32_t>(column(n0 + 8 * g + (lane >> 3)) - n0) * kbytes + (lane & 7) * 16;
  uint8_t *const tile = smem + WAVES * C::kRing * xturn + wave * NT * 2048;
  const uint32_t t_write = (lane >> 3) * 128 + (((lane & 7) ^ (lane >> 3)) << 4), t_read = r * 128 + ((q ^ (r & 7)) << 4);
  const uint8_t *const w0 = p.qw + int64_t(n0) * kbytes;
  auto load_next = [&](Set &s) __attribute__((always_inline)) {
    const uint8_t *const wb = w0 + __builtin_amdgcn_readfirstlane(wave * 128u + w_turn * kTurn);
    static_for<NT>([&](auto G) __attribute__((always_inline)) {
      static_for<2>([&](auto I) __attribute__((always_inline)) { s.w[G][I] = *reinterpret_cast<const v4i *>(wb + wv[G][I]); });
    });
    ++w_turn;
  };
  v4i acc[NT][MT] = {};
  auto product = [&](const v4i &w0, const v4i &w1, const v4i (&x)[MT][2][FragOps<MODE>::H], v4i (&c)[MT]) __attribute__((always_inline)) {
    constexpr int H = FragOps<MODE>::H;
    static_for<2>([&](auto I) __attribute__((always_inline)) {
      v4i w[H];
      FragOps<MODE>::unpack(I ? w1 : w0, w);
      static_for<MT * H>([&](auto J) __attribute__((always_inline)) {
        constexpr int m = J % MT, k = J / MT;
        c[m] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w[k], x[m][I][k], c[m], 0, 0, 0);
      });
    });
  };
  int turn = 0;
  uint32_t x_at = 0;
  auto multiply = [&](Set &s) __attribute__((always_inline)) {
    asm volatile("" : "+v"(s.w[0][0]) : : "memory");  // its weights are there, and so are the token rows
    static_for<2 * NT>([&](auto J) __attribute__((always_inline)) {
      *reinterpret_cast<v4i *>(tile + J * 1024 + t_write) = s.w[J >> 1][J & 1];
    });
    v4i x[MT][2][FragOps<MODE>::H];
    static_for<2 * MT>([&](auto J) __attribute__((always_inline)) {
      FragOps<MODE>::unpack(*reinterpret_cast<const v4i *>(x_ring + x_at + (xo[J >> 1] ^ (64 * (J & 1)))), x[J >> 1][J & 1]);
    });
    static_for<NT>([&](auto G) __attribute__((always_inline)) {
      product(*reinterpret_cast<const v4i *>(tile + G * 2048 + t_read), *reinterpret_cast<const v4i *>(tile + G * 2048 + (t_read ^ 64)), x, acc[G]);
    });
    if (turn + C::kRing < mine) {
      asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");  // (the slot has been read)
      copy_x(x_lds + x_at);
    }
    ++turn;
    x_at += xturn;
    x_at = x_at == static_cast<uint32_t>(C::kRing * xturn) ? 0 : x_at;
  };
  if (mine >= SETS) {
    Set set[SETS];
    static_for<SETS>([&](auto S) __attribute__((always_inline)) { load_next(set[S]); });
    int it = 0;
    for (; it + 2 * SETS <= mine; it += SETS) {
      static_for<SETS>([&](auto S) __attribute__((always_inline)) {
        multiply(set[S]);
        load_next(set[S]);
        __builtin_amdgcn_sched_barrier(0);  // (left alone the scheduler delays the loads behind later turns' products)
      });
    }
    static_for<SETS>([&](auto S) __attribute__((always_inline)) {
      multiply(set[S]);
      if (it + SETS + S < mine) load_next(set[S]);
    });
    static_for<SETS>([&](auto S) __attribute__((always_inline)) {
      if (it + SETS + S < mine) multiply(set[S]);
    });
  } else {
    for (int it = 0; it < mine; ++it) {
      Set s;
      load_next(s);
      multiply(s);
    }
  }
  if ((kbytes & 127) != 0 && wave == chunks % WAVES) {  // the row's last bytes, a multiple of 16
    v4i w[NT][2], x[MT][2][FragOps<MODE>::H];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int64_t at = int64_t(chunks) * 128 + 64 * i + q * 16;
      const int64_t off = at < kbytes ? at : 0;  // (past the row: its first bytes, masked)
      const int keep = at < kbytes ? -1 : 0;
#pragma unroll
      for (int g = 0; g < NT; ++g) {
        const v4i t = *reinterpret_cast<const v4i *>(w0 + int64_t(column(n0 + 16 * g + r) - n0) * kbytes + off);
        w[g][i] = v4i{t.x & keep, t.y & keep, t.z & keep, t.w & keep};
      }
#pragma unroll
      for (int g = 0; g < MT; ++g)
        FragOps<MODE>::unpack(*reinterpret_cast<const v4i *>(p.qx + int64_t(token(16 * g + r)) * kbytes + off), x[g][i]);
    }
    static_for<NT>([&](auto G) __attribute__((always_inline)) { product(w[G][0], w[G][1], x, acc[G]); });
  }

  __syncthreads();  // (the token rows have been read)
  // sums of the waves: [wave][block][lane], 16 bytes each
  uint8_t *const red_i = smem, *const red_f = smem + WAVES * C::BLOCKS * 1024;
  static_for<C::BLOCKS>([&](auto B) __attribute__((always_inline)) {
    *reinterpret_cast<v4i *>(red_i + (wave * C::BLOCKS + B) * 1024 + lane * 16) = acc[B / MT][B % MT];
  });
  if constexpr (FUSED) {
    v4f accf[NT][MT] = {};
    for (int t = wave; t < fsteps; t += WAVES) {
      if (t != wave) load_outlier(t);
      const int keep = t * 64 + q * 16 < fbytes ? -1 : 0;  // (of both: an infinity may stand against a masked zero)
      v4i x[MT];
      static_for<MT>([&](auto J) __attribute__((always_inline)) { x[J] = v4i{fx[J].x & keep, fx[J].y & keep, fx[J].z & keep, fx[J].w & keep}; });
      static_for<NT>([&](auto G) __attribute__((always_inline)) {
        const v4i w = {fw[G].x & keep, fw[G].y & keep, fw[G].z & keep, fw[G].w & keep};
        static_for<MT>([&](auto J) __attribute__((always_inline)) { mma16_outlier<BF16>(x[J], w, accf[G][J]); });
      });
    }
    static_for<C::BLOCKS>([&](auto B) __attribute__((always_inline)) {
      *reinterpret_cast<v4f *>(red_f + (wave * C::BLOCKS + B) * 1024 + lane * 16) = accf[B / MT][B % MT];
    });
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < PW; ++i) {
    const int b = wave + i * WAVES;
    if (b >= C::BLOCKS) break;
    v4i ti = {};
    v4f tf = {};
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      ti += *reinterpret_cast<const v4i *>(red_i + (w * C::BLOCKS + b) * 1024 + lane * 16);
      if constexpr (FUSED) {
        const v4f t = *reinterpret_cast<const v4f *>(red_f + (w * C::BLOCKS + b) * 1024 + lane * 16);
#pragma unroll
        for (int v = 0; v < 4; ++v) tf[v] += t[v];
      }
    }
    const int m = 16 * (b % MT) + r, n = n0 + 16 * (b / MT) + 4 * q;  // four consecutive columns of one token row
    if (m >= p.M || n >= n_end) continue;
    if constexpr (FUSED) {
      const float sr = to_f32<BF16>(e_sr[i]), zs = asym ? to_f32<BF16>(e_zr[i]) + p.shift * sr : 0.0f;
      const float srow = MODE == kInt4 ? sr * 0.00390625f : sr;  // the int4 sums carry a factor of 256
      float val[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const float wr = asym ? to_f32<BF16>(e_wr[i][v]) : 0.0f, bs = p.bias ? to_f32<BF16>(e_bs[i][v]) : 0.0f;
        val[v] = (static_cast<float>(ti[v]) * (srow * to_f32<BF16>(e_sc[i][v])) + tf[v]) + (zs * wr + bs);
      }
      uint16_t *dst = p.out + int64_t(m) * p.ldo + n;
      if (n + 4 <= n_end && (reinterpret_cast<uintptr_t>(dst) & 7) == 0) {
        uint32_t lo = pack2_from_f32<BF16>(val[0], val[1]), hi = pack2_from_f32<BF16>(val[2], val[3]);
        if constexpr (BF16) lo = canonical_bf16_pair(lo), hi = canonical_bf16_pair(hi);
        *reinterpret_cast<uint2 *>(dst) = make_uint2(lo, hi);
      } else {
#pragma unroll
        for (int v = 0; v < 4; ++v)
          if (n + v < n_end) dst[v] = from_f32<BF16>(val[v]);
      }
    } else {
      int32_t *dst = Cm + int64_t(m) * ldc + n;
      const v4i out = MODE == kInt4 ? v4i{ti.x >> 8, ti.y >> 8, ti.z >> 8, ti.w >> 8} : ti;
      if (n + 4 <= n_end && (reinterpret_cast<uintptr_t>(dst) & 15) == 0) {
        *reinterpret_cast<v4i *>(dst) = out;
      } else {
#pragma unroll
        for (int v = 0; v < 4; ++v)
          if (n + v < n_end) dst[v] = out[v];
      }
    }
  }
}

}  // namespace quik
