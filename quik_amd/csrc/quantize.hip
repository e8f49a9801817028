// Per-token activation quantisation for MI355X (gfx950): column map, asymmetric quantize
// with outlier gather, find_meta, quantizeOld and the symmetric quantize.
//
// Arithmetic contract (what the parity tests pin bit for bit):
//   scale = storage(fmaxf((f32(max) - f32(min)) / (2^bits - 1), 1e-6f)), zero = min
//   d     = storage(x - zero)                     one rounding to fp16 / bf16
//   t     = storage(d / scale)                    correctly rounded quotient
//   v     = rne_int(t), NaN -> 0;  code = clamp(v, 0, 2^bits - 1) - 2^(bits-1)
// (reference: src/asymmetric/asymmetric.cu:340-435).
//
// Two kernels implement it.  The streaming kernel (see "Streaming path" below) serves the usual
// layout, ascending int_indices; the gather kernel serves any other order: it copies the row
// to LDS with 16-byte loads while taking min/max over the non-outlier columns (one mask bit per
// column), then each lane gathers two consecutive destination codes per step from LDS through a
// compact source-column table and stores one packed byte (int4) or two bytes (int8).
//
// The quotient.  r = 1/scale is one IEEE division per row.  Pairs of bf16 values take d*r, two roundings
// away (quotient_pair_bf16).  The gather kernel uses q = d*r; e = fma(-q, s, d); q' = fma(e, r, q): q' is within
// 2^-24(1+eps) of d/s relative, while d/s with 11-bit (8-bit for bf16) significands stays more
// than 2^-23 relative away from every rounding boundary of the storage type, so storage(q')
// equals the correctly rounded storage(d/s).  The fp16 streaming path uses fp16(d*r) without
// the correction step: that value can differ from storage(d/s) in the last place (about 1.5e-6
// of all (d, s) pairs) but never across a k + 1/2 boundary, so rne_int gives the same level for
// every fp16 d >= 0 and every fp16 scale >= 1e-6 with both 4 and 8 bits; the tests enumerate
// that whole domain.  Rows whose range overflows the storage type, or whose scale is below
// 1e-20 (bf16 only), take the plain IEEE division instead.
#include <type_traits>

#include "colmap.h"
#include "common.h"
#include "fp6_format.h"
#include "quantize_math.h"

namespace quik {
namespace {

constexpr int kThreads = 256;

// number of non-zero bytes among the low `nbytes` bytes of w
__device__ __forceinline__ uint32_t nonzero_bytes(uint32_t w, int nbytes) {
  uint32_t n = 0;
  for (int b = 0; b < nbytes; ++b) n += ((w >> (8 * b)) & 0xFFu) != 0u;
  return n;
}

// Column map of at most kStreamMaxCols columns: one workgroup of 1024 threads, one 32-column mask word per thread.
//
// The stand-alone quantize gets the index lists with every call, so this kernel stands in front of each of its
// launches and its time is latency, not bandwidth.  The mask lives in LDS, the counts of outliers and of dirty
// groups in front of every word come from one scan over the workgroup (both in one register, 16 bits each), and all
// index loads of a pass are in flight together.  row_major_only: the sections that only operand buffers in tile order
// read (in-place order, units) are left out and the in-place flag stays clear.  Before, every group walked over all mask words in front of it and
// thread 0 walked over all words and units alone: 72 us for 4096 columns with 128 outliers; now 9 us, 6 us
// without the operand sections (the launch alone takes about 2).
struct ColmapOut {
  uint16_t *src_col, *fp_col;
  uint32_t *mask, *grp, *dirty;
  uint16_t *dirty_grp, *kperm;
  uint32_t *patch;
  uint16_t *unit, *gather_unit, *gather_cols;
  uint32_t *flags;
};
constexpr int kBuildThreads = 1024, kBuildBatch = 8;
static_assert(kStreamMaxCols / 32 == kBuildThreads, "one mask word per thread");

// exclusive sum of v over the workgroup (in thread order); `total` = the sum.  parts: one word per wave + 1
__device__ __forceinline__ uint32_t block_scan(uint32_t v, uint32_t *parts, uint32_t &total) {
  constexpr int kWaves = kBuildThreads / 64;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t inc = v;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t up = __shfl_up(inc, d, 64);
    if (lane >= d) inc += up;
  }
  __syncthreads();  // (parts may still be read from the scan before)
  if (lane == 63) parts[wave] = inc;
  __syncthreads();
  uint32_t base = 0, all = 0;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    const uint32_t p = parts[w];
    base += w < wave ? p : 0u;
    all += p;
  }
  total = all;
  return base + inc - v;
}

__global__ __launch_bounds__(kBuildThreads) void colmap_build_kernel(const int64_t *__restrict__ int_idx, int num_int,
                                                                     const int64_t *__restrict__ fp_idx, int num_fp,
                                                                     int cols, ColmapOut o, int row_major_only) {
  __shared__ uint32_t lmask[kBuildThreads + 1];
  __shared__ uint32_t prefix[kBuildThreads + 1];  // in front of word w: outliers | dirty groups << 16
  __shared__ uint32_t parts[kBuildThreads / 64];
  __shared__ int bad;
  const int tid = threadIdx.x, words = (cols + 31) / 32;
  lmask[tid] = 0u;
  if (tid == 0) bad = 0;
  __syncthreads();
  auto clamp = [&](int64_t c) { return static_cast<int>(c < 0 ? 0 : (c >= cols ? cols - 1 : c)); };
  int64_t c[kBuildBatch], next[kBuildBatch];  // (the first batch is requested in front of the outlier list's round trip)
  auto load = [&](int j0) {
#pragma unroll
    for (int b = 0; b < kBuildBatch; ++b) {
      const int j = j0 + b * kBuildThreads;
      c[b] = int_idx[j < num_int ? j : num_int - 1];
      next[b] = int_idx[j + 1 < num_int ? j + 1 : num_int - 1];
    }
  };
  if (num_int > 0) load(tid);
  for (int j = tid; j < num_fp; j += kBuildThreads) {
    const int f = clamp(fp_idx[j]);
    o.fp_col[j] = static_cast<uint16_t>(f);
    atomicOr(&lmask[f >> 5], 1u << (f & 31));
  }
  __syncthreads();
  // int_indices: strictly ascending, in range, none of them an outlier column (the streaming kernels take the integer
  // columns as the complement of the outlier mask, the gather kernels take them from the list)
  bool wrong = false;
  for (int j0 = tid; j0 < num_int; j0 += kBuildThreads * kBuildBatch) {
    if (j0 != tid) load(j0);
#pragma unroll
    for (int b = 0; b < kBuildBatch; ++b) {
      const int j = j0 + b * kBuildThreads;
      if (j >= num_int) continue;
      const int cc = clamp(c[b]);
      if ((j + 1 < num_int && !(c[b] < next[b])) || c[b] != cc || ((lmask[cc >> 5] >> (cc & 31)) & 1u)) wrong = true;
      o.src_col[j] = static_cast<uint16_t>(cc);
    }
  }
  if (wrong) bad = 1;
  const uint32_t word = lmask[tid];
  uint32_t total;
  const uint32_t in_front = block_scan(__popc(word) | (static_cast<uint32_t>(nonzero_bytes(word, 4)) << 16), parts, total);
  prefix[tid] = in_front;
  if (tid == 0) prefix[kBuildThreads] = total;
  if (tid < words) o.mask[tid] = word;
  __syncthreads();
  const bool streams = !bad && cols % 8 == 0 && static_cast<int>(total & 0xFFFFu) == num_fp;
  const bool in_place = streams && !row_major_only && num_int % 32 == 0 && num_fp % 32 == 0;
  // outliers in columns [0, c), c <= cols
  auto before = [&](int c) {
    const uint32_t p = prefix[c >> 5] & 0xFFFFu;
    return static_cast<int>(p + ((c & 31) ? __popc(lmask[c >> 5] & ((1u << (c & 31)) - 1u)) : 0));
  };
  const int holes = in_place ? before(num_int) : 0;  // = integer columns in the tail
  if (in_place) {
    auto is_outlier = [&](int c) { return (lmask[c >> 5] >> (c & 31)) & 1u; };
    uint16_t *hole_col = reinterpret_cast<uint16_t *>(o.patch), *filler_col = hole_col + 1;  // interleaved halves
    for (int c = tid; c < cols; c += kBuildThreads) {
      const int ob = before(c);
      if (c < num_int) {
        if (is_outlier(c)) {
          hole_col[2 * ob] = static_cast<uint16_t>(c);
        } else {
          o.kperm[c] = static_cast<uint16_t>(c - ob);
        }
      } else if (!is_outlier(c)) {
        filler_col[2 * ((c - num_int) - (ob - holes))] = static_cast<uint16_t>(c);
      }
    }
    __syncthreads();
    for (int i = tid; i < holes; i += kBuildThreads) {
      const int f = filler_col[2 * i];
      o.kperm[hole_col[2 * i]] = static_cast<uint16_t>(f - before(f));
    }
  }
  const int groups = (cols + 7) / 8;
  const uint32_t cap = static_cast<uint32_t>(max_dirty_groups(cols, num_fp));
  for (int g = tid; g < groups; g += kBuildThreads) {
    const uint32_t w = lmask[g >> 2], p = prefix[g >> 2];
    const int sh = (g & 3) * 8;
    const uint32_t slot = (p >> 16) + nonzero_bytes(w, g & 3);
    const uint32_t mb = (w >> sh) & 0xFFu;
    const uint32_t dest = static_cast<uint32_t>(g * 8) - ((p & 0xFFFFu) + __popc(w & ((1u << sh) - 1u)));
    if (mb == 0u) {
      o.grp[g] = dest << 8;
    } else {
      o.grp[g] = (slot << 8) | mb;
      if (slot < cap) {
        o.dirty[slot] = (dest << 8) | mb;
        o.dirty_grp[slot] = static_cast<uint16_t>(g);
      }
    }
  }
  // 16-column units of the tile-ordered int8 operand buffers (colmap.h): two per thread
  uint32_t gathered = 0;
  if (streams && !row_major_only && num_int % 16 == 0) {
    const int units = num_int / 16;
    uint32_t c0[2], flag[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int u = 2 * tid + e;
      flag[e] = 0u;
      if (u < units) {
        c0[e] = static_cast<uint32_t>(int_idx[16 * u]);
        flag[e] = static_cast<uint32_t>(int_idx[16 * u + 15]) - c0[e] != 15u ? 1u : 0u;
        o.unit[u] = flag[e] ? uint16_t(0xFFFF) : static_cast<uint16_t>(c0[e]);
      }
    }
    uint32_t n = block_scan(flag[0] + flag[1], parts, gathered);
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      if (!flag[e]) continue;
      const int u = 2 * tid + e;
      if (n < static_cast<uint32_t>(num_fp)) {  // (always: an outlier column lies inside the span of at most one unit)
        o.gather_unit[n] = static_cast<uint16_t>(u);
        for (int t = 0; t < 16; ++t) o.gather_cols[16 * n + t] = static_cast<uint16_t>(int_idx[16 * u + t]);
      }
      ++n;
    }
  }
  if (tid == 0) {
    o.flags[0] = (streams ? 1u : 0u) | (in_place ? 2u : 0u);
    o.flags[1] = total >> 16;
    o.flags[2] = static_cast<uint32_t>(holes);
    o.flags[3] = gathered;
  }
}

// More columns than the streaming kernels take: the gather kernels read src_col, fp_col and the mask only.  One
// workgroup: the mask is cleared before any bit is set.
template <typename IdxT>
__global__ __launch_bounds__(kBuildThreads) void colmap_build_wide_kernel(
    const int64_t *__restrict__ int_idx, int64_t num_int, const int64_t *__restrict__ fp_idx, int64_t num_fp, int64_t cols,
    IdxT *__restrict__ src_col, IdxT *__restrict__ fp_col, uint32_t *__restrict__ mask, uint32_t *__restrict__ flags) {
  auto clamp = [&](int64_t c) { return c < 0 ? 0 : (c >= cols ? cols - 1 : c); };
  for (int64_t w = threadIdx.x; w < (cols + 31) / 32; w += kBuildThreads) mask[w] = 0u;
  for (int64_t j = threadIdx.x; j < num_int; j += kBuildThreads) src_col[j] = static_cast<IdxT>(clamp(int_idx[j]));
  __syncthreads();
  for (int64_t j = threadIdx.x; j < num_fp; j += kBuildThreads) {
    const int64_t c = clamp(fp_idx[j]);
    fp_col[j] = static_cast<IdxT>(c);
    atomicOr(&mask[c >> 5], 1u << (c & 31));
  }
  if (threadIdx.x < 4) flags[threadIdx.x] = 0u;  // (does not stream)
}

// ---------------------------------------------------------------------------------------
// block-wide (min, max) reduction; every thread returns the result
template <int TPR = kThreads>
__device__ __forceinline__ void block_minmax(float &mn, float &mx, float *red) {
  mn = wave_min(mn);
  mx = wave_max(mx);
  __syncthreads();  // protects `red` from the previous use (and orders the callers' LDS row writes)
  if constexpr (TPR > 64) {
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
      red[wave] = mn;
      red[TPR / 64 + wave] = mx;
    }
    __syncthreads();
    mn = red[0];
    mx = red[TPR / 64];
#pragma unroll
    for (int w = 1; w < TPR / 64; ++w) {
      mn = fminf(mn, red[w]);
      mx = fmaxf(mx, red[TPR / 64 + w]);
    }
  }
}

template <typename IdxT, int BITS, bool BF16, int TPR = kThreads>
__device__ __forceinline__ void gather_rows(
    const uint16_t *__restrict__ x, int64_t rows, int64_t cols, const IdxT *__restrict__ src_col,
    const IdxT *__restrict__ fp_col, const uint32_t *__restrict__ mask, int64_t num_int, int64_t num_fp,
    uint8_t *__restrict__ dst, uint16_t *__restrict__ meta, uint16_t *__restrict__ fp_x, int vec_ok,
    uint16_t *row_s, float *red) {
  const int tid = threadIdx.x;
  constexpr float kMaxQ = static_cast<float>((1 << BITS) - 1);
  constexpr uint32_t kFlip = BITS == 4 ? 0x88u : 0x8080u;

  for (int64_t row = blockIdx.x; row < rows; row += gridDim.x) {
    const uint16_t *xr = x + row * cols;
    float mn = __builtin_inff(), mx = -__builtin_inff();
    if (vec_ok) {
      const uint4 *xv = reinterpret_cast<const uint4 *>(xr);
      uint4 *sv = reinterpret_cast<uint4 *>(row_s);
      const int64_t nvec = cols >> 3;
      for (int64_t c8 = tid; c8 < nvec; c8 += TPR) {
        const uint4 v = xv[c8];
        sv[c8] = v;
        uint32_t mb = (mask[c8 >> 2] >> ((c8 & 3) * 8)) & 0xFFu;
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float lo = to_f32<BF16>(static_cast<uint16_t>(w[i] & 0xFFFFu));
          const float hi = to_f32<BF16>(static_cast<uint16_t>(w[i] >> 16));
          if (!(mb & (1u << (2 * i)))) {
            mn = fminf(mn, lo);
            mx = fmaxf(mx, lo);
          }
          if (!(mb & (2u << (2 * i)))) {
            mn = fminf(mn, hi);
            mx = fmaxf(mx, hi);
          }
        }
      }
    } else {
      for (int64_t c = tid; c < cols; c += TPR) {
        const uint16_t v = xr[c];
        row_s[c] = v;
        if (!((mask[c >> 5] >> (c & 31)) & 1u)) {
          const float f = to_f32<BF16>(v);
          mn = fminf(mn, f);
          mx = fmaxf(mx, f);
        }
      }
    }
    block_minmax<TPR>(mn, mx, red);  // also orders the LDS row writes before the gathers below

    RowQuant<BF16> rq;
    rq.init(mn, mx, BITS);
    if (tid == 0) {
      meta[2 * row] = rq.scale_bits;
      meta[2 * row + 1] = rq.zero_bits;
    }

    const int64_t pairs = num_int >> 1;
    if constexpr (BITS == 4) {
      uint8_t *drow = dst + row * pairs;
      for (int64_t p = tid; p < pairs; p += TPR) {
        const IdxT c0 = src_col[2 * p], c1 = src_col[2 * p + 1];
        const uint32_t v0 = RowQuant<BF16>::to_level(rq.quotient(row_s[c0]), kMaxQ);
        const uint32_t v1 = RowQuant<BF16>::to_level(rq.quotient(row_s[c1]), kMaxQ);
        drow[p] = static_cast<uint8_t>((v0 | (v1 << 4)) ^ kFlip);
      }
    } else {
      uint16_t *drow = reinterpret_cast<uint16_t *>(dst + row * num_int);
      for (int64_t p = tid; p < pairs; p += TPR) {
        const IdxT c0 = src_col[2 * p], c1 = src_col[2 * p + 1];
        const uint32_t v0 = RowQuant<BF16>::to_level(rq.quotient(row_s[c0]), kMaxQ);
        const uint32_t v1 = RowQuant<BF16>::to_level(rq.quotient(row_s[c1]), kMaxQ);
        drow[p] = static_cast<uint16_t>((v0 | (v1 << 8)) ^ kFlip);
      }
    }
    if (fp_x != nullptr) {
      uint16_t *frow = fp_x + row * num_fp;
      for (int64_t f = tid; f < num_fp; f += TPR) frow[f] = row_s[fp_col[f]];
    }
    __syncthreads();  // the next row overwrites row_s
  }
}

// ---------------------------------------------------------------------------------------
// Streaming path (ascending int_indices, the layout MixedQLinear.from_float produces).
//
// Works in source order, so nothing is gathered.  Every lane keeps NV 16-byte groups of the row
// in registers.
// All lanes run the same branch-free code on their groups as if they were clean: packed fp16
// min/max (a dirty group's contribution is replaced by the neutral element with one select),
// then 8 codes per group, written as 8 bytes to the group's destination position in an LDS byte
// buffer (only that write is predicated).  Dirty groups are handled a second time by lanes
// 0..ndirty-1, one group each, with per-element masking: that keeps the expensive masked code off
// the all-lanes path, where a divergent branch would make every wave pay for both sides.  Those
// lanes load their group (and every lane its outlier value) straight from the row, right after
// the row's own loads, so the data arrives with them (same cache lines).  A last pass reads 16
// code bytes per lane, packs them to nibbles (int4) and writes 8 or 16 contiguous bytes per lane.
// One row is handled by the TPR threads of one workgroup (a multiple of 64; the launches use 256 and 512),
// which walks over rows blockIdx.x, blockIdx.x + gridDim.x, ...
// SYM: symmetric activations (scale = fp16(max |x| / sym_divisor), one scale per row in meta[row]); fp16 only.

// A lane's row-invariant tables: its NV groups, its first ND dirty groups and outlier columns (so that the per-row loops
// wait on no global load).  Every load is unconditional, from an address that always exists (lanes without an entry read
// the first words of grp): behind a condition each load sits in a branch of its own with its own wait, and the kernel
// starts with one round trip to the L2 after the other.  For the same reason `load` does not wait for the map's flag words:
// it takes as many dirty entries as the map has room for, and `settle` drops those behind the map's own count.
template <int NV, int TPR>
struct StreamTables {
  static constexpr int ND = TPR >= 256 ? 1 : 256 / TPR;
  uint32_t g[NV], dirty[ND], dgrp[ND], fpcol[ND];
  __device__ __forceinline__ void load(const uint32_t *grp, const uint32_t *dirty_map, const uint16_t *dirty_grp,
                                       const uint16_t *fp_col, int64_t cols, int64_t num_fp) {
    const int tid = threadIdx.x, nvec = static_cast<int>(cols >> 3), room = static_cast<int>(max_dirty_groups(cols, num_fp));
    const uint16_t *spare16 = reinterpret_cast<const uint16_t *>(grp);
#pragma unroll
    for (int i = 0; i < NV; ++i) g[i] = grp[tid + i * TPR < nvec ? tid + i * TPR : 0];
#pragma unroll
    for (int k = 0; k < ND; ++k) {
      const int j = tid + k * TPR;
      dirty[k] = *(j < room ? dirty_map + j : grp);
      dgrp[k] = *(j < room ? dirty_grp + j : spare16);
      fpcol[k] = *(j < num_fp ? fp_col + j : spare16);
    }
  }
  // the loads stay in front of whatever follows (the compiler would move them behind a branch that not all paths need
  // them in, and the wait for the branch's condition in front of them)
  __device__ __forceinline__ void pin() {
#pragma unroll
    for (int i = 0; i < NV; ++i) asm volatile("" : "+v"(g[i]));
#pragma unroll
    for (int k = 0; k < ND; ++k) asm volatile("" : "+v"(dirty[k]), "+v"(dgrp[k]), "+v"(fpcol[k]));
  }
  __device__ __forceinline__ void settle(int nvec, int ndirty, int64_t num_fp) {
    const int tid = threadIdx.x;
#pragma unroll
    for (int i = 0; i < NV; ++i) g[i] = tid + i * TPR < nvec ? g[i] : 0xFFFFFFFFu;
#pragma unroll
    for (int k = 0; k < ND; ++k) {
      if (!(tid + k * TPR < ndirty)) dirty[k] = dgrp[k] = 0u;
      if (!(tid + k * TPR < num_fp)) fpcol[k] = 0u;
    }
  }
};

template <int BITS, bool BF16, int NV, int TPR, bool SYM = false, bool PF = false>
__device__ __forceinline__ void stream_rows(const uint16_t *__restrict__ x, int64_t rows, int64_t cols,
                                            StreamTables<NV, TPR> &tables, const uint32_t *__restrict__ dirty,
                                            const uint16_t *__restrict__ dirty_grp, int ndirty,
                                            const uint16_t *__restrict__ fp_col, int64_t num_int, int64_t num_fp,
                                            uint8_t *__restrict__ dst, uint16_t *__restrict__ meta,
                                            uint16_t *__restrict__ fp_x, uint8_t *codes_s, float *red, int vec_out,
                                            float sym_divisor = 1.0f) {
  // vec_out: 0 byte-wise output, 1 16-byte output,
  // 3 (8 bits only): dst is an int8 operand buffer in tile order for gemm_tile8.h, which also takes the outlier
  // values (fp_x is not written); needs num_int % 16 == 0 and num_fp % 32 == 0
  // (the 6-bit operand buffers of gemm_fp6.h are written by quantize_fp6_row_kernel below)
  const Tile8Layout l8 = tile8_layout(rows, num_int, num_fp);
  const bool to8 = BITS == 8 && vec_out == 3;
  const int tid = threadIdx.x;
  const int nvec = static_cast<int>(cols >> 3);
  const float inf = __builtin_inff();
  tables.settle(nvec, ndirty, num_fp);
  constexpr int ND = StreamTables<NV, TPR>::ND;
  const uint32_t(&g)[NV] = tables.g;
  const uint32_t(&my_dirty)[ND] = tables.dirty, (&my_dgrp)[ND] = tables.dgrp, (&my_fpcol)[ND] = tables.fpcol;

  auto load_row = [&](int64_t row, uint4 (&v)[NV]) {
    const uint4 *xv = reinterpret_cast<const uint4 *>(x + row * cols);
#pragma unroll
    for (int i = 0; i < NV; ++i) v[i] = xv[tid + i * TPR < nvec ? tid + i * TPR : nvec - 1];  // (past the end: any group; its g[i] says "not clean")
  };

  // min/max of one dirty group.  fp16: the outlier halves are overwritten with 0xFFFF, a quiet NaN,
  // which the packed min/max skip; bf16: per-element selects on fp32
  auto dirty_minmax = [&](const uint4 &v, uint32_t mb, h2 &pmn, h2 &pmx, float &mn, float &mx) {
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
    if constexpr (!BF16) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const uint32_t lo = static_cast<uint32_t>(__builtin_amdgcn_sbfe(static_cast<int>(mb), 2 * k, 1));
        const uint32_t hi = static_cast<uint32_t>(__builtin_amdgcn_sbfe(static_cast<int>(mb), 2 * k + 1, 1));
        const h2 m = __builtin_bit_cast(h2, w[k] | __builtin_amdgcn_perm(hi, lo, 0x07060100u));
        pmn = __builtin_elementwise_min(pmn, m);
        pmx = __builtin_elementwise_max(pmx, m);
      }
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float f = to_f32<true>(static_cast<uint16_t>(w[e >> 1] >> (16 * (e & 1))));
        const bool out = (mb >> e) & 1u;
        mn = fminf(mn, out ? inf : f);
        mx = fmaxf(mx, out ? -inf : f);
      }
    }
  };
  // SYM: largest |x| pattern of one dirty group, outlier halves zeroed
  auto dirty_absmax = [&](const uint4 &v, uint32_t mb, u2 &amax) {
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint32_t lo = static_cast<uint32_t>(__builtin_amdgcn_sbfe(static_cast<int>(mb), 2 * k, 1));
      const uint32_t hi = static_cast<uint32_t>(__builtin_amdgcn_sbfe(static_cast<int>(mb), 2 * k + 1, 1));
      const uint32_t outl = __builtin_amdgcn_perm(hi, lo, 0x07060100u);  // 0xFFFF in the outlier halves
      amax = __builtin_elementwise_max(amax, __builtin_bit_cast(u2, w[k] & 0x7FFF7FFFu & ~outl));
    }
  };
  // codes of one dirty group, outliers squeezed out
  auto dirty_codes = [&](const uint4 &v, uint32_t info, const RowQuant<BF16> &rq, auto slow_c) {
    constexpr bool SLOW = decltype(slow_c)::value;
    const uint32_t mb = info & 0xFFu;
    const uint2 c = group_codes<BITS, BF16, SLOW, SYM>(v, rq);
    uint8_t *out = codes_s + (info >> 8);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      if (!((mb >> e) & 1u))
        out[e - __popc(mb & ((1u << e) - 1u))] = static_cast<uint8_t>((e < 4 ? c.x : c.y) >> (8 * (e & 3)));
    }
  };

  // one row; `cur` holds its groups, `parity` alternates so that two sets of reduction slots are used
  auto process = [&](int64_t row, const uint4 (&cur)[NV], const uint4 (&dv)[ND], const uint16_t (&fpv)[ND],
                     int parity) {
    const uint4 *xv = reinterpret_cast<const uint4 *>(x + row * cols);
    // ---- all lanes: min / max as if every group were clean
    float mn = inf, mx = -inf;
    const h2 pinf = h2{static_cast<_Float16>(inf), static_cast<_Float16>(inf)};
    h2 pmn = pinf, pmx = -pinf;
    u2 amax = u2{0, 0};  // SYM: largest |x| bit pattern per half (non-negative fp16 patterns order like unsigned integers)
    if constexpr (SYM) {
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const u2 a = __builtin_bit_cast(u2, cur[i].x & 0x7FFF7FFFu), b = __builtin_bit_cast(u2, cur[i].y & 0x7FFF7FFFu);
        const u2 c = __builtin_bit_cast(u2, cur[i].z & 0x7FFF7FFFu), d = __builtin_bit_cast(u2, cur[i].w & 0x7FFF7FFFu);
        const u2 hi = __builtin_elementwise_max(__builtin_elementwise_max(a, b), __builtin_elementwise_max(c, d));
        const bool clean = (g[i] & 0xFFu) == 0u;
        amax = __builtin_elementwise_max(amax, clean ? hi : u2{0, 0});
      }
    } else if constexpr (!BF16) {
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const h2 a = __builtin_bit_cast(h2, cur[i].x), b = __builtin_bit_cast(h2, cur[i].y);
        const h2 c = __builtin_bit_cast(h2, cur[i].z), d = __builtin_bit_cast(h2, cur[i].w);
        const h2 lo = __builtin_elementwise_min(__builtin_elementwise_min(a, b), __builtin_elementwise_min(c, d));
        const h2 hi = __builtin_elementwise_max(__builtin_elementwise_max(a, b), __builtin_elementwise_max(c, d));
        const bool clean = (g[i] & 0xFFu) == 0u;
        pmn = __builtin_elementwise_min(pmn, clean ? lo : pinf);
        pmx = __builtin_elementwise_max(pmx, clean ? hi : -pinf);
      }
    } else {
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const uint32_t w[4] = {cur[i].x, cur[i].y, cur[i].z, cur[i].w};
        float lo = inf, hi = -inf;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const float f0 = __uint_as_float(w[k] << 16), f1 = __uint_as_float(w[k] & 0xFFFF0000u);
          lo = fminf(lo, fminf(f0, f1));
          hi = fmaxf(hi, fmaxf(f0, f1));
        }
        const bool clean = (g[i] & 0xFFu) == 0u;
        mn = fminf(mn, clean ? lo : inf);
        mx = fmaxf(mx, clean ? hi : -inf);
      }
    }
    // ---- outliers, in the caller's order
    auto fp_slot = [&](int64_t f) -> uint16_t * {
      if (to8)
        return reinterpret_cast<uint16_t *>(dst + tile8_offset(l8, row, l8.steps + (f >> 4), static_cast<int>((f >> 3) & 1))) + (f & 7);
      return fp_x + row * num_fp + f;
    };
#pragma unroll
    for (int k = 0; k < ND; ++k)
      if (tid + k * TPR < num_fp) *fp_slot(tid + k * TPR) = fpv[k];
    for (int64_t f = tid + ND * TPR; f < num_fp; f += TPR) *fp_slot(f) = x[row * cols + fp_col[f]];
    // ---- lanes 0 .. ndirty-1: one dirty group each (more when there are more than ND * TPR of them)
    if constexpr (SYM) {
#pragma unroll
      for (int k = 0; k < ND; ++k)
        if (tid + k * TPR < ndirty) dirty_absmax(dv[k], my_dirty[k] & 0xFFu, amax);
      for (int j = tid + ND * TPR; j < ndirty; j += TPR) dirty_absmax(xv[dirty_grp[j]], dirty[j] & 0xFFu, amax);
      mn = 0.0f;
      mx = static_cast<float>(amax.x > amax.y ? amax.x : amax.y);  // a 15-bit integer: exact, ordered like the patterns
    } else {
#pragma unroll
      for (int k = 0; k < ND; ++k)
        if (tid + k * TPR < ndirty) dirty_minmax(dv[k], my_dirty[k] & 0xFFu, pmn, pmx, mn, mx);
      for (int j = tid + ND * TPR; j < ndirty; j += TPR)
        dirty_minmax(xv[dirty_grp[j]], dirty[j] & 0xFFu, pmn, pmx, mn, mx);
      if constexpr (!BF16) {
        mn = fminf(static_cast<float>(pmn.x), static_cast<float>(pmn.y));
        mx = fmaxf(static_cast<float>(pmx.x), static_cast<float>(pmx.y));
      }
    }
    mn = wave_min(mn);
    mx = wave_max(mx);
    if constexpr (TPR > 64) {
      constexpr int NW = TPR / 64;
      float *r = red + parity * 2 * NW;  // two sets: the next row's writes cannot overtake this row's reads
      if ((tid & 63) == 0) {
        r[tid >> 6] = mn;
        r[NW + (tid >> 6)] = mx;
      }
      __syncthreads();
      mn = r[0];
      mx = r[NW];
#pragma unroll
      for (int w = 1; w < NW; ++w) {
        mn = fminf(mn, r[w]);
        mx = fmaxf(mx, r[NW + w]);
      }
    }

    RowQuant<BF16> rq;
    if constexpr (SYM) {
      rq.init_sym(static_cast<uint32_t>(mx), sym_divisor);
      if (tid == 0) meta[row] = rq.scale_bits;
    } else {
      rq.init(mn, mx, BITS);
      if (tid == 0) {
        meta[2 * row] = rq.scale_bits;
        meta[2 * row + 1] = rq.zero_bits;
      }
    }
    // ---- quantise in source order, 8 code bytes per clean group to their destination position
    auto quantise = [&](auto slow_c) {
      constexpr bool SLOW = decltype(slow_c)::value;
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const uint2 c = group_codes<BITS, BF16, SLOW, SYM>(cur[i], rq);
        if ((g[i] & 0xFFu) == 0u) *reinterpret_cast<Bytes8 *>(codes_s + (g[i] >> 8)) = Bytes8{c.x, c.y};
      }
#pragma unroll
      for (int k = 0; k < ND; ++k)
        if (tid + k * TPR < ndirty) dirty_codes(dv[k], my_dirty[k], rq, slow_c);
      for (int j = tid + ND * TPR; j < ndirty; j += TPR) dirty_codes(xv[dirty_grp[j]], dirty[j], rq, slow_c);
    };
    if (__builtin_amdgcn_readfirstlane(rq.slow ? 1 : 0)) {
      quantise(std::true_type{});
    } else {
      quantise(std::false_type{});
    }
    __syncthreads();

    // ---- pack pass: 16 code bytes per lane -> 8 bytes (int4) or 16 bytes (int8)
    const int units = static_cast<int>((num_int + 15) >> 4);
    for (int u = tid; u < units; u += TPR) {
      const uint4 c = *reinterpret_cast<const uint4 *>(codes_s + u * 16);
      const int valid = static_cast<int>(num_int) - u * 16;  // codes of this unit that exist (16 except at the tail)
      if constexpr (BITS == 4) {
        // byte pairs (c0, c1) -> c0 | c1 << 4: t = w | w >> 4 leaves them in bytes 0 and 2
        const uint32_t t0 = c.x | (c.x >> 4), t1 = c.y | (c.y >> 4), t2 = c.z | (c.z >> 4), t3 = c.w | (c.w >> 4);
        const uint2 packed = make_uint2(__builtin_amdgcn_perm(t1, t0, 0x06040200u),
                                        __builtin_amdgcn_perm(t3, t2, 0x06040200u));
        uint8_t *drow = dst + row * (num_int >> 1) + u * 8;
        if (valid >= 16 && vec_out) {
          *reinterpret_cast<uint2 *>(drow) = packed;
        } else {
          for (int b = 0; b < (valid < 16 ? valid : 16) / 2; ++b)
            drow[b] = static_cast<uint8_t>((b < 4 ? packed.x : packed.y) >> (8 * (b & 3)));
        }
      } else {
        uint8_t *drow = to8 ? dst + tile8_offset(l8, row, u >> 1, u & 1) : dst + row * num_int + u * 16;
        if (valid >= 16 && vec_out) {
          *reinterpret_cast<uint4 *>(drow) = c;
        } else {
          for (int b = 0; b < (valid < 16 ? valid : 16); ++b) {
            const uint32_t w = b < 4 ? c.x : (b < 8 ? c.y : (b < 12 ? c.z : c.w));
            drow[b] = static_cast<uint8_t>(w >> (8 * (b & 3)));
          }
        }
      }
    }
  };

  // Without PF: no software prefetch; the launch makes one workgroup per row (up to the grid limit), several of
  // them are resident per CU, and their phases drift apart, so loads, arithmetic and stores of
  // different rows overlap.
  // Tile-ordered output: a cache line of the operand buffer takes pieces of 4 (heads) or 16 (tails) consecutive rows.
  // Workgroups are dealt round-robin to the 8 XCDs, so workgroup w takes row (w % 8) * rows / 8 + w / 8: rows
  // that share lines then run at about the same time on the same XCD and meet in its L2.
  const int64_t per_xcd = (rows + 7) >> 3;
  const int64_t items = to8 ? per_xcd * 8 : rows;
  int parity = 0;
  auto row_of = [&](int64_t w) -> int64_t {
    const int64_t r = to8 ? (w & 7) * per_xcd + (w >> 3) : w;
    return w < items && r < rows ? r : -1;
  };
  auto load_all = [&](int64_t row, uint4 (&v)[NV], uint4 (&dvv)[ND], uint16_t (&fv)[ND]) {
    load_row(row, v);
    const uint4 *xv = reinterpret_cast<const uint4 *>(x + row * cols);
#pragma unroll
    for (int k = 0; k < ND; ++k) {
      dvv[k] = make_uint4(0, 0, 0, 0);
      fv[k] = 0;
      if (tid + k * TPR < ndirty) dvv[k] = xv[my_dgrp[k]];
      if (tid + k * TPR < num_fp) fv[k] = x[row * cols + my_fpcol[k]];
    }
  };
  if constexpr (PF) {
    // Long rows leave room for two workgroups per CU only (registers), so the launch is persistent (a few rows per
    // workgroup) and the next row's loads are issued before the current row's arithmetic: the memory pipeline has
    // work while the workgroup reduces, quantises and stores.
    uint4 cur[NV], nxt[NV], dv[ND], dvn[ND];
    uint16_t fpv[ND], fpvn[ND];
    int64_t w = blockIdx.x;
    int64_t row = row_of(w);
    if (row >= 0) load_all(row, cur, dv, fpv);
    for (; w < items; w += gridDim.x) {
      const int64_t row2 = row_of(w + gridDim.x);
      if (row2 >= 0) load_all(row2, nxt, dvn, fpvn);
      if (row >= 0) {
        parity ^= 1;
        process(row, cur, dv, fpv, parity);
      }
#pragma unroll
      for (int i = 0; i < NV; ++i) cur[i] = nxt[i];
#pragma unroll
      for (int k = 0; k < ND; ++k) {
        dv[k] = dvn[k];
        fpv[k] = fpvn[k];
      }
      row = row2;
    }
  } else {
    for (int64_t w = blockIdx.x; w < items; w += gridDim.x) {
      const int64_t row = row_of(w);
      if (row < 0) continue;
      parity ^= 1;
      uint4 cur[NV], dv[ND];
      uint16_t fpv[ND];
      load_all(row, cur, dv, fpv);
      process(row, cur, dv, fpv, parity);
    }
  }
}

template <typename IdxT, int BITS, bool BF16>
__global__ __launch_bounds__(kThreads) void asym_quantize_kernel(
    const uint16_t *__restrict__ x, int64_t rows, int64_t cols, const IdxT *__restrict__ src_col,
    const IdxT *__restrict__ fp_col, const uint32_t *__restrict__ mask, int64_t num_int, int64_t num_fp,
    uint8_t *__restrict__ dst, uint16_t *__restrict__ meta, uint16_t *__restrict__ fp_x, int vec_ok) {
  extern __shared__ __align__(16) uint16_t row_s[];
  __shared__ float red[8];
  gather_rows<IdxT, BITS, BF16>(x, rows, cols, src_col, fp_col, mask, num_int, num_fp, dst, meta, fp_x, vec_ok, row_s,
                                red);
}

// Shapes that may stream: the column map's flag (known only on the device) picks the path.
// Dynamic LDS: the row (gather path) or one byte per code (streaming path), whichever is larger.
// SYM: symmetric activations; exists on the streaming path only (the host checks the column map's flag first).
template <typename IdxT, int BITS, bool BF16, int NV, int TPR, bool SYM = false, bool PF = false>
__global__ __launch_bounds__(TPR) void asym_quantize_stream_kernel(
    const uint16_t *__restrict__ x, int64_t rows, int64_t cols, const IdxT *__restrict__ src_col,
    const IdxT *__restrict__ fp_col, const uint32_t *__restrict__ mask, const uint32_t *__restrict__ grp,
    const uint32_t *__restrict__ dirty, const uint16_t *__restrict__ dirty_grp, const uint32_t *__restrict__ flags,
    int64_t num_int, int64_t num_fp, uint8_t *__restrict__ dst, uint16_t *__restrict__ meta,
    uint16_t *__restrict__ fp_x, int vec_out, float sym_divisor) {
  static_assert(sizeof(IdxT) == 2, "streaming needs cols <= 32768");
  extern __shared__ __align__(16) uint16_t row_s[];
  __shared__ float red[64];
  // The flag words and the lane's tables in one round trip to memory: the map at this address may be another one at
  // every launch (rebuilt, copied over, replayed in a graph), so the words are the device's, never the host's.
  const uint32_t map_flags = flags[0], ndirty = flags[1];
  StreamTables<NV, TPR> tables;
  tables.load(grp, dirty, dirty_grp, reinterpret_cast<const uint16_t *>(fp_col), cols, num_fp);
  // (with sixteen groups per lane registers count for more: pinned / not, int8 1024 x 28672 27.5 / 26.1 us)
  if constexpr (NV < 16) tables.pin();
  if (map_flags & kColmapStreams) {
    uint8_t *codes_s = reinterpret_cast<uint8_t *>(row_s);
    stream_rows<BITS, BF16, NV, TPR, SYM, PF>(x, rows, cols, tables, dirty, dirty_grp, static_cast<int>(ndirty),
                                              reinterpret_cast<const uint16_t *>(fp_col), num_int, num_fp, dst, meta,
                                              fp_x, codes_s, red, vec_out, sym_divisor);
  } else if constexpr (!SYM) {
    // Tile-ordered output exists on the streaming path only: a column map that does not stream (any other index
    // order) must not reach the row-major gather code with an operand buffer as `dst` and no `fp_x`.  Nothing is
    // written then; the entry points refuse such a column map before launching.
    if (vec_out >= 2) return;
    gather_rows<IdxT, BITS, BF16, TPR>(x, rows, cols, src_col, fp_col, mask, num_int, num_fp, dst, meta, fp_x, 1,
                                       row_s, red);
  }
}

// ---------------------------------------------------------------------------------------
// Rows of more than 16384 columns (the largest down_proj inputs) -> int8 operand buffer in tile order, fp16 input, more rows than CUs.
//
// One workgroup of eight waves per CU walks over its rows; a row is copied global -> LDS with direct copies (no registers, so two rows are in
// flight while a third is worked on) into a ring of two slots.  Per row:
//   wait for this wave's copies of the row, barrier (the row is in LDS)
//   every lane reads its NV groups of 8 columns (and, lanes 0 .. ndirty-1, one group that holds outlier columns;
//   lanes 0 .. num_fp-1 one outlier value, which goes straight to the staging area); barrier (the slot is free)
//   the copies of the row after the next are issued into the slot
//   min / max, barrier, scale and zero
//   8 codes per group -> staging area in SOURCE order (one byte per column, 8 aligned bytes per group; the bytes
//   at outlier columns mean nothing), barrier
//   staging area -> operand buffer in 16-byte units: a unit takes 16 consecutive integer columns, which are 16
//   consecutive staged bytes from an offset that depends on the unit only (the outlier columns in front of it) unless
//   outlier columns lie between them; lanes 0 .. (such units) - 1 gather one of those byte by byte.  The outlier
//   values follow the codes and leave as 16-byte units as well.
// Squeezing the outlier columns out on the way OUT of the staging area keeps every LDS access aligned: 8-byte
// writes at byte offsets that are not multiples of 8 (the compacted position of a group) cost about twice the
// time of aligned ones here, and were half of this kernel's time per row.
// The arithmetic of a row takes less time than its bytes need, so the copies never wait for it; with registers as
// the prefetch target (asym_quantize_stream_kernel's persistent form) two workgroups of four waves fit a CU, a wave
// stalls in the issue of 16 loads per lane while the memory queue is full, and transfer and arithmetic add up.
// Groups past the row's end read 16 bytes of NaN kept behind the slot (min / max skip them).
constexpr int kRingThreads = 512;

// LDS bytes of the ring kernel (host and device agree through these functions)
__host__ __device__ inline int64_t ring_groups_per_lane(int64_t cols) { return (cols / 8 + kRingThreads - 1) / kRingThreads; }
__host__ __device__ inline int64_t ring_slot_bytes(int64_t cols) { return ((cols * 2 + 1023) / 1024) * 1024 + 16; }
__host__ __device__ inline int64_t ring_lds_bytes(int64_t cols, int64_t num_fp) {
  return 2 * ring_slot_bytes(cols) + ring_groups_per_lane(cols) * kRingThreads * 8 + 2 * num_fp + 32 +
         4 * (kRingThreads / 64) * sizeof(float);
}

// codes of the two halves of w in bytes 0 and 2 (int8: code = level - 128 mod 256), rows on the fast path
__device__ __forceinline__ uint32_t ring_code_pair(uint32_t w, h2 zero2, float rcp, uint32_t maxq2) {
  const uint32_t d = __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2, w) - zero2);
  uint32_t tb;
  asm("v_fma_mixlo_f16 %0, %1, %2, 0 op_sel_hi:[1,0,0]\n\t"
      "v_fma_mixhi_f16 %0, %1, %2, 0 op_sel:[1,0,0] op_sel_hi:[1,0,0]"
      : "=&v"(tb)
      : "v"(d), "v"(rcp));
  tb = pk_min_f16(pk_max_f16(tb, 0u), maxq2);  // NaN -> 0
  constexpr _Float16 magic = static_cast<_Float16>(1024 + 128);
  return __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2, tb) + h2{magic, magic});
}

template <int NV>
__global__ __launch_bounds__(kRingThreads) void quantize_tile8_ring_kernel(
    const uint16_t *__restrict__ x, int64_t rows, int64_t cols, const uint16_t *__restrict__ fp_col,
    const uint32_t *__restrict__ grp, const uint32_t *__restrict__ dirty, const uint16_t *__restrict__ dirty_grp,
    const uint16_t *__restrict__ unit, const uint16_t *__restrict__ gather_unit,
    const uint16_t *__restrict__ gather_cols, int ndirty, int ngather, int64_t num_int, int64_t num_fp,
    uint8_t *__restrict__ dst, uint16_t *__restrict__ meta) {
  constexpr int T = kRingThreads, NW = T / 64;
  constexpr int NU = NV / 2 + 1;  // 16-byte units per lane: (codes + outlier values) / 16 / T, at most 512 outliers
  extern __shared__ __align__(16) uint8_t ring_s[];
  treat_all_nans_alike();
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nvec = static_cast<int>(cols >> 3);
  const uint32_t row_bytes = static_cast<uint32_t>(cols) * 2u;
  const uint32_t pieces = (row_bytes + 1023u) >> 10;  // direct copies move 1 KB each
  const uint32_t nan_off = pieces << 10;              // inside a slot: 16 bytes of NaN behind the row
  const uint32_t slot_stride = nan_off + 16u;
  // LDS: slot 0 | slot 1 | codes in source order (8 NV T bytes) | outlier values | 32 spare bytes (the units' second
  // 16-byte read may start there) | reduction slots
  uint8_t *codes_s = ring_s + 2 * slot_stride;
  const uint32_t fp_off = NV * T * 8;
  float *red_s = reinterpret_cast<float *>(codes_s + fp_off + 2 * num_fp + 32);  // [2][2 NW]
  const Tile8Layout l8 = tile8_layout(rows, num_int, num_fp);

  // rows of this workgroup: workgroups are dealt round-robin to the 8 XCDs and the four rows that share the cache
  // lines of the operand buffer should meet in one L2, so XCD k takes the k-th eighth of the rows
  const int64_t per_xcd = (rows + 7) >> 3, stride = gridDim.x >> 3;
  auto row_at = [&](int64_t i) -> int64_t {
    const int64_t idx = (blockIdx.x >> 3) + i * stride;
    const int64_t r = (blockIdx.x & 7) * per_xcd + idx;
    return idx < per_xcd && r < rows ? r : -1;
  };
  const uint32_t ring_lds = lds_address(ring_s);
  // copy k of this wave for a row (every wave issues NV copies per row, the count the waits below rely on: a piece
  // past the last is the last once more)
  auto issue_one = [&](int64_t row, int slot, int k) {
    const uint8_t *src = reinterpret_cast<const uint8_t *>(x + row * cols);
    const uint32_t base = ring_lds + static_cast<uint32_t>(slot) * slot_stride;
    uint32_t piece = static_cast<uint32_t>(wave + NW * k);
    piece = piece < pieces ? piece : pieces - 1u;
    uint32_t off = (piece << 10) + static_cast<uint32_t>(lane) * 16u;
    off = off < row_bytes - 16u ? off : row_bytes - 16u;  // lanes past the row's end repeat its last 16 bytes
    dma_load16(src, off, base + (piece << 10));
  };
  auto issue = [&](int64_t row, int slot) {
#pragma unroll
    for (int k = 0; k < NV; ++k) issue_one(row, slot, k);
  };

  int64_t row = row_at(0);
  if (row < 0) return;
  issue(row, 0);

  // ---- row-invariant tables of this lane, in registers
  // groups: where to read (the NaN block for groups past the row's end) and whether min / max take the group as it
  // is (a group with outlier columns is taken by one of the lanes 0 .. ndirty-1 instead, with those columns masked)
  // (every load is unconditional, from a clamped index: behind a condition each would sit in a branch of its own
  // with its own wait, one round trip to the L2 after the other)
  uint32_t gsrc[NV], keep[NV];
  uint32_t info[NV];
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const int gi = tid + k * T;
    info[k] = grp[gi < nvec ? gi : nvec - 1];
  }
  const bool has_dirty = tid < ndirty, has_fp = tid < num_fp;
  // (lanes without an entry read the first words of grp, which always exist: the other tables may be empty)
  const uint16_t *spare = reinterpret_cast<const uint16_t *>(grp);
  const uint32_t d_info = *(has_dirty ? dirty + tid : grp);
  const uint32_t d_grp = *(has_dirty ? dirty_grp + tid : spare);
  const uint32_t f_col = *(has_fp ? fp_col + tid : spare);
  // units (colmap.h): consecutive columns are 16 consecutive staged bytes from the unit's first column on ("plain");
  // the others are gathered byte by byte, one unit per lane of the first `ngather` lanes
  const int nu_int = static_cast<int>(num_int >> 4), nu = nu_int + static_cast<int>(num_fp >> 3);
  const int unit_pad = static_cast<int>(2 * l8.steps) - nu_int;
  uint32_t ubase[NU], ushift[NU];  // 16-byte-aligned offset into the staging area, byte shift; 0xFFFFFFFF: not plain
  uint32_t ucol[NU];
#pragma unroll
  for (int j = 0; j < NU; ++j) {
    const int u = tid + j * T;
    ucol[j] = unit[u < nu_int ? u : nu_int - 1];  // (num_int >= 64: at least four units)
  }
  const bool has_gather = tid < ngather;
  uint32_t goff[8];  // staged byte offsets (= columns) of the 16 codes of this lane's gathered unit, two per register
  const int gunit = *(has_gather ? gather_unit + tid : spare);
  {
    const uint4 *c = reinterpret_cast<const uint4 *>(has_gather ? gather_cols + 16 * tid : spare);
    const uint4 a = c[0], b = c[1];
    goff[0] = a.x, goff[1] = a.y, goff[2] = a.z, goff[3] = a.w;
    goff[4] = b.x, goff[5] = b.y, goff[6] = b.z, goff[7] = b.w;
  }
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const int gi = tid + k * T;
    gsrc[k] = gi < nvec ? static_cast<uint32_t>(gi) * 16u : nan_off;
    keep[k] = gi >= nvec || (info[k] & 0xFFu) == 0u ? 0xFFFFFFFFu : 0u;
  }
  const uint32_t d_mask = has_dirty ? d_info & 0xFFu : 0xFFu;
  const uint32_t d_src = has_dirty ? d_grp * 16u : nan_off;
  const uint32_t f_src = has_fp ? f_col * 2u : 0u;
#pragma unroll
  for (int j = 0; j < NU; ++j) {
    const int u = tid + j * T;
    uint32_t off = 0xFFFFFFFFu;
    if (u < nu_int) {
      if (ucol[j] != 0xFFFFu) off = ucol[j];
    } else if (u < nu) {
      off = fp_off + static_cast<uint32_t>(u - nu_int) * 16u;
    }
    ubase[j] = off == 0xFFFFFFFFu ? off : off & ~15u;
    ushift[j] = off & 15u;
  }
  if (tid < 4) {
    reinterpret_cast<uint32_t *>(ring_s + nan_off)[tid] = 0xFFFFFFFFu;
    reinterpret_cast<uint32_t *>(ring_s + slot_stride + nan_off)[tid] = 0xFFFFFFFFu;
  }
  // the tables are complete here (this also waits for the first row), not at their first use inside the loop,
  // where a wait for them would wait for the copies in flight as well
#pragma unroll
  for (int k = 0; k < NV; ++k) asm volatile("" ::"v"(gsrc[k]), "v"(keep[k]));
#pragma unroll
  for (int j = 0; j < NU; ++j) asm volatile("" ::"v"(ubase[j]), "v"(ushift[j]));
#pragma unroll
  for (int j = 0; j < 8; ++j) asm volatile("" ::"v"(goff[j]));
  asm volatile("" ::"v"(d_mask), "v"(d_src), "v"(f_src), "v"(gunit));
  {
    const int64_t r1 = row_at(1);
    if (r1 >= 0) issue(r1, 1);
  }

  const uint32_t maxq2 = 0x5BF85BF8u;  // 255.0 in both halves
  for (int64_t i = 0; row >= 0; ++i) {
    const int slot = static_cast<int>(i & 1);
    const int64_t row1 = row_at(i + 1), row2 = row_at(i + 2);
    // This wave's copies of the row have landed.  Memory operations complete in the order of their issue; the NV
    // newest at this point are stores of the last row and, before them, copies of the next row, so "at most NV
    // outstanding" covers the NV copies of this row, which are older than all of those.
    if (row1 >= 0) {
      __builtin_amdgcn_s_waitcnt(vmcnt_imm(NV));
    } else {
      __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
    }
    __syncthreads();
    const uint8_t *slot_s = ring_s + static_cast<uint32_t>(slot) * slot_stride;
    uint4 v[NV];
#pragma unroll
    for (int k = 0; k < NV; ++k) v[k] = *reinterpret_cast<const uint4 *>(slot_s + gsrc[k]);
    const uint4 dv = *reinterpret_cast<const uint4 *>(slot_s + d_src);
    const uint16_t fpv = *reinterpret_cast<const uint16_t *>(slot_s + f_src);
    // (the staging area is free: every wave has finished the last row's stores before the barrier above)
    if (has_fp) reinterpret_cast<uint16_t *>(codes_s + fp_off)[tid] = fpv;
    __syncthreads();

    // ---- min / max; the copies of the row after the next go out between the groups (the address unit takes a
    // copy every 16 cycles: issued in one run, the eight waves would queue behind each other for half a microsecond)
    uint32_t pmn_b = 0x7C007C00u, pmx_b = 0xFC00FC00u;  // +inf / -inf in both halves
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      if (row2 >= 0) issue_one(row2, slot, k);
      const uint32_t lo = pk_min_f16(pk_min_f16(v[k].x, v[k].y), pk_min_f16(v[k].z, v[k].w));
      const uint32_t hi = pk_max_f16(pk_max_f16(v[k].x, v[k].y), pk_max_f16(v[k].z, v[k].w));
      pmn_b = pk_min_f16(pmn_b, (lo & keep[k]) | (0x7C007C00u & ~keep[k]));
      pmx_b = pk_max_f16(pmx_b, (hi & keep[k]) | (0xFC00FC00u & ~keep[k]));
    }
    if (has_dirty) {
      // outlier halves become 0xFFFF, a quiet NaN, which min / max skip
      const uint32_t w[4] = {dv.x, dv.y, dv.z, dv.w};
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const uint32_t lo = static_cast<uint32_t>(__builtin_amdgcn_sbfe(static_cast<int>(d_mask), 2 * k, 1));
        const uint32_t hi = static_cast<uint32_t>(__builtin_amdgcn_sbfe(static_cast<int>(d_mask), 2 * k + 1, 1));
        const uint32_t m = w[k] | __builtin_amdgcn_perm(hi, lo, 0x07060100u);
        pmn_b = pk_min_f16(pmn_b, m);
        pmx_b = pk_max_f16(pmx_b, m);
      }
    }
    const h2 pmn = __builtin_bit_cast(h2, pmn_b), pmx = __builtin_bit_cast(h2, pmx_b);
    float mn = fminf(static_cast<float>(pmn.x), static_cast<float>(pmn.y));
    float mx = fmaxf(static_cast<float>(pmx.x), static_cast<float>(pmx.y));
    mn = wave_min(mn);
    mx = wave_max(mx);
    float *r = red_s + slot * 2 * NW;  // two sets: the next row's writes cannot overtake this row's reads
    if (lane == 0) {
      r[wave] = mn;
      r[NW + wave] = mx;
    }
    __syncthreads();
    mn = r[0];
    mx = r[NW];
#pragma unroll
    for (int w = 1; w < NW; ++w) {
      mn = fminf(mn, r[w]);
      mx = fmaxf(mx, r[NW + w]);
    }
    RowQuant<false> rq;
    rq.init(mn, mx, 8);
    if (tid == 0) {
      meta[2 * row] = rq.scale_bits;
      meta[2 * row + 1] = rq.zero_bits;
    }

    // ---- codes -> staging area, source order
    uint2 *stage8 = reinterpret_cast<uint2 *>(codes_s) + tid;
    if (__builtin_amdgcn_readfirstlane(rq.slow ? 1 : 0)) {
#pragma unroll
      for (int k = 0; k < NV; ++k) stage8[k * T] = group_codes<8, false, true>(v[k], rq);
    } else {
      const _Float16 zh = static_cast<_Float16>(rq.zero);
      const h2 zero2 = h2{zh, zh};
#pragma unroll
      for (int k = 0; k < NV; ++k) {
        const uint32_t p0 = ring_code_pair(v[k].x, zero2, rq.rcp, maxq2), p1 = ring_code_pair(v[k].y, zero2, rq.rcp, maxq2);
        const uint32_t p2 = ring_code_pair(v[k].z, zero2, rq.rcp, maxq2), p3 = ring_code_pair(v[k].w, zero2, rq.rcp, maxq2);
        stage8[k * T] = make_uint2(__builtin_amdgcn_perm(p1, p0, 0x06040200u), __builtin_amdgcn_perm(p3, p2, 0x06040200u));
      }
    }
    __syncthreads();

    // ---- staging area -> operand buffer, 16 bytes per lane and unit
    // chunk (step, h) of the row is at + 2048 step + 16 (h ^ bit 3 of the row) from here (tile8_offset)
    uint8_t *drow = dst + (row >> 6) * l8.block_bytes + ((row >> 5) & 1) * 1024 + (row & 31) * 32;
    const uint32_t swap16 = static_cast<uint32_t>((row >> 3) & 1) << 4;
    auto unit_at = [&](int u) -> uint4 * {
      return reinterpret_cast<uint4 *>(drow + ((static_cast<uint32_t>(u >> 1) << 11) | ((static_cast<uint32_t>(u & 1) << 4) ^ swap16)));
    };
#pragma unroll
    for (int j = 0; j < NU; ++j) {
      if (ubase[j] != 0xFFFFFFFFu) {
        // 16 bytes from byte offset ubase + ushift: two aligned 16-byte reads, then a shift by whole words (two
        // levels of selects) and by bytes
        const uint4 a = *reinterpret_cast<const uint4 *>(codes_s + ubase[j]);
        const uint4 b = *reinterpret_cast<const uint4 *>(codes_s + ubase[j] + 16);
        uint32_t w[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
        // (selects written as bit masks: as conditional moves between array elements the compiler turns them into
        // one dynamically indexed array in scratch memory, whose loads would wait for the copies in flight)
        const uint32_t by2 = 0u - ((ushift[j] >> 3) & 1u), by1 = 0u - ((ushift[j] >> 2) & 1u);
#pragma unroll
        for (int t = 0; t < 6; ++t) w[t] = (w[t + 2] & by2) | (w[t] & ~by2);
#pragma unroll
        for (int t = 0; t < 5; ++t) w[t] = (w[t + 1] & by1) | (w[t] & ~by1);
        uint4 c;
        c.x = __builtin_amdgcn_alignbyte(w[1], w[0], ushift[j]);
        c.y = __builtin_amdgcn_alignbyte(w[2], w[1], ushift[j]);
        c.z = __builtin_amdgcn_alignbyte(w[3], w[2], ushift[j]);
        c.w = __builtin_amdgcn_alignbyte(w[4], w[3], ushift[j]);
        const int u = tid + j * T;  // outlier units start behind the filled-up integer steps
        *unit_at(u < nu_int ? u : u + unit_pad) = c;
      }
    }
    if (has_gather) {
      uint32_t c[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const uint32_t b0 = codes_s[goff[2 * t] & 0xFFFFu], b1 = codes_s[goff[2 * t] >> 16];
        const uint32_t b2 = codes_s[goff[2 * t + 1] & 0xFFFFu], b3 = codes_s[goff[2 * t + 1] >> 16];
        c[t] = b0 | (b1 << 8) | (b2 << 16) | (b3 << 24);
      }
      *unit_at(gunit) = make_uint4(c[0], c[1], c[2], c[3]);
    }
    row = row1;
  }
}

// 4-bit LEVELS (code + 8, 0 .. 15) of the two fp16 halves of w in bytes 0 and 2 of the result, for rows on the fast
// path (finite range, scale >= 1e-6; RowQuant::slow == false); same levels as code_pair gives.
//   asymmetric: d = fp16(x - zero); t = fp16(f32(d) * rcp); t = max(t, 0) (a NaN element becomes 0, as the
//   reference's integer conversion makes it); t + 1024 holds rne(t) in its low mantissa bits.  No upper clamp:
//   on this path t < 15.5 for every fp16 scale (x - zero <= max - min, the scale is at least fp16((max - min) / 15),
//   and over all fp16 scales >= 1e-6 the largest quotient, reached at the smallest, subnormal scale, is 15.47;
//   tests/test_quotient_levels.py enumerates them).
//   symmetric: t = fp16(f32(x) * rcp) with |t| <= 4.2 (scale = fp16(max|x| / 4), at most 3 % below the quotient
//   for the smallest scale); t + 1544 holds rne(t) + 8 in its low mantissa bits.
// (The two v_fma_mix instructions write the low and the high half of one register: the output is early-clobber
// because the second one still reads the inputs after the first has written; VALU to VALU, no wait states needed.)
template <bool SYM, class RQ>
__device__ __forceinline__ uint32_t level_pair_fast(uint32_t w, const RQ &rq) {
  uint32_t d = w, tb;
  if constexpr (!SYM) {
    const _Float16 zh = static_cast<_Float16>(rq.zero);
    d = __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2, w) - h2{zh, zh});
  }
  asm("v_fma_mixlo_f16 %0, %1, %2, 0 op_sel_hi:[1,0,0]\n\t"
      "v_fma_mixhi_f16 %0, %1, %2, 0 op_sel:[1,0,0] op_sel_hi:[1,0,0]"
      : "=&v"(tb)
      : "v"(d), "v"(rq.rcp));
  if constexpr (!SYM) tb = pk_max_f16(tb, 0u);
  constexpr _Float16 magic = static_cast<_Float16>(SYM ? 1544 : 1024);
  return __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2, tb) + h2{magic, magic});
}

// The levels of four bf16 values in the bytes of the result, rows on the fast path.  As above: t = max(t, 0), no upper clamp (x - zero <= max -
// min, rounded up by at most 2^-8, and the scale is at least (max - min) / 15 less 2^-8: the quotient is at most 15.118, t 15.125, which is
// reached: tests/test_quotient_levels_bf16.py), and t + 1.5 2^23 holds rne(t) in its low byte.
// (v_max_f32 by hand: the compiler's fmaxf first quiets an operand that may be a signalling NaN; a converted value is none.  Plain VALU
// instruction, no hazard.)
__device__ __forceinline__ uint32_t level_quad_bf16(uint32_t w0, uint32_t w1, const RowQuant<true> &rq) {
  float t[4];
  rq.quotient_pair_bf16<false>(w0, t[0], t[1]);
  rq.quotient_pair_bf16<false>(w1, t[2], t[3]);
  uint32_t m[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    float c;
    asm("v_max_f32 %0, 0, %1" : "=v"(c) : "v"(t[k]));
    m[k] = __float_as_uint(c + 12582912.0f);
  }
  return __builtin_amdgcn_perm(m[1], m[0], 0x0C0C0400u) | (__builtin_amdgcn_perm(m[3], m[2], 0x0C0C0400u) << 16);
}

// ---- pieces of the kernel that writes 6-bit operand buffers (quantize_fp6_row_kernel)

// Byte offset of source column c inside a row image in LDS.  A copy instruction moves one contiguous kilobyte (64 groups
// of 8 columns = 16 fragments of 32 consecutive columns; whole cache lines) and deals it to the LDS slots transposed:
// slot 16 i + m of the kilobyte holds group 4 m + i, i.e. the i-th group of the kilobyte's fragment m.  The i-th 16-byte
// reads of 16 neighbouring fragments cover 256 consecutive bytes, so all reads are free of bank conflicts.
__device__ __forceinline__ uint32_t img_of_col(uint32_t c) {
  const uint32_t g = c >> 3, f = g >> 2, i = g & 3u;
  return ((f >> 4) << 10) + ((16u * i + (f & 15u)) << 4) + ((c & 7u) << 1);
}
// the four groups of fragment f
__device__ __forceinline__ void img_fragment(const uint8_t *img, int f, uint4 (&v)[4]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = *reinterpret_cast<const uint4 *>(img + ((f >> 4) << 10) + ((16 * i + (f & 15)) << 4));
}
// address of the row, in scalar registers
// (the intrinsic returns int: each half goes through uint32_t, or the low half would be sign-extended)
__device__ __forceinline__ const uint8_t *uniform_row(const uint16_t *x, int64_t row, int cols) {
  const uint64_t a = reinterpret_cast<uint64_t>(x + row * cols);
  const uint32_t a_hi = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(a >> 32)));
  const uint32_t a_lo = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(a & 0xFFFFFFFFu)));
  return reinterpret_cast<const uint8_t *>((static_cast<uint64_t>(a_hi) << 32) | a_lo);
}

// Running min / max (symmetric: largest |x| pattern) over fragments.
template <bool BF16, bool SYM>
struct FragmentRange {
  float mn = __builtin_inff(), mx = -__builtin_inff();
  uint32_t pmn = 0x7C007C00u, pmx = 0xFC00FC00u;  // fp16: +inf / -inf in both halves
  u2 amax = u2{0, 0};
  __device__ __forceinline__ void add(const uint4 (&v)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t w[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
      if constexpr (SYM) {
#pragma unroll
        for (int k = 0; k < 4; ++k) amax = __builtin_elementwise_max(amax, __builtin_bit_cast(u2, w[k] & 0x7FFF7FFFu));
      } else if constexpr (!BF16) {
        // packed fp16 min / max skip NaN operands, as the reference's __hmin / __hmax do
        pmn = pk_min_f16(pmn, pk_min_f16(pk_min_f16(w[0], w[1]), pk_min_f16(w[2], w[3])));
        pmx = pk_max_f16(pmx, pk_max_f16(pk_max_f16(w[0], w[1]), pk_max_f16(w[2], w[3])));
      } else {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const float f0 = __uint_as_float(w[k] << 16), f1 = __uint_as_float(w[k] & 0xFFFF0000u);
          mn = fminf(mn, fminf(f0, f1));
          mx = fmaxf(mx, fmaxf(f0, f1));
        }
      }
    }
  }
  // wave-wide (lo, hi); symmetric: hi is the largest pattern, a 15-bit integer (exact, ordered like the patterns)
  __device__ __forceinline__ void reduce(float &lo, float &hi) const {
    const h2 a = __builtin_bit_cast(h2, pmn), b = __builtin_bit_cast(h2, pmx);
    lo = SYM ? 0.0f : BF16 ? mn : fminf(static_cast<float>(a.x), static_cast<float>(a.y));
    hi = SYM ? static_cast<float>(amax.x > amax.y ? amax.x : amax.y)
             : BF16 ? mx : fmaxf(static_cast<float>(b.x), static_cast<float>(b.y));
    lo = wave_min(lo);
    hi = wave_max(hi);
  }
};

// Scale and zero of a row from its range, written to meta by the one thread that says so.
template <bool BF16, bool SYM>
__device__ __forceinline__ RowQuant<BF16> row_quant4(float lo, float hi, float sym_divisor, bool writes, uint16_t *meta,
                                                     int64_t row) {
  RowQuant<BF16> rq;
  if constexpr (SYM) {
    rq.init_sym(static_cast<uint32_t>(hi), sym_divisor);
    if (writes) meta[row] = rq.scale_bits;
  } else {
    rq.init(lo, hi, 4);
    if (writes) {
      meta[2 * row] = rq.scale_bits;
      meta[2 * row + 1] = rq.zero_bits;
    }
  }
  return rq;
}

// Where the row's fragments go in the operand buffer: the row's part of the address is wave-uniform, the fragment's part is
// the unit f / 2 and its half.
// (4-bit format: the unit is 2048 bytes and has no tails)
template <bool FOUR>
struct Fp6RowOut {
  static constexpr uint32_t kUnit = FOUR ? 2048u : 3072u;
  uint8_t *head, *tail;
  uint32_t swap16;
  template <class Layout>
  __device__ __forceinline__ Fp6RowOut(uint8_t *dst, const Layout &l, int64_t row) {
    uint8_t *rb = dst + (row >> 6) * l.block_bytes;
    head = rb + ((row >> 5) & 1) * 1024 + (row & 31) * 32;
    tail = rb + 2048 + (row & 63) * 8;
    swap16 = static_cast<uint32_t>((row >> 3) & 1) << 4;
  }
};

// One fragment: 32 values -> 32 levels -> 24 bytes (16 in the 4-bit format), stored; returns the sum of its levels.
template <bool BF16, bool SYM, bool SLOW, bool FOUR>
__device__ __forceinline__ int quantise_fragment(const uint4 (&v)[4], const RowQuant<BF16> &rq, int f, const Fp6RowOut<FOUR> &out) {
  uint32_t b[8];  // 32 levels, one per byte
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if constexpr (!SLOW && !BF16) {
      const uint32_t p0 = level_pair_fast<SYM>(v[i].x, rq), p1 = level_pair_fast<SYM>(v[i].y, rq);
      const uint32_t p2 = level_pair_fast<SYM>(v[i].z, rq), p3 = level_pair_fast<SYM>(v[i].w, rq);
      b[2 * i] = __builtin_amdgcn_perm(p1, p0, 0x06040200u);  // bytes 0, 2 of p0 then bytes 0, 2 of p1
      b[2 * i + 1] = __builtin_amdgcn_perm(p3, p2, 0x06040200u);
    } else if constexpr (!SLOW) {
      b[2 * i] = level_quad_bf16(v[i].x, v[i].y, rq);
      b[2 * i + 1] = level_quad_bf16(v[i].z, v[i].w, rq);
    } else {
      const uint2 c = group_codes<4, BF16, SLOW, SYM>(v[i], rq);  // code nibbles (two's complement), one per byte
      b[2 * i] = c.x ^ 0x08080808u;                               // level = code + 8
      b[2 * i + 1] = c.y ^ 0x08080808u;
    }
  }
  int sum = 0;
#pragma unroll
  for (int i = 0; i < 8; ++i) sum = __builtin_amdgcn_udot4(b[i], 0x01010101u, sum, false);
  uint32_t o[6];
  fp6_pack_fragment(b, o);
  const uint32_t unit = static_cast<uint32_t>(f >> 1) * out.kUnit, h = static_cast<uint32_t>(f & 1);
  // (default cache policy: a 128-byte line of the operand buffer takes pieces of 4 (heads) or 16 (tails) rows,
  // which meet in the XCD's L2; as streaming stores every piece went to memory on its own and the launch
  // took 29 us instead of 12)
  if constexpr (FOUR) {
    *reinterpret_cast<uint4 *>(out.head + unit + ((h << 4) ^ out.swap16)) = nib_squeeze(o);
  } else {
    *reinterpret_cast<uint4 *>(out.head + unit + ((h << 4) ^ out.swap16)) = make_uint4(o[0], o[1], o[2], o[3]);
    *reinterpret_cast<uint2 *>(out.tail + unit + h * 512u) = make_uint2(o[4], o[5]);
  }
  return sum;
}

// ---------------------------------------------------------------------------------------
// 6-bit operand buffers (consumer: gemm_fp6.h), written in the in-place order of the column map.
//
// One workgroup per row; a lane owns JT fragments of 32 columns, one for rows of up to 16384 columns (a wave per 2048
// columns).  The row is copied global -> LDS with direct copies (no registers are held while it is in flight).  In the image
// the holes (outlier columns among the first num_int columns) are overwritten with their fillers (integer columns of the
// tail); after that the first num_int columns ARE the integer operand, in place: a lane reads its fragment once, takes
// part in the reduction of the range, turns the fragment into 32 levels in registers, packs them to 24 bytes and stores
// head and tail.
//
// What bounds a launch is the chain of one row (launch, transfer, range, levels, stores) as long as the rows are few, the
// memory system from about 2000 rows on.  A wave per row, two or eight of them in a workgroup and without any barrier, was
// the form before: its two passes over up to five fragments per lane stood behind the transfer, and 64 rows occupied 64 of
// 1024 SIMDs.  Here a pass takes as long as one fragment, for four barriers (image landed, outlier values read, holes
// patched, range exchanged).  us per launch in a graph of twenty on one input, wave per row -> this, 256 outlier columns, fp16:
// 16 x 4096 4.1 -> 3.5, 64 x 8192 5.3 -> 3.7, 128 x 5120 4.7 -> 3.6, 777 x 4096 5.4 -> 4.6, 1024 x 8192 7.9 -> 6.7, 8192 x 8192
// 36.2 -> 31.0, 64 x 28672 12.5 -> 5.6, 2048 x 28672 56.8 -> 32.5; bf16 64 x 8192 9.6 -> 4.2, 777 x 4096 8.7 -> 5.5, 2048 x 28672
// 115 -> 42 (with the rounding of quotient_pair_bf16).
// Slower where the wave form's rows were all resident and each CU had seven or eight of them: 2048 x 8192 10.9 -> 11.3, and fewer
// columns if the input does not come from the cache's last launch (one input / four in turn / 600 MB in turn: 2048 x 4096 6.8 /
// 7.8 / 8.3 -> 6.8 / 8.3 / 9.0, 2048 x 5120 8.7 / 9.2 / 9.9 -> 8.4 / 9.7 / 10.3, 1537 x 4096 6.5 / 7.1 / 7.4 -> 6.2 / 7.4 / 7.9); from nine
// rows per CU on a quarter faster (2304 x 4096 9.9 / 11.3 / 12.5 -> 7.5 / 8.9 / 9.4).  Kept for these counts beside this one, on the
// same pieces, the wave form took 7.3 / 7.8 / 8.5 at 2048 x 4096.
// (Fillers read beside the outlier values and the ranges of all waves in one LDS round trip, not one after the other:
// 64 x 8192 3.68 -> 3.57, 2048 x 8192 12.3 -> 12.1, 64 x 28672 5.71 -> 5.48.)
// (arguments in the order in which they are needed: the first sixteen words are there when a wave starts, the Makefile's
// kernarg-preload-count)
template <bool BF16, bool SYM, int JT, bool FOUR>
__global__ __launch_bounds__(512) void quantize_fp6_row_kernel(
    const uint16_t *__restrict__ x, int64_t first, int count, int cols, const uint32_t *__restrict__ patch,
    const uint16_t *__restrict__ fp_col, int nholes, int num_fp, int num_int, float sym_divisor, uint8_t *__restrict__ dst,
    int64_t rows, uint16_t *__restrict__ meta) {
  static_assert(!(BF16 && SYM), "symmetric activations are fp16");
  extern __shared__ __align__(16) uint8_t img[];
  __shared__ __align__(16) float red[16];  // minimum and maximum of up to eight waves
  __shared__ uint32_t total_s;
  if constexpr (!BF16 && !SYM) treat_all_nans_alike();  // the range uses pk_min_f16 / pk_max_f16 on the raw row
  // (nholes: the column map's count of holes, which the host knows: the entry points look the map's flag words up
  // before launching, and refuse a map without the in-place order; the kernel starts without a dependent load)
  const int tid = threadIdx.x, lane = tid & 63, T = blockDim.x, W = T >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int frags = num_int >> 5, nchunk = num_fp >> 3;
  // Rows [first, first + count); workgroup g takes number (g % 8) * count / 8 + g / 8: a cache line of the operand buffer takes pieces of 4 (heads) or 16
  // (tails) consecutive rows; workgroups are dealt round-robin to the 8 XCDs, so rows that share lines run on the same XCD
  // at about the same time and meet in its L2.
  const int per_xcd = (count + 7) >> 3, at = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if (at >= count) return;
  const int64_t row = first + at;
  {
    const uint8_t *rp = uniform_row(x, row, cols);
    const uint32_t lds0 = lds_address(img);
    const int g_in = 4 * (lane & 15) + (lane >> 4), g_last = (cols >> 3) - 1;
#pragma unroll
    for (int j = 0; j < JT; ++j)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int q = 4 * (wave + j * W) + t, g = 64 * q + g_in;
        dma_load16(rp, static_cast<uint32_t>(g < g_last ? g : g_last) * 16u, lds0 + q * 1024);  // past the row: any valid group
      }
  }
  // (unconditional loads, in flight together with the row)
  constexpr int PREG = 2;
  uint32_t pe[PREG];
#pragma unroll
  for (int k = 0; k < PREG; ++k) pe[k] = patch[tid + k * T < nholes ? tid + k * T : 0];
  const uint4 oc = *reinterpret_cast<const uint4 *>(fp_col + (tid < nchunk ? tid : 0) * 8);
  if (tid == 0) total_s = 0;
  if (tid < 8 && tid >= W) red[tid] = __builtin_inff(), red[8 + tid] = -__builtin_inff();
  const auto layout = [&] {
    if constexpr (FOUR) {
      return tile4_layout(rows, num_int, num_fp);
    } else {
      return fp6_layout(rows, num_int, num_fp);
    }
  };
  const auto l6 = layout();
  auto outlier_offset = [&](int c) {
    if constexpr (FOUR) {
      return tile4_offset(l6, row, l6.steps + (c >> 1), c & 1);
    } else {
      return fp6_outlier_offset(l6, row, c >> 1, c & 1);
    }
  };
  __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
  __syncthreads();

  auto ld16 = [&](uint32_t c) -> uint32_t { return *reinterpret_cast<const uint16_t *>(img + img_of_col(c)); };
  // outlier values first: holes are outlier columns
  auto outliers = [&](int c, const uint4 &cols8) {
    const uint32_t ow[4] = {cols8.x, cols8.y, cols8.z, cols8.w};
    uint32_t o[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) o[k] = ld16(ow[k] & 0xFFFFu) | (ld16(ow[k] >> 16) << 16);
    *reinterpret_cast<uint4 *>(dst + outlier_offset(c)) = make_uint4(o[0], o[1], o[2], o[3]);
  };
  uint32_t filler[PREG];  // read together with the outlier values: integer columns, none of them is a hole
#pragma unroll
  for (int k = 0; k < PREG; ++k) filler[k] = ld16(tid + k * T < nholes ? pe[k] >> 16 : 0);
  if (tid < nchunk) outliers(tid, oc);
  for (int c = tid + T; c < nchunk; c += T) outliers(c, *reinterpret_cast<const uint4 *>(fp_col + c * 8));
  __syncthreads();
  // holes <- fillers
  auto fill = [&](uint32_t e, uint32_t value) {
    *reinterpret_cast<uint16_t *>(img + img_of_col(e & 0xFFFFu)) = static_cast<uint16_t>(value);
  };
#pragma unroll
  for (int k = 0; k < PREG; ++k)
    if (tid + k * T < nholes) fill(pe[k], filler[k]);
  for (int e = tid + PREG * T; e < nholes; e += T) fill(patch[e], ld16(patch[e] >> 16));
  __syncthreads();

  FragmentRange<BF16, SYM> range;
  uint4 v[JT][4];
#pragma unroll
  for (int j = 0; j < JT; ++j)
    if (tid + j * T < frags) {
      img_fragment(img, tid + j * T, v[j]);
      range.add(v[j]);
    }
  float mn, mx;
  range.reduce(mn, mx);
  if (lane == 0) {
    red[wave] = mn;
    red[8 + wave] = mx;
  }
  __syncthreads();
  // all eight slots in one round trip to the LDS (those of waves that are not there are neutral)
  float part[16];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const float4 r = *reinterpret_cast<const float4 *>(red + 4 * k);
    part[4 * k] = r.x, part[4 * k + 1] = r.y, part[4 * k + 2] = r.z, part[4 * k + 3] = r.w;
  }
#pragma unroll
  for (int w = 0; w < 8; ++w) {
    mn = fminf(mn, part[w]);
    mx = fmaxf(mx, part[8 + w]);
  }
  const RowQuant<BF16> rq = row_quant4<BF16, SYM>(mn, mx, sym_divisor, tid == 0, meta, row);
  const Fp6RowOut<FOUR> out(dst, l6, row);
  int sum = 0;
  auto quantise = [&](auto slow_c) {
#pragma unroll
    for (int j = 0; j < JT; ++j)
      if (tid + j * T < frags)
        sum += quantise_fragment<BF16, SYM, decltype(slow_c)::value, FOUR>(v[j], rq, tid + j * T, out);
  };
  if (__builtin_amdgcn_readfirstlane(rq.slow ? 1 : 0)) {
    quantise(std::true_type{});
  } else {
    quantise(std::false_type{});
  }
  // the wave that adds its sum last writes the row's: count in the high byte, sums below 2^19 (32768 columns of level 15)
  sum = wave_sum(sum);
  if (lane == 0) {
    const uint32_t mine = (1u << 24) | static_cast<uint32_t>(sum);
    const uint32_t all = __hip_atomic_fetch_add(&total_s, mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) + mine;
    if ((all >> 24) == static_cast<uint32_t>(W))
      reinterpret_cast<int32_t *>(dst + l6.sums_off)[row] = static_cast<int32_t>(all & 0xFFFFFFu);
  }
}

// ---------------------------------------------------------------------------------------
// Rows -> row-major codes of a layer's few rows (calls of the weight-streaming GEMM, gemm_skinny.h), or int8 operand buffers in tile order, a
// workgroup of eight waves per row.
//
// What bounds such a launch is the chain of one row.  asym_quantize_stream_kernel makes two trips to memory, one for the lane's tables and
// one for the groups and values that they name, and writes the codes at odd places of the LDS.  Here the row goes to the LDS beside the
// one trip for all tables, a lane has its groups of 8 columns whole, outliers masked, and what is squeezed is read on the way out: the codes
// lie in source order, 16 integer columns that follow each other are two aligned reads and a shift (the column map's units), the others
// are gathered by the byte.  The same arithmetic.
// us per forward, asym_quantize_stream_kernel / this: int4 4 x 2048 -> 4096 7.0 / 6.6, 8 x 4096 -> 4096 7.55 / 7.35, 16 x 8192 -> 8192 12.5 / 11.9,
// 3 x 13824 -> 5120 13.9 / 13.1, 16 x 8192 -> 28672 27.5 / 26.9, bf16 8 x 4096 -> 4096 7.95 / 7.5, int8 16 x 13824 -> 5120 19.4 / 18.5, 24 x
// 28672 -> 8192 43.7 / 42.05.  Tile order: 64 x 4096 -> 4096 11.1 / 10.6, 64 x 8192 -> 8192 18.25 / 17.55, 256 x 4096 -> 4096 14.95 / 14.3, 1024 x 13824 ->
// 512 36.5 / 35.4, 2048 x 8192 -> 512 32.4 / 30.9, 8192 x 4096 -> 512 56.0 / 54.9, bf16 64 x 11008 -> 4096 18.6 / 18.0, 2048 x 13824 -> 512 51.85 / 48.0,
// 1536 x 28672 -> 512 97.25 / 95.3; against quantize_tile8_ring_kernel: see asym_quantize_tile8.
constexpr int kUnitThreads = 512, kFewRows = 32;
__host__ __device__ inline int64_t unit_raw_bytes(int64_t cols) { return (cols * 2 + 1023) / 1024 * 1024; }
__host__ __device__ inline int64_t unit_lds_bytes(int64_t cols) { return unit_raw_bytes(cols) + (cols + 47) / 16 * 16; }

// TILED (int8): into an operand buffer in tile order (gemm_tile8.h), outlier values included.
// SYM: symmetric activations, one scale per row, fp16; row-major only.
template <int BITS, bool BF16, int NV, bool TILED, bool SYM = false>
__global__ __launch_bounds__(kUnitThreads) void quantize_units_kernel(
    const uint16_t *__restrict__ x, const uint32_t *__restrict__ grp, const uint16_t *__restrict__ unit, int cols, int num_int, int num_fp,
    int rows, const uint16_t *__restrict__ fp_col, const uint16_t *__restrict__ gather_unit, const uint16_t *__restrict__ gather_cols,
    const uint32_t *__restrict__ flags, uint8_t *__restrict__ dst, uint16_t *__restrict__ fp_x, uint16_t *__restrict__ meta,
    const uint16_t *__restrict__ src_col, const uint32_t *__restrict__ mask, float sym_divisor) {
  extern __shared__ __align__(16) uint8_t lds[];
  __shared__ __align__(16) float red[64];
  static_assert(!SYM || (!BF16 && !TILED), "symmetric activations: fp16, row-major");
  constexpr int T = kUnitThreads, W = T / 64, NU = (NV + 1) / 2;
  static_assert(!TILED || BITS == 8, "tile order: int8");
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // (tile order: rows that share cache lines of the operand buffer on one XCD)
  const int row = TILED ? (blockIdx.x & 7) * ((rows + 7) >> 3) + (blockIdx.x >> 3) : blockIdx.x;
  if (row >= rows) return;
  const int nvec = cols >> 3, nu = num_int >> 4;
  uint8_t *const raw = lds, *const stage = lds + unit_raw_bytes(cols);
  {
    const uint8_t *rp = uniform_row(x, row, cols);
    const uint32_t lds0 = lds_address(raw);
#pragma unroll
    for (int k = 0; k < NV; ++k) {  // (a kilobyte per wave and turn, past the row: its last group)
      const int q = wave + k * W, g = q * 64 + lane;
      if (q * 64 < nvec) dma_load16(rp, static_cast<uint32_t>(g < nvec ? g : nvec - 1) * 16u, lds0 + q * 1024);
    }
  }
  // (unconditional loads from valid addresses, in flight together)
  uint32_t info[NV], first[NU];
#pragma unroll
  for (int k = 0; k < NV; ++k) info[k] = grp[tid + k * T < nvec ? tid + k * T : 0];
#pragma unroll
  for (int k = 0; k < NU; ++k) first[k] = unit[tid + k * T < nu ? tid + k * T : 0];
  const uint16_t *const spare = reinterpret_cast<const uint16_t *>(grp);  // (always there; the other tables may be empty)
  const bool has_f = tid < num_fp;  // (at most num_fp gathered units)
  const uint32_t gunit = *(has_f ? gather_unit + tid : spare), fcol = *(has_f ? fp_col + tid : spare);
  const uint4 *const gc = reinterpret_cast<const uint4 *>(has_f ? gather_cols + 16 * tid : spare);
  const uint4 ga = gc[0], gb = gc[1];
  // The device's words: the map at this address may be another one at every launch.  (A vector load, beside the others: as a scalar one
  // it is waited for with the arguments, 16 x 8192 -> 8192 12.0 instead of 11.85 us per forward.)
  uint32_t none = 0;
  asm volatile("" : "+v"(none));
  const uint4 words = reinterpret_cast<const uint4 *>(flags)[none];
  __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
  __syncthreads();
  const uint32_t map_flags = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(words.x)));
  const uint32_t ngather = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(words.w)));
  if (!(map_flags & kColmapStreams)) {  // any other order of the columns (tile order, SYM: refused before the launch, nothing is written)
    if constexpr (!TILED && !SYM)
      gather_rows<uint16_t, BITS, BF16, T>(x, rows, cols, src_col, fp_col, mask, num_int, num_fp, dst, meta, fp_x, 1, reinterpret_cast<uint16_t *>(lds), red);
    return;
  }
  if constexpr (!BF16 && !SYM) treat_all_nans_alike();  // pk_min_f16 / pk_max_f16 on the raw row

  auto value = [&](uint32_t c) { return reinterpret_cast<const uint16_t *>(raw)[c]; };
  const Tile8Layout l8 = tile8_layout(rows, num_int, num_fp);
  auto outlier = [&](int f) -> uint16_t * {
    if constexpr (TILED)
      return reinterpret_cast<uint16_t *>(dst + tile8_offset(l8, row, l8.steps + (f >> 4), (f >> 3) & 1)) + (f & 7);
    return fp_x + static_cast<int64_t>(row) * num_fp + f;
  };
  if (has_f) *outlier(tid) = value(fcol);
  for (int f = tid + T; f < num_fp; f += T) *outlier(f) = value(fp_col[f]);
  uint4 v[NV];
  uint32_t pmn = 0x7C007C00u, pmx = 0xFC00FC00u;
  u2 amax = u2{0, 0};  // SYM: largest |x| pattern (a NaN's is larger than any number's)
  float mn = __builtin_inff(), mx = -__builtin_inff();
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const int g = tid + k * T;
    v[k] = *reinterpret_cast<const uint4 *>(raw + (g < nvec ? g : 0) * 16);
    const uint32_t w[4] = {v[k].x, v[k].y, v[k].z, v[k].w}, skip = g < nvec ? info[k] : 0xFFu;  // (bit e: column e is an outlier)
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const uint32_t lo = static_cast<uint32_t>(__builtin_amdgcn_sbfe(static_cast<int>(skip), 2 * t, 1));
      const uint32_t hi = static_cast<uint32_t>(__builtin_amdgcn_sbfe(static_cast<int>(skip), 2 * t + 1, 1));
      if constexpr (SYM) {
        amax = __builtin_elementwise_max(amax, __builtin_bit_cast(u2, w[t] & 0x7FFF7FFFu & ~__builtin_amdgcn_perm(hi, lo, 0x07060100u)));
      } else if constexpr (!BF16) {
        const uint32_t m = w[t] | __builtin_amdgcn_perm(hi, lo, 0x07060100u);  // outliers: a NaN, which is skipped
        pmn = pk_min_f16(pmn, m), pmx = pk_max_f16(pmx, m);
      } else {
        const float f0 = __uint_as_float((w[t] << 16) | lo), f1 = __uint_as_float((w[t] & 0xFFFF0000u) | hi);
        mn = fminf(mn, fminf(f0, f1)), mx = fmaxf(mx, fmaxf(f0, f1));
      }
    }
  }
  if constexpr (SYM) {
    mn = 0.0f, mx = static_cast<float>(amax.x > amax.y ? amax.x : amax.y);  // a 15-bit integer: exact
  } else if constexpr (!BF16) {
    const h2 a = __builtin_bit_cast(h2, pmn), b = __builtin_bit_cast(h2, pmx);
    mn = fminf(static_cast<float>(a.x), static_cast<float>(a.y)), mx = fmaxf(static_cast<float>(b.x), static_cast<float>(b.y));
  }
  mn = wave_min(mn), mx = wave_max(mx);
  if (lane == 0) red[wave] = mn, red[W + wave] = mx;
  __syncthreads();
  float part[2 * W];
#pragma unroll
  for (int k = 0; k < 2 * W / 4; ++k) {
    const float4 r = *reinterpret_cast<const float4 *>(red + 4 * k);
    part[4 * k] = r.x, part[4 * k + 1] = r.y, part[4 * k + 2] = r.z, part[4 * k + 3] = r.w;
  }
#pragma unroll
  for (int w = 0; w < W; ++w) mn = fminf(mn, part[w]), mx = fmaxf(mx, part[W + w]);
  RowQuant<BF16> rq;
  if constexpr (SYM) {
    rq.init_sym(static_cast<uint32_t>(mx), sym_divisor);
    if (tid == 0) meta[row] = rq.scale_bits;
  } else {
    rq.init(mn, mx, BITS);
    if (tid == 0) meta[2 * row] = rq.scale_bits, meta[2 * row + 1] = rq.zero_bits;
  }
  auto codes = [&](auto slow_c) {
#pragma unroll
    for (int k = 0; k < NV; ++k)
      if (tid + k * T < nvec) *reinterpret_cast<uint2 *>(stage + (tid + k * T) * 8) = group_codes<BITS, BF16, decltype(slow_c)::value, SYM>(v[k], rq);
  };
  if (__builtin_amdgcn_readfirstlane(rq.slow ? 1 : 0)) {
    codes(std::true_type{});
  } else {
    codes(std::false_type{});
  }
  __syncthreads();

  uint8_t *const drow = dst + static_cast<int64_t>(row) * (BITS == 4 ? num_int >> 1 : num_int);
  auto put = [&](int u, const uint4 &c) {
    if constexpr (TILED) {
      *reinterpret_cast<uint4 *>(dst + tile8_offset(l8, row, u >> 1, u & 1)) = c;
    } else if constexpr (BITS == 8) {
      *reinterpret_cast<uint4 *>(drow + u * 16) = c;
    } else {
      // byte pairs (c0, c1) -> c0 | c1 << 4: t = w | w >> 4 leaves them in bytes 0 and 2
      const uint32_t t0 = c.x | (c.x >> 4), t1 = c.y | (c.y >> 4), t2 = c.z | (c.z >> 4), t3 = c.w | (c.w >> 4);
      *reinterpret_cast<uint2 *>(drow + u * 8) = make_uint2(__builtin_amdgcn_perm(t1, t0, 0x06040200u), __builtin_amdgcn_perm(t3, t2, 0x06040200u));
    }
  };
#pragma unroll
  for (int k = 0; k < NU; ++k) {
    const uint32_t c0 = first[k];
    if (tid + k * T < nu && c0 != 0xFFFFu) {
      // two aligned reads, a shift by whole words (bit-mask selects) and by bytes
      const uint4 a = *reinterpret_cast<const uint4 *>(stage + (c0 & ~15u)), b = *reinterpret_cast<const uint4 *>(stage + (c0 & ~15u) + 16);
      uint32_t w[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
      const uint32_t by2 = 0u - ((c0 >> 3) & 1u), by1 = 0u - ((c0 >> 2) & 1u);
#pragma unroll
      for (int t = 0; t < 6; ++t) w[t] = (w[t + 2] & by2) | (w[t] & ~by2);
#pragma unroll
      for (int t = 0; t < 5; ++t) w[t] = (w[t + 1] & by1) | (w[t] & ~by1);
      put(tid + k * T, make_uint4(__builtin_amdgcn_alignbyte(w[1], w[0], c0), __builtin_amdgcn_alignbyte(w[2], w[1], c0),
                                  __builtin_amdgcn_alignbyte(w[3], w[2], c0), __builtin_amdgcn_alignbyte(w[4], w[3], c0)));
    }
  }
  auto gather = [&](uint32_t u, const uint4 &a, const uint4 &b) {
    const uint32_t at[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    uint32_t c[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const uint32_t b0 = stage[at[2 * t] & 0xFFFFu], b1 = stage[at[2 * t] >> 16], b2 = stage[at[2 * t + 1] & 0xFFFFu], b3 = stage[at[2 * t + 1] >> 16];
      c[t] = b0 | (b1 << 8) | (b2 << 16) | (b3 << 24);
    }
    put(static_cast<int>(u), make_uint4(c[0], c[1], c[2], c[3]));
  };
  if (static_cast<uint32_t>(tid) < ngather) gather(gunit, ga, gb);
  for (uint32_t i = tid + T; i < ngather; i += T) {
    const uint4 *const more = reinterpret_cast<const uint4 *>(gather_cols + 16 * i);
    gather(gather_unit[i], more[0], more[1]);
  }
}

// ---------------------------------------------------------------------------------------
// Stand-alone quantize straight from the index lists: no column map, one launch.
//
// What bounded the two launches it replaces at a few hundred rows was the map: one workgroup builds it, 6.3 us in front of
// 6.2 us of quantizing 512 x 4096.  Here every workgroup loads the integer columns of its code groups itself, once
// (clamped and packed to 16 bits in registers), together with its first row, marks the outlier columns in an LDS mask,
// and then walks over rows blockIdx.x, blockIdx.x + gridDim.x, ..., the next row's loads in flight behind the gathers.
// The results are those of a column map that does not stream (gather_rows), for any lists: minimum and maximum over the
// columns that are not in the outlier list, codes in the order of the integer list, indices outside the row clamped.
// A workgroup reads 8 bytes of list per integer column, which the L2 serves; two workgroups per CU bound that traffic.
// Needs cols % 8 == 0, num_int % 8 == 0, 16-byte aligned rows and 8-byte aligned codes; NV: groups of 8 columns per lane.
//
// Measured (map + quantize -> this kernel, us in a graph, int4): 1 x 4096 9.1 -> 3.7, 512 x 4096 10.9 -> 5.2, 2048 x 8192
// 21.6 -> 16.3, 512 x 13824 18.9 -> 12.8, 2048 x 16384 39.7 -> 29.8; int8 the same within 0.5.  At 2048 rows it is the
// walk over four rows per workgroup that counts, 33 MB in 16 us.
template <int BITS, bool BF16, int NV>
__global__ __launch_bounds__(kThreads) void asym_quantize_list_kernel(
    const uint16_t *__restrict__ x, int rows, int cols, const int64_t *__restrict__ int_idx, int num_int,
    const int64_t *__restrict__ fp_idx, int num_fp, uint8_t *__restrict__ dst, uint16_t *__restrict__ meta,
    uint16_t *__restrict__ fp_x) {
  extern __shared__ __align__(16) uint16_t row_s[];  // the row, the outlier columns, the outlier mask
  __shared__ float red[8];
  const int tid = threadIdx.x, nvec = cols >> 3, groups = num_int >> 3, words = (cols + 31) / 32;
  uint16_t *const fp_s = row_s + cols;
  uint32_t *const mask_s = reinterpret_cast<uint32_t *>(fp_s + (num_fp + 7) / 8 * 8);
  auto clamp = [&](int64_t c) { return static_cast<uint32_t>(c < 0 ? 0 : (c >= cols ? cols - 1 : c)); };
  uint4 next[NV];
  auto load = [&](int row) {
    const uint4 *xv = reinterpret_cast<const uint4 *>(x + int64_t(row < rows ? row : rows - 1) * cols);
#pragma unroll
    for (int i = 0; i < NV; ++i) next[i] = xv[tid + i * kThreads < nvec ? tid + i * kThreads : 0];
  };
  load(blockIdx.x);
  uint32_t src[NV][4];  // this lane's code groups: eight byte offsets into the row
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int64_t *list = int_idx + (tid + i * kThreads < groups ? tid + i * kThreads : 0) * 8;
    int64_t c[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) c[e] = list[e];
#pragma unroll
    for (int e = 0; e < 4; ++e) src[i][e] = clamp(c[2 * e]) * 2u | clamp(c[2 * e + 1]) << 17;
  }
  for (int w = tid; w < words; w += kThreads) mask_s[w] = 0u;
  __syncthreads();
  for (int f = tid; f < num_fp; f += kThreads) {
    const uint32_t c = clamp(fp_idx[f]);
    fp_s[f] = static_cast<uint16_t>(c);
    atomicOr(&mask_s[c >> 5], 1u << (c & 31u));
  }
  __syncthreads();
  uint32_t skip[NV];  // this lane's row groups: their outlier columns
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int g = tid + i * kThreads;
    skip[i] = g < nvec ? (mask_s[g >> 2] >> ((g & 3) * 8)) & 0xFFu : 0xFFu;
  }
  for (int row = blockIdx.x; row < rows; row += gridDim.x) {
    float mn = __builtin_inff(), mx = -__builtin_inff();
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      if (tid + i * kThreads < nvec) reinterpret_cast<uint4 *>(row_s)[tid + i * kThreads] = next[i];
      const uint32_t w[4] = {next[i].x, next[i].y, next[i].z, next[i].w};
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float v = to_f32<BF16>(static_cast<uint16_t>(w[e >> 1] >> (16 * (e & 1))));
        const bool out = (skip[i] >> e) & 1u;
        mn = fminf(mn, out ? __builtin_inff() : v);
        mx = fmaxf(mx, out ? -__builtin_inff() : v);
      }
    }
    load(row + gridDim.x);
    block_minmax<kThreads>(mn, mx, red);  // also orders the row's LDS writes before the gathers
    RowQuant<BF16> rq;
    rq.init(mn, mx, BITS);
    if (tid == 0) {
      meta[2 * row] = rq.scale_bits;
      meta[2 * row + 1] = rq.zero_bits;
    }
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int g = tid + i * kThreads;
      if (g >= groups) continue;
      uint32_t w[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint8_t *base = reinterpret_cast<const uint8_t *>(row_s);
        const uint32_t lo = *reinterpret_cast<const uint16_t *>(base + (src[i][e] & 0xFFFFu));
        const uint32_t hi = *reinterpret_cast<const uint16_t *>(base + (src[i][e] >> 16));
        w[e] = lo | hi << 16;
      }
      const uint4 v = make_uint4(w[0], w[1], w[2], w[3]);
      const uint2 c = rq.slow ? group_codes<BITS, BF16, true>(v, rq) : group_codes<BITS, BF16, false>(v, rq);
      if constexpr (BITS == 4) {
        const uint32_t a = c.x | (c.x >> 4), b = c.y | (c.y >> 4);  // bytes 0 and 2: two codes each
        reinterpret_cast<uint32_t *>(dst + int64_t(row) * (num_int >> 1))[g] = __builtin_amdgcn_perm(b, a, 0x06040200u);
      } else {
        reinterpret_cast<uint2 *>(dst + int64_t(row) * num_int)[g] = c;
      }
    }
    for (int f = tid; f < num_fp; f += kThreads) fp_x[int64_t(row) * num_fp + f] = row_s[fp_s[f]];
    __syncthreads();  // the next row overwrites row_s
  }
}

// Rows too long for LDS: same arithmetic, gathers go to global memory (L2-resident row).
template <typename IdxT, int BITS, bool BF16>
__global__ __launch_bounds__(kThreads) void asym_quantize_longrow_kernel(
    const uint16_t *__restrict__ x, int64_t rows, int64_t cols, const IdxT *__restrict__ src_col,
    const IdxT *__restrict__ fp_col, int64_t num_int, int64_t num_fp, uint8_t *__restrict__ dst,
    uint16_t *__restrict__ meta, uint16_t *__restrict__ fp_x) {
  __shared__ float red[8];
  const int tid = threadIdx.x;
  constexpr float kMaxQ = static_cast<float>((1 << BITS) - 1);
  for (int64_t row = blockIdx.x; row < rows; row += gridDim.x) {
    const uint16_t *xr = x + row * cols;
    float mn = __builtin_inff(), mx = -__builtin_inff();
    for (int64_t j = tid; j < num_int; j += kThreads) {
      const float f = to_f32<BF16>(xr[src_col[j]]);
      mn = fminf(mn, f);
      mx = fmaxf(mx, f);
    }
    block_minmax(mn, mx, red);
    RowQuant<BF16> rq;
    rq.init(mn, mx, BITS);
    if (tid == 0) {
      meta[2 * row] = rq.scale_bits;
      meta[2 * row + 1] = rq.zero_bits;
    }
    const int64_t pairs = num_int >> 1;
    for (int64_t p = tid; p < pairs; p += kThreads) {
      const uint32_t v0 = RowQuant<BF16>::to_level(rq.quotient(xr[src_col[2 * p]]), kMaxQ);
      const uint32_t v1 = RowQuant<BF16>::to_level(rq.quotient(xr[src_col[2 * p + 1]]), kMaxQ);
      if constexpr (BITS == 4) {
        dst[row * pairs + p] = static_cast<uint8_t>((v0 | (v1 << 4)) ^ 0x88u);
      } else {
        reinterpret_cast<uint16_t *>(dst + row * num_int)[p] = static_cast<uint16_t>((v0 | (v1 << 8)) ^ 0x8080u);
      }
    }
    for (int64_t f = tid; f < num_fp; f += kThreads) fp_x[row * num_fp + f] = xr[fp_col[f]];
  }
}

// ---------------------------------------------------------------------------------------
// find_meta: fp16, all columns (reference: src/asymmetric/asymmetric.cu:263-338)
__global__ __launch_bounds__(kThreads) void find_meta_kernel(const uint16_t *__restrict__ x, int64_t rows,
                                                             int64_t cols, int bits, uint16_t *__restrict__ meta) {
  __shared__ float red[8];
  for (int64_t row = blockIdx.x; row < rows; row += gridDim.x) {
    const uint16_t *xr = x + row * cols;
    float mn = __builtin_inff(), mx = -__builtin_inff();
    for (int64_t c = threadIdx.x; c < cols; c += kThreads) {
      const float f = to_f32<false>(xr[c]);
      mn = fminf(mn, f);
      mx = fmaxf(mx, f);
    }
    block_minmax(mn, mx, red);
    if (threadIdx.x == 0) {
      RowQuant<false> rq;
      rq.init(mn, mx, bits);
      meta[2 * row] = rq.scale_bits;
      meta[2 * row + 1] = rq.zero_bits;
    }
  }
}

__device__ __forceinline__ uint32_t old_level(uint16_t xb, uint16_t sb, uint16_t zb, float maxq) {
  const _Float16 d = __builtin_bit_cast(_Float16, xb) - __builtin_bit_cast(_Float16, zb);
  const float q = static_cast<float>(d) / static_cast<float>(__builtin_bit_cast(_Float16, sb));
  return RowQuant<false>::to_level(round_storage<false>(q), maxq);
}

// quantizeOld, 4 bit: flat pairing over the whole array, meta row = idx / colsDst
// (reference: src/asymmetric/asymmetric.cu:13-45)
__global__ __launch_bounds__(kThreads) void quantize_old4_kernel(const uint16_t *__restrict__ x,
                                                                 const uint16_t *__restrict__ meta, int64_t rows,
                                                                 int64_t cols, int64_t cols_dst,
                                                                 uint8_t *__restrict__ dst) {
  const int64_t n_dst = rows * cols_dst, n_src = rows * cols;
  for (int64_t idx = blockIdx.x * int64_t(kThreads) + threadIdx.x; idx < n_dst; idx += int64_t(gridDim.x) * kThreads) {
    const int64_t row = idx / cols_dst;
    const uint16_t sb = meta[2 * row], zb = meta[2 * row + 1];
    uint32_t byte = 0;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int64_t s = idx * 2 + i;
      if (s < n_src) byte |= ((old_level(x[s], sb, zb, 15.0f) ^ 8u) & 0xFu) << (4 * i);
    }
    dst[idx] = static_cast<uint8_t>(byte);
  }
}

__global__ __launch_bounds__(kThreads) void quantize_old8_kernel(const uint16_t *__restrict__ x,
                                                                 const uint16_t *__restrict__ meta, int64_t rows,
                                                                 int64_t cols, uint8_t *__restrict__ dst) {
  const int64_t n = rows * cols;
  for (int64_t idx = blockIdx.x * int64_t(kThreads) + threadIdx.x; idx < n; idx += int64_t(gridDim.x) * kThreads) {
    const int64_t row = idx / cols;
    dst[idx] = static_cast<uint8_t>(old_level(x[idx], meta[2 * row], meta[2 * row + 1], 255.0f) ^ 0x80u);
  }
}

// symmetric quantize (reference: src/symmetric/symmetric.cu:6-61): no clamp, wraps
__device__ __forceinline__ int sym_code(uint16_t xb, float s) {
  const float q = round_storage<false>(to_f32<false>(xb) / s);
  // __half2int_rn: NaN -> 0, saturating
  return __float2int_rn(q);
}

__global__ __launch_bounds__(kThreads) void sym_quantize_kernel(const uint16_t *__restrict__ x,
                                                                const uint16_t *__restrict__ scale, int64_t rows,
                                                                int64_t cols, int bits, uint8_t *__restrict__ dst) {
  const int64_t cols_dst = bits == 4 ? (cols + 1) / 2 : cols;
  for (int64_t row = blockIdx.y; row < rows; row += gridDim.y) {
    const float s = to_f32<false>(scale[row]);
    const uint16_t *xr = x + row * cols;
    uint8_t *dr = dst + row * cols_dst;
    for (int64_t j = blockIdx.x * int64_t(kThreads) + threadIdx.x; j < cols_dst; j += int64_t(gridDim.x) * kThreads) {
      if (bits == 4) {
        uint32_t b = static_cast<uint32_t>(sym_code(xr[2 * j], s)) & 0xFu;
        if (2 * j + 1 < cols) b |= (static_cast<uint32_t>(sym_code(xr[2 * j + 1], s)) & 0xFu) << 4;
        dr[j] = static_cast<uint8_t>(b);
      } else {
        dr[j] = static_cast<uint8_t>(sym_code(xr[j], s) & 0xFF);
      }
    }
  }
}

int grid_for(int64_t work_items, int64_t per_block) {
  int64_t g = (work_items + per_block - 1) / per_block;
  if (g < 1) g = 1;
  if (g > 65535 * 16) g = 65535 * 16;
  return static_cast<int>(g);
}

constexpr int64_t kMaxLdsRowBytes = 128 * 1024;  // of the 160 KB per CU

// Few rows of more than 4096 columns: eight waves per row instead of four, while the rows leave half of the CUs without one
// (us per launch: int8 16 x 13824 5.2 -> 4.9, 32 x 28672 7.5 -> 6.9, bf16 16 x 13824 5.7 -> 5.2, int4 32 x 8192 4.1 -> 3.9; 256 x 28672 bf16
// 11.8 -> 10.7, 512 x 11008 9.3 -> 8.8 but fp16 256 x 8192 4.3 -> 4.4; sixteen waves were slower than eight everywhere).
int64_t wide_rows() { return num_cus() / 2; }

template <typename IdxT, int BITS, bool BF16, int NV, int TPR, bool SYM = false, bool PF = false>
int launch_stream(const void *x, int64_t rows, int64_t cols, const uint8_t *cm, const ColmapLayout &l, int64_t num_int,
                  int64_t num_fp, void *dst, void *meta, void *fp_x, hipStream_t st, bool tiled,
                  float sym_divisor = 1.0f) {
  auto kern = asym_quantize_stream_kernel<IdxT, BITS, BF16, NV, TPR, SYM, PF>;
  // the row (gather path) or one byte per code (streaming path); a tile-ordered launch only ever streams
  const int64_t lds = tiled ? align16(num_int) : align16(cols * 2);
  if (lds > 48 * 1024) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
    if (e != hipSuccess) {
      set_last_hip_error(e);
      return QUIK_ERR_LAUNCH;
    }
  }
  const int64_t items = tiled ? (rows + 7) / 8 * 8 : rows;
  int grid = static_cast<int>(items < (int64_t(1) << 30) ? items : (int64_t(1) << 30));
  if (PF && grid > 2 * num_cus()) grid = 2 * num_cus();  // persistent: the workgroups that are resident at once
  // tiled: dst is an operand buffer in tile order (6-bit levels for 4 bits, int8 for 8 bits)
  const int vec_out = tiled ? (BITS == 4 ? 2 : 3) : (num_int % 16 == 0 && reinterpret_cast<uintptr_t>(dst) % 16 == 0);
  hipLaunchKernelGGL(kern, dim3(grid), dim3(TPR), static_cast<size_t>(lds), st,
                     static_cast<const uint16_t *>(x), rows, cols, reinterpret_cast<const IdxT *>(cm),
                     reinterpret_cast<const IdxT *>(cm + l.off_fp), reinterpret_cast<const uint32_t *>(cm + l.off_mask),
                     reinterpret_cast<const uint32_t *>(cm + l.off_grp),
                     reinterpret_cast<const uint32_t *>(cm + l.off_dirty),
                     reinterpret_cast<const uint16_t *>(cm + l.off_slot),
                     reinterpret_cast<const uint32_t *>(cm + l.off_flags), num_int, num_fp,
                     static_cast<uint8_t *>(dst), static_cast<uint16_t *>(meta), static_cast<uint16_t *>(fp_x), vec_out,
                     sym_divisor);
  return check_launch();
}

// symmetric activations through the streaming kernel (fp16; the caller has checked that the column map streams)
template <int BITS>
int launch_sym_stream(const void *x, int64_t rows, int64_t cols, const uint8_t *cm, const ColmapLayout &l,
                      int64_t num_int, int64_t num_fp, void *dst, void *scale, void *fp_x, hipStream_t st, bool tiled,
                      float divisor) {
  const int64_t groups = cols / 8;
#define QUIK_SYM_STREAM(NV, TPR)                                                                             \
  return launch_stream<uint16_t, BITS, false, NV, TPR, true>(x, rows, cols, cm, l, num_int, num_fp, dst, scale, \
                                                             fp_x, st, tiled, divisor)
  if (groups <= 512) QUIK_SYM_STREAM(2, kThreads);
  if (rows <= wide_rows()) {
    if (groups <= 1024) QUIK_SYM_STREAM(2, 512);
    if (groups <= 2048) QUIK_SYM_STREAM(4, 512);
    QUIK_SYM_STREAM(8, 512);
  }
  if (groups <= 1024) QUIK_SYM_STREAM(4, kThreads);
  if (groups <= 2048) QUIK_SYM_STREAM(8, kThreads);
  QUIK_SYM_STREAM(16, kThreads);
#undef QUIK_SYM_STREAM
}

// Long fp16 rows -> int8 operand buffer through the LDS ring (quantize_tile8_ring_kernel).  `ndirty`: groups of 8
// columns that hold outlier columns, from the host's copy of the column map's flag words.
constexpr int64_t kLdsPerCu = 160 * 1024;
// rows of more than 16384 columns (against quantize_units_kernel: asym_quantize_tile8); against the streaming kernel at 2048 rows, kernel
// time from a cold cache: 28672 columns 41.6 against 51.0 us
constexpr int64_t kRingMinGroups = 4 * kRingThreads + 1;
bool ring_fits(int64_t cols, int64_t num_int, int64_t num_fp, int64_t ndirty) {
  const int64_t groups = cols / 8;
  return groups >= kRingMinGroups && groups <= 8 * kRingThreads && ndirty >= 0 && ndirty <= kRingThreads &&
         num_fp <= kRingThreads && num_int % 16 == 0 && ring_lds_bytes(cols, num_fp) <= kLdsPerCu;
}
template <int NV>
int launch_tile8_ring_nv(const void *x, int64_t rows, int64_t cols, const uint8_t *cm, const ColmapLayout &l,
                         int64_t num_int, int64_t num_fp, int ndirty, int ngather, void *dst, void *meta,
                         hipStream_t st) {
  auto kern = quantize_tile8_ring_kernel<NV>;
  const int64_t lds = ring_lds_bytes(cols, num_fp);
  if (hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                                         hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
      e != hipSuccess) {
    set_last_hip_error(e);
    return QUIK_ERR_LAUNCH;
  }
  const int64_t per_xcd = (rows + 7) / 8;
  // the ring takes most of a CU's LDS: one workgroup each; a multiple of the XCDs
  int64_t grid = num_cus() / 8 * 8;
  if (grid < 8) grid = 8;
  if (grid > per_xcd * 8) grid = per_xcd * 8;
  hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(grid)), dim3(kRingThreads), static_cast<size_t>(lds), st,
                     static_cast<const uint16_t *>(x), rows, cols, reinterpret_cast<const uint16_t *>(cm + l.off_fp),
                     reinterpret_cast<const uint32_t *>(cm + l.off_grp),
                     reinterpret_cast<const uint32_t *>(cm + l.off_dirty),
                     reinterpret_cast<const uint16_t *>(cm + l.off_slot),
                     reinterpret_cast<const uint16_t *>(cm + l.off_unit),
                     reinterpret_cast<const uint16_t *>(cm + l.off_gunit),
                     reinterpret_cast<const uint16_t *>(cm + l.off_gcols), ndirty, ngather, num_int, num_fp,
                     static_cast<uint8_t *>(dst), static_cast<uint16_t *>(meta));
  return check_launch();
}
int launch_tile8_ring(const void *x, int64_t rows, int64_t cols, const uint8_t *cm, const ColmapLayout &l,
                      int64_t num_int, int64_t num_fp, int ndirty, int ngather, void *dst, void *meta,
                      hipStream_t st) {
  switch ((cols / 8 + kRingThreads - 1) / kRingThreads) {
    case 5: return launch_tile8_ring_nv<5>(x, rows, cols, cm, l, num_int, num_fp, ndirty, ngather, dst, meta, st);
    case 6: return launch_tile8_ring_nv<6>(x, rows, cols, cm, l, num_int, num_fp, ndirty, ngather, dst, meta, st);
    case 7: return launch_tile8_ring_nv<7>(x, rows, cols, cm, l, num_int, num_fp, ndirty, ngather, dst, meta, st);
    default: return launch_tile8_ring_nv<8>(x, rows, cols, cm, l, num_int, num_fp, ndirty, ngather, dst, meta, st);
  }
}

template <typename IdxT, int BITS, bool BF16>
int launch_asym(const void *x, int64_t rows, int64_t cols, const uint8_t *cm, const ColmapLayout &l, int64_t num_int,
                int64_t num_fp, void *dst, void *meta, void *fp_x, hipStream_t st) {
  const IdxT *src_col = reinterpret_cast<const IdxT *>(cm);
  const IdxT *fp_col = reinterpret_cast<const IdxT *>(cm + l.off_fp);
  const uint32_t *mask = reinterpret_cast<const uint32_t *>(cm + l.off_mask);
  if constexpr (sizeof(IdxT) == 2) if (cols <= kStreamMaxCols && cols % 8 == 0 && reinterpret_cast<uintptr_t>(x) % 16 == 0) {
    // Four waves per row, or eight (wide_rows), one row per workgroup: more, shorter waves hide the load and LDS latencies
    // better than fewer waves with less per-row fixed work (64 and 128 threads were slower).
    const int64_t groups = cols / 8;
#define QUIK_STREAM(NV, TPR) \
  return launch_stream<IdxT, BITS, BF16, NV, TPR>(x, rows, cols, cm, l, num_int, num_fp, dst, meta, fp_x, st, false)
    if (groups > 512 && rows <= wide_rows()) {
      if (groups <= 1024) QUIK_STREAM(2, 512);
      if (groups <= 2048) QUIK_STREAM(4, 512);
      QUIK_STREAM(8, 512);
    }
    if (groups <= 512) QUIK_STREAM(2, kThreads);
    if (groups <= 1024) QUIK_STREAM(4, kThreads);
    if (groups <= 2048) QUIK_STREAM(8, kThreads);
    QUIK_STREAM(16, kThreads);
#undef QUIK_STREAM
  }
  const int grid = static_cast<int>(rows < 65535 * 8 ? rows : 65535 * 8);
  const int64_t lds = align16(cols * 2);
  if (lds <= kMaxLdsRowBytes) {
    auto kern = asym_quantize_kernel<IdxT, BITS, BF16>;
    if (lds > 48 * 1024) {
      hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                                         hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
      if (e != hipSuccess) {
        set_last_hip_error(e);
        return QUIK_ERR_LAUNCH;
      }
    }
    const int vec_ok = (cols % 8 == 0) && (reinterpret_cast<uintptr_t>(x) % 16 == 0);
    hipLaunchKernelGGL(kern, dim3(grid), dim3(kThreads), static_cast<size_t>(lds), st,
                       static_cast<const uint16_t *>(x), rows, cols, src_col, fp_col, mask, num_int, num_fp,
                       static_cast<uint8_t *>(dst), static_cast<uint16_t *>(meta), static_cast<uint16_t *>(fp_x),
                       vec_ok);
  } else {
    hipLaunchKernelGGL((asym_quantize_longrow_kernel<IdxT, BITS, BF16>), dim3(grid), dim3(kThreads), 0, st,
                       static_cast<const uint16_t *>(x), rows, cols, src_col, fp_col, num_int, num_fp,
                       static_cast<uint8_t *>(dst), static_cast<uint16_t *>(meta), static_cast<uint16_t *>(fp_x));
  }
  return check_launch();
}


// 6-bit (FOUR: 4-bit) operand output through quantize_fp6_row_kernel; meta: (scale, zero) pairs, or one scale per row (SYM)
template <bool BF16, bool SYM, bool FOUR>
int launch_fp6_row(const void *x, int64_t rows, int64_t cols, const uint8_t *cm, const ColmapLayout &l, int64_t num_int,
                   int64_t num_fp, void *dst, void *meta, hipStream_t st, float sym_divisor) {
  uint32_t words[4];
  if (int rc = colmap_words(cm, cols, num_int, num_fp, st, words)) return rc;
  if ((words[0] & (kColmapStreams | kColmapInPlace)) != (kColmapStreams | kColmapInPlace)) return QUIK_ERR_COLMAP;
  auto go = [&](auto kern, int jt) {
    const int per_wave = 64 * 32 * jt, W = static_cast<int>((cols + per_wave - 1) / per_wave);
    if (int rc = prepare(kern, 8 * jt * 4096)) return rc;
    constexpr int64_t kMost = 1 << 20;  // rows per launch: a grid holds fewer than 2^32 threads
    for (int64_t first = 0; first < rows; first += kMost) {
      const int64_t count = rows - first < kMost ? rows - first : kMost;
      hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>((count + 7) / 8 * 8)), dim3(64 * W),
                         static_cast<size_t>(W * jt * 4096), st, static_cast<const uint16_t *>(x), first,
                         static_cast<int>(count), static_cast<int>(cols), reinterpret_cast<const uint32_t *>(cm + l.off_patch),
                         reinterpret_cast<const uint16_t *>(cm + l.off_fp), static_cast<int>(words[2]), static_cast<int>(num_fp),
                         static_cast<int>(num_int), sym_divisor, static_cast<uint8_t *>(dst), rows, static_cast<uint16_t *>(meta));
      if (int rc = check_launch()) return rc;
    }
    return static_cast<int>(QUIK_OK);
  };
  // at most eight waves per workgroup; kStreamMaxCols columns are two fragments per lane
  return cols <= 8 * 64 * 32 ? go(quantize_fp6_row_kernel<BF16, SYM, 1, FOUR>, 1)
                             : go(quantize_fp6_row_kernel<BF16, SYM, 2, FOUR>, 2);
}
// asym_quantize_list_kernel: calls that it takes (everything else, and every error, is left to the column map's path).
// Up to 16384 columns it was the faster one at every row count from 1 to 2048 (2048 x 11008 27.1 -> 25.5, the least); with
// 16 groups per lane only where a CU has one row (256 x 28672 26.0 -> 18.0 us, 512 rows 31.0 -> 33.8).
bool list_quantize_ok(const void *x, int dtype, int64_t rows, int64_t cols, const int64_t *int_idx, int64_t num_int,
                      const int64_t *fp_idx, int64_t num_fp, int bits, const void *colmap, const void *dst, const void *meta,
                      const void *fp_x) {
  if ((bits != 4 && bits != 8) || (dtype != QUIK_F16 && dtype != QUIK_BF16)) return false;
  if (rows <= 0 || rows >= (1 << 30) || cols <= 0 || cols > kStreamMaxCols || num_int <= 0 || num_fp < 0 || num_int + num_fp != cols) return false;
  if (cols > 16384 && rows > num_cus()) return false;
  if (!x || !int_idx || !colmap || !dst || !meta || (num_fp > 0 && (!fp_idx || !fp_x))) return false;
  return cols % 8 == 0 && num_int % 8 == 0 && reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(dst) % 8 == 0;
}
int launch_list(const void *x, int dtype, int64_t rows, int64_t cols, const int64_t *int_idx, int64_t num_int,
                const int64_t *fp_idx, int64_t num_fp, int bits, void *dst, void *meta, void *fp_x, hipStream_t st) {
  // the row, the outlier columns and their mask: most with 32768 columns that are all outliers but eight
  constexpr int64_t kMost = kStreamMaxCols * 2 + kStreamMaxCols * 2 + kStreamMaxCols / 8;
  static_assert(kMost + 1024 <= kLdsBytes, "with the static LDS of the reductions");
  const int64_t lds = cols * 2 + (num_fp + 7) / 8 * 16 + (cols + 31) / 32 * 4;
  const int64_t grid = rows < 2 * num_cus() ? rows : 2 * num_cus();
  auto go = [&](auto kern) {
    if (lds > 48 * 1024) {
      if (int rc = prepare(kern, static_cast<int>(kMost))) return rc;
    }
    hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(grid)), dim3(kThreads), static_cast<size_t>(lds), st,
                       static_cast<const uint16_t *>(x), static_cast<int>(rows), static_cast<int>(cols), int_idx,
                       static_cast<int>(num_int), fp_idx, static_cast<int>(num_fp), static_cast<uint8_t *>(dst),
                       static_cast<uint16_t *>(meta), static_cast<uint16_t *>(fp_x));
    return static_cast<int>(check_launch());
  };
#define QUIK_LIST_NV(BITS, BF16)                                                   \
  return cols <= 4096    ? go(asym_quantize_list_kernel<BITS, BF16, 2>)            \
         : cols <= 8192  ? go(asym_quantize_list_kernel<BITS, BF16, 4>)            \
         : cols <= 16384 ? go(asym_quantize_list_kernel<BITS, BF16, 8>)            \
                         : go(asym_quantize_list_kernel<BITS, BF16, 16>)
  if (bits == 4) {
    if (dtype == QUIK_F16) QUIK_LIST_NV(4, false);
    QUIK_LIST_NV(4, true);
  }
  if (dtype == QUIK_F16) QUIK_LIST_NV(8, false);
  QUIK_LIST_NV(8, true);
#undef QUIK_LIST_NV
}
}  // namespace
}  // namespace quik

using namespace quik;

extern "C" int64_t quik_colmap_bytes(int64_t cols, int64_t num_int, int64_t num_fp) {
  if (cols <= 0 || num_int < 0 || num_fp < 0 || num_int + num_fp != cols) return 0;
  return colmap_layout(cols, num_int, num_fp).bytes;
}

static int build_colmap(const int64_t *int_indices, int64_t num_int, const int64_t *fp_indices, int64_t num_fp, int64_t cols,
                        void *colmap, void *stream, int row_major_only) {
  if (cols <= 0 || num_int < 0 || num_fp < 0 || num_int + num_fp != cols) return QUIK_ERR_SHAPE;
  if (!colmap || (num_int > 0 && !int_indices) || (num_fp > 0 && !fp_indices)) return QUIK_ERR_NULL;
  if (cols > (int64_t(1) << 31)) return QUIK_ERR_RANGE;
  colmap_forget(colmap);  // whatever was known about a map at this address is void
  const ColmapLayout l = colmap_layout(cols, num_int, num_fp);
  uint8_t *cm = static_cast<uint8_t *>(colmap);
  hipStream_t st = as_stream(stream);
  const auto u16 = [cm](int64_t off) { return reinterpret_cast<uint16_t *>(cm + off); };
  const auto u32 = [cm](int64_t off) { return reinterpret_cast<uint32_t *>(cm + off); };
  if (cols <= kStreamMaxCols) {
    const ColmapOut o{u16(0),          u16(l.off_fp),    u32(l.off_mask),  u32(l.off_grp),  u32(l.off_dirty),  u16(l.off_slot),
                      u16(l.off_kperm), u32(l.off_patch), u16(l.off_unit), u16(l.off_gunit), u16(l.off_gcols), u32(l.off_flags)};
    hipLaunchKernelGGL(colmap_build_kernel, dim3(1), dim3(kBuildThreads), 0, st, int_indices, static_cast<int>(num_int),
                       fp_indices, static_cast<int>(num_fp), static_cast<int>(cols), o, row_major_only);
    return check_launch();
  }
  if (l.idx16)
    hipLaunchKernelGGL(colmap_build_wide_kernel<uint16_t>, dim3(1), dim3(kBuildThreads), 0, st, int_indices, num_int,
                       fp_indices, num_fp, cols, u16(0), u16(l.off_fp), u32(l.off_mask), u32(l.off_flags));
  else
    hipLaunchKernelGGL(colmap_build_wide_kernel<uint32_t>, dim3(1), dim3(kBuildThreads), 0, st, int_indices, num_int,
                       fp_indices, num_fp, cols, u32(0), u32(l.off_fp), u32(l.off_mask), u32(l.off_flags));
  return check_launch();
}

extern "C" int quik_colmap_build(const int64_t *int_indices, int64_t num_int, const int64_t *fp_indices,
                                 int64_t num_fp, int64_t cols, void *colmap, void *stream) {
  return build_colmap(int_indices, num_int, fp_indices, num_fp, cols, colmap, stream, 0);
}

extern "C" int quik_asym_quantize_indexed(const void *x, int dtype, int64_t rows, int64_t cols, const int64_t *int_indices,
                                          int64_t num_int, const int64_t *fp_indices, int64_t num_fp, int bits,
                                          void *colmap_workspace, void *dst, void *meta, void *fp_x, void *stream) {
  if (rows == 0) return QUIK_OK;
  if (list_quantize_ok(x, dtype, rows, cols, int_indices, num_int, fp_indices, num_fp, bits, colmap_workspace, dst, meta, fp_x))
    return launch_list(x, dtype, rows, cols, int_indices, num_int, fp_indices, num_fp, bits, dst, meta, fp_x, as_stream(stream));
  if (int rc = build_colmap(int_indices, num_int, fp_indices, num_fp, cols, colmap_workspace, stream, 1)) return rc;
  return quik_asym_quantize(x, dtype, rows, cols, colmap_workspace, num_int, num_fp, bits, dst, meta, fp_x, stream);
}

extern "C" int quik_asym_quantize(const void *x, int dtype, int64_t rows, int64_t cols, const void *colmap,
                                  int64_t num_int, int64_t num_fp, int bits, void *dst, void *meta, void *fp_x,
                                  void *stream) {
  if (bits != 4 && bits != 8) return QUIK_ERR_BITS;
  if (dtype != QUIK_F16 && dtype != QUIK_BF16) return QUIK_ERR_DTYPE;
  if (rows < 0 || cols <= 0 || num_int <= 0 || num_fp < 0 || num_int + num_fp != cols) return QUIK_ERR_SHAPE;
  if (num_int % 2 != 0) return QUIK_ERR_ALIGN;
  if (rows == 0) return QUIK_OK;
  if (!x || !colmap || !dst || !meta || (num_fp > 0 && !fp_x)) return QUIK_ERR_NULL;
  if (cols > (int64_t(1) << 31)) return QUIK_ERR_RANGE;
  const ColmapLayout l = colmap_layout(cols, num_int, num_fp);
  const uint8_t *cm = static_cast<const uint8_t *>(colmap);
  hipStream_t st = as_stream(stream);
#define QUIK_DISPATCH(IDX)                                                                                     \
  if (bits == 4) {                                                                                             \
    return dtype == QUIK_F16                                                                                   \
               ? launch_asym<IDX, 4, false>(x, rows, cols, cm, l, num_int, num_fp, dst, meta, fp_x, st)       \
               : launch_asym<IDX, 4, true>(x, rows, cols, cm, l, num_int, num_fp, dst, meta, fp_x, st);       \
  } else {                                                                                                     \
    return dtype == QUIK_F16                                                                                   \
               ? launch_asym<IDX, 8, false>(x, rows, cols, cm, l, num_int, num_fp, dst, meta, fp_x, st)       \
               : launch_asym<IDX, 8, true>(x, rows, cols, cm, l, num_int, num_fp, dst, meta, fp_x, st);       \
  }
  if (l.idx16) {
    QUIK_DISPATCH(uint16_t)
  } else {
    QUIK_DISPATCH(uint32_t)
  }
#undef QUIK_DISPATCH
}

extern "C" int quik_colmap_streaming(const void *colmap, int64_t cols, int64_t num_int, int64_t num_fp, void *stream) {
  if (!colmap || cols <= 0 || num_int < 0 || num_fp < 0 || num_int + num_fp != cols) return QUIK_ERR_SHAPE;
  uint32_t flags = 0;
  if (int rc = colmap_flags(colmap, cols, num_int, num_fp, as_stream(stream), &flags)) return rc;
  return (flags & kColmapStreams) ? 1 : 0;
}

int quik::asym_quantize_fp6(const void *x, int dtype, int64_t rows, int64_t cols, const void *colmap, int64_t num_int,
                            int64_t num_fp, void *out6, void *meta, void *stream, int64_t k_multiple, bool four) {
  if (dtype != QUIK_F16 && dtype != QUIK_BF16) return QUIK_ERR_DTYPE;
  if (rows < 0 || cols <= 0 || num_int <= 0 || num_fp < 0 || num_int + num_fp != cols) return QUIK_ERR_SHAPE;
  if (num_int % k_multiple != 0 || num_fp % 32 != 0 || cols > kStreamMaxCols) return QUIK_ERR_ALIGN;
  if (rows == 0) return QUIK_OK;
  if (!x || !colmap || !out6 || !meta) return QUIK_ERR_NULL;
  if (reinterpret_cast<uintptr_t>(x) % 16 != 0 || reinterpret_cast<uintptr_t>(out6) % 256 != 0) return QUIK_ERR_ALIGN;
  if (int rc = colmap_require(colmap, cols, num_int, num_fp, as_stream(stream), kColmapStreams | kColmapInPlace)) return rc;
  const ColmapLayout l = colmap_layout(cols, num_int, num_fp);
  const uint8_t *cm = static_cast<const uint8_t *>(colmap);
  hipStream_t st = as_stream(stream);
  auto go = [&](auto launch) { return launch(x, rows, cols, cm, l, num_int, num_fp, out6, meta, st, 1.0f); };
  if (four) return dtype == QUIK_F16 ? go(launch_fp6_row<false, false, true>) : go(launch_fp6_row<true, false, true>);
  return dtype == QUIK_F16 ? go(launch_fp6_row<false, false, false>) : go(launch_fp6_row<true, false, false>);
}

namespace {
constexpr int64_t kUnitRows = 1 << 20;  // rows per launch: a grid holds fewer than 2^32 threads
bool units_ok(const void *x, int64_t cols, int64_t num_int, const void *dst) {
  return cols % 8 == 0 && cols <= kStreamMaxCols && num_int % 16 == 0 && reinterpret_cast<uintptr_t>(x) % 16 == 0 &&
         reinterpret_cast<uintptr_t>(dst) % 16 == 0;
}
template <int BITS, bool BF16, bool TILED, bool SYM = false>
int launch_units(const void *x, int64_t rows, int64_t cols, const void *colmap, int64_t num_int, int64_t num_fp, void *dst, void *meta,
                 void *fp_x, hipStream_t st, float sym_divisor = 1.0f) {
  const ColmapLayout l = colmap_layout(cols, num_int, num_fp);
  const uint8_t *cm = static_cast<const uint8_t *>(colmap);
  auto go = [&](auto kern) {
    if (int rc = prepare(kern, static_cast<int>(unit_lds_bytes(kStreamMaxCols)))) return rc;
    hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(TILED ? (rows + 7) / 8 * 8 : rows)), dim3(kUnitThreads),
                       static_cast<size_t>(unit_lds_bytes(cols)), st, static_cast<const uint16_t *>(x),
                       reinterpret_cast<const uint32_t *>(cm + l.off_grp), reinterpret_cast<const uint16_t *>(cm + l.off_unit),
                       static_cast<int>(cols), static_cast<int>(num_int), static_cast<int>(num_fp), static_cast<int>(rows),
                       reinterpret_cast<const uint16_t *>(cm + l.off_fp), reinterpret_cast<const uint16_t *>(cm + l.off_gunit),
                       reinterpret_cast<const uint16_t *>(cm + l.off_gcols), reinterpret_cast<const uint32_t *>(cm + l.off_flags),
                       static_cast<uint8_t *>(dst), static_cast<uint16_t *>(fp_x), static_cast<uint16_t *>(meta),
                       reinterpret_cast<const uint16_t *>(cm), reinterpret_cast<const uint32_t *>(cm + l.off_mask), sym_divisor);
    return check_launch();
  };
  const int64_t groups = cols / 8;
  if (groups <= 512) return go(quantize_units_kernel<BITS, BF16, 1, TILED, SYM>);
  if (groups <= 1024) return go(quantize_units_kernel<BITS, BF16, 2, TILED, SYM>);
  if (groups <= 2048) return go(quantize_units_kernel<BITS, BF16, 4, TILED, SYM>);
  return go(quantize_units_kernel<BITS, BF16, 8, TILED, SYM>);
}
}  // namespace

// A layer's few rows: quantize_units_kernel where it takes the shape, else as quik_asym_quantize.
int quik::asym_quantize_few(const void *x, int dtype, int64_t rows, int64_t cols, const void *colmap, int64_t num_int, int64_t num_fp, int bits,
                            void *dst, void *meta, void *fp_x, void *stream) {
  hipStream_t st = as_stream(stream);
  if (rows > 0 && rows <= kFewRows && num_int > 0 && num_fp >= 0 && num_int + num_fp == cols && (bits == 4 || bits == 8) &&
      (dtype == QUIK_F16 || dtype == QUIK_BF16) && x && colmap && dst && meta && (num_fp == 0 || fp_x) &&
      units_ok(x, cols, num_int, dst)) {
    auto go = [&](auto launch) { return launch(x, rows, cols, colmap, num_int, num_fp, dst, meta, fp_x, st, 1.0f); };
    if (bits == 4) return dtype == QUIK_F16 ? go(launch_units<4, false, false>) : go(launch_units<4, true, false>);
    return dtype == QUIK_F16 ? go(launch_units<8, false, false>) : go(launch_units<8, true, false>);
  }
  return quik_asym_quantize(x, dtype, rows, cols, colmap, num_int, num_fp, bits, dst, meta, fp_x, stream);
}

extern "C" int quik_asym_quantize_tile4(const void *x, int dtype, int64_t rows, int64_t cols, const void *colmap,
                                        int64_t num_int, int64_t num_fp, void *out4, void *meta, void *stream) {
  return quik::asym_quantize_fp6(x, dtype, rows, cols, colmap, num_int, num_fp, out4, meta, stream, kLayerK4, true);
}

extern "C" int quik_asym_quantize_fp6(const void *x, int dtype, int64_t rows, int64_t cols, const void *colmap,
                                      int64_t num_int, int64_t num_fp, void *out6, void *meta, void *stream) {
  return quik::asym_quantize_fp6(x, dtype, rows, cols, colmap, num_int, num_fp, out6, meta, stream, 128);
}

int quik::asym_quantize_tile8(const void *x, int dtype, int64_t rows, int64_t cols, const void *colmap, int64_t num_int,
                              int64_t num_fp, void *out8, void *meta, void *stream, int64_t k_multiple) {
  if (dtype != QUIK_F16 && dtype != QUIK_BF16) return QUIK_ERR_DTYPE;
  if (rows < 0 || cols <= 0 || num_int <= 0 || num_fp < 0 || num_int + num_fp != cols) return QUIK_ERR_SHAPE;
  if (num_int % k_multiple != 0 || num_fp % 32 != 0 || cols > kStreamMaxCols) return QUIK_ERR_ALIGN;
  if (rows == 0) return QUIK_OK;
  if (!x || !colmap || !out8 || !meta) return QUIK_ERR_NULL;
  if (reinterpret_cast<uintptr_t>(x) % 16 != 0 || reinterpret_cast<uintptr_t>(out8) % 256 != 0) return QUIK_ERR_ALIGN;
  uint32_t words[4];
  if (int rc = colmap_words(colmap, cols, num_int, num_fp, as_stream(stream), words)) return rc;
  if (!(words[0] & kColmapStreams)) return QUIK_ERR_COLMAP;
  hipStream_t st = as_stream(stream);
  // fp16 rows of more than 16384 columns, eight groups per lane, where a CU has more than one: quantize_tile8_ring_kernel, whose next row is
  // on its way while one is worked on (us per forward, units / ring: 256 x 28672 -> 1024 29.2 / 29.7, 512 x 28672 -> 512 40.65 / 39.45, 2048 x
  // 28672 -> 512 100 / 85; 768 x 16384 -> 512 32.55 / 34.05, 2048 x 13824 -> 512 46.05 / 47.15)
  if (dtype == QUIK_BF16 || cols <= 16384 || rows <= num_cus()) {
    auto go = [&](auto launch) {
      static_assert(kUnitRows % 64 == 0, "whole blocks of the operand buffer");
      const int64_t block = tile8_layout(rows, num_int, num_fp).block_bytes;
      for (int64_t first = 0; first < rows; first += kUnitRows) {
        const int64_t count = rows - first < kUnitRows ? rows - first : kUnitRows;
        if (int rc = launch(static_cast<const uint16_t *>(x) + first * cols, count, cols, colmap, num_int, num_fp,
                            static_cast<uint8_t *>(out8) + first / 64 * block, static_cast<uint16_t *>(meta) + 2 * first, nullptr, st, 1.0f))
          return rc;
      }
      return static_cast<int>(QUIK_OK);
    };
    return dtype == QUIK_F16 ? go(launch_units<8, false, true>) : go(launch_units<8, true, true>);
  }
  const ColmapLayout l = colmap_layout(cols, num_int, num_fp);
  const uint8_t *cm = static_cast<const uint8_t *>(colmap);
  if (ring_fits(cols, num_int, num_fp, words[1]) && words[3] <= kRingThreads)
    return launch_tile8_ring(x, rows, cols, cm, l, num_int, num_fp, static_cast<int>(words[1]), static_cast<int>(words[3]), out8, meta, st);
  // What the ring does not take (more outlier columns or groups that hold some than lanes, rows whose ring exceeds the LDS): 180
  // registers per lane leave room for two workgroups per CU, so the launch is persistent and requests the next row beside this one
  // (2048 x 28672 inside the forward, 67 -> 61 us)
  return launch_stream<uint16_t, 8, false, 16, kThreads, false, true>(x, rows, cols, cm, l, num_int, num_fp, out8, meta, nullptr, st, true);
}

extern "C" int quik_asym_quantize_tile8(const void *x, int dtype, int64_t rows, int64_t cols, const void *colmap,
                                        int64_t num_int, int64_t num_fp, void *out8, void *meta, void *stream) {
  return quik::asym_quantize_tile8(x, dtype, rows, cols, colmap, num_int, num_fp, out8, meta, stream, 64);
}

int quik::sym_quantize_mapped(const void *x, int64_t rows, int64_t cols, const void *colmap, int64_t num_int, int64_t num_fp,
                              int bits, float divisor, int tiled, void *dst, void *scale, void *fp_x, void *stream,
                              int64_t k_multiple) {
  if (bits != 4 && bits != 8) return QUIK_ERR_BITS;
  if (rows < 0 || cols <= 0 || num_int <= 0 || num_fp < 0 || num_int + num_fp != cols) return QUIK_ERR_SHAPE;
  if (cols % 8 != 0 || cols > kStreamMaxCols || !(divisor > 0.0f)) return QUIK_ERR_SHAPE;
  if (tiled && (num_int % k_multiple != 0 || num_fp % 32 != 0)) return QUIK_ERR_ALIGN;
  if (bits == 4 && num_int % 2 != 0) return QUIK_ERR_ALIGN;
  if (rows == 0) return QUIK_OK;
  if (!x || !colmap || !dst || !scale || (!tiled && num_fp > 0 && !fp_x)) return QUIK_ERR_NULL;
  if (reinterpret_cast<uintptr_t>(x) % 16 != 0 || reinterpret_cast<uintptr_t>(dst) % (tiled ? 256 : 1) != 0)
    return QUIK_ERR_ALIGN;
  if (int rc = colmap_require(colmap, cols, num_int, num_fp, as_stream(stream),
                              kColmapStreams | (bits == 4 && tiled ? kColmapInPlace : 0u)))
    return rc;
  const ColmapLayout l = colmap_layout(cols, num_int, num_fp);
  const uint8_t *cm = static_cast<const uint8_t *>(colmap);
  hipStream_t st = as_stream(stream);
  if (bits == 4 && tiled == QUIK_TILED_4)
    return launch_fp6_row<false, true, true>(x, rows, cols, cm, l, num_int, num_fp, dst, scale, st, divisor);
  if (bits == 4 && tiled) return launch_fp6_row<false, true, false>(x, rows, cols, cm, l, num_int, num_fp, dst, scale, st, divisor);
  // few rows: as asym_quantize_few (us per forward, streaming kernel / units: 16 x 8192 -> 8192 12.4 / 12.0, 3 x 13824 -> 5120 13.75 / 13.3,
  // 16 x 28672 -> 8192 28.05 / 26.95, 24 x 2048 -> 2048 7.35 / 7.15, 32 x 4096 -> 4096 8.85 / 8.7; 5120 columns the same)
  if (!tiled && rows <= kFewRows && units_ok(x, cols, num_int, dst))
    return bits == 4 ? launch_units<4, false, false, true>(x, rows, cols, colmap, num_int, num_fp, dst, scale, fp_x, st, divisor)
                     : launch_units<8, false, false, true>(x, rows, cols, colmap, num_int, num_fp, dst, scale, fp_x, st, divisor);
  return bits == 4 ? launch_sym_stream<4>(x, rows, cols, cm, l, num_int, num_fp, dst, scale, fp_x, st, tiled != 0, divisor)
                   : launch_sym_stream<8>(x, rows, cols, cm, l, num_int, num_fp, dst, scale, fp_x, st, tiled != 0, divisor);
}

extern "C" int quik_sym_quantize_mapped(const void *x, int64_t rows, int64_t cols, const void *colmap, int64_t num_int,
                                        int64_t num_fp, int bits, float divisor, int tiled, void *dst, void *scale,
                                        void *fp_x, void *stream) {
  return quik::sym_quantize_mapped(x, rows, cols, colmap, num_int, num_fp, bits, divisor, tiled, dst, scale, fp_x, stream,
                                   bits == 8 ? 64 : tiled == QUIK_TILED_4 ? kLayerK4 : 128);
}

extern "C" int quik_asym_find_meta(const void *x, int64_t rows, int64_t cols, int bits, void *meta, void *stream) {
  if (bits != 4 && bits != 8) return QUIK_ERR_BITS;
  if (rows < 0 || cols <= 0) return QUIK_ERR_SHAPE;
  if (rows == 0) return QUIK_OK;
  if (!x || !meta) return QUIK_ERR_NULL;
  const int grid = static_cast<int>(rows < 65535 ? rows : 65535);
  hipLaunchKernelGGL(find_meta_kernel, dim3(grid), dim3(kThreads), 0, as_stream(stream),
                     static_cast<const uint16_t *>(x), rows, cols, bits, static_cast<uint16_t *>(meta));
  return check_launch();
}

extern "C" int quik_asym_quantize_old(const void *x, const void *meta, int64_t rows, int64_t cols, int bits,
                                      void *dst, void *stream) {
  if (bits != 4 && bits != 8) return QUIK_ERR_BITS;
  if (rows < 0 || cols <= 0) return QUIK_ERR_SHAPE;
  if (rows == 0) return QUIK_OK;
  if (!x || !meta || !dst) return QUIK_ERR_NULL;
  if (bits == 4) {
    const int64_t cols_dst = (cols + 1) / 2;
    hipLaunchKernelGGL(quantize_old4_kernel, dim3(grid_for(rows * cols_dst, kThreads * 4)), dim3(kThreads), 0,
                       as_stream(stream), static_cast<const uint16_t *>(x), static_cast<const uint16_t *>(meta), rows,
                       cols, cols_dst, static_cast<uint8_t *>(dst));
  } else {
    hipLaunchKernelGGL(quantize_old8_kernel, dim3(grid_for(rows * cols, kThreads * 4)), dim3(kThreads), 0,
                       as_stream(stream), static_cast<const uint16_t *>(x), static_cast<const uint16_t *>(meta), rows,
                       cols, static_cast<uint8_t *>(dst));
  }
  return check_launch();
}

extern "C" int quik_sym_quantize(const void *x, const void *scale, int64_t rows, int64_t cols, int bits, void *dst,
                                 void *stream) {
  if (bits != 4 && bits != 8) return QUIK_ERR_BITS;
  if (rows < 0 || cols <= 0) return QUIK_ERR_SHAPE;
  if (rows == 0) return QUIK_OK;
  if (!x || !scale || !dst) return QUIK_ERR_NULL;
  const int64_t cols_dst = bits == 4 ? (cols + 1) / 2 : cols;
  int gx = grid_for(cols_dst, kThreads);
  if (gx > 64) gx = 64;
  const int gy = static_cast<int>(rows < 65535 ? rows : 65535);
  hipLaunchKernelGGL(sym_quantize_kernel, dim3(gx, gy), dim3(kThreads), 0, as_stream(stream),
                     static_cast<const uint16_t *>(x), static_cast<const uint16_t *>(scale), rows, cols, bits,
                     static_cast<uint8_t *>(dst));
  return check_launch();
}
