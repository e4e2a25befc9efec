// Persistent bf16 GEMM core for gfx950 shared by the SwiGLU and LM-head
// kernels and the plain products around them: D[m][n] = sum_k X(m, k) W(n, k)
// in tiles of 256 rows x BN (256 or 320) columns, fp32 accumulation, with the
// epilogue supplied by the caller.
//
// Either operand is ROW (k contiguous: X [M, K], W [N, K]) or COL (k-major:
// X [K, M], W [K, N]); PAIRED takes W's columns from two COL matrices (128
// columns of each per tile: the SwiGLU gate and up weights).
//
// A workgroup (8 waves, two per SIMD, one workgroup per CU) owns a tile and
// walks k in windows of 64 staged in a two-slot LDS ring (64 or 72 KiB per slot)
// by the LDS DMA.  Wave (wm, wn), wm = w % WM, wn = w / WM, accumulates TI row
// blocks of 32 from block TI wm on against the TJ column blocks from TJ wn on
// or (PAIRED) block wn of the first and of the second matrix.  acc[b][i] is
// the 32 x 32 product of column block b and row block i (lane: row 32i +
// (lane & 31); register 4q + e: column 8q + 4(lane/32) + e of the block).
//
// What bounds it, and the layout that follows from it.  The products alone
// run at 1.79 PFLOP/s here (the clock falls to ~1.75 GHz under them); timing
// copies made the path that feeds the ring the next limit (8192^3 now 1.24-1.39
// PFLOP/s by layout; hipBLASLt 1.61, 1.42 and 1.23), so:
//   * every copy moves whole 128-byte lines (64 k of one row, or 64 columns
//     of one k): with 64-byte pieces (32 k per window) the copies alone took
//     1500 clocks per 32 k and the 8192^3 products ran at 1.22-1.25 PFLOP/s;
//     with whole lines 1100 clocks, 1.30-1.42 PFLOP/s;
//   * the eight copies of a wave and its LDS reads are dealt out between its
//     products (batch()), not issued together after the barrier, where they
//     stall every wave's issue at once;
//   * a window's last k step is in registers before the barrier that hands
//     its slot to the copies, and the first k step of the next window is read
//     right after it, so no product waits on the LDS behind the barrier;
//   * outputs that the next kernel does not find in a cache anyway leave with
//     non-temporal stores: ordinary ones displace the operands from the L2
//     (16384 x 49152 x 1280, bf16 output: 1.79 -> 1.62 ms).
// LDS panels are 4 KiB: 32 rows x 64 k (ROW) or 32 k x 64 columns (COL), 128
// bytes per LDS row, the 16-byte chunks of row r permuted by chunk ^ s(r) so
// that the row reads (ds_read_b128) and the transposed reads
// (ds_read_b64_tr_b16) are conflict-free.
#pragma once
#include <type_traits>

#include "mm1_common.h"

namespace mm1 {
namespace gemm {

enum Layout { ROW, COL };

constexpr int BM = 256;                    // rows of a tile
constexpr int BK = 64;                     // k per ring slot
constexpr int WAVES = 8;
constexpr int PANEL = 4096;
constexpr int X_BYTES = BM * BK * 2;       // X of one slot

// How the 8 waves share a tile: WM x WN waves of TI row and TJ column blocks
// of 32.  Wide320 is for widths that 320 divides better than 256 (1280 = 4 x
// 320: at 16,384 rows 256 tiles, one per CU, where 256 columns make 320).
template <int WM_, int WN_, int TI_, int TJ_, int STAGE>
struct Shape {
  static constexpr int WM = WM_, WN = WN_, TI = TI_, TJ = TJ_;
  static constexpr int BN = WN * TJ * 32;
  static constexpr int W_BYTES = BN * BK * 2;                         // W of one slot
  static constexpr int RING = 2 * (X_BYTES + W_BYTES);                // X slots 0, 1; W slots 0, 1
  static constexpr int STAGE_BYTES = STAGE;                           // the epilogue's, per wave
  static constexpr size_t LDS_BYTES = RING + (size_t)WAVES * STAGE;
  static_assert(WM * WN == WAVES && WM * TI * 32 == BM && LDS_BYTES <= 160 * 1024, "tile shape");
};
using Wide256 = Shape<2, 4, 4, 2, 4096>;
using Wide320 = Shape<4, 2, 2, 5, 2048>;
constexpr long CACHED_BYTES = 192L << 20;  // outputs up to this size are taken to survive in the memory-side cache
constexpr int GROUP = 8;                   // row blocks per group of the tile order

template <int V>
using ic = std::integral_constant<int, V>;

// f(ic<0>), .., f(ic<N - 1>)
template <int N, int I = 0, class F>
__device__ __forceinline__ void for_each_ic(F&& f) {
  if constexpr (I < N) {
    f(ic<I>{});
    for_each_ic<N, I + 1>(f);
  }
}

// Per-lane LDS addresses of an operand's fragments (block blk of the wave, k
// step kk): a lane base plus a constant that folds into the ds offset field.
// s(r) of the panels: ROW (r >> 1) & 7, COL 4((r >> 1) & 1) | (r >> 2) & 3
// (a transposed read touches 4 consecutive rows x 64 bytes per half wave).
template <Layout L>
struct Frag;

template <>
struct Frag<ROW> {
  uint32_t base;
  __device__ __forceinline__ Frag(int lane, uint32_t region, int first_block) {
    const int l32 = lane & 31, h = lane >> 5, s = (l32 >> 1) & 7;
    base = region + first_block * PANEL + l32 * 128 + 16 * (h ^ s);
  }
  // the base of k step KK, made anew for each (one instruction, opaque to the
  // compiler, which would otherwise hold four bases per operand in registers)
  template <int KK>
  __device__ __forceinline__ uint32_t at() const {
    if constexpr (KK == 0) return base;
    uint32_t r;
    __asm__ volatile("v_xor_b32 %0, %1, %2" : "=v"(r) : "n"(32 * KK), "v"(base));
    return r;
  }
  // row 32blk + (lane & 31), k = 16kk + 8(lane/32) + 0..7
  template <int SLOT_OFF, int BLK, int KK>
  __device__ __forceinline__ bf16x8 get(uint32_t at_kk) const {
    return *reinterpret_cast<const MM1_LDS bf16x8*>((const MM1_LDS char*)(uintptr_t)at_kk + (SLOT_OFF + BLK * PANEL));
  }
};

template <>
struct Frag<COL> {
  uint32_t off[2][2];   // [block parity][half r]: k rows 16kk + 8h + 4r + j/4
  __device__ __forceinline__ Frag(int lane, uint32_t region, int first_block) {
    const int h = lane >> 5, g = (lane >> 4) & 1, j = lane & 15, jj = j >> 2;
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const int blk = first_block + b;
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        const int row = 8 * h + 4 * r + jj, s = (((jj >> 1) & 1) << 2) | ((2 * h + r) & 3);
        const int chunk = 4 * (blk & 1) + 2 * g + ((j & 3) >> 1);
        off[b][r] = region + (blk >> 1) * 2 * PANEL + row * 128 + 16 * (chunk ^ s) + 8 * (j & 1);
      }
    }
  }
  template <int KK>
  __device__ __forceinline__ uint32_t at() const { return 0; }
  // column 32blk + (lane & 31), k = 16kk + 8(lane/32) + 0..7
  template <int SLOT_OFF, int BLK, int KK>
  __device__ __forceinline__ bf16x8 get(uint32_t) const {
    bf16x8 out;
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const bf16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
          (MM1_LDS bf16x4*)((const MM1_LDS char*)(uintptr_t)off[BLK & 1][r] +
                            (SLOT_OFF + (BLK >> 1) * 2 * PANEL + (KK >> 1) * PANEL + 2048 * (KK & 1))));
#pragma unroll
      for (int q = 0; q < 4; ++q) out[4 * r + q] = v[q];
    }
    return out;
  }
};

struct Operand {
  const __bf16* p;
  long ld;    // row stride in elements
  int n;      // rows (ROW) or columns (COL, a multiple of 8) that exist; later ones are clamped
};

struct Problem {
  Operand x, w;
  // PAIRED: the second weight matrix.  Else, with k_cut > 0 (a multiple of
  // 64): W's part from k = k_cut on, W = [w | w1] along k.  Stride as w's.
  const __bf16* w1;
  int k_cut;
  int K;              // reduction length, a multiple of 128 (any with both operands COL)
  int n_mblk, n_nblk;
};

// Windows of a reduction over K: whole pairs (the ring's two slots).
__host__ __device__ inline int windows_of(int K) { return (K + 2 * BK - 1) / (2 * BK) * 2; }

// Source of the copies past a ragged K.
__device__ __attribute__((aligned(16))) static const uint32_t kZeros[4] = {0, 0, 0, 0};

// The host's bound on the copies' 32-bit byte offsets from a tile's base.
constexpr long SPAN = 1L << 30;            // elements
inline bool offsets_fit(Layout l, long ld, int n, int K) {
  return l == ROW ? BM * ld + K < SPAN : BK * ld + n < SPAN;
}

// Byte offset of element k of row `row` of a ROW operand, unsigned: a tile's W
// has up to Wide320::BN rows, which at the longest stride pass 2^31.
__host__ __device__ constexpr uint32_t row_off(int row, long ld, int k) {
  return (uint32_t)row * (uint32_t)(2 * ld) + (uint32_t)(2 * k);
}
constexpr long LD_MAX = SPAN / BM - 8;     // the longest stride that fits
static_assert(row_off(Wide320::BN - 1, LD_MAX, BK) == 2 * ((Wide320::BN - 1) * LD_MAX + BK), "offsets of the widest tile");

__device__ __forceinline__ void tile_coords(int t, int n_mblk, int n_nblk, int& mb, int& nb) {
  const int per_group = GROUP * n_nblk;
  const int group = t / per_group, first = group * GROUP;
  const int gm = min(GROUP, n_mblk - first);
  const int local = t - group * per_group;
  mb = first + local % gm;
  nb = local / gm;
}

// Launch geometry: one workgroup per CU, a multiple of the 8 XCDs.
inline int persistent_grid(int cus, int total_tiles) {
  int grid = ((cus > 0 ? cus : 256) + 7) & ~7;
  const int cap = (total_tiles + 7) & ~7;
  return grid < cap ? grid : cap;
}

// One piece of a workgroup's work: windows k0 .. k0 + nk - 1 (nk even) of
// `tile`.  half: -1 the whole tile, else the half of its columns kept.
// part: -1 the tile's result, else the slot its partial sums go to.
struct Item {
  int tile, half, k0, nk, part;
};

// Whole tiles dealt to the 8 XCDs in contiguous runs of a grouped order (8
// row blocks, then the next column block), so an XCD's concurrent tiles share
// X rows and W columns in its L2.  Ragged last round: when at most half of
// this XCD's workgroups would get one more tile, its rem leftover tiles are
// split by columns into 2 rem half tiles, one for each of the first 2 rem
// workgroups (the waves of the other half skip the products and the
// epilogue), so no workgroup runs a whole extra tile alone.
struct WholeTiles {
  int first, n_wg, n_full, n, t_split, j, n_kt;
  bool split;
  __device__ __forceinline__ WholeTiles(int total, int n_kt_) : n_kt(n_kt_) {
    const int xcd = blockIdx.x & 7;
    n_wg = gridDim.x >> 3;
    j = (int)(blockIdx.x >> 3);
    const int t0 = (int)(((long)xcd * total) >> 3), t1 = (int)(((long)(xcd + 1) * total) >> 3);
    first = t0 + j;
    n_full = (t1 - t0) / n_wg;
    const int rem = (t1 - t0) % n_wg;
    split = rem > 0 && 2 * rem <= n_wg;
    t_split = t0 + n_full * n_wg;
    n = split ? n_full + (j < 2 * rem ? 1 : 0) : (first < t1 ? (t1 - first + n_wg - 1) / n_wg : 0);
  }
  __device__ __forceinline__ int windows() const { return n * n_kt; }
  __device__ __forceinline__ Item at(int i) const {
    if (split && i == n_full) return {t_split + (j >> 1), j & 1, 0, n_kt, -1};
    return {first + i * n_wg, -1, 0, n_kt, -1};
  }
};

// Full rounds of whole tiles, then the leftover tiles (fewer than the grid's
// workgroups) split along k into equal runs of window pairs, one run per
// workgroup: a run is shorter than a tile, so it touches at most two.  The
// partial sums of leftover tile l that workgroup g computed go to slot g + l
// (a run's second piece and the next workgroup's first never share one), and
// split_sum_kernel adds them in workgroup order.
struct SplitTiles {
  int q, g, n_g, left0, upt, n_kt, u0, u1;
  int n;
  __device__ __host__ static long unit(long g, long left, long upt, long n_g) { return g * left * upt / n_g; }
  __device__ __forceinline__ SplitTiles(int total, int n_kt_) : n_kt(n_kt_) {
    const int n_wg = gridDim.x >> 3;
    n_g = gridDim.x;
    g = (int)(blockIdx.x & 7) * n_wg + (int)(blockIdx.x >> 3);     // an XCD's workgroups in a row
    q = total / n_g;
    left0 = q * n_g;
    upt = n_kt / 2;
    u0 = (int)unit(g, total - left0, upt, n_g);
    u1 = (int)unit(g + 1, total - left0, upt, n_g);
    n = q + (u1 > u0 ? (u1 - 1) / upt - u0 / upt + 1 : 0);
  }
  __device__ __forceinline__ int windows() const { return q * n_kt + 2 * (u1 - u0); }
  __device__ __forceinline__ Item at(int i) const {
    if (i < q) {
      const int n_wg = n_g >> 3, xcd = g / n_wg;
      return {xcd * q * n_wg + i * n_wg + (g - xcd * n_wg), -1, 0, n_kt, -1};
    }
    const int l = u0 / upt + (i - q);
    const int a = max(u0, l * upt), b = min(u1, (l + 1) * upt);
    return {left0 + l, -1, 2 * (a - l * upt), 2 * (b - a), g + l};
  }
};

// The persistent loop of one workgroup (512 threads, all of which must call
// it), over the items of Tiles; pro(mb, nb) runs in each item's first window
// (its loads land during the products), epi(mb, nb, acc, part) at its end
// with acc[TJ][TI] as described above.
template <Layout LX, Layout LW, bool PAIRED, class S, class Tiles, class Pro, class Epi>
__device__ __forceinline__ void run(const Problem& p, char* smem, Pro&& pro, Epi&& epi) {
  static_assert(!PAIRED || (LW == COL && std::is_same<S, Wide256>::value), "paired weights are k-major");
  constexpr int TI = S::TI, TJ = S::TJ, BN = S::BN;
  constexpr int NCX = X_BYTES / 1024 / WAVES;          // copies (1 KiB) of X per wave and window
  constexpr int NC = NCX + S::W_BYTES / 1024 / WAVES;  // ... and of both operands
  constexpr int W0 = 2 * X_BYTES;                      // W's ring
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = w % S::WM, wn = w / S::WM;
  constexpr bool RAGGED_K = LX == COL && LW == COL;    // k rows past K read as zeros
  const Tiles tiles(p.n_mblk * p.n_nblk, RAGGED_K ? windows_of(p.K) : p.K / BK);
  if (tiles.n == 0) return;
  const int n_win = tiles.windows();
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_addr(smem));

  // Copies: copy c of wave w fills piece w & 3 (8 LDS rows) of panel
  // (w >> 2) + 2c of its operand; lane L fills chunk position L & 7 of row
  // 8(w & 3) + L/8.  Successive copies lie 64 rows (ROW) or 64 columns (COL)
  // apart, so in a tile inside the operand every copy takes one per-lane
  // offset and its own scalar base; in a tile that crosses the operand's edge
  // the rows or columns past it are clamped per lane.
  const int lr = 8 * (w & 3) + (lane >> 3);
  const int crow = 8 * ((lane & 7) ^ ((lr >> 1) & 7));                                  // ROW: first k of the chunk
  const int ccol = 8 * ((lane & 7) ^ ((((lr >> 1) & 1) << 2) | ((lr >> 2) & 3)));       // COL: its first column
  const int prow = 32 * (w >> 2) + lr;                                                  // ROW: row; COL: k
  auto lane_off = [&](auto layout, long ld) MM1_INLINE {
    return (uint32_t)((prow * ld + (decltype(layout)::value == ROW ? crow : ccol)) * 2);
  };
  const uint32_t xoff = lane_off(ic<LX>{}, p.x.ld), woff = lane_off(ic<LW>{}, p.w.ld);
  const long xstep = LX == ROW ? 2 * BK : 2 * BK * p.x.ld, wstep = LW == ROW ? 2 * BK : 2 * BK * p.w.ld;   // window
  const long xcopy = LX == ROW ? 128 * p.x.ld : 128, wcopy = LW == ROW ? 128 * p.w.ld : 128;               // copy
  const int cut = !PAIRED && p.k_cut > 0 ? p.k_cut / BK : 0x7fffffff;    // window at which W changes over
  const char *xbase = nullptr, *wbase = nullptr, *wbase1 = nullptr;
  long w_tile = 0;                 // byte offset of the tile's first row or column of W
  int xroom = 0, wroom = 0;        // rows or columns of the operand from the tile's first on
  int iss_item = 0, iss_kt = 0, iss_end = 0;
  auto set_item = [&]() MM1_INLINE {
    const Item it = tiles.at(iss_item);
    int mb, nb;
    tile_coords(it.tile, p.n_mblk, p.n_nblk, mb, nb);
    const int m0 = mb * BM, n0 = nb * (PAIRED ? BN / 2 : BN);
    xroom = p.x.n - m0;
    wroom = p.w.n - n0;
    iss_kt = it.k0;
    iss_end = it.k0 + it.nk;
    xbase = reinterpret_cast<const char*>(p.x.p) + (LX == ROW ? 2L * m0 * p.x.ld : 2L * m0) + it.k0 * xstep;
    w_tile = LW == ROW ? 2L * n0 * p.w.ld : 2L * n0;
    if (PAIRED) {
      wbase = reinterpret_cast<const char*>(p.w.p) + w_tile + it.k0 * wstep;
      wbase1 = reinterpret_cast<const char*>(p.w1) + w_tile + it.k0 * wstep;
    } else {
      wbase = it.k0 >= cut ? reinterpret_cast<const char*>(p.w1) + w_tile + (it.k0 - cut) * wstep
                           : reinterpret_cast<const char*>(p.w.p) + w_tile + it.k0 * wstep;
    }
  };
  auto issue_begin = [&]() MM1_INLINE {
    if (iss_kt == iss_end) set_item();
  };
  // copy n of an operand in a tile that crosses its edge (`room` >= 1)
  auto edge_off = [&](auto layout, int n, int room, long ld) MM1_INLINE {
    if constexpr (decltype(layout)::value == ROW)
      return row_off(min(prow + 64 * n, room - 1), ld, crow);
    else
      return (uint32_t)(prow * (int)(2 * ld) + 2 * min(64 * n + ccol, room - 8));
  };
  // copy n of an operand (layout, `room` rows or columns from the tile's first
  // on, `full` of them in a tile), whose window starts at base
  auto copy_one = [&](auto layout, int n, int room, int full, long ld, uint32_t lane, long step, const char* base,
                      uint32_t dst) MM1_INLINE {
    if constexpr (RAGGED_K) {
      const int k_left = p.K - iss_kt * BK;
      if (k_left < BK) {
        const char* src = room >= full ? base + n * step + lane : base + edge_off(layout, n, room, ld);
        dma16(prow < k_left ? src : reinterpret_cast<const char*>(kZeros), dst);
        return;
      }
    }
    if (room >= full) dma16_sbase(lane, base + n * step, dst);
    else dma16_sbase(edge_off(layout, n, room, ld), base, dst);
  };
  auto issue = [&](int slot, auto copy) MM1_INLINE {
    constexpr int C = decltype(copy)::value;
    if constexpr (C < NCX) {
      copy_one(ic<LX>{}, C, xroom, BM, p.x.ld, xoff, xcopy, xbase, lds0 + slot * X_BYTES + (w + WAVES * C) * 1024);
    } else {
      constexpr int N = C - NCX;
      const uint32_t dst = lds0 + W0 + slot * S::W_BYTES + (w + WAVES * N) * 1024;
      if constexpr (PAIRED)        // 128 columns of each matrix, always inside
        dma16_sbase(woff, (N < 2 ? wbase : wbase1) + (N & 1) * wcopy, dst);
      else
        copy_one(ic<LW>{}, N, wroom, BN, p.w.ld, woff, wcopy, wbase, dst);
    }
  };
  auto issue_end = [&]() MM1_INLINE {
    xbase += xstep;
    wbase += wstep;
    if (PAIRED) wbase1 += wstep;
    ++iss_kt;
    if (!PAIRED && iss_kt == cut) wbase = reinterpret_cast<const char*>(p.w1) + w_tile;
    if (iss_kt == iss_end) ++iss_item;
  };

  const Frag<LX> fx(lane, lds0, TI * wm);
  // PAIRED: block wn of the first matrix, and the same block 128 columns on
  const Frag<LW> fw(lane, lds0 + W0, PAIRED ? wn : TJ * wn);
  constexpr int NM = TI * TJ, NF = TI + TJ;
  struct Frags {
    bf16x8 x[TI], w[TJ];
  };
  Frags f[2];
  auto read = [&](auto slot, auto kk, auto n, uint32_t xat, uint32_t wat, Frags& g) MM1_INLINE {
    constexpr int U = decltype(slot)::value, KK = decltype(kk)::value, N = decltype(n)::value;
    if constexpr (N < TJ) {
      if constexpr (PAIRED) g.w[N] = fw.template get<U * S::W_BYTES, 4 * N, KK>(wat);   // block parity: wn & 1 is in the base
      else g.w[N] = fw.template get<U * S::W_BYTES, N, KK>(wat);
    } else {
      g.x[N - TJ] = fx.template get<U * X_BYTES, N - TJ, KK>(xat);
    }
  };

#pragma unroll
  for (int t = 0; t < 2; ++t) {
    if (t < n_win) {
      issue_begin();
      for_each_ic<NC>([&](auto c) MM1_INLINE { issue(t, c); });
      issue_end();
    }
  }
  __asm__ volatile("s_waitcnt vmcnt(%0)" ::"n"(NC) : "memory");   // nk >= 2: two windows were issued
  lds_barrier();
  for_each_ic<NF>([&](auto n) MM1_INLINE { read(ic<0>{}, ic<0>{}, n, fx.template at<0>(), fw.template at<0>(), f[0]); });

  f32x16 acc[TJ][TI];
  int win = 0;
  // k step KK of window `win` in slot U: NM products, and between them the
  // reads of the next k step and, in the batch after the barrier and the one
  // behind it, half each of the copies into the slot the barrier freed.
  // ACTIVE: this wave computes (see WholeTiles); it copies in any case.
  auto batch = [&](auto u, auto kk, auto active) MM1_INLINE {
    constexpr int U = decltype(u)::value, KK = decltype(kk)::value;
    constexpr bool ACTIVE = decltype(active)::value;
    const Frags& cur = f[KK & 1];
    Frags& nxt = f[(KK + 1) & 1];
    constexpr bool NEXT = KK == 3;                       // reads and copies of the next window
    if constexpr (NEXT) {
      wait_dma();        // this wave's copies of window win + 1 have landed
      lds_barrier();     // ... and everyone's, and every read of slot U is done
      if (win + 2 < n_win) issue_begin();
    }
    constexpr int C0 = KK == 3 ? 0 : (NC + 1) / 2, CN = KK == 3 ? (NC + 1) / 2 : NC / 2;   // its copies
    const bool copy = KK == 3 ? win + 2 < n_win : KK == 0 && win > 0 && win + 1 < n_win;
    constexpr int ISLOT = KK == 3 ? U : U ^ 1;
    const uint32_t xat = fx.template at<(KK + 1) & 3>(), wat = fw.template at<(KK + 1) & 3>();
    for_each_ic<NM>([&](auto m) MM1_INLINE {
      constexpr int M = decltype(m)::value;
      if constexpr (ACTIVE) {
        if constexpr (M < NF) read(ic<NEXT ? U ^ 1 : U>{}, ic<(KK + 1) & 3>{}, m, xat, wat, nxt);
        __builtin_amdgcn_sched_barrier(0);
        acc[M % TJ][M / TJ] = mfma32(cur.w[M % TJ], cur.x[M / TJ], acc[M % TJ][M / TJ]);
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr ((KK == 3 || KK == 0) && M % 2 == 0 && M / 2 < CN) {
        if (copy) issue(ISLOT, ic<C0 + M / 2>{});
      }
      __builtin_amdgcn_sched_barrier(0);
    });
    static_assert(NF < NM && (NC + 1) / 2 <= (NM + 1) / 2, "reads and copies fit between the products");
    if constexpr (KK == 0) {
      if (copy) issue_end();
    }
  };
  auto window = [&](auto u, auto active) MM1_INLINE {
    batch(u, ic<0>{}, active);
    batch(u, ic<1>{}, active);
    batch(u, ic<2>{}, active);
    batch(u, ic<3>{}, active);
    ++win;
  };
  for (int i = 0; i < tiles.n; ++i) {
    const Item it = tiles.at(i);
    int mb, nb;
    tile_coords(it.tile, p.n_mblk, p.n_nblk, mb, nb);
    pro(mb, nb);
    // the half of the columns a wave holds: columns BN/2 * (2wn / WN) .. of
    // the tile, or (PAIRED) columns 64 (wn >> 1) .. of both matrices
    if (it.half < 0 || (2 * wn) / S::WN == it.half) {
#pragma unroll
      for (int a = 0; a < TJ; ++a) {
#pragma unroll
        for (int b = 0; b < TI; ++b) acc[a][b] = zero16();
      }
      for (int kt = 0; kt < it.nk; kt += 2) {
        window(ic<0>{}, std::true_type{});
        window(ic<1>{}, std::true_type{});
      }
      epi(mb, nb, acc, it.part);
    } else {
      for (int kt = 0; kt < it.nk; kt += 2) {
        window(ic<0>{}, std::false_type{});
        window(ic<1>{}, std::false_type{});
      }
    }
  }
}

// Stores one bf16 output of a wave's tile, 128 rows x 32 columns (PAIRED),
// whose values the lane holds as val(i, q): the bf16x4 of columns 8q +
// 4(lane/32) .. +3 of row 32i + (lane & 31) (the accumulator layout above).
// Stored directly, an instruction writes 32 separate 16-byte pieces; here
// they go through `lds` (4 KiB owned by the wave) in two rounds of 64 rows,
// after which each lane holds 16 bytes of one 64-byte row and an instruction
// writes 16 rows.  row(r) is the global address of the first column of row r
// (0..127) of the tile, or nullptr for a row outside the tensor.  The 16-byte
// chunks of LDS row r are permuted by chunk ^ ((r >> 2) & 3), which spreads
// the writes over the banks.  wave_sync() orders the lanes' exchange, which
// the compiler's per-thread view of memory does not see.  NT: non-temporal.
template <bool NT>
__device__ __forceinline__ void store8(__bf16* p, const bf16x8& v) {
  if constexpr (NT) __builtin_nontemporal_store(v, reinterpret_cast<bf16x8*>(p));
  else *reinterpret_cast<bf16x8*>(p) = v;
}

template <bool NT, class Val, class Row>
__device__ __forceinline__ void store_rows64(char* lds, int lane, Val&& val, Row&& row) {
  const int l32 = lane & 31, h = lane >> 5;
#pragma unroll
  for (int half = 0; half < 2; ++half) {
#pragma unroll
    for (int ii = 0; ii < 2; ++ii) {
      const int r = 32 * ii + l32;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const bf16x4 v = val(2 * half + ii, q);
        *reinterpret_cast<bf16x4*>(lds + r * 64 + ((q ^ ((r >> 2) & 3)) << 4) + 8 * h) = v;
      }
    }
    wave_sync();
    bf16x8 x[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int r = 16 * k + (lane >> 2), c = lane & 3;
      x[k] = *reinterpret_cast<const bf16x8*>(lds + r * 64 + ((c ^ ((r >> 2) & 3)) << 4));
    }
    wave_sync();
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int r = 16 * k + (lane >> 2), c = lane & 3;
      __bf16* p = row(64 * half + r);
      if (p) store8<NT>(p + 8 * c, x[k]);
    }
  }
}

// The same for 32 rows x 32 columns through 2 KiB: val(q) as above.
template <bool NT, class Val, class Row, class ChunkOk>
__device__ __forceinline__ void store_block64(char* lds, int lane, Val&& val, Row&& row, ChunkOk&& chunk_ok) {
  const int l32 = lane & 31, h = lane >> 5;
#pragma unroll
  for (int q = 0; q < 4; ++q)
    *reinterpret_cast<bf16x4*>(lds + l32 * 64 + ((q ^ ((l32 >> 2) & 3)) << 4) + 8 * h) = val(q);
  wave_sync();
  bf16x8 x[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int r = 16 * k + (lane >> 2), c = lane & 3;
    x[k] = *reinterpret_cast<const bf16x8*>(lds + r * 64 + ((c ^ ((r >> 2) & 3)) << 4));
  }
  wave_sync();
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int r = 16 * k + (lane >> 2), c = lane & 3;
    __bf16* p = row(r);
    if (p && chunk_ok(c)) store8<NT>(p + 8 * c, x[k]);
  }
}

// The same for 32 rows x 64 columns (two 32-column blocks, the single-matrix
// layout): val(b, q) is the bf16x4 of columns 32b + 8q + 4(lane/32) .. +3 of
// row lane & 31.  Each lane then holds 16 bytes of one 128-byte row and an
// instruction writes 8 rows.  chunk_ok(c) says whether the 8 columns
// 8c .. 8c+7 exist.  Chunks of LDS row r are permuted by chunk ^ ((r >> 1) & 7).
template <bool NT, class Val, class Row, class ChunkOk>
__device__ __forceinline__ void store_block128(char* lds, int lane, Val&& val, Row&& row, ChunkOk&& chunk_ok) {
  const int l32 = lane & 31, h = lane >> 5;
#pragma unroll
  for (int b = 0; b < 2; ++b) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const bf16x4 v = val(b, q);
      const int chunk = (4 * b + q) ^ ((l32 >> 1) & 7);
      *reinterpret_cast<bf16x4*>(lds + l32 * 128 + (chunk << 4) + 8 * h) = v;
    }
  }
  wave_sync();
  bf16x8 x[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int r = 8 * k + (lane >> 3), c = lane & 7;
    x[k] = *reinterpret_cast<const bf16x8*>(lds + r * 128 + ((c ^ ((r >> 1) & 7)) << 4));
  }
  wave_sync();
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int r = 8 * k + (lane >> 3), c = lane & 7;
    __bf16* p = row(r);
    if (p && chunk_ok(c)) store8<NT>(p + 8 * c, x[k]);
  }
}

// 32 rows x 32 columns in fp32, ROWS (16 or 32) rows at a time through ROWS x
// 128 bytes: val(q) is the f32x4 of columns 8q + 4(lane/32) .. +3 of row
// lane & 31, row(r) the global address of row r's first column or nullptr,
// chunk_ok(c) whether columns 4c .. 4c+3 exist.  An instruction writes 8 whole
// 128-byte rows; stored directly it writes 32 bytes of each of 32 rows
// (49152 x 1280 x 1000, fp32 output past the caches: 184 -> 165 us with it, x
// 2000 276 -> 249, x 500 98 -> 93; weight gradients of a few MB unchanged).
template <int ROWS, bool NT, class Val, class Row, class ChunkOk>
__device__ __forceinline__ void store_block_f32(char* lds, int lane, Val&& val, Row&& row, ChunkOk&& chunk_ok) {
  const int l32 = lane & 31, h = lane >> 5;
#pragma unroll
  for (int r0 = 0; r0 < 32; r0 += ROWS) {
    const int wr = l32 - r0;
    if (wr >= 0 && wr < ROWS) {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<f32x4*>(lds + wr * 128 + (((2 * q + h) ^ ((wr >> 1) & 7)) << 4)) = val(q);
    }
    wave_sync();
    f32x4 x[ROWS / 8];
#pragma unroll
    for (int k = 0; k < ROWS / 8; ++k) {
      const int r = 8 * k + (lane >> 3), c = lane & 7;
      x[k] = *reinterpret_cast<const f32x4*>(lds + r * 128 + ((c ^ ((r >> 1) & 7)) << 4));
    }
    wave_sync();
#pragma unroll
    for (int k = 0; k < ROWS / 8; ++k) {
      const int r = 8 * k + (lane >> 3), c = lane & 7;
      float* p = row(r0 + r);
      if (p && chunk_ok(c)) {
        if constexpr (NT) __builtin_nontemporal_store(x[k], reinterpret_cast<f32x4*>(p + 4 * c));
        else *reinterpret_cast<f32x4*>(p + 4 * c) = x[k];
      }
    }
  }
}

// A wave's 128 rows x 64 columns in four rounds of 32 rows: val(i, b, q) as
// above for row 32i + (lane & 31), row(r) for r = 0..127.
template <bool NT, class Val, class Row, class ChunkOk>
__device__ __forceinline__ void store_rows128(char* lds, int lane, Val&& val, Row&& row, ChunkOk&& chunk_ok) {
#pragma unroll
  for (int i = 0; i < 4; ++i)
    store_block128<NT>(
        lds, lane, [&](int b, int q) { return val(i, b, q); }, [&](int r) { return row(32 * i + r); }, chunk_ok);
}

// ---------------------------------------------------------------------------
// Small tiles: 64 rows x 64 columns per workgroup of 4 waves, for products
// with too few 256-wide tiles to occupy the CUs, whose time is the latency of
// one workgroup's walk over k.  An eight-slot ring (16 KiB per 64-k window)
// keeps seven windows in flight, against one in the large tile; the LDS panels
// and swizzles are the same.  Wave w of the plain form owns the 32 x 32 block
// (w & 1, w >> 1); PAIRED (32 columns of each of two matrices) gives wave w
// rows 32 (w & 1) and both column blocks for the k steps 2 (w >> 1), +1 of
// every window, so that a lane holds the same (row, column) of both; the two k
// halves are summed through LDS (small_sum_halves).
constexpr int SMALL = 64, SMALL_WAVES = 4, SMALL_SLOTS = 8;
constexpr int SMALL_SLOT = 4 * PANEL;                     // X panels 0, 1; W panels 0, 1
constexpr int SMALL_LDS = SMALL_SLOTS * SMALL_SLOT;

// Fragment reads of one 32-row (column) block with a run-time slot offset.
template <Layout L>
struct SmallFrag;

template <>
struct SmallFrag<ROW> {
  uint32_t base;
  __device__ __forceinline__ SmallFrag(int lane, uint32_t region, int blk) {
    const int l32 = lane & 31, h = lane >> 5;
    base = region + blk * PANEL + l32 * 128 + 16 * (h ^ ((l32 >> 1) & 7));
  }
  __device__ __forceinline__ bf16x8 get(int slot_off, int kk) const {
    return *reinterpret_cast<const MM1_LDS bf16x8*>((const MM1_LDS char*)(uintptr_t)((base ^ (32 * kk)) + slot_off));
  }
};

template <>
struct SmallFrag<COL> {
  uint32_t off[2];
  __device__ __forceinline__ SmallFrag(int lane, uint32_t region, int blk) {
    const int h = lane >> 5, g = (lane >> 4) & 1, j = lane & 15, jj = j >> 2;
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const int row = 8 * h + 4 * r + jj, s = (((jj >> 1) & 1) << 2) | ((2 * h + r) & 3);
      off[r] = region + row * 128 + 16 * ((4 * blk + 2 * g + ((j & 3) >> 1)) ^ s) + 8 * (j & 1);
    }
  }
  __device__ __forceinline__ bf16x8 get(int slot_off, int kk) const {
    bf16x8 out;
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const bf16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
          (MM1_LDS bf16x4*)((const MM1_LDS char*)(uintptr_t)off[r] + (slot_off + (kk >> 1) * PANEL + 2048 * (kk & 1))));
#pragma unroll
      for (int q = 0; q < 4; ++q) out[4 * r + q] = v[q];
    }
    return out;
  }
};

// Windows w0 .. w0 + nw - 1 of the tile (mb, nb): acc[0] the wave's block, or
// (PAIRED) acc[0], acc[1] the blocks of the two matrices over the wave's k
// half.  All 256 threads call it; it ends with a barrier, so the ring is free.
template <Layout LX, Layout LW, bool PAIRED>
__device__ __forceinline__ void run_small(const Problem& p, char* smem, int mb, int nb, int w0, int nw,
                                          f32x16 (&acc)[PAIRED ? 2 : 1]) {
  constexpr bool RAGGED_K = LX == COL && LW == COL;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_addr(smem));
  // copies: piece w (8 LDS rows) of X panels 0, 1 and W panels 0, 1
  const int lr = 8 * w + (lane >> 3);
  const int crow = 8 * ((lane & 7) ^ ((lr >> 1) & 7));
  const int ccol = 8 * ((lane & 7) ^ ((((lr >> 1) & 1) << 2) | ((lr >> 2) & 3)));
  const __bf16* src[4];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const int x0 = mb * SMALL;
    src[c] = LX == ROW ? p.x.p + (long)min(x0 + 32 * c + lr, p.x.n - 1) * p.x.ld + crow + (long)w0 * BK
                       : p.x.p + (long)(w0 * BK + 32 * c + lr) * p.x.ld + min(x0 + ccol, p.x.n - 8);
    if (PAIRED) {      // 32 columns of each matrix
      src[2 + c] = (ccol < 32 ? p.w.p : p.w1) + (long)(w0 * BK + 32 * c + lr) * p.w.ld + nb * 32 + (ccol & 31);
    } else {
      const int n0 = nb * SMALL;
      src[2 + c] = LW == ROW ? p.w.p + (long)min(n0 + 32 * c + lr, p.w.n - 1) * p.w.ld + crow + (long)w0 * BK
                             : p.w.p + (long)(w0 * BK + 32 * c + lr) * p.w.ld + min(n0 + ccol, p.w.n - 8);
    }
  }
  const long xstep = LX == ROW ? BK : BK * p.x.ld, wstep = LW == ROW ? BK : BK * p.w.ld;
  int k_left = p.K - w0 * BK;      // of the window being issued
  auto issue = [&](int slot) MM1_INLINE {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const __bf16* s = src[c];
      if (RAGGED_K && k_left < BK && 32 * (c & 1) + lr >= k_left) s = reinterpret_cast<const __bf16*>(kZeros);
      dma16(s, lds0 + slot * SMALL_SLOT + c * PANEL + w * 1024);
      src[c] += c < 2 ? xstep : wstep;
    }
    k_left -= BK;
  };
  const SmallFrag<LX> fx(lane, lds0, w & 1);
  const SmallFrag<LW> fw(lane, lds0 + 2 * PANEL, PAIRED ? 0 : w >> 1);
  const SmallFrag<LW> fw1(lane, lds0 + 2 * PANEL, 1);     // PAIRED: the second matrix
#pragma unroll
  for (int a = 0; a < (PAIRED ? 2 : 1); ++a) acc[a] = zero16();
  for (int i = 0; i < SMALL_SLOTS - 1 && i < nw; ++i) issue(i);
  for (int i = 0; i < nw; ++i) {
    // window i has landed; the newer ones stay in flight
    if (i + SMALL_SLOTS - 2 < nw)
      __asm__ volatile("s_waitcnt vmcnt(%0)" ::"n"(4 * (SMALL_SLOTS - 2)) : "memory");
    else
      wait_dma();
    lds_barrier();     // ... everyone's, and every read of window i - 1 is done
    if (i + SMALL_SLOTS - 1 < nw) issue((i + SMALL_SLOTS - 1) % SMALL_SLOTS);
    const int so = (i % SMALL_SLOTS) * SMALL_SLOT;
    if constexpr (PAIRED) {
      const int kk0 = 2 * (w >> 1);
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const bf16x8 x = fx.get(so, kk0 + j);
        acc[0] = mfma32(fw.get(so, kk0 + j), x, acc[0]);
        acc[1] = mfma32(fw1.get(so, kk0 + j), x, acc[1]);
      }
    } else {
      bf16x8 x[4], y[4];
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) {
        x[kk] = fx.get(so, kk);
        y[kk] = fw.get(so, kk);
      }
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) acc[0] = mfma32(y[kk], x[kk], acc[0]);
    }
  }
  __syncthreads();
}

// PAIRED: adds the second k half's accumulators (waves 2, 3) to the first's
// (waves 0, 1, for which it returns true).
__device__ __forceinline__ bool small_sum_halves(char* smem, f32x16 (&acc)[2]) {
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  f32x4* buf = reinterpret_cast<f32x4*>(smem) + (w & 1) * 512 + lane;
  if (w >> 1) {
#pragma unroll
    for (int a = 0; a < 2; ++a) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        f32x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = acc[a][4 * q + e];
        buf[(4 * a + q) * 64] = v;
      }
    }
  }
  __syncthreads();
  if (w >> 1) return false;
#pragma unroll
  for (int a = 0; a < 2; ++a) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const f32x4 v = buf[(4 * a + q) * 64];
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[a][4 * q + e] += v[e];
    }
  }
  return true;
}

}  // namespace gemm
}  // namespace mm1
