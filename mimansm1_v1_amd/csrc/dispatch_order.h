// Workgroup dispatch order for the causal forward and dQ grids.
//
// The row blocks of a causal grid carry very different amounts of work: row
// block i walks about i key tiles.  How gfx950 deals workgroups out
// (measured with a per-workgroup probe of XCC / SE / CU ids and timestamps):
// launch slot b goes to XCD b % 8; each XCD hands its k-th workgroup to
// shader engine k % 4 (4 SEs of 8 CUs) and waits, in order, until that SE
// has a free CU.  With one workgroup per CU and 2-3 per CU in total (the
// training shapes) the longest-first order then ends in a ragged last round.
//
// Instead, the host deals each XCD's items to its 4 SE lanes (longest first,
// in a snake, so every lane gets the same mix), packs each lane into its
// SE's CUs (bins of near-equal modelled work), lists each lane's items in
// the order in which those CUs would ask for them, and interleaves the lanes
// position by position so the SEs progress together.  Launch slot b runs
// item order.item[b]; b % 8 is the XCD the default order gives that item, so
// each XCD works on the same (batch, KV head) set as before.  The order only
// permutes which workgroup does which row block: the results are bitwise the
// same.
//
// The table travels in the kernel arguments (no device memory, no copy).  It
// is built once per shape and cached.  The default order (order.n == 0) is
// kept for non-causal grids (equal items), tilings with two workgroups per
// CU (the two share the CU's throughput, which this model does not capture;
// the packed order measured slower for them), shapes with more items than
// the table holds, and shapes where the model finds no gain.  The per-head
// dK/dV grid is not reordered: its items are closer in size, and the model's
// gain there (about 1%) did not show in measurement.  The grouped dK/dV grid
// (below) is: its chunks run about two per CU.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mm1 {

constexpr int kOrderCap = 1536;            // items a table holds
constexpr uint16_t kNoItem = 0xFFFF;       // a launch slot without an item

struct DispatchOrder {
  int n;                                   // launch slots; 0: default order
  uint16_t item[kOrderCap];                // item of launch slot b, in the default numbering
};

// Item of this workgroup in the default numbering (blockIdx.x when the order
// is the default one), or -1 when its launch slot carries no item.
__device__ __forceinline__ int dispatch_item(const DispatchOrder& ord) {
  if (ord.n == 0) return (int)blockIdx.x;
  const int it = ord.item[blockIdx.x];
  return it == kNoItem ? -1 : it;
}

// A row-block grid: item j = (tile n_tiles-1-j/nbg, bg j%nbg) of `rows`
// packed query rows, walking 64-key tiles; `wg_per_cu` resident workgroups.
struct GridShape {
  int B, S, H, Hkv;
  int rows;
  int wg_per_cu;
};

// The grid of the forward launcher for a tiling index (1 = 128 rows, 2
// workgroups per CU; 0, 2 = 256 rows, 3 = 128, 4 = 64, 1 per CU) and of the
// dQ launcher (0 = 128 rows, 2 per CU; 1 = 256 rows, 2 = 128, 3 = 64, 1 per CU).
GridShape row_block_grid(int variant, int B, int S, int H, int Hkv);
GridShape dq_grid(int variant, int B, int S, int H, int Hkv);

// Cached order for the current device (its CU count); a table with n == 0
// when the default order applies (see above, or the MM1_DISPATCH_ORDER=0
// switch).
const DispatchOrder& dispatch_order(const GridShape& g, bool causal);

// Same for a given CU count (the host-side model; no device needed).
const DispatchOrder& dispatch_order_for(const GridShape& g, bool causal, int cus);

// ---------------------------------------------------------------------------
// Grouped dK/dV grid.  A workgroup owns one 128-key tile of one (batch, KV
// head) and walks the 32-query tiles of all G query heads of the group
// (position-major: position tiles from the sequence end down, the G heads of
// each in turn), so K and V are loaded once per group and the group sum
// happens in registers.  Key tile kt has
// len(kt) = G * n_qt(kt) query tiles; the plan splits it into
// nc(kt) = min(C, ceil(len / L)) interleaved chunks (chunk c walks tiles c,
// c + nc, c + 2*nc, ... of the position-major walk, so all chunks start at
// the sequence end and stream the same rows together), so that the long key
// tiles of a causal grid do not set the finish time.  A key tile with one chunk writes bf16
// dK/dV directly; the chunks of a split key tile write fp32 partials to
// workspace slot c, summed (in slot order) by the reduction.
//
// Default item numbering: j = (kt * C + c) * (B * Hkv) + (b * Hkv + g), key
// tiles ascending (longest first when causal); items with c >= nc(kt) are
// empty.

// Query tiles of 32 rows that key tile kt meets in one head.
__host__ __device__ inline int dkdv_n_qt(int S, int kt, bool causal) {
  const int q_begin = causal ? 128 * kt : 0;
  return (S - q_begin + 31) / 32;
}

// Chunks of a key tile with `len` query tiles.
__host__ __device__ inline int dkdv_chunks(int len, int L, int C) {
  const int n = (len + L - 1) / L;
  return n < 1 ? 1 : (n > C ? C : n);
}

// dK/dV tilings (mm1_attn_tile_desc order) that run the grouped grid and so
// leave the chunked partial-sum layout: 0 (the per-head tiling is 1).
__host__ __device__ inline bool dkdv_grouped(int variant) { return variant == 0; }

// Partial-sum slots of a dK/dV tiling in the backward workspace.
struct WsSlots {
  long stride;   // floats per slot
  int rows;      // key rows per batch element in a slot
  int slots;     // slots of dK (then as many of dV)
};

struct DkdvPlan {
  int L;            // target query tiles per chunk
  int C;            // chunks per key tile at most (<= G: the workspace holds G slots)
  int split_keys;   // keys [0, split_keys) of each batch lie in split key tiles
  int n_items;      // items in the default numbering (n_kt * C * B * Hkv)
  DispatchOrder order;   // n == 0: default order, n_items launch slots
};

// Cached plan for the current device's CU count / for a given CU count.
const DkdvPlan& dkdv_plan(int B, int S, int H, int Hkv, bool causal);
const DkdvPlan& dkdv_plan_for(int B, int S, int H, int Hkv, bool causal, int cus);

// Workspace slots of dK/dV tiling `variant` (grouped: the plan's C chunks of
// its split keys; per-head: G heads of all keys), and their bytes (0 for
// G == 1, where no partials are written).
WsSlots ws_slots(int B, int S, int H, int Hkv, bool causal, int variant);
size_t bwd_partials_bytes(int B, int S, int H, int Hkv, bool causal, int variant);

}  // namespace mm1
