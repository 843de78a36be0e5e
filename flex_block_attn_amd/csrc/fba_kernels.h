// Host-visible parameter blocks and launchers of the gfx950 kernels.  Internal to the shared library; the public
// surface is the C ABI in include/fba.h.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace fba {

// Active-block lists, as produced by the compaction kernel.
//   q_cnt [mask_bh, nQ], q_idx [mask_bh, nQ, nK]: for every query block the ascending selected key blocks.
//   k_cnt [mask_bh, nK], k_idx [mask_bh, nK, nQ]: for every key block the ascending query blocks that select it.
// mask_bh is B*Hq, or 1 when one 2-D mask is shared by every (batch, head).

// Tail splitting.  Work-groups are handed to free slots in index order, so the last (items % slots) items of a launch
// would run as a partial round with most compute units idle.  With a workspace, those items are cut into `parts` ranges of
// their lists, each run by its own work-group at the end of the grid; the work-groups store fp32 partial results into the
// workspace and a small merge kernel combines them in a fixed order.  Items [0, first) run whole.
//
// How many parts pay depends on how long the lists are, which only the device knows.  The host plans for the longest possible ones and
// says from which length on which number pays; the kernel looks at the lists (split_parts in fba_common.h) and leaves a note for the
// merge.  Work-groups that are not needed exit at once; with one part the items are done whole and nothing is merged.

// Length of an item's list in steps of the kernel: entries of its list row(s) times the steps of an entry.
struct ListLengths {
  const int32_t* cnt;  // [1 or heads * group, rows_per_head]; null: the plan's number of parts stands
  int shared;          // one row set for all heads
  int tile_rows, list_rows, rows_per_head;  // rows of an item, rows that share a list row, list rows per head
  int group;           // rows of `group` consecutive heads add up (dK/dV: query heads of a kv head)
  int steps;           // of an entry
  const uint8_t* mask = nullptr;  // instead of cnt: the rows' masks, of `blocks` bytes each
  int blocks = 0;
};

constexpr int kMostParts = 8;  // of a split item

// Which lists the device looks at, and the line in units of what it finds: n entries in a lane, one list or four of a group.
struct ListLook {
  const int32_t* cnt;        // null: the plan's number of parts stands, unless there are masks
  const uint8_t* mask;       // null, or rows of `blocks` bytes, one of them for a block that is listed
  int blocks;
  int first, stride, last;   // rows first + 0..3, first + stride + 0..3, ... first + 15 stride + 0..3, none of them beyond first + last
  int group, rows_per_head;  // see ListLengths; row numbers count one head of a group
  // Where the split items are the last of an order of their own (dK/dV), their rows instead: item order[i] has row order[i] / row_tiles.  Else null.
  const int32_t* order;
  int row_tiles, shared;
  float step;                // steps of an entry
  // Whole items take as long as a list of  mean + spread (largest - mean)  entries, call it L, parts as long as one of  mean + 0.4 (L - mean).
  float spread, whole, cut, least;  // parts are made where whole * (the first) - cut * (the second) >= least,
  int fewest;                       // at least as many as this,
  float more[kMostParts - 2];       // and one more for each of these that the second reaches
};

struct SplitPlan {
  float* ws;      // null: nothing is split
  int first;      // first item that is split
  int parts;      // work-groups per split item, at most (>= 2 when ws is set)
  int main_wgs;   // work-groups in front of the split ones (a multiple of the XCD count)
  int items;      // that are split
  int share;      // consecutive items that read the same keys and values
  uint32_t grouped;  // bit n: n parts are dealt to the XCDs by what they read (split_position)
  ListLook look;
  int32_t* note;  // behind the parts' results: how many parts the kernel made, for the merge
};

// What a step of a list takes, in units of what one part's results cost (see fba_split.hip): in a work-group alone on its compute unit,
// in a launch where few share one and where all do.
struct StepCost {
  double alone, few, full;
  bool scans = false;     // a part reads its whole list before it takes its own steps (tile lists)
  bool own_pace = true;   // a whole round ends with its longest list (false: bound by memory, which the short ones leave to the long ones)
};

// Items and work-group slots of a launch -> plan (first = num_items, parts = 1 when nothing is split).  `slot_bytes` is
// what one part stores; the workspace must hold (num_items - first) * parts of them.  `max_steps` is the longest possible list
// of an item.  main_wgs is left to the launcher.
SplitPlan plan_split(int num_items, int wgs_per_cu, int max_steps, StepCost step, int64_t slot_bytes, void* ws, int64_t ws_bytes,
                     const ListLengths& lengths);

// What a launch with the plan `split` leaves to be merged.
struct Merge;
struct PartialOut;
struct Pieces;
Merge merge_of(const SplitPlan& split, int64_t slot_floats, int rows, const PartialOut* outs, int n_outs, const int32_t* order, const Pieces& pieces);

// Sets share and grouped: `tiles` consecutive items read the same `bytes`.
void group_parts(SplitPlan& plan, int tiles, int64_t bytes);

// The plans of the launches below, from the sizes, q_cnt / k_cnt, split.ws and split_ws_bytes of their parameters: num_items and split are set.
struct FwdParams;
struct BwdParams;
void plan_fwd(FwdParams& p);
void plan_bwd_dq(BwdParams& p);
int plan_bwd_dq_from_ds(BwdParams& p);  // waves of a work-group
// dK/dV: key rows of an item, its step's cost (see StepCost), bytes that a part stores (dV, then dK)
struct KeyTiles {
  int rows;
  double step;
  int64_t slot_bytes;
};
constexpr KeyTiles kKeyTiles128{128, 14, 2 * 128 * 128 * 4};  // block lists: dkdv64_kernel, dkdv_kernel
constexpr KeyTiles kKeyTiles64{64, 22, 2 * 64 * 128 * 4};     // tile lists: dkdv_slab_kernel
void plan_bwd_dkdv(BwdParams& p, const KeyTiles& tiles);

// Work-groups of a launch that merges parts: each does every so many blocks of eight rows, so that little is launched where
// the lists turn out too short for parts.
inline int merge_grid(int blocks) { return blocks < 1024 ? blocks : 1024; }

// How the whole items of a launch are dealt to the XCDs (see xcd_remap): contiguous spans when the launch has at least
// one (batch, head) per XCD, work-group order otherwise.  Sets items_per_xcd and the number of work-groups that come
// before the split ones.
inline void plan_xcd_mapping(int heads, int whole_items, int& items_per_xcd, int& main_wgs) {
  constexpr int kXcds = 8;
  if (heads >= kXcds) {
    items_per_xcd = (whole_items + kXcds - 1) / kXcds;
    main_wgs = items_per_xcd * kXcds;
  } else {
    items_per_xcd = 0;
    main_wgs = whole_items;
  }
}

constexpr int kSplitMaxSlots = 512;                           // two work-groups on each of 256 compute units
constexpr int64_t kSplitSlotBytes = 128 * 128 * 4 * 2;        // dK and dV partials of a key tile; forward: O^T + (m, l)
constexpr int64_t kSplitWsBytes = kSplitMaxSlots * kSplitSlotBytes + (1 << 20);

struct FwdParams {
  const __bf16* q;
  const __bf16* k;
  const __bf16* v;
  __bf16* o;
  float* lse;  // [B, Hq, Sq], natural log
  const int32_t* q_cnt;
  const int32_t* q_idx;
  int64_t mask_bh;
  int B, Hq, Hkv, Sq, Skv, nQ, nK, q_block, k_block;
  float scale_log2e;  // log2(e) / sqrt(head_dim)
  int num_items, items_per_xcd;
  // tiled = 1: q_cnt / q_idx are tile lists (qt_cnt [mask_bh, Sq/128], qt_ent [mask_bh, Sq/128, nK], see
  // tile_lists_kernel) instead of block lists
  int tiled;
  // null, or the block mask [mask_bh, nQ, nK] to be read in place of q_cnt / q_idx (block lists, up to kMaskBlocks key blocks)
  const uint8_t* mask;
  // lists that are to be made from it on the way, for a backward pass (q_cnt null: none), by so many work-groups
  struct {
    int32_t *q_cnt, *q_idx, *k_cnt, *k_idx;
    int wgs;
  } make;
  int64_t split_ws_bytes;  // size of split.ws as handed in by the caller
  int variant;  // 0: 384-row work-groups where q_block allows (measurement of that variant); 1: 128-row work-groups
  SplitPlan split;
};

// Forward straight from the block mask (fwd_mask_kernel): mask [mask_bh, nQ, nK], one byte per entry, any block sizes and lengths
// the operator takes.
struct FwdMaskParams {
  const __bf16* q;
  const __bf16* k;
  const __bf16* v;
  __bf16* o;
  float* lse;
  const uint8_t* mask;
  int64_t mask_bh;
  int B, Hq, Hkv, Sq, Skv, nQ, nK, q_block, k_block;
  float scale_log2e;
  int num_items, items_per_xcd;
  uint8_t* mask_copy;  // null, or where a copy of the mask goes
  int o_rows;          // from a head of o to the next, Sq or more
};

// Backward straight from the block mask (bwd_mask_kernel).
struct BwdMaskParams {
  const __bf16* q;
  const __bf16* k;
  const __bf16* v;
  const __bf16* o;
  const __bf16* d_o;
  const float* lse;
  __bf16* dq;
  __bf16* dk;
  __bf16* dv;
  const uint8_t* mask;
  int64_t mask_bh;
  int B, Hq, Hkv, Sq, Skv, nQ, nK, q_block, k_block;
  int o_rows;  // from a head of o to the next
  float scale, scale_log2e;
  int key_items, key_wgs, key_per_xcd, query_items, query_per_xcd;  // key tiles, the work-groups for them, query tiles
};

// Backward statistics (see stats_rows in fba_split.hip); stats null: there are some already.
struct BwdStats {
  const __bf16* o;
  const __bf16* d_o;
  const float* lse;
  float* stats;  // [2, rows]
  int64_t rows;
  // null, or where dO goes that has given_rows of the head_rows rows of a head, with rows of zeros for the rest
  __bf16* filled = nullptr;
  int head_rows = 0, given_rows = 0;
};

// A dK/dV launch whose lists differ so much that the longest of them would set its time: all items as pieces, long ones first.  Made on the
// device (plan_pieces in fba_split.hip), because only there the lists are known.
struct Piece {
  int32_t item, begin, slabs;  // slabs begin .. begin + slabs - 1 of the item's list
  int32_t slot;                // where the partial results go, or -1: the item is whole
};
struct CutItem {
  int32_t item, slot, pieces, unused;  // the item's pieces have consecutive slots
};
struct Pieces {  // in the caller's workspace
  const int32_t* header;  // number of pieces (0: the launch runs as the host has planned it), of items that are cut; null: no launch of this kind
  const Piece* list;
  const CutItem* cut;
};

// One output of the split items: where the sums go, what they are multiplied by, where in a part's slot they lie (floats); rows of a head
// that the items have and those of them that the output has (0: all).
struct PartialOut {
  __bf16* out;
  float scale;
  int64_t offset;
  int head_rows = 0, out_rows = 0;
};

// The parts of a launch that are to be summed (merge_parts in fba_common.h).  dQ does not need dK and dV, so their merge rides in the dQ launch, as
// work-groups behind its own: by itself it took 5 to 7 us, also where the device had made no parts.  Steps, a launch of its own / along: H12 S3072,
// 128-token blocks, a third kept 131.1 / 126.6 us; H12 S3456 153.1 / 147.5; H2 S6144, 384-token blocks, half kept 140.4 / 138.6; H2 S7680 190.3 / 186.4; nothing
// beyond noise in steps of a millisecond (B2 H16/4 S8192 1013.9 / 1013.2).  (In front of dQ's work-groups instead, in launches of two rounds and more: the same.)
struct Merge {
  const float* ws = nullptr;
  const int32_t* note = nullptr;  // how many parts there are; null: `parts`
  int first = 0, items = 0, parts = 1;
  int rows = 0;  // of an item
  int64_t slot_floats = 0;
  int n_outs = 0;
  PartialOut out[2] = {};
  const int32_t* order = nullptr;  // or the item of every grid index
  Pieces pieces = {};
  int wgs = 0;  // work-groups for it, a multiple of n_outs; 0: there is nothing to merge
  int64_t results_end = 0, kept_from = 0;  // bytes of the workspace that the parts' results take, from where on it holds what the merge reads besides
};

struct BwdParams {
  const __bf16* q;
  const __bf16* k;
  const __bf16* v;
  const __bf16* d_o;
  const float* stats;  // [2, B, Hq, Sq]: lse * log2(e), then -delta = -rowsum(dO o O)
  __bf16* dq;
  __bf16* dk;
  __bf16* dv;
  const int32_t* q_cnt;
  const int32_t* q_idx;
  const int32_t* k_cnt;
  const int32_t* k_idx;
  int64_t mask_bh;
  int B, Hq, Hkv, Sq, Skv, nQ, nK, q_block, k_block;
  int out_q, out_kv;  // rows of a head of dq and of dk, dv; with tile lists they may have fewer than q and k: none for what fills up the last tile
  float scale;        // 1 / sqrt(head_dim)
  float scale_log2e;  // log2(e) / sqrt(head_dim)
  int num_items, items_per_xcd;
  // tiled = 1: q_cnt / q_idx are qt_cnt / qt_ent and k_cnt / k_idx are kt_cnt [mask_bh, Skv/128] /
  // kt_ent [mask_bh, Skv/128, Sq/32] (see tile_lists_kernel)
  int tiled;
  // dS hand-over (null when unused).  The key-major kernel stores dS of every selected block pair into ds_ws and the
  // query-major kernel reads it back instead of recomputing S and dP.  Block lists:
  //   pair_base [mask_bh * nK + 1]: exclusive prefix sum of k_cnt; the last entry is the number of pairs in the lists
  //   q_slot    [mask_bh, nQ, nK]:  pair number of entry e of query block I, i.e. pair_base[m, J] + position of I in
  //                                 k_idx[m, J, :] for J = q_idx[m, I, e]; -1 beyond q_cnt
  // Pair n of head bh lives at ds_ws + (n + (mask_bh == 1 ? bh * pairs : 0)) * q_block * k_block * 2 bytes.
  // Tile lists (see tile_slots_kernel): the pairs are (128-row query tile, 128-key tile) pairs of 32 KiB,
  //   pair_base [mask_bh * Skv/128 + 1]:        exclusive prefix sum of the listed tile pairs per key tile
  //   k_slot    [mask_bh, Skv/128, Sq/32]:      pair number of every kt_ent entry
  //   q_slot    [mask_bh, Sq/128, Skv/128]:     pair number of (query tile, key tile), -1 where nothing is listed
  //   zero_unit: 2 KiB of zeros in device memory, read in place of half a dS unit that no wave stored
  // pair_base null: dense numbering, a place for every pair whether selected or not, (bh * nK + J) * nQ + I (tile lists:
  // (bh * Skv/128 + U) * Sq/128 + T) with bh over all heads; q_slot and k_slot are not read
  __bf16* ds_ws;
  int64_t ws_pairs;  // pairs ds_ws has room for
  const int32_t* pair_base;
  const int32_t* q_slot;
  const int32_t* k_slot;
  const char* zero_unit;
  SplitPlan split;
  // dkdv64_kernel: claim counters, one per XCD, in the caller's tail-splitting workspace (null: work-group i does grid
  // index i), and the number of grid indices there are to claim (see claim_work)
  int* queue;
  int total_work;
  // dkdv64_kernel, dkdv_kernel on block lists: the item of every grid index, long lists first (null: items in xcd_remap's
  // order; see order_items)
  const int32_t* order;
  int64_t split_ws_bytes;  // size of split.ws as handed in by the caller
  Pieces pieces;           // dkdv64_kernel
  int64_t results_end, kept_from;  // see Merge
  BwdStats make;           // statistics that are to be formed in front of the dK/dV kernel
};

// How a backward call hands dS over: not at all (dQ recomputes), through pairs numbered in list order, or through a place
// for every pair (dense numbering, see BwdParams).
constexpr int kRecompute = 0, kNumbered = 1, kDense = 2;

hipError_t launch_mask_compact(const uint8_t* mask, int64_t mask_bh, int nQ, int nK, int32_t* q_cnt, int32_t* q_idx,
                               int32_t* k_cnt, int32_t* k_idx, hipStream_t stream);
hipError_t launch_tile_lists(const uint8_t* mask, int64_t mask_bh, int mask_q, int mask_k, int nK, int q_block, int k_block, int n_qt,
                             int n_kt, int n_qs, int32_t* qt_cnt, int32_t* qt_ent, int32_t* kt_cnt, int32_t* kt_ent,
                             hipStream_t stream);
// Sliding window over blocks that are the tiles of a (t, h, w) grid of `n` tiles, T-major: tile j is in the window of tile i when on every
// axis it is at most `half` away from i's coordinate, which is first moved into [low, high] (shifted in at the borders).
// n[0] = 0: no window.
struct TileWindow {
  int n[3], half[3], low[3], high[3];
  __host__ __device__ bool holds(int i, int j) const {
    const int a[3] = {i / (n[1] * n[2]), i / n[2] % n[1], i % n[2]}, b[3] = {j / (n[1] * n[2]), j / n[2] % n[1], j % n[2]};
    bool in = true;
    for (int x = 0; x < 3; ++x) {
      int c = a[x] < low[x] ? low[x] : a[x];
      c = c > high[x] ? high[x] : c;
      const int d = c > b[x] ? c - b[x] : b[x] - c;
      in = in && d <= half[x];
    }
    return in;
  }
};

// Means of the blocks of one tensor, or of two in one launch (the second with n_blocks = 0: there is none).
struct BlockMeans {
  const __bf16* x;
  float* out;
  int64_t n_blocks;
  int block;
};
hipError_t launch_block_mean(const BlockMeans (&of)[2], hipStream_t stream);
hipError_t launch_ssta_mask(const float* q_mean, const float* k_mean, const uint8_t* base, uint8_t* mask, int64_t BH, int Hq, int Hkv, int nQ,
                            int nK, int q_block, int k_block, int topk, int band, int sink, const TileWindow& window, hipStream_t stream);
hipError_t launch_tile_gather(int n, const void* const* x, void* const* out, float* const* mean, const int64_t* n_seq, int T, int H, int W, int tT,
                              int tH, int tW, int to_tiles, hipStream_t stream);
hipError_t launch_tile_permute(const void* x, void* out, int64_t n_seq, int T, int H, int W, int tT, int tH, int tW,
                               int to_tiles, hipStream_t stream);
hipError_t launch_resize_rows(int n, const void* const* src, void* const* dst, const int64_t* n_seq, const int32_t* src_len, const int32_t* dst_len,
                              hipStream_t stream);
hipError_t launch_resize_mask(const uint8_t* src, uint8_t* dst, int64_t M, int src_q, int src_k, int dst_q, int dst_k, hipStream_t stream);
constexpr int kMaskBlocks = 256, kMakeRows = 1024;  // of lists that forward makes on the way, at most
hipError_t launch_fwd(FwdParams p, hipStream_t stream);
hipError_t launch_fwd_mask(FwdMaskParams p, hipStream_t stream);
bool fwd_takes_mask(int64_t rows, int64_t kv_len);
bool fwd_takes_halves(int64_t rows, int64_t kv_len);  // of block masks in fwd_half_kernel; rows: of 128-row tiles
hipError_t launch_bwd_mask(BwdMaskParams p, hipStream_t stream);
bool bwd_takes_mask(int64_t heads, int64_t kv_heads, int64_t q_len, int64_t kv_len);
hipError_t launch_bwd_stats(const BwdStats& s, hipStream_t stream);
// dK/dV launches leave their merge, if any, in *later (null: they launch it); dQ launches take one along.
hipError_t launch_bwd_dq(BwdParams p, hipStream_t stream, Merge before = {});
hipError_t launch_bwd_dkdv(BwdParams p, hipStream_t stream, Merge* later = nullptr);
hipError_t launch_bwd_dkdv64(BwdParams p, hipStream_t stream, Merge* later = nullptr);  // block lists only: 64 keys per wave, one wave per SIMD
hipError_t launch_bwd_dkdv_slab(BwdParams p, hipStream_t stream, Merge* later = nullptr);  // tile lists only: 64 keys per work-group
hipError_t launch_bwd_dq_from_ds(BwdParams p, hipStream_t stream, Merge before = {});
// Shape of a dK/dV launch over key tiles of `tile_rows` rows, whose parts store `slot_bytes` each: sets p.num_items, split,
// items_per_xcd, order, queue and total_work and the number of work-groups, and launches what has to run in front, p.make's statistics
// among it.
hipError_t plan_key_tiles(BwdParams& p, const KeyTiles& tiles, int& grid, hipStream_t stream, bool takes_pieces = false);
int device_compute_units();
// For plans without a device: as long as it lives, this thread plans for so many compute units (0: those there are).
struct AssumedUnits {
  explicit AssumedUnits(int units);
  ~AssumedUnits();
  AssumedUnits(const AssumedUnits&) = delete;
  const int before;
};
// Merges parts in a launch of its own, or of dK/dV with `later` set leaves that to the dQ launch (see Merge).
hipError_t launch_merge(const Merge& m, hipStream_t stream);
// For a dQ launch with the plan `split`, whose parts store `slot_bytes` each: it takes `before` along, with the results of its own parts behind
// those that are still to be merged, or where they do not fit there `before` is launched now and cleared.
hipError_t take_along(SplitPlan& split, int64_t slot_bytes, Merge& before, hipStream_t stream);
bool put_behind(SplitPlan& split, int64_t slot_bytes, const Merge& before);  // false where they do not fit
// Where a whole backward pass with p.split.ws keeps what (fba_split_regions in include/fba.h).
struct SplitRegions {
  int64_t parts_end, pieces_end, dq_from, dq_end, kept_from;
};
SplitRegions plan_split_regions(BwdParams p, bool from_ds);
hipError_t launch_probe_mfma(const float* src, float* sink, int work_groups, int iters, hipStream_t stream);
hipError_t launch_probe_read(const void* src, int64_t bytes, uint32_t* sink, int work_groups, hipStream_t stream);
hipError_t launch_pair_slots(const int32_t* q_cnt, const int32_t* q_idx, const int32_t* k_cnt, const int32_t* k_idx, int64_t mask_bh,
                             int nQ, int nK, int32_t* pair_base, int32_t* q_slot, int32_t* bounds, hipStream_t stream);
hipError_t launch_tile_slots(const int32_t* kt_cnt, const int32_t* kt_ent, int64_t mask_bh, int n_qt, int n_kt, int n_qs,
                             int32_t* pair_base, int32_t* kt_slot, int32_t* slot_table, int32_t* bounds, hipStream_t stream);

}  // namespace fba
