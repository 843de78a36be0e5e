// Backward, dK and dV on tile lists: gfx950, head_dim 128, bf16 in / fp32 accumulate / bf16 out, no atomics.
//
// Same mathematics as the kernels on block lists (fba_bwd_dkdv.hip).  Block sizes that are not multiples of 128 give the
// two 64-key halves of a 128-key tile query slabs of their own (with independent random 64-token blocks at 40 % density the
// tile's list is 64 % long and a half needs 62 % of its entries), so here a work-group owns 64 keys, which always lie in one
// key block, and walks exactly the slabs that select them.
//
// Work-group = 64 key rows of one (batch, kv head), eight waves, two per SIMD.  Wave w works on keys 32 (w % 2) .. +31 and on
// every fourth 32-query slab (w / 2 = position in a group of four), lane = key:
//   S = Q K^T, dP = dO V^T             A = Q / dO slab rows from LDS, B = K rows in registers / V rows from LDS
//   P = exp2(c S - lse2[q]),  dS = P o (dP - delta[q])
//   dV^T += dO^T P,  dK^T += Q^T dS    A = dO / Q slab through transposing LDS fetches, B = P / dS packed to bf16
// The list is first compacted into LDS: the entries of the 128-key tile whose predicate bits name this half, up to kChapter
// at a time (a longer list is worked off in several such chapters), so that a step costs one LDS read instead of a walk.
// The four waves of a key group hold partial sums over their slabs, which meet in LDS at the end.
// LDS: ring of two steps x four (Q slab | dO slab | lse2 | -delta) buffers, the V rows (16 KiB), the compacted list.
//
// Bound by the matrix pipe and the arithmetic between its instructions (two waves per SIMD take turns), like the 32-key
// kernel on block lists.  Two waves share a slab instead of four, so a quarter more bytes travel L2 -> LDS than with
// 128-key work-groups that walk the union of their halves' lists with the idle half skipping, but every wave works in every
// step: B1 H24 S30720, independent 64 x 64 blocks, 40 % kept, dK/dV + dQ 19.2 -> 14.5 ms.  It wins where all halves of a tile
// agree as well (15.7 -> 14.4 ms with 64-row query blocks and 128-key blocks, 14.8 -> 13.4 when the rows agree too).
#include <type_traits>

#include "fba_common.h"
#include "fba_kernels.h"

namespace fba {

namespace {

constexpr int kSlab = 32;
constexpr int kSlabBytes = kSlab * kRowBytes;       // 8 KiB
constexpr int kStatBytes = 2 * kSlab * 4;           // lse2[32] | -delta[32]
constexpr int kStageBytes = 2 * kSlabBytes + kStatBytes;
constexpr int kPar = 4;                             // slabs per step
constexpr int kTK = 64;                             // keys per work-group
constexpr int kTileBase = 2 * kPar * kStageBytes;   // V rows, behind the ring (two buffers per position in a step)
constexpr int kListBase = kTileBase + kTK * kRowBytes;
constexpr int kRound = 512;                         // list entries scanned at a time: 64 per wave
constexpr int kChapter = 2 * kRound;                // entries the LDS list holds, 8 bytes each
constexpr int kCountBase = kListBase + kChapter * 8;  // two sets of eight counts, one per wave
constexpr int kClaimBase = kCountBase + 64;
constexpr int kSmemBytes = kClaimBase + 16;
constexpr int kSlotFloats = 2 * kTK * kHeadDim;     // partial result of one part of a split item: dV rows, then dK rows
static_assert(kKeyTiles64.rows == kTK && kKeyTiles64.slot_bytes == kSlotFloats * 4);

template <int N>
using IC = std::integral_constant<int, N>;

}  // namespace

// kHandOver: every wave also stores the bf16 dS it forms to p.ds_ws (tile pairs of 16 units, see fba_common.h).
// kHalves: q_block is an odd multiple of 16, so that 16-row groups select for themselves.  The list then holds the groups that select
// these keys, and a slab is two neighbours of the list, wherever in the sequence their rows lie: the matrix instructions sum dV and dK
// over 16 rows each, S and dP take the 32 rows as they come, and the two halves of a dS unit are stored apart.  With slabs of rows that follow
// each other, half of such a slab was often masked (16-row blocks, a quarter kept: 42 % of the slabs worked on for 24 % of the
// rows): B2 H8/2 S3136 q16 k64, 12 of 49 kept, step 241 -> 208 us; B1 H22/11 S14080 q16 k64, 131 of 220 kept 8.02 -> 6.99 ms.
template <bool kHandOver, bool kHalves>
__global__ __attribute__((amdgpu_flat_work_group_size(512, 512), amdgpu_waves_per_eu(2, 2))) void dkdv_slab_kernel(const BwdParams p) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kg = wave & 1, par = wave >> 1;  // 32-key group, position in a step
  // the grid index this work-group works on: its own, or one it claims (a launch with claim counters)
  int grid_index = (int)blockIdx.x;
  if (p.queue != nullptr) {
    volatile int* claimed = reinterpret_cast<volatile int*>(smem + kClaimBase);
    if (tid == 0) *claimed = claim_work(p.queue, xcd_id(), p.total_work);
    __syncthreads();
    grid_index = __builtin_amdgcn_readfirstlane(*claimed);
    if (grid_index < 0) return;
  }
  // whole items first (dealt to the XCDs in contiguous spans), then the parts of the split items
  int item, part = 0, parts = 1;
  const int slot = grid_index - p.split.main_wgs;  // where a part's results go
  if (slot < 0) {
    item = xcd_remap(grid_index, p.items_per_xcd);
    if (item >= p.split.first) return;
  } else if (!split_position<Look::kNever>(p.split, nullptr, slot, item, part, parts)) {
    return;
  }
  const int tiles_per_head = p.Skv / kTK;
  const int bhk = item / tiles_per_head;
  const int kt = item - bhk * tiles_per_head;
  const int half = kt & 1;  // of the 128-key tile whose lists these are
  const int b = bhk / p.Hkv, hkv = bhk - b * p.Hkv;
  const int group = p.Hq / p.Hkv;
  const int64_t krow0 = (int64_t)bhk * p.Skv + (int64_t)kt * kTK;
  const int row_len = p.Sq / kSlab;  // entries per list row
  const int lists_per_head = p.Skv / 128;
  {
    const bool numbered = kHandOver && p.pair_base != nullptr;
    const ConstIdx pb = const_idx(numbered ? p.pair_base : p.k_cnt);
    read_ahead(const_idx(p.k_cnt)[(p.mask_bh == 1 ? 0 : (int64_t)b * p.Hq + hkv * group) * lists_per_head + (kt >> 1)], pb[0],
               pb[numbered ? p.mask_bh * lists_per_head : 0]);
  }
  // lists that number more pairs than the workspace holds: no slab is touched, and the outputs become NaN
  bool fits = true;
  if constexpr (kHandOver) fits = workspace_holds_lists(p);

  const uint32_t lds0 = lds_addr(smem);
  // the two waves of a position bring in its slab together, 16 rows (four wave-level copies) each
  uint32_t dma_off[4];
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const int row = 4 * g + (lane >> 4);  // of the 16
    dma_off[g] = (uint32_t)(row * kRowBytes + (((lane & 15) ^ swz(row)) << 4));
  }
  {  // V rows: wave w brings in rows 8 w .. 8 w + 7 (two copies)
    const char* src = reinterpret_cast<const char*>(p.v) + (krow0 + 8 * wave) * kRowBytes;
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      const int row = 8 * wave + 4 * g + (lane >> 4);
      dma16(lds0 + kTileBase + (8 * wave + 4 * g) * kRowBytes, src, (uint32_t)((4 * g + (lane >> 4)) * kRowBytes + (((lane & 15) ^ swz(row)) << 4)));
    }
  }
  // K rows of the wave as B operands, in registers for the whole list: lane holds key l32, d = 16 ks + 8 h .. +7
  bf16x8 kreg[8];
  {
    const __bf16* kp = p.k + (krow0 + 32 * kg + l32) * kHeadDim + 8 * h;
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) kreg[ks] = *reinterpret_cast<const bf16x8*>(kp + 16 * ks);
  }

  // Compaction of the tile's lists (one per query head of the group) into LDS, a round of kRound entries at a time: every wave
  // tests 64 of them and the waves' counts give each its place.  The scan position is scalar state, the same in all waves.
  // An LDS entry is {number over all heads, tile-pair number} of a slab, or of a 16-row group (kHalves: two threads to a list entry).
  int scan_g = fits ? 0 : group, scan_e = 0, seen = 0, flip_count = 0;
  int2* const list = reinterpret_cast<int2*>(smem + kListBase);
  constexpr int kScan = kHalves ? kRound / 2 : kRound;  // list entries of a round
  const int scan_at = kHalves ? tid >> 1 : tid, scan_half = kHalves ? tid & 1 : 0;
  // Places the entries of this half numbered [lo, hi) that follow the scan position, as many rounds as fit; returns how many.
  auto fill = [&](int lo, int hi) -> int {
    int n = 0;
    while (scan_g < group) {
      const int64_t bh = (int64_t)b * p.Hq + hkv * group + scan_g;
      const int64_t lr = (p.mask_bh == 1 ? 0 : bh) * lists_per_head + (kt >> 1);
      const int cnt = const_idx(p.k_cnt)[lr];
      // entries are asked for a round ahead, the first ones before the count is there
      auto load = [&](const int32_t* x, int e) { return e < row_len ? x[lr * row_len + e] : 0; };
      int ent_ahead = load(p.k_idx, scan_e + scan_at), pair_ahead = 0;
      if constexpr (kHandOver) pair_ahead = p.pair_base != nullptr ? load(p.k_slot, scan_e + scan_at) : 0;
      while (scan_e < cnt) {
        if (n > kChapter - kRound || seen >= hi) return n;
        const int e = scan_e + scan_at;
        const int ent = e < cnt ? ent_ahead : 0;
        int pair = pair_ahead;
        ent_ahead = load(p.k_idx, e + kScan);
        if constexpr (kHandOver) {
          if (p.pair_base == nullptr) {  // dense numbering
            pair = (int)((bh * lists_per_head + (kt >> 1)) * (p.Sq / 128)) + (ent >> 10);
          } else {
            pair_ahead = load(p.k_slot, e + kScan);
            if (p.mask_bh == 1) pair += (int)(bh * const_idx(p.pair_base)[lists_per_head]);
          }
        }
        const int bits = (ent >> (4 * half + scan_half)) & (kHalves ? 1 : 3);
        const unsigned long long on = __ballot(bits != 0);
        int* counts = reinterpret_cast<int*>(smem + kCountBase) + 8 * flip_count;
        flip_count ^= 1;
        if (lane == 0) counts[wave] = __popcll(on);
        __syncthreads();
        int before = 0, all = 0;
#pragma unroll
        for (int w = 0; w < 8; ++w) {
          const int c = __builtin_amdgcn_readfirstlane(counts[w]);
          before += w < wave ? c : 0;
          all += c;
        }
        const int first = seen > lo ? seen : lo, last = seen + all < hi ? seen + all : hi;
        const int at = seen + before + __popcll(on & ((1ull << lane) - 1ull));
        if (bits != 0 && at >= first && at < last) {
          int2 v;
          v.x = (int)(bh * row_len) + (ent >> 8);
          if constexpr (kHalves) v.x = 2 * v.x + scan_half;
          v.y = pair;
          list[n + at - first] = v;
        }
        n += last > first ? last - first : 0;
        seen += all;
        scan_e += kScan;
      }
      scan_e = 0;
      ++scan_g;
    }
    return n;
  };
  int lo = 0, hi = 0x7fffffff;
  if (parts > 1) {  // this work-group's share of the slabs that select these keys
    while (scan_g < group) fill(0, 0x7fffffff);
    const int total = seen;
    scan_g = fits ? 0 : group;
    scan_e = seen = 0;
    constexpr int kWhole = kHalves ? -2 : -1;  // pairs of 16-row groups stay together
    lo = (int)((int64_t)total * part / parts) & kWhole;
    hi = part + 1 == parts ? total : (int)((int64_t)total * (part + 1) / parts) & kWhole;
    __syncthreads();  // what the counting scan left in the list is not mixed with what follows
  }

  int n = fill(lo, hi);
  f32x16 acc_k[4], acc_v[4];
#pragma unroll
  for (int mb = 0; mb < 4; ++mb)
#pragma unroll
    for (int r = 0; r < 16; ++r) { acc_k[mb][r] = 0.f; acc_v[mb][r] = 0.f; }

  RowMajorOffsets rm;
  rm.init(lane);
  TransposedOffsets tr;
  tr.init(lane);
  const char* const qbase = reinterpret_cast<const char*>(p.q);
  const char* const dobase = reinterpret_cast<const char*>(p.d_o);
  const char* const stbase = reinterpret_cast<const char*>(p.stats);
  const int64_t rows_total = (int64_t)p.B * p.Hq * p.Sq;
  // statistics copy: lanes 0..31 fetch lse2 of the slab's 32 rows, lanes 32..63 -delta
  const uint32_t stat_off = (uint32_t)((lane >> 5) * rows_total * 4 + (lane & (kHalves ? 15 : 31)) * 4);
  const uint32_t ho_off0 = (uint32_t)ds_unit_store_off(0, lane);
  const float c = p.scale_log2e;
  // ring buffer of position `par`, step parity s: byte (2 par + s) * kStageBytes
  const uint32_t ring_dst = lds0 + 2 * par * kStageBytes;
  // per-lane fetch addresses with the wave's share folded in; what remains is a compile-time displacement
  const LdsPtr lds = lds_ptr(smem);
  LdsPtr q_ptr[8], v_ptr[8], t_ptr[4][2];
#pragma unroll
  for (int ks = 0; ks < 8; ++ks) {
    q_ptr[ks] = lds + rm.rd[ks] + 2 * par * kStageBytes;
    v_ptr[ks] = lds + rm.rd[ks] + kTileBase + kg * kSlabBytes;
  }
#pragma unroll
  for (int mb = 0; mb < 4; ++mb) {
    t_ptr[mb][0] = lds + tr.rd[mb][0] + 2 * par * kStageBytes;
    t_ptr[mb][1] = lds + tr.rd[mb][1] + 2 * par * kStageBytes;
  }
  const LdsPtr st_ptr = lds + 2 * par * kStageBytes + 2 * kSlabBytes + 16 * h;

  // A slab of the list: first row / 16 and tile-pair number of its two 16-row groups, which follow each other unless kHalves; `both` is
  // false where a list of an odd number of groups leaves the second place empty (the first group is copied there once more).
  struct Slab {
    int row[2], pair[2];
    bool both;
  };
  // Copy i (0..8) of the nine that a wave owes for its slab of a step: Q rows, dO rows, statistics.
  auto copy_part = [&](int i, uint32_t dst, const Slab& t) {
    const int64_t row = (int64_t)(kg == 0 ? t.row[0] : t.row[1]) * 16;
    if (i < 4) dma16(dst + (16 * kg + 4 * i) * kRowBytes, qbase + row * kRowBytes, dma_off[i]);
    else if (i < 8) dma16(dst + kSlabBytes + (16 * kg + 4 * (i - 4)) * kRowBytes, dobase + row * kRowBytes, dma_off[i - 4]);
    else dma4(dst + 2 * kSlabBytes, stbase + (int64_t)t.row[0] * 64, kHalves && (lane & 16) != 0 ? stat_off + (t.row[1] - t.row[0]) * 64 : stat_off);  // both waves copy the same 256 bytes
  };

  // One slab against this wave's 32 keys.  The copies of the next step's slab are issued in between the matrix
  // instructions of S and dP.
  auto compute = [&](auto buf_c, const Slab& cur, const Slab& next) {
    constexpr int so = decltype(buf_c)::value * kStageBytes;
    constexpr int no = kStageBytes - so;
    f32x16 s, dp;
    // accumulator element 4g + e of half-wave h is query row 8g + 4h + e of the slab; dP starts from -delta of its row
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const f32x4 d4 = lds_read_f32x4(st_ptr + so + 4 * kSlab + 32 * g);
#pragma unroll
      for (int e = 0; e < 4; ++e) { s[4 * g + e] = 0.f; dp[4 * g + e] = d4[e]; }
    }
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
      s = mfma32(lds_read_b128(q_ptr[ks] + so), kreg[ks], s);
      dp = mfma32(lds_read_b128(q_ptr[ks] + so + kSlabBytes), lds_read_b128(v_ptr[ks]), dp);
      copy_part(ks, ring_dst + no, next);
    }
    copy_part(8, ring_dst + no, next);
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const f32x4 l4 = lds_read_f32x4(st_ptr + so + 32 * g);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float pv = fast_exp2(__builtin_fmaf(s[4 * g + e], c, -l4[e]));
        s[4 * g + e] = pv;
        dp[4 * g + e] = pv * dp[4 * g + e];
      }
    }
    bf16x8 pk[2], dsk[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      pk[j] = pack8(s[8 * j + 0], s[8 * j + 1], s[8 * j + 2], s[8 * j + 3], s[8 * j + 4], s[8 * j + 5], s[8 * j + 6], s[8 * j + 7]);
      dsk[j] = pack8(dp[8 * j + 0], dp[8 * j + 1], dp[8 * j + 2], dp[8 * j + 3], dp[8 * j + 4], dp[8 * j + 5], dp[8 * j + 6], dp[8 * j + 7]);
    }
    if constexpr (kHandOver) {
      // 16 units per tile pair, ordered (32-key slab, 32-row slab); streaming stores: written once, read once much later
      auto unit = [&](int f) {
        return reinterpret_cast<char*>(p.ds_ws) + (int64_t)cur.pair[f] * (16 * kDsUnitBytes) + ((2 * half + kg) * 4 + ((cur.row[f] >> 1) & 3)) * kDsUnitBytes;
      };
      if constexpr (kHalves) {  // the halves of a unit are those of its rows: ds_unit_store_off(1, l) is ds_unit_store_off(0, l) ^ 128, and 1024 on
        store16_stream(unit(0) + (cur.row[0] & 1) * 1024, ho_off0 ^ (uint32_t)((cur.row[0] & 1) << 7), dsk[0]);
        if (cur.both) store16_stream(unit(1) + (cur.row[1] & 1) * 1024, ho_off0 ^ (uint32_t)((cur.row[1] & 1) << 7), dsk[1]);
      } else {
        store16_stream(unit(0), ho_off0, dsk[0]);
        store16_stream_second(unit(0), ho_off0, dsk[1]);
      }
    }
    if constexpr (kHalves) {  // (whole bits, so that inf and NaN go as well)
      const u32x4 keep = cur.both ? ~0u : 0u;
      pk[1] = __builtin_bit_cast(bf16x8, __builtin_bit_cast(u32x4, pk[1]) & keep);
      dsk[1] = __builtin_bit_cast(bf16x8, __builtin_bit_cast(u32x4, dsk[1]) & keep);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int mb = 0; mb < 4; ++mb) {
        const int roff = so + 16 * j * kRowBytes;
        const bf16x8 adv = cat(lds_read_tr(t_ptr[mb][0] + kSlabBytes + roff), lds_read_tr(t_ptr[mb][1] + kSlabBytes + roff));
        acc_v[mb] = mfma32(adv, pk[j], acc_v[mb]);
        const bf16x8 adk = cat(lds_read_tr(t_ptr[mb][0] + roff), lds_read_tr(t_ptr[mb][1] + roff));
        acc_k[mb] = mfma32(adk, dsk[j], acc_k[mb]);
      }
  };

  // Every chapter of the list: entry 4 i + par is this wave's slab of step i (past the end: the last entry, copied into a
  // buffer nobody reads, so that every wave has the same number of copies in flight at every wait).
  while (n > 0) {
    __syncthreads();  // the list is complete
    const int slabs = kHalves ? (n + 1) / 2 : n;
    const int nsteps = (slabs + kPar - 1) / kPar;
    struct Entry {
      int2 e[2];
      bool both;
    };
    auto entry_of = [&](int step) -> Entry {
      const int at = kPar * step + par, s = at < slabs ? at : slabs - 1;
      if constexpr (!kHalves) return {{list[s], {}}, true};
      const bool both = 2 * s + 1 < n;
      return {{list[2 * s], list[both ? 2 * s + 1 : 2 * s]}, both};
    };
    auto uniform = [](const Entry& e) -> Slab {
      auto u = [](int x) { return __builtin_amdgcn_readfirstlane(x); };
      if constexpr (!kHalves) {
        const int r = 2 * u(e.e[0].x), y = u(e.e[0].y);
        return {{r, r + 1}, {y, y}, true};
      }
      return {{u(e.e[0].x), u(e.e[1].x)}, {u(e.e[0].y), u(e.e[1].y)}, e.both};
    };
    Slab cur = uniform(entry_of(0)), nxt = uniform(entry_of(1));
#pragma unroll
    for (int i = 0; i < 9; ++i) copy_part(i, ring_dst, cur);
    wait_vmem<0>();
    __syncthreads();
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) pin(kreg[ks]);
    auto step = [&](auto buf_c, int i) {
      const Entry after = entry_of(i + 2);  // read ahead, used behind the barrier
      const bool worked = kPar * i + par < slabs;
      if (worked) {
        compute(buf_c, cur, nxt);
      } else {
#pragma unroll
        for (int j = 0; j < 9; ++j) copy_part(j, ring_dst + kStageBytes - decltype(buf_c)::value * kStageBytes, nxt);
      }
      // the copies of the next step's slab must have landed; the two dS stores, if any, are younger and may still fly (the
      // counter covers loads and stores alike and runs down in issue order)
      if (kHandOver && worked && cur.both) wait_vmem<2>(); else wait_vmem<0>();
      __syncthreads();  // everybody is done with this step's buffers and everybody's copies for the next have landed
      cur = nxt;
      nxt = uniform(after);
    };
    for (int i = 0; i < nsteps; i += 2) {
      step(IC<0>{}, i);
      if (i + 1 < nsteps) step(IC<1>{}, i + 1);
    }
    wait_vmem<0>();
    __syncthreads();  // no copy is writing LDS any more, and nobody reads the list
    // Most lists are one chapter.  Whatever is live across a further scan goes to scratch on the way, so that scan sits here
    // and not at the top of the loop, where every work-group would pass it: there it spilled 165 registers per lane in front
    // of the first chapter, and B2 H22 S3584, q64 k128, 57 % kept took 883 us instead of 498.
    n = __builtin_expect(scan_g < group && seen < hi, 0) ? fill(lo, hi) : 0;
  }
  wait_vmem<0>();
  __syncthreads();

  // The four waves of a key group add up their partial sums through LDS, first of dV and then of dK: every wave puts its 32 x 128
  // tile there (16 KiB, chunk c of row r at slot c ^ r, so that neither side meets bank conflicts) and thread t forms columns
  // 8 (t % 16) .. +7 of rows t / 16 and t / 16 + 32, so that a store fills whole lines.  (Half of the waves adding what the others
  // had put there, in three rounds, and stores of 8 bytes to 32 rows, before / now: B2 H16 S8192, 64-token blocks, 16 and 32 of 128
  // kept 442 / 424 and 707 / 691 us.  What is left beside the slabs is 2 us for the claim, 6.2 to 6.7 until the first products, 4 here.)
  const float poison = kHandOver ? poison_unless_fit(p) : 1.f;
  const int64_t out_row0 = krow0 - (int64_t)bhk * (p.Skv - p.out_kv);
  const int out_left = p.out_kv - kt * kTK;
  auto finish = [&](const f32x16 (&a)[4], int which, __bf16* out, float oscale) {
    f32x4* dst = reinterpret_cast<f32x4*>(smem + wave * 16384) + l32 * 32;
#pragma unroll
    for (int mb = 0; mb < 4; ++mb)
#pragma unroll
      for (int g = 0; g < 4; ++g) dst[(8 * mb + 2 * g + h) ^ l32] = (f32x4){a[mb][4 * g + 0], a[mb][4 * g + 1], a[mb][4 * g + 2], a[mb][4 * g + 3]};
    __syncthreads();
    const int r = tid >> 4, c8 = 2 * (tid & 15);
    float* const part_out = p.split.ws + (int64_t)slot * kSlotFloats + which * (kTK * kHeadDim);
#pragma unroll
    for (int k2 = 0; k2 < 2; ++k2) {  // the two key groups
      f32x4 sum[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const f32x4* src = reinterpret_cast<const f32x4*>(smem + k2 * 16384) + r * 32 + ((c8 + j) ^ r);  // two waves to the next position
        sum[j] = (src[0] + src[4 * 1024]) + (src[2 * 1024] + src[6 * 1024]);
        sum[j] *= oscale;
      }
      const int row = 32 * k2 + r;
      if (parts > 1) {  // of a split item: fp32 partial sums, dV rows, then dK rows
        *reinterpret_cast<f32x4*>(part_out + row * kHeadDim + 4 * c8) = sum[0];
        *reinterpret_cast<f32x4*>(part_out + row * kHeadDim + 4 * c8 + 4) = sum[1];
      } else {
        if (row < out_left)
          *reinterpret_cast<bf16x8*>(out + (out_row0 + row) * kHeadDim + 4 * c8) =
              pack8(sum[0][0], sum[0][1], sum[0][2], sum[0][3], sum[1][0], sum[1][1], sum[1][2], sum[1][3]);
      }
    }
  };
  finish(acc_v, 0, p.dv, poison);
  __syncthreads();
  finish(acc_k, 1, p.dk, parts > 1 ? poison : p.scale * poison);
}

hipError_t launch_bwd_dkdv_slab(BwdParams p, hipStream_t stream, Merge* later) {
  const bool hand_over = p.ds_ws != nullptr, halves = p.q_block % 32 != 0;
  void (*fn)(const BwdParams) = hand_over ? (halves ? &dkdv_slab_kernel<true, true> : &dkdv_slab_kernel<true, false>)
                                          : (halves ? &dkdv_slab_kernel<false, true> : &dkdv_slab_kernel<false, false>);
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, kSmemBytes);
  if (e != hipSuccess) return e;
  int grid;
  if ((e = plan_key_tiles(p, kKeyTiles64, grid, stream)) != hipSuccess) return e;
  hipLaunchKernelGGL(fn, dim3(grid), dim3(512), kSmemBytes, stream, p);
  if (p.num_items > p.split.first || p.pieces.header != nullptr) {
    const PartialOut outs[2] = {{p.dv, 1.f, 0, p.Skv, p.out_kv}, {p.dk, p.scale, kTK * kHeadDim, p.Skv, p.out_kv}};
    Merge m = merge_of(p.split, kSlotFloats, kTK, outs, 2, p.order, p.pieces);
    m.results_end = p.results_end;
    m.kept_from = p.kept_from;
    if (later == nullptr) return launch_merge(m, stream);
    *later = m;
  }
  return hipGetLastError();
}

}  // namespace fba
