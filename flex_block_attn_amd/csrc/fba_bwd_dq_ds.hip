// Backward, dQ from handed-over dS: gfx950, head_dim 128, bf16 in / fp32 accumulate / bf16 out, no atomics.
//
//   dQ = dS K                                   (reference: flex_block_attn_h100.cu:750-753)
// The reference forms dS and dQ in one key-major kernel and adds dQ into an fp32 buffer with reducing stores
// (:707-708).  Here the key-major kernel (dkdv64_kernel; dkdv_slab_kernel on tile lists) stores the bf16 dS of every selected block pair
// once, and this query-major kernel reads it back: two products per pair instead of the six of dq_kernel, which
// recomputes S and dP.  Every dQ element is still written exactly once, by the work-group that owns its row.
//
// Work-group = kWaves waves of 32 query rows, lane = query row (128 rows, two work-groups per CU; 256 or 384 rows, one per CU):
//   dQ^T += K^T dS^T                   A = K slab through transposing LDS fetches, B = dS^T through transposing LDS
//                                      fetches of the wave's own dS unit (layout: fba_common.h)
// A wave does 8 MFMAs per 2 KiB of dS and its share of a K slab, so the kernel runs at the speed of memory: K slabs (8 KiB, shared
// by the waves, mostly L2 hits) and dS units (2 KiB per wave, each read exactly once from HBM) travel global -> LDS directly
// into a ring of four stages; stage t+4 is requested when stage t is dead.  More rows per work-group share a K slab among more
// waves: half (256 rows) or a third (384) of the K bytes, and with 384 rows half as much dS again in flight per CU.
#include <algorithm>
#include <mutex>
#include <type_traits>

#include "fba_common.h"
#include "fba_kernels.h"

namespace fba {

namespace {

constexpr int kSlab = 32;
constexpr int kSlabBytes = kSlab * kRowBytes;        // 8 KiB: one K slab, or the four dS units of a step
constexpr int stage_bytes(int waves) { return kSlabBytes + waves * kDsUnitBytes; }  // K slab | dS units
constexpr int kRing = 4;

template <int N>
using IC = std::integral_constant<int, N>;

}  // namespace

template <int kMode, int kWaves>  // kMode: kNumbered or kDense
__global__ __attribute__((amdgpu_flat_work_group_size(64 * kWaves, 64 * kWaves), amdgpu_waves_per_eu(kWaves == 12 ? 3 : 2, kWaves == 12 ? 3 : 2))) void dq_from_ds_kernel(
    const BwdParams p, const Merge before) {
  extern __shared__ __attribute__((aligned(16))) char smem[];  // ring [4] of (K slab | dS units)
  constexpr int TQ = 32 * kWaves;
  constexpr int kStageBytes = stage_bytes(kWaves);
  const int own_wgs = (int)gridDim.x - before.wgs;
  if ((int)blockIdx.x >= own_wgs) return merge_parts<64 * kWaves>(before, (int)blockIdx.x - own_wgs, before.wgs);

  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // whole items first (dealt to the XCDs in contiguous spans), then the parts of the split items
  int item, part = 0, parts = 1;
  int ws_slot = (int)blockIdx.x - p.split.main_wgs;  // of a part's results
  if (ws_slot < 0) {
    item = xcd_remap(blockIdx.x, p.items_per_xcd);
    if (item >= p.split.first) return;
  } else if (!split_position<kWaves == 4 ? Look::kSingle : Look::kNever>(p.split, ws_slot, item, part, parts)) {
    return;
  }
  const int tiles_per_head = p.Sq / TQ;
  const int bh = item / tiles_per_head;
  const int qt = item - bh * tiles_per_head;
  const int b = bh / p.Hq, hq = bh - b * p.Hq;
  const int hkv = hq / (p.Hq / p.Hkv);

  const int64_t qrow0 = (int64_t)bh * p.Sq + (int64_t)qt * TQ + wave * 32;
  const char* kp = reinterpret_cast<const char*>(p.k + ((int64_t)(b * p.Hkv + hkv) * p.Skv) * kHeadDim);

  const int qblk = (qt * TQ) / p.q_block;
  // the 128-row tile of the query block that this wave's rows lie in
  const int tq = (qt * TQ - qblk * p.q_block) / 128 + (wave >> 2);
  const int64_t mrow = (p.mask_bh == 1 ? 0 : (int64_t)bh) * p.nQ + qblk;
  constexpr bool dense = kMode == kDense;
  {
    const int32_t* const base = dense ? p.q_cnt : p.pair_base;
    const int32_t* const slot_row = dense ? p.q_cnt : p.q_slot + mrow * p.nK;
    read_ahead(const_idx(p.q_cnt)[mrow], const_idx(p.q_idx)[mrow * p.nK], const_idx(slot_row)[0], const_idx(base)[0],
               const_idx(base)[dense ? 0 : p.mask_bh * p.nK]);
  }
  // lists that number more pairs than the workspace holds: nothing is fetched, and the output becomes NaN
  const int cnt = dense || workspace_holds_lists(p) ? const_idx(p.q_cnt)[mrow] : 0;
  const ConstIdx idx = const_idx(p.q_idx + mrow * p.nK);
  // pair number per list entry
  const ConstIdx slots = const_idx(dense ? nullptr : p.q_slot + mrow * p.nK);
  auto slot = [&](int e) -> int64_t {
    if constexpr (!dense) return slots[e];
    else return ((int64_t)bh * p.nK + idx[e]) * p.nQ + qblk;
  };
  const int nsub = p.k_block / kSlab;
  // this work-group's range of 32-key steps of the list: all of it, or part `part` of `parts` (boundaries on whole rings)
  const int steps_all = cnt * nsub;
  const int t_begin = parts == 1 ? 0 : 4 * (int)(((int64_t)(steps_all / 4) * part) / parts);
  const int t_end = parts == 1 ? steps_all : 4 * (int)(((int64_t)(steps_all / 4) * (part + 1)) / parts);
  const int nsteps = t_end - t_begin;
  const int e_begin = t_begin / nsub, sub_begin = t_begin - e_begin * nsub;
  const int64_t pair_bytes = (int64_t)p.q_block * p.k_block * 2;
  // dS of this wave's 32 rows: pair base + (tq * nsub + t) * 4 units + wave, t = 32-key slab inside the key block
  const int64_t head_pairs = p.mask_bh == 1 && !dense ? (int64_t)bh * const_idx(p.pair_base)[p.nK] : 0;
  const char* ds_base = reinterpret_cast<const char*>(p.ds_ws) + head_pairs * pair_bytes + ((int64_t)tq * nsub * 4 + (wave & 3)) * kDsUnitBytes;

  TransposedOffsets tr;
  tr.init(lane);
  // K slab: two copies of four rows by each of four waves, or one by each of the first eight
  const bool copies_k = kWaves <= 8 || wave < 8;
  uint32_t k_off_lane[2];
#pragma unroll
  for (int g = 0; g < 2; ++g) {
    const int row = 4 * (kWaves == 4 ? 2 * wave + g : wave & 7) + (lane >> 4);
    k_off_lane[g] = (uint32_t)(row * kRowBytes + (((lane & 15) ^ swz(row)) << 4));
  }
  const uint32_t k_dst_wave = (uint32_t)((kWaves == 4 ? 2 * wave : wave & 7) * 4 * kRowBytes);
  // until the copies of all but the `n` youngest stages have landed
  auto wait_stages = [&](auto n_c) {
    constexpr int n = decltype(n_c)::value;
    if constexpr (kWaves == 4) wait_vmem<4 * n>();
    else if (copies_k) wait_vmem<3 * n>();
    else wait_vmem<2 * n>();
  };
  const uint32_t ring_dst = lds_addr(smem);
  // Transposing fetches of the B operand from the wave's unit.  Group G = lane / 16 of the wave serves query rows
  // 16 (G % 2) .. +15 and the key half 4 (G / 2) .. +3 of each 8 keys; source lane s = lane % 16 addresses the slot of
  // key (16 jj + 8 rr + 4 (G / 2) + s / 4) and query group 4 (G % 2) + s % 4.
  int ds_off[2][2];
#pragma unroll
  for (int jj = 0; jj < 2; ++jj)
#pragma unroll
    for (int rr = 0; rr < 2; ++rr) {
      const int G = lane >> 4, s = lane & 15;
      ds_off[jj][rr] = kSlabBytes + wave * kDsUnitBytes + ds_unit_slot_off(16 * jj + 8 * rr + 4 * (G >> 1) + (s >> 2), 4 * (G & 1) + (s & 3));
    }

  f32x16 acc[4];
#pragma unroll
  for (int mb = 0; mb < 4; ++mb)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[mb][r] = 0.f;

  // sources of the next stage to request, in list order; the following list entry is read one block ahead
  const int64_t block_bytes = (int64_t)p.k_block * kRowBytes;
  int e_next = e_begin + 1, rem = nsub - sub_begin;
  int64_t k_off = nsteps > 0 ? idx[e_begin] * block_bytes + (int64_t)sub_begin * kSlabBytes : 0;
  int64_t ds_off_g = nsteps > 0 ? slot(e_begin) * pair_bytes + (int64_t)sub_begin * (4 * kDsUnitBytes) : 0;
  int blk_next = e_next < cnt ? idx[e_next] : 0;
  int64_t slot_next = e_next < cnt ? slot(e_next) : 0;
  const uint32_t lane16 = (uint32_t)lane * 16;
  auto copy_next = [&](auto ring_c) {
    constexpr int ring = decltype(ring_c)::value;
    const uint32_t dst = ring_dst + ring * kStageBytes;
    if constexpr (kWaves == 4) {
      dma16(dst + k_dst_wave, kp + k_off, k_off_lane[0]);
      dma16(dst + k_dst_wave + 4 * kRowBytes, kp + k_off, k_off_lane[1]);
    } else {
      if (copies_k) dma16(dst + k_dst_wave, kp + k_off, k_off_lane[0]);
    }
    const char* src = ds_base + ds_off_g;
    dma16_stream(dst + kSlabBytes + wave * kDsUnitBytes, src, lane16);
    dma16_stream(dst + kSlabBytes + wave * kDsUnitBytes + 1024, src, lane16 + 1024);
    if (--rem == 0) {
      rem = nsub;
      k_off = blk_next * block_bytes;
      ds_off_g = slot_next * pair_bytes;
      ++e_next;
      blk_next = e_next < cnt ? idx[e_next] : 0;
      slot_next = e_next < cnt ? slot(e_next) : 0;
    } else {
      k_off += kSlabBytes;
      ds_off_g += 4 * kDsUnitBytes;
    }
  };

  if (nsteps > 0) {
    if (0 < nsteps) copy_next(IC<0>{});
    if (1 < nsteps) copy_next(IC<1>{});
    if (2 < nsteps) copy_next(IC<2>{});
    if (3 < nsteps) copy_next(IC<3>{});
    // stage 0
    if (3 < nsteps) wait_stages(IC<3>{}); else wait_vmem<0>();
    __syncthreads();

    // step t (t % 4 == R): dQ += K_t^T dS_t
    auto step = [&](auto ring_c, int t) {
      constexpr int R = decltype(ring_c)::value;
      const char* stage = smem + R * kStageBytes;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const bf16x8 dsk = cat(lds_read_tr(stage, ds_off[j][0]), lds_read_tr(stage, ds_off[j][1]));
#pragma unroll
        for (int mb = 0; mb < 4; ++mb) {
          const int roff = 16 * j * kRowBytes;
          const bf16x8 a = cat(lds_read_tr(stage, tr.rd[mb][0] + roff), lds_read_tr(stage, tr.rd[mb][1] + roff));
          acc[mb] = mfma32(a, dsk, acc[mb]);
        }
      }
      // stage t+1 must have landed (first read in step t+1); the copies of stages t+2 and t+3 may still fly
      if (t + 3 < nsteps) wait_stages(IC<2>{}); else if (t + 2 < nsteps) wait_stages(IC<1>{}); else wait_stages(IC<0>{});
      __syncthreads();
      if (t + 4 < nsteps) copy_next(IC<R>{});
    };
    for (int t = 0; t < nsteps; t += 4) {  // nsteps is a multiple of 4
      step(IC<0>{}, t);
      step(IC<1>{}, t + 1);
      step(IC<2>{}, t + 2);
      step(IC<3>{}, t + 3);
    }
  }

  const float poison = dense ? 1.f : poison_unless_fit(p);
  if (parts > 1) {  // part of a split item: unscaled fp32 partial sums go to the workspace
    float* prow = p.split.ws + (int64_t)ws_slot * (TQ * kHeadDim) + (wave * 32 + l32) * kHeadDim;
#pragma unroll
    for (int mb = 0; mb < 4; ++mb)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<f32x4*>(prow + 32 * mb + 8 * g + 4 * h) = 
            (f32x4){acc[mb][4 * g + 0] * poison, acc[mb][4 * g + 1] * poison, acc[mb][4 * g + 2] * poison, acc[mb][4 * g + 3] * poison};
    return;
  }
  // (the ring is free: the last step ended with a barrier and requested nothing)
  store_tile_bf16(smem + wave * kSlabBytes, acc, p.scale * poison, p.dq + qrow0 * kHeadDim, lane);
}

// dQ from dS on tile lists.  The workspace is divided into (128-row query tile, 128-key tile) pairs of 16 units; the list of the work-group's
// query tile names key blocks with a predicate per 16 rows.
//
// Work-group = the 128 rows of a list, four waves of 32, two work-groups per CU.  It steps through the key blocks that some row selects, 64 keys at a
// time, with K in a ring of two chunks, and a wave none of whose rows select a block leaves its matrix work out.  dS is fetched by every wave for itself,
// only where its rows select: room for three chunks of 64 keys by 32 rows, the next requested as soon as one is used up, so that a wave with work in
// two steps of five has the dS of the next seven on its way.  Where only 16 of the rows select a chunk, the other half of its units was never
// stored and zeros are copied instead.
//
// Every wave walks the list twice, for K and for its dS, each time with 64 chunks in registers, one per lane, so that no step waits for a scalar load
// (a block of 64 keys asked for three every two steps, and every wait for one waits for the LDS reads in flight as well).
//
// Bound by what a step takes from barrier to barrier in launches of about a round (B2 H8/2 S3136 q16 k64: 36 of 46 us without any copy),
// by memory in large ones.  In steps of 32 keys, with zeros for every wave that has no dS there, so that all waves have as many copies in flight, / so:
// steps of H24 S30720, 64-token blocks, 192 of 480 kept 18.97 / 18.53 ms; B2 H8/2 S3136 q16 k64, 12 of 49 kept 188.7 / 180.6 us; B2 H8/4 S9472 q64 k128, 42 of
// 74 1817 / 1759; H22 S4096, 64-token blocks, 16 of 64 308 / 301, but 40 of 64 549 / 558 (with
// parts behind the round and dK/dV's merge in the launch 549 / 545).  Steps of 32 keys with dS as here 592 / 571 us (B2 H3 S7168 q16 k128); the copies of
// dS in between the next step's matrix instructions 18.97 / 19.39 ms for the first.
namespace {

constexpr int kAhead = 3;                         // chunks of dS that a wave has room for
constexpr int kChunkUnits = 2 * kDsUnitBytes;     // 64 keys by 32 rows
constexpr int kTilesRing = 2;                     // chunks of K
constexpr int kTilesSmem = kTilesRing * 2 * kSlabBytes + 4 * kAhead * kChunkUnits;  // 80 KiB

// The chunks of a tile list in order: key chunk << 8 | predicate bits of its block (0 past the end).
struct TileChunks {
  const int32_t* list;
  int blocks, total, lane;  // chunks of a key block, chunks up to the end
  FBA_DEVICE uint32_t load(int from) const {
    const int c = from + lane;
    if (c >= total) return 0;
    const int e = c / blocks, entry = list[e];
    return (uint32_t)((entry >> 8) * blocks + c - e * blocks) << 8 | (entry & 255);
  }
};

}  // namespace

template <int kMode>  // kNumbered or kDense
__global__ __attribute__((amdgpu_flat_work_group_size(256, 256), amdgpu_waves_per_eu(2, 2))) void dq_tiles_kernel(const BwdParams p, const Merge before) {
  extern __shared__ __attribute__((aligned(16))) char smem[];  // K chunks [2] | dS [wave][kAhead]
  const int own_wgs = (int)gridDim.x - before.wgs;
  if ((int)blockIdx.x >= own_wgs) return merge_parts<256>(before, (int)blockIdx.x - own_wgs, before.wgs);
  constexpr bool dense = kMode == kDense;
  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int item, part = 0, parts = 1;
  int ws_slot = (int)blockIdx.x - p.split.main_wgs;  // of a part's results
  if (ws_slot < 0) {
    item = xcd_remap(blockIdx.x, p.items_per_xcd);
    if (item >= p.split.first) return;
  } else if (!split_position<Look::kSingle>(p.split, ws_slot, item, part, parts)) {
    return;
  }
  const int tiles_per_head = p.Sq / 128, n_kt = p.Skv / 128;
  const int bh = item / tiles_per_head;
  const int qt = item - bh * tiles_per_head;
  const int b = bh / p.Hq, hq = bh - b * p.Hq;
  const int hkv = hq / (p.Hq / p.Hkv);
  const int64_t qrow0 = (int64_t)bh * p.Sq + (int64_t)qt * 128 + wave * 32;
  const char* const kp = reinterpret_cast<const char*>(p.k + ((int64_t)(b * p.Hkv + hkv) * p.Skv) * kHeadDim);
  const int64_t mrow = (p.mask_bh == 1 ? 0 : (int64_t)bh) * tiles_per_head + qt;
  {
    const int32_t* const base = dense ? p.q_cnt : p.pair_base;
    read_ahead(const_idx(p.q_cnt)[mrow], const_idx(base)[0], const_idx(base)[dense ? 0 : p.mask_bh * n_kt]);
  }
  // lists that number more pairs than the workspace holds: nothing is fetched, and the output becomes NaN
  const int cnt = dense || workspace_holds_lists(p) ? const_idx(p.q_cnt)[mrow] : 0;
  const int listed = cnt * (p.k_block / 64);
  const int t_begin = (int)((int64_t)listed * part / parts), t_end = (int)((int64_t)listed * (part + 1) / parts);
  const TileChunks chunks{p.q_idx + mrow * p.nK, p.k_block / 64, t_end, lane};
  const int nsteps = t_end - t_begin;

  // dS of this wave's rows: pair base + 32-key slab of the key tile * 4 units + wave
  constexpr int64_t pair_bytes = 16 * kDsUnitBytes;
  const int64_t head_pairs = p.mask_bh == 1 && !dense ? (int64_t)bh * const_idx(p.pair_base)[n_kt] : 0;
  const char* const ds_base = reinterpret_cast<const char*>(p.ds_ws) + head_pairs * pair_bytes + wave * kDsUnitBytes;
  const int32_t* const slots = dense ? nullptr : p.q_slot + mrow * n_kt;  // by key tile
  const int slot0 = dense ? (int)(bh * n_kt * tiles_per_head + qt) : 0;   // dense pairs: of key tile 0
  const uint32_t wave_bits = 3u << (2 * wave);  // predicate bits of this wave's two 16-row groups in a list entry

  TransposedOffsets tr;
  tr.init(lane);
  uint32_t k_off_lane[4];  // K chunk: wave w brings in rows 16 w .. 16 w + 15
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const int row = 4 * (4 * wave + g) + (lane >> 4);
    k_off_lane[g] = (uint32_t)(row * kRowBytes + (((lane & 15) ^ swz(row)) << 4));
  }
  const uint32_t k_dst = lds_addr(smem) + 4 * wave * 4 * kRowBytes;
  const int ds_lds = kTilesRing * 2 * kSlabBytes + wave * kAhead * kChunkUnits;
  const uint32_t ds_dst = lds_addr(smem) + ds_lds;
  // B operand from a unit: see dq_from_ds_kernel
  int ds_off[2][2];
#pragma unroll
  for (int jj = 0; jj < 2; ++jj)
#pragma unroll
    for (int rr = 0; rr < 2; ++rr) {
      const int G = lane >> 4, s = lane & 15;
      ds_off[jj][rr] = ds_lds + ds_unit_slot_off(16 * jj + 8 * rr + 4 * (G >> 1) + (s >> 2), 4 * (G & 1) + (s & 3));
    }

  f32x16 acc[4];
#pragma unroll
  for (int mb = 0; mb < 4; ++mb)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[mb][r] = 0.f;

  if (nsteps > 0) {
    // K: the chunk to be requested next
    int k_base = t_begin, k_at = 0;
    uint32_t k_now = chunks.load(k_base), k_ahead = chunks.load(k_base + 64);
    auto request_k = [&](auto ring_c) -> uint32_t {  // past the end of the list chunk 0 once more, selected by nobody
      constexpr int ring = decltype(ring_c)::value;
      if (k_at == 64) {
        k_base += 64;
        k_at = 0;
        k_now = k_ahead;
        k_ahead = chunks.load(k_base + 64);
      }
      const uint32_t chunk = (uint32_t)__builtin_amdgcn_readlane((int)k_now, k_at++);
      const char* const src = kp + (int64_t)(chunk >> 8) * (2 * kSlabBytes);
#pragma unroll
      for (int i = 0; i < 4; ++i) dma16(k_dst + ring * 2 * kSlabBytes + i * 4 * kRowBytes, src, k_off_lane[i]);
      return chunk;
    };
    // dS: the chunks this wave selects and has not requested, among the 64 at ds_at
    int ds_at = t_begin, pair_now, pair_ahead = 0;
    uint32_t ds_now, ds_ahead = 0;
    unsigned long long left;
    auto ds_load = [&](int from) {
      ds_ahead = chunks.load(from);
      const int kt = (int)(ds_ahead >> 9);
      if (from + lane < chunks.total) pair_ahead = dense ? slot0 + kt * tiles_per_head : slots[kt];
    };
    auto ds_take = [&] {
      ds_now = ds_ahead;
      pair_now = pair_ahead;
      left = __builtin_amdgcn_ballot_w64((ds_now & wave_bits) != 0);
      ds_load(ds_at + 64);
    };
    ds_load(ds_at);
    ds_take();
    const uint32_t lane16 = (uint32_t)lane * 16;
    auto request_ds = [&](int place) -> bool {
      while (left == 0) {
        if (ds_at + 64 >= chunks.total) return false;
        ds_at += 64;
        ds_take();
      }
      const int i = __builtin_ctzll(left);
      left &= left - 1;
      const uint32_t of = (uint32_t)__builtin_amdgcn_readlane((int)ds_now, i);
      const char* const src = ds_base + __builtin_amdgcn_readlane(pair_now, i) * pair_bytes + (of >> 8 & 1) * (8 * kDsUnitBytes);
      const uint32_t dst = ds_dst + place * kChunkUnits;
      // the halves of a unit are the dS of its two 16-row groups
      const bool first = (of >> (2 * wave) & 1) != 0, second = (of >> (2 * wave) & 2) != 0;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        dma16_stream(dst + j * kDsUnitBytes, first ? src + j * (4 * kDsUnitBytes) : p.zero_unit, lane16);
        dma16_stream(dst + j * kDsUnitBytes + 1024, second ? src + j * (4 * kDsUnitBytes) : p.zero_unit, lane16 + 1024);
      }
      return true;
    };

    uint32_t bits[2];  // of the chunks in the two places of K
    bool all = request_ds(0);
    bits[0] = request_k(IC<0>{});
    all = all && request_ds(1);
    bits[1] = request_k(IC<1>{});
    all = all && request_ds(2);
    if (all) wait_vmem<12>(); else wait_vmem<0>();  // the first chunk of dS and of K
    __syncthreads();

    int place = 0;     // of the next dS chunk to be used
    bool req = false;  // was dS requested at the end of the last step?
    // step t (t % 2 == R): dQ += K_t^T dS_t
    auto step = [&](auto ring_c) {
      constexpr int R = decltype(ring_c)::value;
      const bool mine = (bits[R] & wave_bits) != 0;
      if (mine) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const char* const k_stage = smem + (2 * R + u) * kSlabBytes;
          const char* const ds_stage = smem + place * kChunkUnits + u * kDsUnitBytes;
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            const bf16x8 dsk = cat(lds_read_tr(ds_stage, ds_off[j][0]), lds_read_tr(ds_stage, ds_off[j][1]));
#pragma unroll
            for (int mb = 0; mb < 4; ++mb) {
              const int roff = 16 * j * kRowBytes;
              const bf16x8 a = cat(lds_read_tr(k_stage, tr.rd[mb][0] + roff), lds_read_tr(k_stage, tr.rd[mb][1] + roff));
              acc[mb] = mfma32(a, dsk, acc[mb]);
            }
          }
        }
      }
      // K_{t+1} must have landed, requested at the end of step t - 1; the dS requested after it may still fly.  dS that step t + 1 reads is older: a chunk
      // is requested where one is used up, with the two chunks between them still to come.
      if (req) wait_vmem<4>(); else wait_vmem<0>();
      __syncthreads();
      bits[R] = request_k(IC<R>{});
      req = mine && request_ds(place);
      if (mine) place = place == kAhead - 1 ? 0 : place + 1;
    };
    for (int t = 0; t < nsteps; t += 2) {  // (an odd number of chunks: the last step has nothing to do)
      step(IC<0>{});
      step(IC<1>{});
    }
  }
  wait_vmem<0>();  // no copy is writing LDS any more
  __syncthreads();
  const float poison = dense ? 1.f : poison_unless_fit(p);
  if (parts > 1) {  // part of a split item: unscaled fp32 partial sums go to the workspace
    float* prow = p.split.ws + (int64_t)ws_slot * (128 * kHeadDim) + (wave * 32 + l32) * kHeadDim;
#pragma unroll
    for (int mb = 0; mb < 4; ++mb)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<f32x4*>(prow + 32 * mb + 8 * g + 4 * h) =
            (f32x4){acc[mb][4 * g + 0] * poison, acc[mb][4 * g + 1] * poison, acc[mb][4 * g + 2] * poison, acc[mb][4 * g + 3] * poison};
    return;
  }
  store_tile_bf16(smem + wave * kSlabBytes, acc, p.scale * poison, p.dq + (qrow0 - (int64_t)bh * (p.Sq - p.out_q)) * kHeadDim, lane, p.out_q - qt * 128 - wave * 32);
}

namespace {

// What a wave copies in place of half a dS unit that nobody stored (tile lists).  Part of the library's device image and never
// written; host code reaches it only through the address hipGetSymbolAddress returns for the current device.
__device__ __attribute__((aligned(256))) char g_zero_unit[kDsUnitBytes];

hipError_t zero_unit_address(const char** out) {
  constexpr int kMaxDevices = 64;
  static std::mutex mu;
  static const char* cache[kMaxDevices] = {};
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(mu);
  if (cache[dev] == nullptr) {
    void* ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(g_zero_unit));
    if (e != hipSuccess) return e;
    cache[dev] = static_cast<const char*>(ptr);
  }
  *out = cache[dev];
  return hipSuccess;
}

}  // namespace

__global__ __attribute__((amdgpu_flat_work_group_size(256, 256))) void merge_kernel(const Merge m) { merge_parts<256>(m, blockIdx.x, gridDim.x); }

Merge merge_of(const SplitPlan& split, int64_t slot_floats, int rows, const PartialOut* outs, int n_outs, const int32_t* order, const Pieces& pieces) {
  Merge m;
  m.ws = split.ws;
  m.note = split.look.cnt == nullptr ? nullptr : split.note;
  m.first = split.first; m.items = split.items; m.parts = split.parts;
  m.rows = rows; m.slot_floats = slot_floats;
  m.n_outs = n_outs;
  for (int i = 0; i < n_outs; ++i) m.out[i] = outs[i];
  m.order = order; m.pieces = pieces;
  m.wgs = std::max(merge_grid(split.items * (rows / 8)), pieces.header != nullptr ? 128 : 0) * n_outs;
  return m;
}

hipError_t launch_merge(const Merge& m, hipStream_t stream) {
  if (m.wgs > 0) hipLaunchKernelGGL(merge_kernel, dim3(m.wgs), dim3(256), 0, stream, m);
  return hipGetLastError();
}

hipError_t take_along(SplitPlan& split, int64_t slot_bytes, Merge& before, hipStream_t stream) {
  if (before.wgs == 0) return hipSuccess;
  if (!put_behind(split, slot_bytes, before)) {
    const hipError_t e = launch_merge(before, stream);
    before = {};
    return e;
  }
  before.wgs = std::min(before.wgs, 128 * before.n_outs);  // a work-group or so to a compute unit, while others work on dQ
  return hipSuccess;
}

// Tail splitting on block lists (two work-groups of four waves per compute unit, one of more); a part stores a tile of fp32 sums.
//
// Wide work-groups where the query blocks allow them and the launch has two rounds of them: smaller launches fill the chip
// better with 128 rows.  Backward, 128 rows everywhere / wide, 40 % kept: H24 S30720, 384-token blocks 12.49 -> 12.31 ms (dQ
// 3.36 -> 3.18 ms), 256-token blocks 12.49 -> 12.25 ms; H24 S115200 sliding window, step 51.5 -> 50.9 ms.
int plan_bwd_dq_from_ds(BwdParams& p) {
  const int64_t rows = (int64_t)p.B * p.Hq * p.Sq, enough = 2LL * device_compute_units();  // work-groups
  const int waves = p.tiled ? 4 : p.q_block % 384 == 0 && rows / 384 >= enough ? 12 : p.q_block % 256 == 0 && rows / 256 >= enough ? 8 : 4;
  const int tile = 32 * waves;
  p.num_items = p.B * p.Hq * (p.Sq / tile);
  if (p.tiled) {
    // Steps of 64 keys.  Parts behind a whole round only: B2 H8/4 S9472 q64 k64, 60 of 148 kept, 1184 tiles, step whole / in parts 1372 / 1337 us; in launches of less
    // than one they give nothing: B2 H3 S7168 q16 k128 358 / 359 us, H4 S6144 q32 k64 170.5 / 171.0, H8 S2944 q64 121.5 / 121.7, H2 S3072 q64 45.2 / 44.9.
    const bool rounds = p.num_items > enough;
    const ListLengths lengths{p.q_cnt, p.mask_bh == 1, tile, 128, p.Sq / 128, 1, p.k_block / 64};
    p.split = plan_split(p.num_items, 2, p.Skv / 64, StepCost{22, 28, 36, /*scans=*/false, /*own_pace=*/false}, (int64_t)tile * kHeadDim * 4, rounds ? p.split.ws : nullptr,
                         p.split_ws_bytes, lengths);
    return waves;
  }
  const ListLengths lengths{waves == 4 ? p.q_cnt : nullptr, p.mask_bh == 1, tile, p.q_block, p.nQ, 1, p.k_block / kSlab};
  p.split = plan_split(p.num_items, waves == 4 ? 2 : 1, p.Skv / 32, StepCost{10, 14, 18, /*scans=*/false, /*own_pace=*/false}, (int64_t)tile * kHeadDim * 4, p.split.ws,
                       p.split_ws_bytes, lengths);
  group_parts(p.split, p.Hq / p.Hkv * (p.Sq / tile), (int64_t)p.Skv * kRowBytes);
  return waves;
}

namespace {

template <int kWaves>
hipError_t launch_dq_rows(BwdParams p, hipStream_t stream, Merge before) {
  constexpr int kRows = 32 * kWaves, kSmem = kRing * stage_bytes(kWaves);
  plan_xcd_mapping(p.B * p.Hq, p.split.first, p.items_per_xcd, p.split.main_wgs);
  const int split_items = p.num_items - p.split.first;
  const bool dense = p.pair_base == nullptr;
  void (*fn)(const BwdParams, const Merge) = dense ? &dq_from_ds_kernel<kDense, kWaves> : &dq_from_ds_kernel<kNumbered, kWaves>;
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, kSmem);
  if (e != hipSuccess || (e = take_along(p.split, kRows * kHeadDim * 4, before, stream)) != hipSuccess) return e;
  hipLaunchKernelGGL(fn, dim3(p.split.main_wgs + split_items * p.split.parts + before.wgs), dim3(64 * kWaves), kSmem, stream, p, before);
  if (split_items > 0) {
    const PartialOut out{p.dq, p.scale, 0};
    return launch_merge(merge_of(p.split, kRows * kHeadDim, kRows, &out, 1, nullptr, {}), stream);
  }
  return hipGetLastError();
}

hipError_t launch_dq_tiles(BwdParams p, hipStream_t stream, Merge before) {
  plan_xcd_mapping(p.B * p.Hq, p.split.first, p.items_per_xcd, p.split.main_wgs);
  const int split_items = p.num_items - p.split.first;
  hipError_t e = zero_unit_address(&p.zero_unit);
  if (e != hipSuccess) return e;
  void (*fn)(const BwdParams, const Merge) = p.pair_base == nullptr ? &dq_tiles_kernel<kDense> : &dq_tiles_kernel<kNumbered>;
  if ((e = hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, kTilesSmem)) != hipSuccess) return e;
  if ((e = take_along(p.split, 128 * kHeadDim * 4, before, stream)) != hipSuccess) return e;
  hipLaunchKernelGGL(fn, dim3(p.split.main_wgs + split_items * p.split.parts + before.wgs), dim3(256), kTilesSmem, stream, p, before);
  if (split_items > 0) {
    const PartialOut out{p.dq, p.scale, 0, p.Sq, p.out_q};
    return launch_merge(merge_of(p.split, 128 * kHeadDim, 128, &out, 1, nullptr, {}), stream);
  }
  return hipGetLastError();
}

}  // namespace

hipError_t launch_bwd_dq_from_ds(BwdParams p, hipStream_t stream, Merge before) {
  if (p.ds_ws == nullptr) return hipErrorInvalidValue;
  const int waves = plan_bwd_dq_from_ds(p);
  if (p.tiled) return launch_dq_tiles(p, stream, before);
  return waves == 12 ? launch_dq_rows<12>(p, stream, before) : waves == 8 ? launch_dq_rows<8>(p, stream, before) : launch_dq_rows<4>(p, stream, before);
}

}  // namespace fba
