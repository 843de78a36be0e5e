// Forward kernel: block-sparse softmax attention for gfx950, head_dim 128, bf16 in / fp32 accumulate.
//
// One work-group of 4 waves owns 128 consecutive query rows of one (batch, head); wave w owns rows [32w, 32w+32).
// The work-group walks the active-key-block list of its query block and streams every selected key block through
// LDS as 32-key slabs of K and V (a ring of four 8 KiB buffers each).
//
// Everything is kept "transposed" so that softmax statistics are per-lane scalars (lane = query row):
//   S^T[key, q]  = K[key, :] . Q[q, :]            A = K slab rows from LDS (128-bit fetches), B = Q in registers
//   P^T          = exp2(c * S^T - c * m[q])        fp32, c = log2(e) / sqrt(128); running reference m and sum l per lane
//   O^T[d, q]   += V^T[d, key] . P^T[key, q]       A = V slab through transposing LDS fetches, B = P^T packed to bf16
// The reference computes the same quantities per selected tile (flex_block_attn_h100.cu:245-290, online softmax
// :199-221, final O / l at :292); here LSE is stored as the natural-log value m/sqrt(128) + ln(l).
//
// Software pipeline.  The unit of work is a 32-key slab t.  While the VALU turns S_t into P_t, the matrix pipe computes
// S_{t+1} and adds P_{t-1} V_{t-1} into O; the three are independent, so one wave keeps both pipes busy.
// K and V slabs travel global -> LDS directly (no registers) into two rings of four 8 KiB buffers: after step t the
// buffers of K_{t+1} and V_{t-1} are dead and receive K_{t+5} and V_{t+3}, i.e. every slab is requested four steps
// before its first use.  One barrier per step orders all LDS traffic; before it each wave waits until its own copies
// of the slabs needed next have landed (all but the two youngest batches of four).
#include <algorithm>
#include <type_traits>

#include "fba_common.h"
#include "fba_kernels.h"

namespace fba {

namespace {

constexpr int kSlab = 32;                      // keys per LDS slab
constexpr int kSlabBytes = kSlab * kRowBytes;  // 8 KiB
constexpr int kRing = 4;                       // slabs per ring
constexpr float kLazy = 8.f;                   // log2 headroom before the softmax reference is raised
constexpr int kFwdSlotBytes = (128 * kHeadDim + 2 * 128) * 4;  // partial result of one part of a split item

template <int N>
using IC = std::integral_constant<int, N>;

struct FwdState {
  bf16x8 qreg[8];
  f32x16 acc_o[4];
  float l_run;  // sum over the keys this half-wave has seen of bf16(P) for the lane's query row
  float m_run;
  RowMajorOffsets rm;
  TransposedOffsets tr;
  float c;
};

// S^T for 32 keys: 8 MFMAs.  k_half points at the first of the 32 key rows inside a swizzled slab.
FBA_DEVICE f32x16 qk_half(const FwdState& st, const char* k_half) {
  f32x16 s;
#pragma unroll
  for (int r = 0; r < 16; ++r) s[r] = 0.f;
#pragma unroll
  for (int ks = 0; ks < 8; ++ks) s = mfma32(lds_read_b128(k_half, st.rm.rd[ks]), st.qreg[ks], s);
  return s;
}

// O^T += V^T P^T for 32 keys: 8 MFMAs; consecutive MFMAs go to different accumulators.  `between(i)` runs behind matrix
// instruction i: the place for the global -> LDS copies a step owes, which take a wave tens of cycles each to issue.
template <typename Between>
FBA_DEVICE void pv_half(FwdState& st, const char* v_half, const bf16x8 (&pk)[2], Between between) {
#pragma unroll
  for (int j = 0; j < 2; ++j) {
#pragma unroll
    for (int mb = 0; mb < 4; ++mb) {
      const int roff = 16 * j * kRowBytes;
      const bf16x8 a = cat(lds_read_tr(v_half, st.tr.rd[mb][0] + roff), lds_read_tr(v_half, st.tr.rd[mb][1] + roff));
      st.acc_o[mb] = mfma32(a, pk[j], st.acc_o[mb]);
      between(4 * j + mb);
    }
  }
}
FBA_DEVICE void pv_half(FwdState& st, const char* v_half, const bf16x8 (&pk)[2]) {
  pv_half(st, v_half, pk, [](int) {});
}

// Raise the softmax reference if some row of the wave would otherwise see exponents above kLazy.  Until then
// P = exp2(c (S - m)) may exceed 1, which fp32 sums and bf16 P both carry.
// `active` is false for a query row whose own mask block does not select the current key block (q_block no multiple of 64 only).
FBA_DEVICE void softmax_reference(FwdState& st, const f32x16& s, bool active) {
  float mx = s[0];
#pragma unroll
  for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[r]);
  mx = active ? mx : -INFINITY;
  // every half-wave tests the 16 keys it holds; the row maximum over both halves is formed only when the reference rises
  if (__builtin_amdgcn_ballot_w64((mx - st.m_run) * st.c > kLazy) != 0) {
    const float m_new = fmaxf(st.m_run, max_halves(mx));
    const float alpha = fast_exp2((st.m_run - m_new) * st.c);
    st.m_run = m_new;
    st.l_run *= alpha;
#pragma unroll
    for (int mb = 0; mb < 4; ++mb)
#pragma unroll
      for (int r = 0; r < 16; ++r) st.acc_o[mb][r] *= alpha;
  }
}

// P^T = exp2(c S^T - c m), packed to bf16 as the B operand of the two 16-key MFMA steps.
template <bool kRows>
FBA_DEVICE void softmax_exp(FwdState& st, f32x16& s, bf16x8 (&pk)[2], bool active) {
  const float mc = st.m_run * st.c;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    s[r] = fast_exp2(__builtin_fmaf(s[r], st.c, -mc));
    if constexpr (kRows) s[r] = active ? s[r] : 0.f;
  }
#pragma unroll
  for (int j = 0; j < 2; ++j)
    pk[j] = pack8(s[8 * j + 0], s[8 * j + 1], s[8 * j + 2], s[8 * j + 3], s[8 * j + 4], s[8 * j + 5], s[8 * j + 6], s[8 * j + 7]);
  // denominator: the sum of the same bf16 P that weighs V, two values per dot-product instruction
  const bf16x2 one2 = {(__bf16)1.f, (__bf16)1.f};
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int t = 0; t < 4; ++t)
      st.l_run = __builtin_amdgcn_fdot2_f32_bf16((bf16x2){pk[j][2 * t], pk[j][2 * t + 1]}, one2, st.l_run, false);
}

}  // namespace

// Block lists: q_block and k_block are multiples of 128, the list of a work-group is that of its query block.
// kWaves = 4: 128 query rows per work-group, two work-groups per CU.  kWaves = 12 (q_block a multiple of 384):
// 384 rows, one work-group per CU with three waves per SIMD; every K / V slab brought into LDS then feeds three
// times as many matrix instructions (the reference shares its K / V tiles between three consumer groups for the same
// reason, flex_block_attn_h100.cu:912-928).
//
// kMask: the list is read from the block mask, so that a call without gradients needs no launch that makes
// lists: H8 S4096, 128-token blocks, 12 of 32 kept 32.7 -> 30.4 us, H12 S3072 32.8 -> 30.6, H2 S10240 68.5 -> 67.2, H24/6 768 rows against 30720 keys 128.0 ->
// 126.4 (launches of a millisecond: nothing beyond noise, H24 S11520, all blocks, 1381.6 / 1381.8).  Steps that number no pairs have it make their lists on the way, a wave to a row in work-groups behind the others:
// H4 S3840 115.1 -> 112.3 us, H2 S6144 139.5 -> 137.0, H12 S3456 146.6 -> 144.4.
template <int kWaves, bool kMask>
__global__ __attribute__((amdgpu_flat_work_group_size(64 * kWaves, 64 * kWaves), amdgpu_waves_per_eu(kWaves == 12 ? 3 : 2, kWaves == 12 ? 3 : 2))) void fwd_kernel(const FwdParams p) {
  extern __shared__ __attribute__((aligned(16))) char smem[];  // K ring [4][8 KiB] | V ring [4][8 KiB]
  constexpr int TQ = 32 * kWaves;

  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  if constexpr (kMask) {
    const int own_wgs = (int)gridDim.x - p.make.wgs;
    if ((int)blockIdx.x >= own_wgs)
      return compact_row(p.mask, p.mask_bh, p.nQ, p.nK, p.make.q_cnt, p.make.q_idx, p.make.k_cnt, p.make.k_idx, ((int)blockIdx.x - own_wgs) * 4 + wave);
  }
  // whole items first (dealt to the XCDs in contiguous spans), then the parts of the split items
  int item, part = 0, parts = 1;
  int ws_slot = (int)blockIdx.x - p.split.main_wgs;  // of a part's results
  if (ws_slot < 0) {
    item = xcd_remap(blockIdx.x, p.items_per_xcd);
    if (item >= p.split.first) return;
  } else if (!split_position<kMask ? Look::kMasks : Look::kSingle>(p.split, ws_slot, item, part, parts)) {
    return;
  }
  const int tiles_per_head = p.Sq / TQ;
  const int bh = item / tiles_per_head;
  const int qt = item - bh * tiles_per_head;
  const int b = bh / p.Hq, hq = bh - b * p.Hq;
  const int hkv = hq / (p.Hq / p.Hkv);

  const int64_t qrow0 = (int64_t)bh * p.Sq + (int64_t)qt * TQ + wave * 32;
  const __bf16* qp = p.q + qrow0 * kHeadDim;
  const char* kp = reinterpret_cast<const char*>(p.k + ((int64_t)(b * p.Hkv + hkv) * p.Skv) * kHeadDim);
  const char* vp = reinterpret_cast<const char*>(p.v + ((int64_t)(b * p.Hkv + hkv) * p.Skv) * kHeadDim);

  const int64_t mrow = (p.mask_bh == 1 ? 0 : (int64_t)bh) * p.nQ + (qt * TQ) / p.q_block;
  const ConstIdx idx = const_idx(kMask ? nullptr : p.q_idx + mrow * p.nK);
  MaskList list;
  int cnt;
  if constexpr (kMask) {
    list.load(p.mask + mrow * p.nK, p.nK, lane);
    cnt = list.count();
  } else {
    cnt = const_idx(p.q_cnt)[mrow];
    read_ahead(cnt, idx[0]);
  }
  // key block of entry e, in order from e_begin on; 0 past the end
  auto entry = [&](int e) -> int {
    if constexpr (kMask) return list.take();
    else return e < cnt ? idx[e] : 0;
  };
  const int nsub = p.k_block / kSlab;
  // this work-group's range of 32-key steps of the list: all of it, or part `part` of `parts` (even boundaries)
  const int steps_all = cnt * nsub;
  const int t_begin = parts == 1 ? 0 : 2 * (int)(((int64_t)(steps_all / 2) * part) / parts);
  const int t_end = parts == 1 ? steps_all : 2 * (int)(((int64_t)(steps_all / 2) * (part + 1)) / parts);
  const int nsteps = t_end - t_begin;
  const int e_begin = t_begin / nsub, sub_begin = t_begin - e_begin * nsub;

  FwdState st;
  // Q as the B operand: lane holds row l32, d = 16 ks + 8 h .. +7
#pragma unroll
  for (int ks = 0; ks < 8; ++ks) st.qreg[ks] = *reinterpret_cast<const bf16x8*>(qp + (int64_t)l32 * kHeadDim + 16 * ks + 8 * h);
  st.rm.init(lane);
  st.tr.init(lane);
  st.c = p.scale_log2e;
  st.m_run = -INFINITY;
  st.l_run = 0.f;
#pragma unroll
  for (int mb = 0; mb < 4; ++mb)
#pragma unroll
    for (int r = 0; r < 16; ++r) st.acc_o[mb][r] = 0.f;

  SlabDmaShared<kWaves> dma;
  dma.init(wave, lane);
  char* const k_lds = smem;
  char* const v_lds = smem + kRing * kSlabBytes;
  const uint32_t k_dst = lds_addr(k_lds);
  const uint32_t v_dst = lds_addr(v_lds);

  // Slab source offsets, in list order.  The list entry of the following key block is read one block ahead, so that
  // the scalar load is off the critical path.  V requests trail K requests by two slabs and reuse their offsets.
  const int64_t block_bytes = (int64_t)p.k_block * kRowBytes;
  int e_next = e_begin + 1, rem = nsub - sub_begin;
  if constexpr (kMask) list.skip(e_begin);
  int64_t src_off = nsteps > 0 ? entry(e_begin) * block_bytes + (int64_t)sub_begin * kSlabBytes : 0;
  int blk_next = entry(e_next);
  auto next_off = [&]() -> int64_t {
    const int64_t off = src_off;
    if (--rem == 0) {
      rem = nsub;
      src_off = blk_next * block_bytes;
      ++e_next;
      blk_next = entry(e_next);
    } else {
      src_off += kSlabBytes;
    }
    return off;
  };
  // K slabs and V slabs are brought in by different (overlapping, for 12 waves) sets of waves
  auto copy_k = [&](uint32_t dst, const char* src) { dma.copy_k(dst, src); };
  auto copy_v = [&](uint32_t dst, const char* src) { dma.copy_v(dst, src); };

  if (nsteps > 0) {
    // prologue: K_0..K_3 and V_0..V_2 requested, S_0 computed, then K_4 into the buffer of K_0
    int64_t off[5] = {0, 0, 0, 0, 0};
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (j < nsteps) {
        off[j] = next_off();
        copy_k(k_dst + j * kSlabBytes, kp + off[j]);
      }
#pragma unroll
    for (int j = 0; j < 3; ++j)
      if (j < nsteps) copy_v(v_dst + j * kSlabBytes, vp + off[j]);
    wait_vmem<0>();
    __syncthreads();
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) pin(st.qreg[ks]);
    f32x16 s_cur = qk_half(st, k_lds);
    pin(s_cur);
    __syncthreads();
    if (4 < nsteps) {
      off[4] = next_off();
      copy_k(k_dst, kp + off[4]);
    }
    int64_t hist0 = off[4], hist1 = off[3];  // offsets of the two youngest K requests

    bf16x8 p_prev[2];
    // The copies a step requests (K_{t+5} into the buffer of K_{t+1}, V_{t+3} into that of V_{t-1}, both free behind the
    // step's barrier) are issued by the following step, in between its first matrix instructions where the work-group
    // has four waves: a copy takes a wave tens of cycles to issue, which the matrix pipe then covers.
    // Every step requests both, so that the counter of copies in flight means the same thing at every wait; past the end
    // of the list they repeat a listed slab into a buffer that nobody reads any more.
    uint32_t owed_k_dst = 0, owed_v_dst = 0;
    const char* owed_k_src = kp;
    const char* owed_v_src = vp;
    bool owed = false;
    constexpr bool kSpread = kWaves == 4;

    // step t (t % 4 == R): O += P_{t-1} V_{t-1} | softmax(S_t) | S_{t+1} = K_{t+1} Q^T
    auto step = [&](auto ring_c, auto first_c, int t) {
      constexpr int R = decltype(ring_c)::value;
      constexpr bool kFirst = decltype(first_c)::value;
      // P_{t-1} was formed against the reference m of step t-1, so it must reach O before step t may raise m
      if constexpr (kSpread && !kFirst) {
        pv_half(st, v_lds + ((R + 3) & 3) * kSlabBytes, p_prev, [&](int i) {
          if (i == 0) dma.copy_piece(0, owed_k_dst, owed_k_src);
          if (i == 2) dma.copy_piece(1, owed_k_dst, owed_k_src);
          if (i == 4) dma.copy_piece(0, owed_v_dst, owed_v_src);
          if (i == 6) dma.copy_piece(1, owed_v_dst, owed_v_src);
        });
      } else {
        if (owed) {
          copy_k(owed_k_dst, owed_k_src);
          copy_v(owed_v_dst, owed_v_src);
        }
        if constexpr (!kFirst) pv_half(st, v_lds + ((R + 3) & 3) * kSlabBytes, p_prev);
      }
      softmax_reference(st, s_cur, true);
      f32x16 s_nxt = qk_half(st, k_lds + ((R + 1) & 3) * kSlabBytes);  // past the last slab: stale data, unused
      softmax_exp<false>(st, s_cur, p_prev, true);  // p_prev := P_t
      // P_t is only consumed after the barrier; without the pins its arithmetic sinks there, away from the MFMAs it is
      // meant to overlap with
      pin(p_prev[0]);
      pin(p_prev[1]);
      s_cur = s_nxt;
      // K_{t+2} and V_t must have landed; the copies requested by steps t-2 and t-1 may still fly
      dma.wait_two_steps();
      __syncthreads();
      owed_v_src = vp + hist1;
      owed_v_dst = v_dst + ((R + 3) & 3) * kSlabBytes;
      hist1 = hist0;
      hist0 = next_off();
      owed_k_src = kp + hist0;
      owed_k_dst = k_dst + ((R + 1) & 3) * kSlabBytes;
      owed = true;
    };
    step(IC<0>{}, std::true_type{}, 0);
    step(IC<1>{}, std::false_type{}, 1);
    // Where the loop lies in the 64-byte lines of the instruction cache counts where a wave has its SIMD to itself (launches of less than a
    // round): H12 S2048, all blocks, 37.0 us with the loop 24 or 56 bytes into a line, 36.1 at 8, 40 or 60; it follows 24 bytes behind this point.
    asm volatile(".p2align 6\n.fill 12, 4, 0xbf800000");
    for (int t = 2; t < nsteps; t += 4) {  // nsteps is even
      step(IC<2>{}, std::false_type{}, t);
      step(IC<3>{}, std::false_type{}, t + 1);
      if (t + 2 >= nsteps) break;
      step(IC<0>{}, std::false_type{}, t + 2);
      step(IC<1>{}, std::false_type{}, t + 3);
    }
    // O += P_{n-1} V_{n-1}
    pv_half(st, v_lds + ((nsteps - 1) & 3) * kSlabBytes, p_prev);
    wait_vmem<0>();  // no copy may still be writing LDS when the work-group gives it back
  }

  const float l = sum_halves(st.l_run);
  if (parts > 1) {
    // part of a split item: unnormalised O^T, the softmax reference in log2 units and the denominator go to the workspace
    float* slot = p.split.ws + (int64_t)ws_slot * (kFwdSlotBytes / 4);
    float* prow = slot + (wave * 32 + l32) * kHeadDim;
#pragma unroll
    for (int mb = 0; mb < 4; ++mb)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<f32x4*>(prow + 32 * mb + 8 * g + 4 * h) =
            (f32x4){st.acc_o[mb][4 * g + 0], st.acc_o[mb][4 * g + 1], st.acc_o[mb][4 * g + 2], st.acc_o[mb][4 * g + 3]};
    if (h == 0) {
      slot[TQ * kHeadDim + wave * 32 + l32] = st.m_run * st.c;
      slot[TQ * kHeadDim + TQ + wave * 32 + l32] = l;
    }
    return;
  }
  // epilogue: O = O^T / l, LSE = ln2 * (c m + log2 l)
  if (h == 0) p.lse[qrow0 + l32] = l > 0.f ? (st.m_run * st.c + __builtin_log2f(l)) * 0.6931471805599453f : -INFINITY;
  __syncthreads();  // everybody is done with the rings, and no copy is on its way into them
  store_tile_bf16(smem + wave * kSlabBytes, st.acc_o, l > 0.f ? 1.f / l : 0.f, p.o + qrow0 * kHeadDim, lane);
}

// Forward on tile lists (q_block or k_block no multiple of 128), and on block masks in small launches.
//
// Work-group = 64 query rows, four waves, two work-groups per CU.  The unit of work is a chunk of 64 keys; wave w owns rows
// 32 (w % 2) .. +31 against keys 32 (w / 2) .. +31 of every chunk, with the same pipeline as fwd_kernel (P_{t-1} V_{t-1} |
// softmax of S_t | S_{t+1}).  The two waves of a row group keep softmax statistics and O of their own, which meet in LDS at
// the end.  Rings of three K chunks and two V chunks (80 KiB, half of a CU's LDS): step t requests V_t and K_{t+3}.
// The list is that of the 128-row tile; every wave keeps 64 of its entries in a register, one per lane, with a scalar mask of
// those that name this half, and takes them in order: no list in LDS, no scalar loads to wait for, only selected chunks.
//
// Bound like fwd_kernel by the matrix pipe, the softmax between its instructions and the clock these allow.  A chunk feeds half
// as many matrix instructions per byte copied as there, but with 128-row work-groups a chunk that one half selects kept the
// waves of the other waiting: B1 H24 S30720, independent 64 x 64 blocks, 40 % kept, a tile's list holds 64 % of the blocks and
// the step took 21.98 ms, now 19.30; B2 H8/2 S3136 q16 k64, a quarter kept, 301 -> 289 us.  Where the halves agree it is ahead as
// well, of a 128-row kernel that reads its tile list entry by entry: forward, 128-row query blocks and 64-key blocks, H24 S30720
// 5.18 -> 4.83 ms, H8 S4096 48 -> 37 us.
//
// kFrom: tile lists, or block masks in small launches (takes_halves).
// kRows: q_block is no multiple of 64, so the four 16-row groups of a half differ as well: a wave leaves out the matrix work
// of chunks that neither of its groups selects, rows switched off inside an active wave are dealt with by selects.
constexpr int kChunkBytes = 2 * kSlabBytes;  // 64 keys
constexpr int kHalfRows = 64;
constexpr int kHalfSlotBytes = (kHalfRows * kHeadDim + 2 * kHalfRows) * 4;  // partial result of one part of a split item
constexpr int kHalfSmem = 5 * kChunkBytes;
// Softmax reference of a row that has met no score yet.  Finite, so that exp2 never sees inf - inf where all keys of a slab are masked out or have scores of
// -inf, also when only one of a row group's two waves meets others, and below every finite score that counts (a difference to it may be infinite: its exp2 is 0).
constexpr float kNoReference = -3e38f;

// The entries of a tile list that name one 64-row half, in order; or the selected blocks of a mask row, which all name it.
// All lanes of a wave call everything together.
enum class From { kTiles, kMask };
template <From kFrom>
struct HalfList {
  const int32_t* list;
  const uint8_t* row;
  int cnt, half_mask, lane;  // cnt: entries; blocks of a mask row
  int head[4];               // this lane's entries among the first 256
  int base;                  // position of `entries` in the list
  int entries, ahead;        // this lane's entry among the 64 at `base` and the 64 behind them
  unsigned long long left;   // lanes whose entry names the half and has not been taken

  FBA_DEVICE int entry_at(int i) const {  // (within the row)
    if constexpr (kFrom == From::kMask) return row[i] != 0 ? i << 8 | 255 : 0;
    else return list[i];
  }
  FBA_DEVICE int load(int at) const { return at + lane < cnt ? entry_at(at + lane) : 0; }
  FBA_DEVICE unsigned long long named(int e) const { return __builtin_amdgcn_ballot_w64((e & half_mask) != 0); }
  // The head of the list, asked for before the count has come back (two round trips less in front of the first copy), and the count.
  FBA_DEVICE void read_head(int row_len, const int32_t* count) {
    const int at_count = kFrom == From::kMask ? row_len : const_idx(count)[0];
#pragma unroll
    for (int i = 0; i < 4; ++i) head[i] = 64 * i + lane < row_len ? entry_at(64 * i + lane) : 0;
    cnt = at_count;
#pragma unroll
    for (int i = 0; i < 4; ++i) head[i] = 64 * i + lane < cnt ? head[i] : 0;
  }
  FBA_DEVICE int total() const {
    int n = __popcll(named(head[0])) + __popcll(named(head[1])) + __popcll(named(head[2])) + __popcll(named(head[3]));
    for (int at = 256; at < cnt; at += 256) {  // four loads in flight
      const int e0 = load(at), e1 = load(at + 64), e2 = load(at + 128), e3 = load(at + 192);
      n += __popcll(named(e0)) + __popcll(named(e1)) + __popcll(named(e2)) + __popcll(named(e3));
    }
    return n;
  }
  // next() gives entry number `skip` of those that name the half
  FBA_DEVICE void start(int skip) {
    base = 0;
    entries = head[0];
    ahead = head[1];
    left = named(entries);
    while (__popcll(left) <= skip && base + 64 < cnt) {
      skip -= __popcll(left);
      refill();
    }
    for (; skip > 0; --skip) left &= left - 1;
  }
  FBA_DEVICE void refill() {
    base += 64;
    entries = ahead;
    ahead = load(base + 64);
    left = named(entries);
  }
  FBA_DEVICE bool next(int& entry) {
    while (left == 0) {
      if (base + 64 >= cnt) return false;
      refill();
    }
    entry = __builtin_amdgcn_readlane(entries, __builtin_ctzll(left));
    left &= left - 1;
    return true;
  }
};

template <bool kRows, From kFrom>
__global__ __attribute__((amdgpu_flat_work_group_size(256, 256), amdgpu_waves_per_eu(2, 2))) void fwd_half_kernel(const FwdParams p) {
  extern __shared__ __attribute__((aligned(16))) char smem[];  // K ring [3][16 KiB] | V ring [2][16 KiB]
  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rg = wave & 1, par = wave >> 1;  // row group, 32-key slab of a chunk
  if constexpr (kFrom == From::kMask) {
    const int own_wgs = (int)gridDim.x - p.make.wgs;
    if ((int)blockIdx.x >= own_wgs)
      return compact_row(p.mask, p.mask_bh, p.nQ, p.nK, p.make.q_cnt, p.make.q_idx, p.make.k_cnt, p.make.k_idx, ((int)blockIdx.x - own_wgs) * 4 + wave);
  }
  int item, part = 0, parts = 1;
  int ws_slot = (int)blockIdx.x - p.split.main_wgs;  // of a part's results
  if (ws_slot < 0) {
    item = xcd_remap(blockIdx.x, p.items_per_xcd);
    if (item >= p.split.first) return;
  } else if (kFrom != From::kTiles || !split_position<Look::kSingle>(p.split, ws_slot, item, part, parts)) {
    return;
  }
  const int tiles_per_head = p.Sq / kHalfRows;
  const int bh = item / tiles_per_head;
  const int qt = item - bh * tiles_per_head;
  const int half = qt & 1;  // of the 128-row tile whose list this is
  const int b = bh / p.Hq, hq = bh - b * p.Hq;
  const int hkv = hq / (p.Hq / p.Hkv);
  const int64_t qrow0 = (int64_t)bh * p.Sq + (int64_t)qt * kHalfRows + rg * 32;
  const __bf16* qp = p.q + qrow0 * kHeadDim;
  const char* kp = reinterpret_cast<const char*>(p.k + ((int64_t)(b * p.Hkv + hkv) * p.Skv) * kHeadDim);
  const char* vp = reinterpret_cast<const char*>(p.v + ((int64_t)(b * p.Hkv + hkv) * p.Skv) * kHeadDim);

  const int64_t mrow = kFrom == From::kTiles ? (p.mask_bh == 1 ? 0 : (int64_t)bh) * (p.Sq / 128) + (qt >> 1) : (p.mask_bh == 1 ? 0 : (int64_t)bh) * p.nQ + qt * kHalfRows / p.q_block;
  HalfList<kFrom> cursor;
  cursor.list = p.q_idx + mrow * p.nK;
  cursor.row = p.mask + mrow * p.nK;
  cursor.half_mask = 15 << (4 * half);
  cursor.lane = lane;
  cursor.read_head(p.nK, p.q_cnt + mrow);

  FwdState st;
#pragma unroll
  for (int ks = 0; ks < 8; ++ks) st.qreg[ks] = *reinterpret_cast<const bf16x8*>(qp + (int64_t)l32 * kHeadDim + 16 * ks + 8 * h);
  const int per_block = p.k_block / 64;
  const int chunks = cursor.total() * per_block;
  const int t_begin = (int)((int64_t)chunks * part / parts), t_end = (int)((int64_t)chunks * (part + 1) / parts);
  const int nsteps = t_end - t_begin;

  st.rm.init(lane);
  st.tr.init(lane);
#pragma unroll
  for (int ks = 0; ks < 8; ++ks) st.rm.rd[ks] += par * kSlabBytes;
#pragma unroll
  for (int mb = 0; mb < 4; ++mb) {
    st.tr.rd[mb][0] += par * kSlabBytes;
    st.tr.rd[mb][1] += par * kSlabBytes;
  }
  st.c = p.scale_log2e;
  st.m_run = kNoReference;
  st.l_run = 0.f;
#pragma unroll
  for (int mb = 0; mb < 4; ++mb)
#pragma unroll
    for (int r = 0; r < 16; ++r) st.acc_o[mb][r] = 0.f;

  char* const k_lds = smem;
  char* const v_lds = smem + 3 * kChunkBytes;
  // wave w brings in rows 16 w .. 16 w + 15 of every chunk, four copies each of K and V
  uint32_t dma_off[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = 16 * wave + 4 * i + (lane >> 4);
    dma_off[i] = (uint32_t)(row * kRowBytes + (((lane & 15) ^ swz(row)) << 4));
  }
  const uint32_t k_dst = lds_addr(k_lds) + 16 * wave * kRowBytes, v_dst = lds_addr(v_lds) + 16 * wave * kRowBytes;

  if (nsteps > 0) {
    // a chunk: number of its first key / 64, predicate bits of the half's four row groups in the low bits
    cursor.start(t_begin / per_block);
    int entry = 0;
    cursor.next(entry);
    int chunk = (((entry >> 8) * per_block + t_begin % per_block) << 4) | ((entry >> (4 * half)) & 15);
    int rem = per_block - t_begin % per_block;
    auto next_chunk = [&]() -> int {  // past the end: the last one again
      const int now = chunk;
      if (--rem > 0) {
        chunk += 16;
      } else if (cursor.next(entry)) {
        rem = per_block;
        chunk = ((entry >> 8) * per_block << 4) | ((entry >> (4 * half)) & 15);
      } else {
        rem = 1;
      }
      return now;
    };
    auto source = [](const char* base, int c) { return base + (int64_t)(c >> 4) * kChunkBytes; };
    auto copy_piece = [&](int i, uint32_t dst, const char* src) { dma16(dst + 4 * i * kRowBytes, src, dma_off[i]); };
    int c0 = next_chunk(), c1 = next_chunk(), c2 = next_chunk();
#pragma unroll
    for (int i = 0; i < 4; ++i) copy_piece(i, k_dst, source(kp, c0));
#pragma unroll
    for (int i = 0; i < 4; ++i) copy_piece(i, k_dst + kChunkBytes, source(kp, c1));
#pragma unroll
    for (int i = 0; i < 4; ++i) copy_piece(i, k_dst + 2 * kChunkBytes, source(kp, c2));
    int c3 = next_chunk();
    wait_vmem<4>();  // K_0 and K_1
    __syncthreads();
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) pin(st.qreg[ks]);
    f32x16 s_cur = qk_half(st, k_lds);
    pin(s_cur);
    __syncthreads();  // K_3 goes where K_0 was

    bf16x8 p_prev[2];
    const int wave_bits = 3 << (2 * rg), group_bit = 1 << (2 * rg + (l32 >> 4));
    bool w_prev = false;  // did this wave form P for the previous chunk?
    // step t, RK = t % 3, RV = t % 2
    auto step = [&](auto rk_c, auto rv_c, auto first_c) {
      constexpr int RK = decltype(rk_c)::value, RV = decltype(rv_c)::value;
      constexpr bool kFirst = decltype(first_c)::value;
      const bool w_cur = !kRows || (c0 & wave_bits) != 0, w_nxt = !kRows || (c1 & wave_bits) != 0;
      const char* const k_src = source(kp, c3);
      const char* const v_src = source(vp, c0);
      auto copies = [&](int i) {
        if (i < 4) copy_piece(i, v_dst + RV * kChunkBytes, v_src);
        else copy_piece(i - 4, k_dst + RK * kChunkBytes, k_src);
      };
      if (!kFirst && (!kRows || w_prev)) {
        pv_half(st, v_lds + (1 - RV) * kChunkBytes, p_prev, copies);
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) copies(i);
      }
      const bool active = !kRows || (c0 & group_bit) != 0;
      if (w_cur) softmax_reference(st, s_cur, active);
      f32x16 s_nxt;
      if (w_nxt) s_nxt = qk_half(st, k_lds + ((RK + 1) % 3) * kChunkBytes);  // past the last chunk: stale data, unused
      else s_nxt = s_cur;
      if (w_cur) softmax_exp<kRows>(st, s_cur, p_prev, active);
      w_prev = w_cur;
      pin(p_prev[0]);
      pin(p_prev[1]);
      s_cur = s_nxt;
      c0 = c1;
      c1 = c2;
      c2 = c3;
      c3 = next_chunk();
      // V_t and K_{t+2} must have landed; the four copies of K_{t+3} may still fly.  (A list load among them only makes the
      // wait stricter.)
      wait_vmem<4>();
      __syncthreads();
    };
    step(IC<0>{}, IC<0>{}, std::true_type{});
    for (int t = 1; t < nsteps; t += 6) {
      step(IC<1>{}, IC<1>{}, std::false_type{});
      if (t + 1 >= nsteps) break;
      step(IC<2>{}, IC<0>{}, std::false_type{});
      if (t + 2 >= nsteps) break;
      step(IC<0>{}, IC<1>{}, std::false_type{});
      if (t + 3 >= nsteps) break;
      step(IC<1>{}, IC<0>{}, std::false_type{});
      if (t + 4 >= nsteps) break;
      step(IC<2>{}, IC<1>{}, std::false_type{});
      if (t + 5 >= nsteps) break;
      step(IC<0>{}, IC<0>{}, std::false_type{});
    }
    if (!kRows || w_prev) pv_half(st, v_lds + ((nsteps - 1) & 1) * kChunkBytes, p_prev);
  }
  wait_vmem<0>();  // no copy is writing LDS any more
  __syncthreads();

  // The two waves of a row group: each hands the other half of its O^T (64 of the 128 columns) and its statistics
  const int keep = 2 * par;  // this wave ends up with accumulators keep, keep + 1
  {
    f32x4* dst = reinterpret_cast<f32x4*>(smem + wave * kSlabBytes) + lane;
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const f32x16& a = par ? st.acc_o[mb] : st.acc_o[mb + 2];
        dst[(mb * 4 + g) * 64] = (f32x4){a[4 * g + 0], a[4 * g + 1], a[4 * g + 2], a[4 * g + 3]};
      }
    float* stat = reinterpret_cast<float*>(smem + 4 * kSlabBytes) + wave * 128;
    stat[lane] = st.m_run;
    stat[64 + lane] = st.l_run;
  }
  __syncthreads();
  const int other = wave ^ 2;
  const float* stat = reinterpret_cast<const float*>(smem + 4 * kSlabBytes) + other * 128;
  const float m_other = stat[lane];
  const float m = fmaxf(st.m_run, m_other);
  const float w_own = fast_exp2((st.m_run - m) * st.c);
  const float w_other = fast_exp2((m_other - m) * st.c);
  const float l = sum_halves(w_own * st.l_run + w_other * stat[64 + lane]);
  f32x4 out[2][4];
  {
    const f32x4* src = reinterpret_cast<const f32x4*>(smem + other * kSlabBytes) + lane;
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const f32x16& a = par ? st.acc_o[mb + 2] : st.acc_o[mb];
        const f32x4 o = src[(mb * 4 + g) * 64];
#pragma unroll
        for (int e = 0; e < 4; ++e) out[mb][g][e] = w_own * a[4 * g + e] + w_other * o[e];
      }
  }
  // Results go through the LDS this wave has just read, 32 rows of 64 columns, so that a store fills whole lines: a lane holds pieces of one
  // row, 8 bytes to each of 32 rows per store.  (With this and the head of the list read ahead: H24 S30720, 64-token blocks, 192 of 480 kept
  // 4.85 -> 4.70 ms; B2 H8/2 S3136, 16 x 64 blocks, 12 of 49 kept 82.0 -> 79.5 us.)
  char* const own = smem + other * kSlabBytes;
  if (parts > 1) {  // as in fwd_kernel; rows of 256 bytes, 16-byte chunk c of row r at slot c ^ r % 16
    float* slot = p.split.ws + (int64_t)ws_slot * (kHalfSlotBytes / 4);
    float* prow = slot + rg * 32 * kHeadDim + 32 * keep;
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
      for (int g = 0; g < 4; ++g) *reinterpret_cast<f32x4*>(own + l32 * 256 + (((8 * mb + 2 * g + h) ^ (l32 & 15)) << 4)) = out[mb][g];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int row = 4 * i + (lane >> 4);
      *reinterpret_cast<f32x4*>(prow + row * kHeadDim + 4 * (lane & 15)) = *reinterpret_cast<const f32x4*>(own + row * 256 + (((lane ^ row) & 15) << 4));
    }
    if (h == 0 && par == 0) {
      slot[kHalfRows * kHeadDim + rg * 32 + l32] = m * st.c;
      slot[kHalfRows * kHeadDim + kHalfRows + rg * 32 + l32] = l;
    }
    return;
  }
  const float inv = l > 0.f ? 1.f / l : 0.f;
  if (h == 0 && par == 0) p.lse[qrow0 + l32] = l > 0.f ? (m * st.c + __builtin_log2f(l)) * 0.6931471805599453f : -INFINITY;
  __bf16* orow = p.o + qrow0 * kHeadDim + 32 * keep;
#pragma unroll
  for (int mb = 0; mb < 2; ++mb)
#pragma unroll
    for (int g = 0; g < 4; ++g)  // rows of 128 bytes, 16-byte chunk c of row r at slot c ^ r % 8
      *reinterpret_cast<bf16x4*>(own + l32 * 128 + (((4 * mb + g) ^ (l32 & 7)) << 4) + 8 * h) =
          pack4(out[mb][g][0] * inv, out[mb][g][1] * inv, out[mb][g][2] * inv, out[mb][g][3] * inv);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = 8 * i + (lane >> 3);
    *reinterpret_cast<bf16x8*>(orow + row * kHeadDim + 8 * (lane & 7)) = *reinterpret_cast<const bf16x8*>(own + row * 128 + (((lane ^ row) & 7) << 4));
  }
}

// Forward on tile lists whose 16-row groups select for themselves, or their 32-row groups in large launches (see takes_rows).
//
// Work-group = the 128 query rows of a tile list, eight waves of 16 rows, two work-groups per CU, so four waves per SIMD.  The work-group
// brings every chunk of 64 keys that some row selects into LDS, and the waves whose rows do work on it:
//   S^T[key, q] = K[key, :] . Q[q, :], O^T[d, q] += V^T[d, key] . P^T[key, q]      16x16x32 matrix instructions, lane = query row
// with the pipeline of fwd_kernel (P_{t-1} V_{t-1} | softmax of S_t | S_{t+1}).
// Row r of a 16-key tile of S^T is key pi(r), bits 2 and 3 of r swapped: the accumulator of lane group g then holds keys
// 0..3, 8..11, 4..7, 12..15 for g = 0..3, and the transposing fetch of V, which takes 4 rows for each of two groups at a time, meets 64
// different banks.
// Rings of three K chunks and two V chunks (80 KiB): step t requests V_t and K_{t+3}.
//
// Few rows of a chunk's 128 select it (with 16-row blocks, a quarter kept, 2.2 of 8 groups), so a launch of one round is bound by how
// long a wave takes from barrier to barrier, and one of many by LDS: a 16-row wave fetches a chunk's 32 KiB for itself, 256 of its
// cycles.  Copies alone would take a third of that (25 TB/s from L2).  Without gradients, fwd_half_kernel / this: B2 H8/2 S3136 q16 k64, 12 of 49
// kept 83.0 / 66.3 us (18 of them in front); B1 H22/11 S14080 q16 k64, 131 of 220 kept 2.25 / 1.58 ms.  With the three parts of a step
// one behind the other 79.6 us and 1.71 ms; with steps of 32 keys and rings of five 83.7 and 1.87.
constexpr int kRowsWaves = 8;
constexpr int kRowsOf = 16;  // rows of a wave
constexpr int kRowsTile = kRowsWaves * kRowsOf;
constexpr int kRowsSmem = 5 * kChunkBytes;

// The chunks of 64 keys of a tile list, in order: key chunk << 8 | predicate bits of its key block.  Every wave keeps 64 of them in a
// register, one per lane, and the 64 behind them; all lanes of a wave call everything together.
struct ChunkList {
  const int32_t* list;
  int row_len, per_block, lane;
  int base, now, ahead;

  FBA_DEVICE int load(int from) const {  // (needs no count: what lies past the end is not asked for)
    const int c = from + lane, e = c / per_block;
    const int entry = e < row_len ? list[e] : 0;
    return ((entry >> 8) * per_block + c - e * per_block) << 8 | (entry & 255);
  }
  FBA_DEVICE void start(int first) {
    base = first;
    now = load(first);
    ahead = load(first + 64);
  }
  FBA_DEVICE int at(int t) {  // t rises by at most one from call to call
    if (t == base + 64) {
      base = t;
      now = ahead;
      ahead = load(t + 64);
    }
    return __builtin_amdgcn_readlane(now, t - base);
  }
};

__global__ __attribute__((amdgpu_flat_work_group_size(64 * kRowsWaves, 64 * kRowsWaves), amdgpu_waves_per_eu(4, 4))) void fwd_rows_kernel(const FwdParams p) {
  extern __shared__ __attribute__((aligned(16))) char smem[];  // K ring [3][16 KiB] | V ring [2][16 KiB]
  const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int item, part = 0, parts = 1;
  int ws_slot = (int)blockIdx.x - p.split.main_wgs;  // of a part's results
  if (ws_slot < 0) {
    item = xcd_remap(blockIdx.x, p.items_per_xcd);
    if (item >= p.split.first) return;
  } else if (!split_position<Look::kSingle>(p.split, ws_slot, item, part, parts)) {
    return;
  }
  const int tiles_per_head = p.Sq / kRowsTile;
  const int bh = item / tiles_per_head;
  const int qt = item - bh * tiles_per_head;
  const int b = bh / p.Hq, hq = bh - b * p.Hq;
  const int hkv = hq / (p.Hq / p.Hkv);
  const int64_t qrow0 = (int64_t)bh * p.Sq + (int64_t)qt * kRowsTile + wave * kRowsOf;
  const char* const kp = reinterpret_cast<const char*>(p.k + ((int64_t)(b * p.Hkv + hkv) * p.Skv) * kHeadDim);
  const char* const vp = reinterpret_cast<const char*>(p.v + ((int64_t)(b * p.Hkv + hkv) * p.Skv) * kHeadDim);

  const int64_t mrow = (p.mask_bh == 1 ? 0 : (int64_t)bh) * tiles_per_head + qt;
  const int per_block = p.k_block / 64;
  ChunkList list{p.q_idx + mrow * p.nK, p.nK, per_block, lane};

  const int chunks = const_idx(p.q_cnt)[mrow] * per_block;
  bf16x8 qreg[4];  // Q as the B operand: lane holds row l16, d = 32 ks + 8 g .. +7
  {
    const __bf16* qp = p.q + (qrow0 + l16) * kHeadDim + 8 * g;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) qreg[ks] = *reinterpret_cast<const bf16x8*>(qp + 32 * ks);
  }
  const int t_begin = (int)((int64_t)chunks * part / parts), t_end = (int)((int64_t)chunks * (part + 1) / parts);
  const int nsteps = t_end - t_begin;

  const float c = p.scale_log2e;
  float m_run = kNoReference, l_run = 0.f;
  f32x4 acc[8];  // O^T: lane holds row l16, columns 16 db + 4 g .. +3
#pragma unroll
  for (int db = 0; db < 8; ++db) acc[db] = (f32x4){0.f, 0.f, 0.f, 0.f};

  // wave w brings in rows 8 w .. 8 w + 7 of every chunk, two copies each of K and V
  uint32_t dma_off[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int row = 8 * wave + 4 * i + (lane >> 4);
    dma_off[i] = (uint32_t)(row * kRowBytes + (((lane & 15) ^ swz(row)) << 4));
  }
  const uint32_t k_dst = lds_addr(smem) + 8 * wave * kRowBytes, v_dst = k_dst + 3 * kChunkBytes;
  // fetches: K row pi(l16) of a 16-key tile, chunk 4 ks + g; V rows pi(4 g) .. +3 and 16 on, columns 16 db .. +15
  // (the chunk number only flips bits of an address: one register each, with the rest formed where it is used)
  uint32_t k_base, v_base;
  {
    const int row = (l16 & 3) | (l16 & 4) << 1 | (l16 & 8) >> 1, vrow = (l16 >> 2) | (g & 1) << 3 | (g & 2) << 1;
    k_base = lds_addr(smem) + tile_off(row, g);
    v_base = lds_addr(smem) + 3 * kChunkBytes + tile_off(vrow, (lane & 3) >> 1) + 8 * (lane & 1);
  }
  auto k_ptr = [&](int ks) { return (LdsPtr)(uintptr_t)(k_base ^ (uint32_t)(ks << 6)); };
  auto v_ptr = [&](int db) { return (LdsPtr)(uintptr_t)(v_base ^ (uint32_t)(db << 5)); };

  if (nsteps > 0) {
    list.start(t_begin);
    int t_ahead = t_begin;
    auto next_chunk = [&]() -> int { return list.at(min(t_ahead++, t_end - 1)); };  // past the end: the last one again
    auto piece = [&](int i, uint32_t dst, const char* base, int of) { dma16(dst + 4 * i * kRowBytes, base + (int64_t)(of >> 8) * kChunkBytes, dma_off[i]); };
    // S^T of chunk `of`, where the wave's rows select it
    auto scores = [&](f32x4 (&s)[4], int ko) {
#pragma unroll
      for (int t = 0; t < 4; ++t) s[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) s[t] = mfma16(lds_read_b128(k_ptr(ks) + ko + t * 16 * kRowBytes), qreg[ks], s[t]);
    };
    bf16x8 pk[2];
    auto add_pv = [&](int vo, auto between) {
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int db = 0; db < 8; ++db) {
          const int off = vo + 32 * u * kRowBytes;
          acc[db] = mfma16(cat(lds_read_tr(v_ptr(db) + off), lds_read_tr(v_ptr(db) + off + 16 * kRowBytes)), pk[u], acc[db]);
          between(8 * u + db);
        }
    };
    int c0 = next_chunk(), c1 = next_chunk(), c2 = next_chunk();
#pragma unroll
    for (int i = 0; i < 2; ++i) piece(i, k_dst, kp, c0);
#pragma unroll
    for (int i = 0; i < 2; ++i) piece(i, k_dst + kChunkBytes, kp, c1);
#pragma unroll
    for (int i = 0; i < 2; ++i) piece(i, k_dst + 2 * kChunkBytes, kp, c2);
    int c3 = next_chunk();
    wait_vmem<2>();  // K_0 and K_1
    __syncthreads();
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) pin(qreg[ks]);
    f32x4 s_cur[4];
    scores(s_cur, 0);
#pragma unroll
    for (int t = 0; t < 4; ++t) pin(s_cur[t]);
    __syncthreads();  // K_3 goes where K_0 was

    bool w_prev = false;  // did this wave form P for the previous chunk?
    // step t, RK = t % 3, RV = t % 2
    auto step = [&](auto rk_c, auto rv_c) {
      constexpr int RK = decltype(rk_c)::value, RV = decltype(rv_c)::value;
      const bool w_cur = (c0 >> wave & 1) != 0, w_nxt = (c1 >> wave & 1) != 0;
      auto copies = [&](int i) {
        if (i < 2) piece(i, v_dst + RV * kChunkBytes, vp, c0);
        else piece(i - 2, k_dst + RK * kChunkBytes, kp, c3);
      };
      if (w_prev) {
        add_pv((1 - RV) * kChunkBytes, [&](int i) { if (i % 3 == 1 && i < 12) copies(i / 3); });
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) copies(i);
      }
      if (w_cur) {
        float mx = s_cur[0][0];
#pragma unroll
        for (int i = 1; i < 16; ++i) mx = fmaxf(mx, s_cur[i >> 2][i & 3]);
        // every lane tests the 16 keys it holds; the row's maximum is formed only when the reference rises (see softmax_reference)
        if (__builtin_amdgcn_ballot_w64((mx - m_run) * c > kLazy) != 0) {
          mx = fmaxf(mx, __shfl_xor(mx, 16));
          const float m_new = fmaxf(m_run, max_halves(mx));
          const float alpha = fast_exp2((m_run - m_new) * c);
          m_run = m_new;
          l_run *= alpha;
#pragma unroll
          for (int db = 0; db < 8; ++db) acc[db] *= alpha;
        }
      }
      f32x4 s_nxt[4];
      if (w_nxt) {
        scores(s_nxt, (RK + 1) % 3 * kChunkBytes);  // past the last chunk: stale data, unused
      } else {
#pragma unroll
        for (int t = 0; t < 4; ++t) s_nxt[t] = s_cur[t];
      }
      if (w_cur) {
        const float mc = m_run * c;
#pragma unroll
        for (int i = 0; i < 16; ++i) s_cur[i >> 2][i & 3] = fast_exp2(__builtin_fmaf(s_cur[i >> 2][i & 3], c, -mc));
        const bf16x2 one2 = {(__bf16)1.f, (__bf16)1.f};
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const f32x4 lo = s_cur[2 * u], hi = s_cur[2 * u + 1];
          pk[u] = pack8(lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]);
#pragma unroll
          for (int t = 0; t < 4; ++t) l_run = __builtin_amdgcn_fdot2_f32_bf16((bf16x2){pk[u][2 * t], pk[u][2 * t + 1]}, one2, l_run, false);
        }
      }
      w_prev = w_cur;
      pin(pk[0]);
      pin(pk[1]);
#pragma unroll
      for (int t = 0; t < 4; ++t) s_cur[t] = s_nxt[t];
      c0 = c1;
      c1 = c2;
      c2 = c3;
      c3 = next_chunk();
      // V_t and K_{t+2} must have landed; the two copies of K_{t+3} may still fly.  (A list load among them only makes the wait stricter.)
      wait_vmem<2>();
      __syncthreads();
    };
    for (int t = 0; t < nsteps; t += 6) {
      step(IC<0>{}, IC<0>{});
      if (t + 1 >= nsteps) break;
      step(IC<1>{}, IC<1>{});
      if (t + 2 >= nsteps) break;
      step(IC<2>{}, IC<0>{});
      if (t + 3 >= nsteps) break;
      step(IC<0>{}, IC<1>{});
      if (t + 4 >= nsteps) break;
      step(IC<1>{}, IC<0>{});
      if (t + 5 >= nsteps) break;
      step(IC<2>{}, IC<1>{});
    }
    if (w_prev) add_pv(((nsteps - 1) & 1) * kChunkBytes, [](int) {});
  }
  wait_vmem<0>();  // no copy is writing LDS any more
  __syncthreads();

  l_run += __shfl_xor(l_run, 16);
  const float l = sum_halves(l_run);
  if (parts > 1) {  // as in fwd_kernel
    float* slot = p.split.ws + (int64_t)ws_slot * (kFwdSlotBytes / 4);
    float* prow = slot + (wave * kRowsOf + l16) * kHeadDim + 4 * g;
#pragma unroll
    for (int db = 0; db < 8; ++db) *reinterpret_cast<f32x4*>(prow + 16 * db) = acc[db];
    if (g == 0) {
      slot[kRowsTile * kHeadDim + wave * kRowsOf + l16] = m_run * c;
      slot[kRowsTile * kHeadDim + kRowsTile + wave * kRowsOf + l16] = l;
    }
    return;
  }
  const float inv = l > 0.f ? 1.f / l : 0.f;
  if (g == 0) p.lse[qrow0 + l16] = l > 0.f ? (m_run * c + __builtin_log2f(l)) * 0.6931471805599453f : -INFINITY;
  char* const own = smem + wave * kRowsOf * kRowBytes;  // so that a store fills four whole rows
#pragma unroll
  for (int db = 0; db < 8; ++db)
    *reinterpret_cast<bf16x4*>(own + tile_off(l16, 2 * db + (g >> 1)) + 8 * (g & 1)) = pack4(acc[db][0] * inv, acc[db][1] * inv, acc[db][2] * inv, acc[db][3] * inv);
#pragma unroll
  for (int i = 0; i < 4; ++i)
    *reinterpret_cast<bf16x8*>(p.o + (qrow0 + 4 * i) * kHeadDim + lane * 8) = lds_read_b128(own, tile_off(4 * i + (lane >> 4), lane & 15));
}

// Forward straight from the block mask, for problems too small to fill the GPU: no lists, no parts, one launch.
//
// Work-group = 32 query rows, eight waves, one work-group per CU.  Every wave reads the mask row of these rows itself (64 key
// blocks to a ballot) and takes every eighth of the selected 32-key slabs; it brings in its K and V slab on its own (16 KiB of LDS
// per wave, no barrier in the loop), with softmax statistics and O of its own, and the eight meet in LDS at the end.  Rows
// past the end of a sequence that is no whole number of 32 are loaded as copies of the last row and not stored.
//
// Such a call is bound by latency: a chain of launches (lists, attention, merge of the parts) that each wait for the one in
// front, and inside a kernel of loads that wait for loads.  Calls without gradients, lists and parts / from the mask: H1 S768,
// 128-token blocks, 40 % kept 15.6 / 7.0 us, H2 S1536 384-token blocks 18.6 / 9.6, H1 S6144 30.3 / 17.5, H3 S2048 against 3840 keys
// 24.3 / 16.8 us.  In longer lists a step of all eight waves takes 1.3 us, what the copies of 128 KiB take (a slab feeds 16 matrix
// instructions here and 64 with 128 rows), so the line is drawn where that begins to count (fwd_takes_mask).  K rows straight to
// registers, two slabs ahead, take 3 us a step: every load touches 32 rows.
constexpr int kMaskWaves = 8;
constexpr int kMaskRows = 32;
constexpr int kMaskStatBase = kMaskWaves * 2 * kSlabBytes;                  // softmax references, then denominators [wave][row]
constexpr int kMaskSmem = kMaskStatBase + 2 * kMaskWaves * kMaskRows * 4;

template <bool kTwo>  // q_block is an odd multiple of 16: the two 16-row halves have mask rows of their own
__global__ __attribute__((amdgpu_flat_work_group_size(64 * kMaskWaves, 64 * kMaskWaves), amdgpu_waves_per_eu(2, 2))) void fwd_mask_kernel(const FwdMaskParams p) {
  extern __shared__ __attribute__((aligned(16))) char smem[];  // [wave](K slab | V slab), statistics
  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int item = xcd_remap(blockIdx.x, p.items_per_xcd);
  if (item >= p.num_items) return;
  const int tiles_per_head = (p.Sq + kMaskRows - 1) / kMaskRows;
  const int bh = item / tiles_per_head;
  const int row0 = (item - bh * tiles_per_head) * kMaskRows;
  const int b = bh / p.Hq, hq = bh - b * p.Hq;
  const int64_t kv_row0 = (int64_t)(b * p.Hkv + hq / (p.Hq / p.Hkv)) * p.Skv;
  const char* kp = reinterpret_cast<const char*>(p.k + kv_row0 * kHeadDim);
  const char* vp = reinterpret_cast<const char*>(p.v + kv_row0 * kHeadDim);

  MaskCursor<kTwo> cursor;
  const uint8_t* mask = p.mask + (p.mask_bh == 1 ? 0 : (int64_t)bh * p.nQ * p.nK);
  cursor.row0 = mask + (int64_t)(row0 / p.q_block) * p.nK;
  cursor.row1 = kTwo ? mask + (int64_t)(min(row0 + 16, p.Sq - 1) / p.q_block) * p.nK : cursor.row0;
  cursor.nK = p.nK;
  cursor.nsub = p.k_block / kSlab;
  cursor.lane = lane;
  cursor.start();

  if (p.mask_copy != nullptr && (p.mask_bh > 1 || bh == 0)) {  // the rows of the query blocks that begin here
    const int64_t at = (p.mask_bh == 1 ? 0 : (int64_t)bh * p.nQ * p.nK);
    for (int i = (row0 + p.q_block - 1) / p.q_block; i * p.q_block < min(row0 + kMaskRows, p.Sq); ++i)
      for (int j = tid; j < p.nK; j += 64 * kMaskWaves) p.mask_copy[at + (int64_t)i * p.nK + j] = mask[(int64_t)i * p.nK + j];
  }

  FwdState st;
  {
    const __bf16* qp = p.q + ((int64_t)bh * p.Sq + min(row0 + l32, p.Sq - 1)) * kHeadDim;
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) st.qreg[ks] = *reinterpret_cast<const bf16x8*>(qp + 16 * ks + 8 * h);
  }
  st.rm.init(lane);
  st.tr.init(lane);
  st.c = p.scale_log2e;
  st.m_run = kNoReference;
  st.l_run = 0.f;
#pragma unroll
  for (int mb = 0; mb < 4; ++mb)
#pragma unroll
    for (int r = 0; r < 16; ++r) st.acc_o[mb][r] = 0.f;

  // copy i (0..7) of a slab fills its rows 4 i .. 4 i + 3; the swizzle repeats after 16 rows
  uint32_t dma_off[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = 4 * i + (lane >> 4);
    dma_off[i] = (uint32_t)(row * kRowBytes + (((lane & 15) ^ swz(row)) << 4));
  }
  const char* const k_lds = smem + wave * 2 * kSlabBytes;
  const char* const v_lds = k_lds + kSlabBytes;
  const uint32_t k_dst = lds_addr(k_lds), v_dst = lds_addr(v_lds);
  auto copy_slab = [&](uint32_t dst, const char* src) {
#pragma unroll
    for (int i = 0; i < 8; ++i) dma16(dst + 4 * i * kRowBytes, src + (i >> 2) * 16 * kRowBytes, dma_off[i & 3]);
  };
  // The compiler knows of no order between the copies and its LDS reads: no read moves up across a fence, and reads of a buffer
  // have returned before it is filled again.
  auto fence = [] { asm volatile("" ::: "memory"); };
  auto reads_done = [] { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); };

  bool more = cursor.skip(wave);
  if (more) {
    const int64_t off = (int64_t)cursor.slab() * kSlabBytes;
    copy_slab(k_dst, kp + off);
    copy_slab(v_dst, vp + off);
  }
  while (more) {
    const int halves = cursor.halves();
    more = cursor.skip(kMaskWaves);
    const int64_t off = more ? (int64_t)cursor.slab() * kSlabBytes : 0;
    const bool active = !kTwo || ((halves >> (l32 >> 4)) & 1) != 0;
    wait_vmem<8>();  // K has landed; the eight copies of V, requested last, may still fly
    fence();
    f32x16 s = qk_half(st, k_lds);
    pin(s);
    reads_done();
    if (more) copy_slab(k_dst, kp + off);
    bf16x8 pk[2];
    softmax_reference(st, s, active);
    softmax_exp<kTwo>(st, s, pk, active);
    if (more) wait_vmem<8>(); else wait_vmem<0>();
    fence();
    pv_half(st, v_lds, pk);
#pragma unroll
    for (int mb = 0; mb < 4; ++mb) pin(st.acc_o[mb]);
    reads_done();
    if (more) copy_slab(v_dst, vp + off);
  }

  // Every wave hands in its O^T (16 KiB in place of its slabs, chunk c of row r at slot c ^ r, so that neither side meets bank
  // conflicts) and its statistics; thread t forms columns 8 (t % 16) .. +7 of row t / 16.
  {
    f32x4* dst = reinterpret_cast<f32x4*>(smem + wave * 2 * kSlabBytes) + l32 * 32;
#pragma unroll
    for (int mb = 0; mb < 4; ++mb)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        dst[(8 * mb + 2 * g + h) ^ l32] = (f32x4){st.acc_o[mb][4 * g + 0], st.acc_o[mb][4 * g + 1], st.acc_o[mb][4 * g + 2], st.acc_o[mb][4 * g + 3]};
    float* stat = reinterpret_cast<float*>(smem + kMaskStatBase);
    const float l = sum_halves(st.l_run);
    if (h == 0) {
      stat[wave * kMaskRows + l32] = st.m_run;
      stat[(kMaskWaves + wave) * kMaskRows + l32] = l;
    }
  }
  __syncthreads();
  const int r = tid >> 4, c8 = 2 * (tid & 15);
  const float* stat = reinterpret_cast<const float*>(smem + kMaskStatBase) + r;
  float m = stat[0];
#pragma unroll
  for (int w = 1; w < kMaskWaves; ++w) m = fmaxf(m, stat[w * kMaskRows]);
  float l = 0.f;
  f32x4 out[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
  for (int w = 0; w < kMaskWaves; ++w) {
    const float weight = fast_exp2((stat[w * kMaskRows] - m) * st.c);
    l += weight * stat[(kMaskWaves + w) * kMaskRows];
    const f32x4* src = reinterpret_cast<const f32x4*>(smem + w * 2 * kSlabBytes) + r * 32;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const f32x4 o = src[(c8 + j) ^ r];
#pragma unroll
      for (int e = 0; e < 4; ++e) out[j][e] += weight * o[e];
    }
  }
  if (row0 + r >= p.Sq) return;
  const float inv = l > 0.f ? 1.f / l : 0.f;
  *reinterpret_cast<bf16x8*>(p.o + ((int64_t)bh * p.o_rows + row0 + r) * kHeadDim + 4 * c8) =
      pack8(out[0][0] * inv, out[0][1] * inv, out[0][2] * inv, out[0][3] * inv, out[1][0] * inv, out[1][1] * inv, out[1][2] * inv, out[1][3] * inv);
  if (c8 == 0) p.lse[(int64_t)bh * p.Sq + row0 + r] = l > 0.f ? (m * st.c + __builtin_log2f(l)) * 0.6931471805599453f : -INFINITY;
}

// Combines the parts of the split items: O = sum_p 2^(m_p - m) O_p / sum_p 2^(m_p - m) l_p with m = max_p m_p, in part
// order.  One thread per (query row, four head-dim columns).  Bound by latency: whatever the parts hold is requested at once (part after
// part, each waiting for the one in front: H7 384 rows against 46720 keys, eight parts, 7.1 us, so 4.6).
template <int kTileRows>
__global__ __attribute__((amdgpu_flat_work_group_size(256, 256))) void fwd_merge_kernel(const FwdParams p) {
  const int tid = threadIdx.x;
  constexpr int kSlotFloats = kTileRows * kHeadDim + 2 * kTileRows;
  const int parts = parts_made(p.split);
  if (parts == 1) return;  // done whole
  for (int block = blockIdx.x; block < p.split.items * (kTileRows / 8); block += gridDim.x) {
    const int row = block * 8 + (tid >> 5), c4 = (tid & 31) * 4;  // row among the kTileRows * (split items) rows
    const int it = row / kTileRows, r = row % kTileRows;
    const int item = p.split.first + it;
    const float* slot = p.split.ws + (int64_t)it * parts * kSlotFloats;
    float mq[kMostParts], lq[kMostParts];
    f32x4 oq[kMostParts];
#pragma unroll
    for (int q = 0; q < kMostParts; ++q)
      if (q < parts) {
        mq[q] = slot[kTileRows * kHeadDim + r];
        lq[q] = slot[kTileRows * kHeadDim + kTileRows + r];
        oq[q] = *reinterpret_cast<const f32x4*>(slot + r * kHeadDim + c4);
        slot += kSlotFloats;
      }
    float m = -INFINITY;
#pragma unroll
    for (int q = 0; q < kMostParts; ++q)
      if (q < parts) m = fmaxf(m, mq[q]);
    float l = 0.f;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int q = 0; q < kMostParts; ++q)
      if (q < parts) {
        const float w = mq[q] == -INFINITY ? 0.f : fast_exp2(mq[q] - m);
        l += w * lq[q];
        acc += w * oq[q];
      }
    const float inv = l > 0.f ? 1.f / l : 0.f;
    const int64_t orow = (int64_t)item * kTileRows + r;  // items are consecutive tiles of [B, Hq, Sq]
    *reinterpret_cast<bf16x4*>(p.o + orow * kHeadDim + c4) = pack4(acc[0] * inv, acc[1] * inv, acc[2] * inv, acc[3] * inv);
    if (c4 == 0) p.lse[orow] = l > 0.f ? (m + __builtin_log2f(l)) * 0.6931471805599453f : -INFINITY;
  }
}

namespace {

// Does a forward pass on tile lists go to fwd_rows_kernel?  Its 128-row work-groups leave out every 16 rows that do not select a chunk, and
// bring in chunks that any of the 128 rows selects; fwd_half_kernel works on 32 rows and 64.  No gradients, fwd_half_kernel / fwd_rows_kernel, 64-token key
// blocks, 12, 25 and 50 % kept (chunks of a compute unit alone in a launch of few work-groups come slowly, so those stay):
//   16-row blocks: 256 tiles (H8 S4096) 35.4 / 43.5, 55.2 / 60.9, 78.1 / 78.1 us; 320 (H10 S4096) 50.4 / 50.5, 74.7 / 71.4, 102.2 / 93.3; 512 (H16
//     S4096) 62.6 / 51.0, 101 / 72.5, 147 / 101; 704 (H22 S4096) 86.4 / 84.4, 141 / 119, 208 / 161; at 90 % 704 240 / 214.  Launches of 64-row work-groups that
//     are little more than a round cut long lists into parts, so the line rises with the keys.  15 (320 tiles: 12), 60 and 90 % kept: 320 tiles, 2048 keys 35.4 / 33.0,
//     67.7 / 57.1, 72.0 / 67.6, 4096 keys 50.6 / 51.4, 104.9 / 100.8, 112.2 / 122.8, 8192 keys 77.8 / 84.6, 193 / 190, 207 / 233; 336 tiles, 4096 keys 62.0 / 57.7,
//     123 / 102, 132 / 124, 5120 keys 76.6 / 67.9, 137 / 125, 146 / 151; 344 tiles, 8192 keys 105 / 100, 221 / 191, 236 / 234, 30720 keys 378 / 380, 799 / 693, 877 / 852.
//   32-row blocks: 320 tiles 39.3 / 39.5, 54.2 / 59.8, 78.8 / 88.8 us; 704 57.4 / 62.3, 92.0 / 97.4, 154 / 153; 1080 (H9 S15360) 245 / 237, 437 / 409, 772 / 682;
//     2880 (H24 S15360) 652 / 634, 1147 / 1112, 2027 / 1894.  Two and a half rounds of long lists with little kept are the worst case: H10 S16384, 6, 12 and 18 %
//     159 / 167, 283 / 289, 391 / 391.
//   64-row blocks: H24 S30720, 40 % kept 4.54 / 5.10 ms.
bool takes_rows(const FwdParams& p) {
  const int64_t tiles = (int64_t)p.B * p.Hq * (p.Sq / kRowsTile), units = device_compute_units();
  if (p.q_block % 32 == 0) return p.q_block % 64 != 0 && tiles >= 4 * units;
  const int thousands = std::min(std::max((p.Skv + 1023) / 1024, 2), 5);  // of keys
  return 32 * tiles >= (38 + thousands) * units;  // 320, 328, 336 and 344 tiles where there are 256 compute units
}

// Does a block mask go to fwd_half_kernel, whole?  Where 128-row work-groups would leave half of the compute units without one, and parts, which fill them, pay
// for their results and the merge: 64 rows at 64 keys a step take as long for a step as 128 rows at 32 keys, a work-group alone on its compute unit.  Long lists are
// better off in more than two parts.  No gradients, 128-token blocks, 128 rows and parts / 64 rows, at 12, 35, 60 and 90 % kept: H6 S1408 (66 tiles) 9.4 / 6.6, 15.1 / 10.2,
// 22.3 / 13.4 and 23.8 / 16.3 us; H3 S3456 (81) 13.1 / 8.9, 23.8 / 15.5, 27.9 / 22.5, 33.2 / 30.6; H3 S4736 (111) 15.9 / 10.8, 27.8 / 20.9, 35.3 / 29.6, 45.1 / 40.8; H6 S2688
// (126) 13.8 / 12.4, 21.2 / 15.0, 28.8 / 20.8, 34.0 / 27.2.  Longer: H1 S8448 (66) 21.8 / 14.6, 30.6 / 30.0, 41.1 / 47.2, 49.1 / 66.7.  More tiles: H3 S5504 (129) 18.0 / 15.8,
// 36.0 / 31.5, 45.9 / 47.2, 58.6 / 67.6, H6 S3072 (144) 11.6 / 15.2, 20.7 / 21.7, 32.0 / 30.5, 45.8 / 42.8.  Steps: H6 S1408 58.7 / 52.6, H5 S3200 96.3 / 87.5.
bool takes_halves(const FwdParams& p) { return p.mask != nullptr && fwd_takes_halves((int64_t)p.B * p.Hq * p.Sq, p.Skv); }

}  // namespace

bool fwd_takes_halves(int64_t rows, int64_t kv_len) {
  const int64_t tiles = rows / 128, units = device_compute_units();
  return 2 * tiles <= units && kv_len / kSlab <= (8 * tiles >= 3 * units ? 148 : 112);
}

// Tail splitting (two work-groups per compute unit); the 384-row kernel does without.
void plan_fwd(FwdParams& p) {
  if (p.tiled && takes_rows(p)) {  // (steps of 64 keys against 128 rows; lines of 30 to 48 units cut the same launches)
    p.num_items = p.B * p.Hq * (p.Sq / kRowsTile);
    const ListLengths lengths{p.q_cnt, p.mask_bh == 1, kRowsTile, 128, p.Sq / 128, 1, p.k_block / 64};
    p.split = plan_split(p.num_items, 2, p.Skv / 64, StepCost{22, 30, 40}, kFwdSlotBytes, p.split.ws, p.split_ws_bytes, lengths);
    group_parts(p.split, p.Hq / p.Hkv * (p.Sq / kRowsTile), 2LL * p.Skv * kRowBytes);
    return;
  }
  if (p.tiled) {  // a step is as long as one of fwd_kernel, a part's results are half as large
    p.num_items = p.B * p.Hq * (p.Sq / kHalfRows);
    const ListLengths lengths{p.q_cnt, p.mask_bh == 1, kHalfRows, 128, p.Sq / 128, 1, p.k_block / 64};  // of the 128-row tile's list
    p.split = plan_split(p.num_items, 2, p.Skv / 64, StepCost{32, 45, 60, /*scans=*/true}, kHalfSlotBytes, p.split.ws, p.split_ws_bytes, lengths);
    group_parts(p.split, p.Hq / p.Hkv * (p.Sq / kHalfRows), 2LL * p.Skv * kRowBytes);
    return;
  }
  const bool wide = p.q_block % 384 == 0 && p.variant != 1 && p.mask == nullptr, halves = takes_halves(p);
  const int rows = wide ? 384 : halves ? kHalfRows : 128;
  p.num_items = p.B * p.Hq * (p.Sq / rows);
  const ListLengths lengths{p.q_cnt, p.mask_bh == 1, rows, p.q_block, p.nQ, 1, p.k_block / kSlab, p.mask, p.nK};
  p.split = plan_split(p.num_items, 2, p.Skv / 32, StepCost{16, 22.5, 30}, kFwdSlotBytes, wide || halves ? nullptr : p.split.ws, p.split_ws_bytes, lengths);
  group_parts(p.split, p.Hq / p.Hkv * (p.Sq / rows), 2LL * p.Skv * kRowBytes);
}

namespace {

hipError_t launch_fwd_tiled(FwdParams p, hipStream_t stream) {
  const bool rows = takes_rows(p);
  void (*fn)(const FwdParams) = rows ? &fwd_rows_kernel : p.q_block % 64 != 0 ? &fwd_half_kernel<true, From::kTiles> : &fwd_half_kernel<false, From::kTiles>;
  const int smem = rows ? kRowsSmem : kHalfSmem, threads = rows ? 64 * kRowsWaves : 256;
  plan_fwd(p);
  plan_xcd_mapping(p.B * p.Hq, p.split.first, p.items_per_xcd, p.split.main_wgs);
  const int split_items = p.num_items - p.split.first;
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, smem);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(fn, dim3(p.split.main_wgs + split_items * p.split.parts), dim3(threads), smem, stream, p);
  if (split_items > 0) {
    if (rows) hipLaunchKernelGGL(fwd_merge_kernel<kRowsTile>, dim3(merge_grid(split_items * kRowsTile / 8)), dim3(256), 0, stream, p);
    else hipLaunchKernelGGL(fwd_merge_kernel<kHalfRows>, dim3(merge_grid(split_items * kHalfRows / 8)), dim3(256), 0, stream, p);
  }
  return hipGetLastError();
}

}  // namespace

// Is a problem small enough for fwd_mask_kernel?  Calls without gradients, lists / mask, at 10, 40 and 90 % kept (cross lengths: 10, 50
// and 90 %), 128-token blocks unless noted.  One round of work-groups: n = 192 of 32 rows against 192 slabs (H1 S6144) 24.1 / 9.1,
// 30.3 / 17.5, 41.0 / 30.7 us, n = 12 against 120 slabs (H3, 128 rows, 3840 keys) 16.3 / 7.4, 19.3 / 13.6, 21.6 / 19.7; n = 12 against 480
// 18.3 / 12.6, 29.6 / 42.7, 40.6 / 72.1: the fewer rows, the more parts the kernels on lists make of them.  Two rounds: n = 288 against 72
// (H4 S2304, all blocks) 30.9 / 33.1, n = 576 against 24 (H24 S768) 11.5 / 15.1, 13.4 / 18.1, 18.9 / 23.7.
bool fwd_takes_mask(int64_t rows, int64_t kv_len) {
  const int64_t n = rows / kMaskRows, slabs = kv_len / kSlab;  // of whole work-groups; at most that many slabs to a row
  return n <= device_compute_units() && 5 * slabs <= 600 + 2 * n;
}

hipError_t launch_fwd_mask(FwdMaskParams p, hipStream_t stream) {
  void (*fn)(const FwdMaskParams) = p.q_block % 32 != 0 ? &fwd_mask_kernel<true> : &fwd_mask_kernel<false>;
  p.num_items = p.B * p.Hq * ((p.Sq + kMaskRows - 1) / kMaskRows);
  int grid;
  plan_xcd_mapping(p.B * p.Hq, p.num_items, p.items_per_xcd, grid);
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, kMaskSmem);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(fn, dim3(grid), dim3(64 * kMaskWaves), kMaskSmem, stream, p);
  return hipGetLastError();
}

hipError_t launch_fwd(FwdParams p, hipStream_t stream) {
  if (p.tiled) return launch_fwd_tiled(p, stream);
  const bool wide = p.q_block % 384 == 0 && p.variant != 1 && p.mask == nullptr, halves = takes_halves(p);
  const int smem = halves ? kHalfSmem : (wide ? 12 : 2 * kRing) * kSlabBytes;  // the rings; the results of twelve waves
  void (*fn)(const FwdParams) = halves ? &fwd_half_kernel<false, From::kMask>
                                : wide ? &fwd_kernel<12, false> : p.mask != nullptr ? &fwd_kernel<4, true> : &fwd_kernel<4, false>;
  const int threads = wide ? 768 : 256;
  plan_fwd(p);
  plan_xcd_mapping(p.B * p.Hq, p.split.first, p.items_per_xcd, p.split.main_wgs);
  const int split_wgs = (p.num_items - p.split.first) * p.split.parts;
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, smem);
  if (e != hipSuccess) return e;
  p.make.wgs = p.make.q_cnt != nullptr ? (int)((p.mask_bh * (p.nQ + p.nK) + 3) / 4) : 0;
  hipLaunchKernelGGL(fn, dim3(p.split.main_wgs + split_wgs + p.make.wgs), dim3(threads), smem, stream, p);
  if (split_wgs > 0) hipLaunchKernelGGL(fwd_merge_kernel<128>, dim3(merge_grid((p.num_items - p.split.first) * 16)), dim3(256), 0, stream, p);
  return hipGetLastError();
}

}  // namespace fba
