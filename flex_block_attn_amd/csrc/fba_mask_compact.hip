// Mask compaction: bool block mask [mask_bh, nQ, nK] -> ascending active-index lists in both orientations.
//
// The reference never materialises such lists: every CTA rescans its mask row in the tile loop
// (flex_block_attn_h100.cu:134-135, :247-248) and the backward pass needs a transposed copy of the mask
// (flex_block_attn_interface.py:85-86; scan at flex_block_attn_h100.cu:672, :738).  Here one launch emits
//   q_cnt[m, i], q_idx[m, i, 0..q_cnt) = { j : mask[m, i, j] }   ascending, padded with -1 to nK entries
//   k_cnt[m, j], k_idx[m, j, 0..k_cnt) = { i : mask[m, i, j] }   ascending, padded with -1 to nQ entries
// One wave per output row (compact_row in fba_common.h).
#include "fba_common.h"
#include "fba_kernels.h"

namespace fba {

__global__ __attribute__((amdgpu_flat_work_group_size(256, 256))) void mask_compact_kernel(
    const uint8_t* __restrict__ mask, int64_t mask_bh, int nQ, int nK, int32_t* __restrict__ q_cnt,
    int32_t* __restrict__ q_idx, int32_t* __restrict__ k_cnt, int32_t* __restrict__ k_idx) {
  compact_row(mask, mask_bh, nQ, nK, q_cnt, q_idx, k_cnt, k_idx, (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6));
}

hipError_t launch_mask_compact(const uint8_t* mask, int64_t mask_bh, int nQ, int nK, int32_t* q_cnt, int32_t* q_idx,
                               int32_t* k_cnt, int32_t* k_idx, hipStream_t stream) {
  const int64_t waves = mask_bh * ((int64_t)nQ + (k_cnt != nullptr ? nK : 0));
  const int64_t blocks = (waves + 3) / 4;
  if (blocks <= 0) return hipSuccess;
  if (blocks > 0x7fffffffLL) return hipErrorInvalidValue;
  hipLaunchKernelGGL(mask_compact_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, mask, mask_bh, nQ, nK, q_cnt,
                     q_idx, k_cnt, k_idx);
  return hipGetLastError();
}

// Tile lists for block sizes that do not align with the kernels' 128-row tiles (q_block or k_block not a multiple of
// 128).  The attention kernels then work on 128-row tiles that straddle mask blocks, so every list entry carries a
// predicate per 16-row group (query side) or per (wave, 16-row half-slab) pair (key side):
//   qt_ent[m, T, 0..qt_cnt) = (J << 8) | bits, ascending J: key block J is selected by at least one of the eight 16-row
//       groups of query tile T; bit g is mask[m, (128 T + 16 g) / q_block, J].                       (forward, dQ)
//   kt_ent[m, U, 0..kt_cnt) = (s << 8) | bits, ascending s: 32-row query slab s touches key tile U; bit 2w + f is
//       mask[m, (32 s + 16 f) / q_block, (128 U + 32 w) / k_block], w = wave (32 keys), f = half of the slab.  (dK/dV)
// One wave per output row, same ballot / prefix-popcount compaction as above; unused entries are -1.  The mask itself may have fewer rows
// and columns (mask_q, mask_k): lengths that are no whole tiles, where blocks that nothing selects fill the last tile up.
//
// What bounds it are the key side's loads: bytes of a column, each in a line of its own.  A tile meets two columns at most (k_block is a multiple
// of 64), a slab one mask row unless its halves have different ones, so one or two rows of two bytes are read and not all eight of the bits' places, and the
// loads of four steps go out side by side: 24 masks of 480 x 480, 64-token blocks 71 -> 38 us.
constexpr int kSideBySide = 4;
__global__ __attribute__((amdgpu_flat_work_group_size(256, 256))) void tile_lists_kernel(
    const uint8_t* __restrict__ mask, int64_t mask_bh, int mask_q, int mask_k, int nK, int q_block, int k_block, int n_qt, int n_kt,
    int n_qs, int32_t* __restrict__ qt_cnt, int32_t* __restrict__ qt_ent, int32_t* __restrict__ kt_cnt,
    int32_t* __restrict__ kt_ent) {
  const int lane = threadIdx.x & 63;
  const int64_t w = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int64_t n_qrows = mask_bh * n_qt, n_krows = mask_bh * n_kt;
  if (w >= n_qrows + n_krows) return;
  const bool q_pass = w < n_qrows;
  const int64_t r = q_pass ? w : w - n_qrows;
  const int per = q_pass ? n_qt : n_kt;
  const int64_t m = r / per;
  const int tile = (int)(r - m * per);
  const uint8_t* base = mask + m * (int64_t)mask_q * mask_k;
  auto selects = [&](int i, int j) -> int {  // (no branch around the load)
    const bool in = i < mask_q && j < mask_k;
    return base[in ? (int64_t)i * mask_k + j : 0] != 0 && in ? 1 : 0;
  };
  const bool halves = q_block % 32 != 0;                                             // a slab's two have mask rows of their own
  const int col0 = 128 * tile / k_block, col1 = (128 * tile + 64) / k_block;  // of the tile's halves
  const int len = q_pass ? nK : n_qs;
  int32_t* out = (q_pass ? qt_ent : kt_ent) + r * (int64_t)len;

  int cnt = 0;
  for (int t0 = 0; t0 < len; t0 += 64 * kSideBySide) {
    int bits[kSideBySide];
#pragma unroll
    for (int c = 0; c < kSideBySide; ++c) {
      const int t = t0 + 64 * c + lane;
      bits[c] = 0;
      if (t < len) {
        if (q_pass) {
#pragma unroll
          for (int g = 0; g < 8; ++g) bits[c] |= selects((128 * tile + 16 * g) / q_block, t) << g;
        } else {
          const int i0 = 32 * t / q_block, i1 = halves ? (32 * t + 16) / q_block : i0;
          bits[c] = 0x05 * selects(i0, col0) | 0x50 * selects(i0, col1);
          if (halves) bits[c] |= 0x0a * selects(i1, col0) | 0xa0 * selects(i1, col1);
          else bits[c] |= bits[c] << 1;
        }
      }
    }
#pragma unroll
    for (int c = 0; c < kSideBySide; ++c) {
      const bool on = bits[c] != 0;
      const unsigned long long bal = __ballot(on);
      if (on) out[cnt + __popcll(bal & ((1ull << lane) - 1ull))] = ((t0 + 64 * c + lane) << 8) | bits[c];
      cnt += __popcll(bal);
    }
  }
  for (int t = cnt + lane; t < len; t += 64) out[t] = -1;
  if (lane == 0) (q_pass ? qt_cnt : kt_cnt)[r] = cnt;
}

hipError_t launch_tile_lists(const uint8_t* mask, int64_t mask_bh, int mask_q, int mask_k, int nK, int q_block, int k_block, int n_qt,
                             int n_kt, int n_qs, int32_t* qt_cnt, int32_t* qt_ent, int32_t* kt_cnt, int32_t* kt_ent,
                             hipStream_t stream) {
  const int64_t waves = mask_bh * ((int64_t)n_qt + n_kt);
  const int64_t blocks = (waves + 3) / 4;
  if (blocks <= 0) return hipSuccess;
  if (blocks > 0x7fffffffLL) return hipErrorInvalidValue;
  hipLaunchKernelGGL(tile_lists_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, mask, mask_bh, mask_q, mask_k, nK, q_block, k_block,
                     n_qt, n_kt, n_qs, qt_cnt, qt_ent, kt_cnt, kt_ent);
  return hipGetLastError();
}

// Pair numbering for the dS hand-over of backward.  Every selected (query block, key block) pair gets a number in
// key-major list order: pair_base = exclusive prefix sum of k_cnt over the flattened (m, J) rows (the last entry is the
// total), pair (m, J, e) = pair_base[m, J] + e.  q_slot gives the same numbers in query-major list order, so that the
// query-major kernel finds what the key-major kernel stored: for J = q_idx[m, I, e], q_slot[m, I, e] = pair_base[m, J] +
// position of I in the ascending row k_idx[m, J, :] (binary search).  Integer work, independent of scheduling.
__global__ __attribute__((amdgpu_flat_work_group_size(1024, 1024))) void pair_base_kernel(const int32_t* __restrict__ k_cnt, int64_t n,
                                                                                          int32_t* __restrict__ pair_base, int64_t head_rows,
                                                                                          int32_t* __restrict__ bounds) {
  __shared__ int32_t wave_sum[16];
  __shared__ int32_t carry_s;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  if (tid == 0) carry_s = 0;
  __syncthreads();
  for (int64_t t0 = 0; t0 < n; t0 += 1024) {
    const int64_t t = t0 + tid;
    const int32_t x = t < n ? k_cnt[t] : 0;
    int32_t incl = x;  // inclusive scan inside the wave
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int32_t y = __shfl_up(incl, d);
      if (lane >= d) incl += y;
    }
    if (lane == 63) wave_sum[wv] = incl;
    __syncthreads();
    int32_t before = carry_s;
    for (int w = 0; w < wv; ++w) before += wave_sum[w];
    if (t < n) pair_base[t] = before + incl - x;
    if (bounds != nullptr && t < n && t % head_rows == 0) bounds[t / head_rows] = before + incl - x;
    __syncthreads();
    if (tid == 1023) carry_s = before + incl;
    __syncthreads();
  }
  if (tid == 0) {
    pair_base[n] = carry_s;
    if (bounds != nullptr) bounds[n / head_rows] = carry_s;
  }
}

// Where I, which is in it, lies in an ascending list (the two orientations describe one mask): a quarter is left after every step, from
// three loads side by side.
FBA_DEVICE int position_of(const int32_t* __restrict__ list, int count, int I) {
  int lo = 0, hi = count - 1;
  while (lo < hi) {
    const int step = (hi - lo + 4) / 4, a = lo + step, b = min(a + step, hi), c = min(b + step, hi);
    const int at_a = list[a], at_b = list[b], at_c = list[c];
    if (I < at_a) hi = a - 1;
    else if (I < at_b) { lo = a; hi = b - 1; }
    else if (I < at_c) { lo = b; hi = c - 1; }
    else lo = c;
  }
  return lo;
}

// Both steps in one launch, where there are so few rows that every work-group can add up what lies in front of its head by itself.  Bound by
// latency: each of two launches waited for a chain of loads (4.4 and 4.9 us and a gap; together 5.5 to 6.5).
constexpr int kMostOwnRows = 16384;  // of k_cnt
constexpr int kMostOwnBlocks = 2048;  // of a head
// One round of work-groups: with more of them the sums are formed over and over (24 heads of 540 x 180 blocks 36 us, in two launches 9 + 19).
constexpr int64_t kMostOwnGroups = 2048;
__global__ __attribute__((amdgpu_flat_work_group_size(256, 256))) void pair_slots_kernel(
    const int32_t* __restrict__ q_cnt, const int32_t* __restrict__ q_idx, const int32_t* __restrict__ k_cnt, const int32_t* __restrict__ k_idx,
    int64_t mask_bh, int nQ, int nK, int blocks_per_head, int32_t* __restrict__ pair_base, int32_t* __restrict__ q_slot, int32_t* __restrict__ bounds) {
  __shared__ int32_t base[kMostOwnBlocks];  // of the head's key blocks, from its first pair on
  __shared__ int32_t sums[4];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int m = (int)blockIdx.x / blocks_per_head, part = (int)blockIdx.x - m * blocks_per_head;
  // this thread's entry: where query block I lies in the list of key block J
  const int entry = part * 256 + tid;
  const bool in = entry < nQ * nK;
  const int I = in ? entry / nK : 0, e = entry - I * nK;
  const int64_t row = (int64_t)m * nQ + I;
  const bool listed = in && e < q_cnt[row];
  const int J = listed ? q_idx[row * nK + e] : 0;
  const int32_t* const list = k_idx + ((int64_t)m * nK + J) * nQ;
  const int count = listed ? k_cnt[(int64_t)m * nK + J] : 0;

  int before = 0;
  const int rows = m * nK;
  for (int t = tid; t < rows; t += 256) before += k_cnt[t];
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) before += __shfl_xor(before, d);
  if (lane == 0) sums[wv] = before;
  __syncthreads();
  const int first = sums[0] + sums[1] + sums[2] + sums[3];
  int carry = 0;
  for (int t0 = 0; t0 < nK; t0 += 256) {
    const int x = t0 + tid < nK ? k_cnt[rows + t0 + tid] : 0;
    int incl = x;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int y = __shfl_up(incl, d);
      if (lane >= d) incl += y;
    }
    __syncthreads();
    if (lane == 63) sums[wv] = incl;
    __syncthreads();
    int at = carry + incl - x;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      at += w < wv ? sums[w] : 0;
      carry += sums[w];
    }
    if (t0 + tid < nK) base[t0 + tid] = at;
  }
  __syncthreads();
  if (part == 0) {
    for (int j = tid; j < nK; j += 256) pair_base[rows + j] = first + base[j];
    if (tid == 0) {
      if (bounds != nullptr) bounds[m] = first;
      if (m + 1 == mask_bh) {
        pair_base[rows + nK] = first + carry;
        if (bounds != nullptr) bounds[m + 1] = first + carry;
      }
    }
  }
  const int at = listed ? position_of(list, count, I) : 0;
  if (in) q_slot[row * nK + e] = listed ? first + base[J] + at : -1;
}

__global__ __attribute__((amdgpu_flat_work_group_size(256, 256))) void q_slot_kernel(
    const int32_t* __restrict__ q_cnt, const int32_t* __restrict__ q_idx, const int32_t* __restrict__ k_cnt,
    const int32_t* __restrict__ k_idx, const int32_t* __restrict__ pair_base, int64_t mask_bh, int nQ, int nK,
    int32_t* __restrict__ q_slot) {
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (t >= mask_bh * nQ * nK) return;
  const int e = (int)(t % nK);
  const int64_t row = t / nK;  // m * nQ + I
  const int I = (int)(row % nQ);
  const int64_t m = row / nQ;
  int32_t out = -1;
  if (e < q_cnt[row]) {
    const int J = q_idx[t];
    const int64_t krow = m * nK + J;
    out = pair_base[krow] + position_of(k_idx + krow * nQ, k_cnt[krow], I);
  }
  q_slot[t] = out;
}

hipError_t launch_pair_slots(const int32_t* q_cnt, const int32_t* q_idx, const int32_t* k_cnt, const int32_t* k_idx, int64_t mask_bh,
                             int nQ, int nK, int32_t* pair_base, int32_t* q_slot, int32_t* bounds, hipStream_t stream) {
  const int64_t n = mask_bh * nK, entries = mask_bh * nQ * nK;
  if (n <= 0 || entries <= 0) return hipSuccess;
  const int64_t blocks = (entries + 255) / 256;
  if (blocks > 0x7fffffffLL) return hipErrorInvalidValue;
  const int64_t per_head = ((int64_t)nQ * nK + 255) / 256;
  if (n <= kMostOwnRows && nK <= kMostOwnBlocks && mask_bh * per_head <= kMostOwnGroups) {
    hipLaunchKernelGGL(pair_slots_kernel, dim3((unsigned)(mask_bh * per_head)), dim3(256), 0, stream, q_cnt, q_idx, k_cnt, k_idx, mask_bh, nQ, nK, (int)per_head,
                       pair_base, q_slot, bounds);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(pair_base_kernel, dim3(1), dim3(1024), 0, stream, k_cnt, n, pair_base, (int64_t)nK, bounds);
  hipLaunchKernelGGL(q_slot_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, q_cnt, q_idx, k_cnt, k_idx, pair_base, mask_bh, nQ, nK, q_slot);
  return hipGetLastError();
}

// Tile-pair numbering for the dS hand-over on tile lists.  The unit of the workspace is a (128-row query tile T, 128-key
// tile U) pair, listed when some 32-row slab of T appears in kt_ent[m, U, :]; pairs are numbered in key-major order:
// pair_base = exclusive prefix sum of the listed pairs per (m, U) row (last entry = total), pair (m, U, r) =
// pair_base[m, U] + r for the r-th distinct query tile of the ascending row.  kt_slot gives every kt_ent entry the number
// of its pair (what the key-major kernel needs, next to the entry); slot_table [m, T, U] gives the query-major kernel
// the same number by position (-1 where nothing is listed).  One wave per row; integer work, independent of scheduling.
__global__ __attribute__((amdgpu_flat_work_group_size(256, 256))) void tile_pair_count_kernel(
    const int32_t* __restrict__ kt_cnt, const int32_t* __restrict__ kt_ent, int64_t rows, int n_qs, int32_t* __restrict__ row_cnt) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const int cnt = kt_cnt[row];
  const int32_t* list = kt_ent + row * n_qs;
  int total = 0;
  for (int t0 = 0; t0 < cnt; t0 += 64) {
    const int e = t0 + lane;
    const bool first = e < cnt && (e == 0 || (list[e] >> 10) != (list[e - 1] >> 10));  // entry = slab << 8 | bits, tile = slab / 4
    total += __popcll(__ballot(first));
  }
  if (lane == 0) row_cnt[row] = total;
}

__global__ __attribute__((amdgpu_flat_work_group_size(256, 256))) void fill_i32_kernel(int32_t* __restrict__ out, int64_t n, int32_t value) {
  for (int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x; t < n; t += (int64_t)gridDim.x * 256) out[t] = value;
}

__global__ __attribute__((amdgpu_flat_work_group_size(256, 256))) void tile_slots_kernel(
    const int32_t* __restrict__ kt_cnt, const int32_t* __restrict__ kt_ent, const int32_t* __restrict__ pair_base, int64_t rows,
    int n_qt, int n_kt, int n_qs, int32_t* __restrict__ kt_slot, int32_t* __restrict__ slot_table) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const int64_t m = row / n_kt;
  const int U = (int)(row - m * n_kt);
  const int cnt = kt_cnt[row];
  const int32_t* list = kt_ent + row * n_qs;
  const int32_t base = pair_base[row];
  int seen = 0;  // distinct query tiles before this chunk
  for (int t0 = 0; t0 < n_qs; t0 += 64) {
    const int e = t0 + lane;
    const bool in = e < cnt;
    const int T = in ? list[e] >> 10 : 0;
    const bool first = in && (e == 0 || (list[e - 1] >> 10) != T);
    const unsigned long long bal = __ballot(first);
    const int32_t slot = base + seen + __popcll(bal & (~0ull >> (63 - lane))) - 1;  // firsts up to and including this lane
    if (e < n_qs) kt_slot[row * n_qs + e] = in ? slot : -1;
    if (first) slot_table[(m * n_qt + T) * n_kt + U] = slot;
    seen += __popcll(bal);
  }
}

hipError_t launch_tile_slots(const int32_t* kt_cnt, const int32_t* kt_ent, int64_t mask_bh, int n_qt, int n_kt, int n_qs,
                             int32_t* pair_base, int32_t* kt_slot, int32_t* slot_table, int32_t* bounds, hipStream_t stream) {
  const int64_t rows = mask_bh * n_kt, table = mask_bh * n_qt * n_kt;
  if (rows <= 0 || table <= 0 || n_qs <= 0) return hipSuccess;
  const int64_t blocks = (rows + 3) / 4;
  if (blocks > 0x7fffffffLL) return hipErrorInvalidValue;
  // the per-row counts rest in the first `rows` entries of kt_slot (which has rows * n_qs >= rows entries) until the
  // prefix sum has read them
  hipLaunchKernelGGL(tile_pair_count_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, kt_cnt, kt_ent, rows, n_qs, kt_slot);
  hipLaunchKernelGGL(pair_base_kernel, dim3(1), dim3(1024), 0, stream, kt_slot, rows, pair_base, (int64_t)n_kt, bounds);
  const int64_t fill_blocks = (table + 255) / 256;
  hipLaunchKernelGGL(fill_i32_kernel, dim3((unsigned)(fill_blocks < 4096 ? fill_blocks : 4096)), dim3(256), 0, stream, slot_table, table, -1);
  hipLaunchKernelGGL(tile_slots_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, kt_cnt, kt_ent, pair_base, rows, n_qt, n_kt, n_qs,
                     kt_slot, slot_table);
  return hipGetLastError();
}

}  // namespace fba
