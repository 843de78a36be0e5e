// Tail splitting: which items of a launch are cut into parts (see SplitPlan in fba_kernels.h).
#include <algorithm>
#include <cstdlib>
#include <mutex>

#include "fba_kernels.h"

namespace fba {

namespace {

// Compute units of the current device (looked up once per device).
int compute_units() {
  constexpr int kMaxDevices = 64;
  static std::mutex mu;
  static int cache[kMaxDevices] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return 256;
  std::lock_guard<std::mutex> lock(mu);
  if (cache[dev] == 0) {
    int n = 0;
    cache[dev] = hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && n > 0 ? n : 256;
  }
  return cache[dev];
}

}  // namespace

int device_compute_units() { return compute_units(); }

// The hardware hands work-groups to free slots in index order.  With n items on s slots the last n % s items form a
// partial round; when that round would fill at most half of the slots, each of its items is cut into up to floor(s / (n % s))
// parts (at most 8), so that the parts fill the slots once and take 1 / parts of a round.  Launches smaller than the
// machine (n < s) are split the same way.
//
// How many parts pay: every part writes its partial results, and the merge reads them back, so with m items of at most
// max_steps steps each the round takes about  max_steps step_cost / parts + m parts  in units of what one part's results
// cost, least at parts = sqrt(max_steps step_cost / m).  The lists are on the device: step_cost assumes that 40 % of the
// longest possible list is there.  One part's 64 KiB cost 27 ns at what the stores and the merge sustain (2.4 TB/s) and a
// forward step of such a round 0.65 us, so forward has step_cost 9, and 18 on tile lists, whose parts store half as much.  dK/dV
// has 6 with 128 keys (0.9 us a slab, 128 KiB a part) and 9 with 64 keys (0.6 us, 64 KiB); dQ has forward's 9 where it recomputes
// S and dP and 4 from dS, whose step is two products instead of six.  Times with a quarter / half / once / twice / four times each
// value: forward (9) H8 S768 60 % kept 14.8 / 14.6 / 14.4 / 18.9 / 19.5 us, H4 S4096 20 % kept 21.2 / 20.7 / 28.6 / 29.4 / 29.3, 60 %
// kept 45.6 / 45.1 / 42.2 / 41.1 / 40.9; (18) H4 S4096 60 % kept 36.3 / 35.1 / 34.7 / 40.3 / 39.6; steps, (6) H4 S4096 60 % kept 157 /
// 156 / 144 / 144 / 144; (4) 145 / 144 / 144 / 143 / 154; (9, 64 keys) H2 S4096 60 % kept 132 / 130 / 127 / 128 / 128.  No value is
// ahead at every density: short lists want fewer parts, long ones more.  Measured, forward / backward in us (always as many
// parts as slots allow, against this rule): B1 H8 S768, 128-token blocks, half kept 22.0 / 54.9 -> 15.8 / 43.0; H4 S1536
// 23.9 / 58.5 -> 19.8 / 54.7; H8 S4096, a quarter kept 43.2 / 104.8 -> 37.0 / 92.9.
SplitPlan plan_split(int num_items, int wgs_per_cu, int max_steps, double step_cost, int64_t slot_bytes, void* ws, int64_t ws_bytes) {
  SplitPlan plan{nullptr, num_items, 1, 0};
  if (ws == nullptr || num_items <= 0) return plan;
  int slots = compute_units() * wgs_per_cu;
  if (slots > kSplitMaxSlots) slots = kSplitMaxSlots;
  const int rest = num_items % slots;
  if (rest == 0 || 2 * rest > slots) return plan;
  int parts = slots / rest;
  if (parts > 8) parts = 8;
  const double whole = max_steps * step_cost;
  while (parts >= 2 && (double)parts * parts * rest > whole) --parts;
  while (parts >= 2 && (int64_t)rest * parts * slot_bytes > ws_bytes) --parts;
  if (parts < 2 || whole / parts + (double)rest * parts > 0.9 * whole) return plan;
  plan.ws = static_cast<float*>(ws);
  plan.first = num_items - rest;
  plan.parts = parts;
  return plan;
}

namespace {

constexpr int kQueueBytes = 256;
constexpr int kRankItems = 64;      // items a block of the ordering launch places
constexpr int kMostOrdered = 2048;  // items of a launch that is ordered at all: eight rounds

__global__ void queue_reset_kernel(int* queue) { queue[threadIdx.x] = 0; }

// Which item every grid index of a dK/dV launch works on: long lists first.  The lists of a random mask differ by 10-20 %
// in length, so with items in index order the last round of work-groups ends with the longest list that happened to start
// last; in falling order of length the last ones to start are the short ones.  An item's key is the number of listed
// query blocks over the query heads of its group.
//
// The items are dealt to `spans` runs (one per XCD, whose work-groups get the grid indices XCD, XCD + 8, ..., or a single one),
// every run is cut into segments of `segment` items counted from its end, and each segment is sorted by counting, for every
// item, the items of the segment in front of it (longer, or as long with a lower number): no atomics, one result.  Segments
// keep the heads of a large launch one after the other, so that work-groups that run together still share Q and dO in L2.
// Lists of one length keep index order, so for them the launch is all cost: it has to be short.  Four lanes share the counting of
// an item, with eight LDS reads in flight each; with one lane per item and a read at a time the chain of reads set the time.
// Grid: spans * ceil(longest run / 64) blocks.
__global__ __attribute__((amdgpu_flat_work_group_size(256, 256))) void order_items_kernel(const BwdParams p, int spans, int segment, int32_t* order) {
  __shared__ int lens[kMostOrdered];
  const int tid = threadIdx.x;
  if (p.queue != nullptr && blockIdx.x == 0 && tid < kQueueBytes / 4) p.queue[tid] = 0;
  const int span = blockIdx.x % spans, i0 = blockIdx.x / spans * kRankItems;
  const int start = span * (p.num_items / spans) + min(span, p.num_items % spans);
  const int count = p.num_items / spans + (span < p.num_items % spans);
  if (i0 >= count) return;
  const int tiles_per_head = p.Skv / 128, group = p.Hq / p.Hkv;
  auto length = [&](int i) {  // of item i of the run
    const int item = start + i;
    const int bhk = item / tiles_per_head, kblk = (item - bhk * tiles_per_head) * 128 / p.k_block;
    if (p.mask_bh == 1) return p.k_cnt[kblk];
    const int64_t row = (int64_t)bhk * group * p.nK + kblk;  // query heads of a kv head are consecutive
    int n = 0;
    for (int g = 0; g < group; ++g) n += p.k_cnt[row + (int64_t)g * p.nK];
    return n;
  };
  auto segment_end = [&](int i) { return count - (count - 1 - i) / segment * segment; };
  const int from = max(0, segment_end(i0) - segment), to = segment_end(min(i0 + kRankItems, count) - 1);  // of all items of the block
  for (int j = from + tid; j < to; j += 256) lens[j - from] = length(j);
  __syncthreads();
  const int i = min(i0 + (tid >> 2), count - 1);
  const int own = lens[i - from], hi = segment_end(i), lo = max(0, hi - segment);
  int before = 0;
#pragma unroll 8
  for (int j = lo + (tid & 3); j < hi; j += 4) {
    const int other = lens[j - from];
    before += other > own || (other == own && j < i);
  }
  before += __shfl_xor(before, 1);
  before += __shfl_xor(before, 2);
  if ((tid & 3) == 0 && i0 + (tid >> 2) < count) order[(int64_t)(lo + before) * spans + span] = start + i;
}

}  // namespace

hipError_t plan_key_tiles(BwdParams& p, int tile_rows, double step_cost, int64_t slot_bytes, int& grid, hipStream_t stream) {
  const int slots = compute_units();  // one work-group per compute unit
  const int heads = p.B * p.Hkv;
  char* const ws = reinterpret_cast<char*>(p.split.ws);  // whether or not anything is split
  p.num_items = heads * (p.Skv / tile_rows);
  p.split = plan_split(p.num_items, 1, p.Hq / p.Hkv * (p.Sq / 32), step_cost, slot_bytes, ws, p.split_ws_bytes);
  plan_xcd_mapping(heads, p.split.first, p.items_per_xcd, p.split.main_wgs);
  const int parts = (p.num_items - p.split.first) * p.split.parts;
  p.queue = nullptr;
  p.order = nullptr;

  // What else lives in the workspace, from its end: the claim counters, then the order of the items.
  int64_t top = ws == nullptr ? 0 : (p.split_ws_bytes - kQueueBytes) & ~(int64_t)15;
  const int64_t bottom = parts * slot_bytes;
  int* const queue = ws != nullptr && top >= bottom ? reinterpret_cast<int*>(ws + top) : nullptr;
  top = (top - (int64_t)p.num_items * 4) & ~(int64_t)15;
  // Items are ordered where they start in more than one round and in at most eight.  One round starts everything at once; over
  // many rounds the spread of the last one no longer counts, while tiles in index order share more of their lists in L2
  // (structured masks).  Steps, items in index order / ordered: masks that choose per head, a quarter kept, H8 S8192 (2 rounds)
  // 344 / 314 us, H24 S6144 (4.5) 599 / 585, B2 H16/4 S8192 (2) 1088 / 1065, 40 % kept, H24 S30720 (7.5 per chunk) 16.53 / 16.04
  // ms; causal H8 S15360 (3.75) 2341 / 2116 us; H24 S69120 top-k (17) 25.3 / 25.2 ms, H24 S115200 sliding window (28) 52.1 / 52.9
  // ms.  Where all lists are equally long it gains nothing and costs the launch (6.6 us for 1920 items, rocprofv3), or next to
  // nothing where a launch has to clear the claim counters anyway: all blocks, H8 S9216 1371 / 1376 us, H24 S6144 1740 / 1734.  So
  // without claims the longest possible list has to have 192 slabs, with them 128: bands of a quarter, H12 S4096 (128 slabs, 1.5
  // rounds) 174 / 179 us, which the 179 / 176 us of a random mask of that size do not make up for, H32 S4096 (4 rounds) 365 / 367
  // against 377 / 359 us; a random mask at H8 S6144 (192 slabs, 1.5 rounds) 302 / 297 us, 308 / 289 where all
  // heads share it.
  const int longest = p.Hq / p.Hkv * (p.Sq / 32);
  const bool ordered = !p.tiled && queue != nullptr && top >= bottom && p.num_items > slots && p.num_items <= std::min(8 * slots, kMostOrdered) &&
                       longest >= (p.split.first + parts >= 4 * slots ? 128 : 192);
  if (ordered) p.split.main_wgs = p.split.first;

  // Launches of four rounds and more let the work-groups claim their grid indices, with some more work-groups than indices,
  // so that an XCD that is through early takes over from the others (claim_work; either mapping deals grid index i to XCD
  // i % 8, which is all a claim relies on).  FBA_CLAIM_WORK=0 switches claiming off, for measurements.
  p.total_work = p.split.main_wgs + parts;
  grid = p.total_work;
  const char* claim = getenv("FBA_CLAIM_WORK");
  if (queue != nullptr && !(claim != nullptr && claim[0] == '0') && p.total_work >= 4 * slots) {
    p.queue = queue;
    grid += (p.total_work / 8 + 7) / 8 * 8;  // an eighth more work-groups, a whole number per XCD
  }
  if (ordered) {
    const int spans = heads >= 8 ? 8 : 1;
    const int tiles_per_head = p.Skv / tile_rows, two_rounds = 2 * slots / spans;
    const int segment = (two_rounds + tiles_per_head - 1) / tiles_per_head * tiles_per_head;
    const int blocks = spans * (((p.num_items + spans - 1) / spans + kRankItems - 1) / kRankItems);
    int32_t* const order = reinterpret_cast<int32_t*>(ws + top);
    hipLaunchKernelGGL(order_items_kernel, dim3(blocks), dim3(256), 0, stream, p, spans, segment, order);
    p.order = order;
  } else if (p.queue != nullptr) {
    hipLaunchKernelGGL(queue_reset_kernel, dim3(1), dim3(kQueueBytes / 4), 0, stream, p.queue);
  }
  return hipGetLastError();
}

}  // namespace fba
