// Tail splitting: which items of a launch are cut into parts (see SplitPlan in fba_kernels.h).
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <mutex>

#include "fba_common.h"
#include "fba_kernels.h"

namespace fba {

namespace {

thread_local int assumed_units = 0;  // see AssumedUnits

// Compute units of the current device (looked up once per device).
int compute_units() {
  if (assumed_units > 0) return assumed_units;
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

AssumedUnits::AssumedUnits(int units) : before(assumed_units) { assumed_units = units; }
AssumedUnits::~AssumedUnits() { assumed_units = before; }

// The hardware hands work-groups to free slots in index order.  With n items on s slots the last n % s items form a
// partial round; the lists of these items are cut into parts (at most 8) where parts fill the slots better.  Launches smaller than the
// machine (n < s) are split the same way.
//
// How many parts pay: every part writes its partial results and the merge reads them back, so with m items of L steps a round
// takes  L slope(parts) + m parts  in units of what one part's results cost, 27 ns for 64 KiB at what the stores and the merge
// sustain (2.4 TB/s; taken a quarter dearer, since the parts of a launch end together).  slope is what a step takes times the rounds
// the parts make, over their number.  A forward step takes 0.50 us in a work-group alone on its compute unit, 0.73 us where the
// first share one and 0.95 us where all do (16, 22.5 and 30 units), so 72 items are better off in 3 parts than in 7: H24 384 rows
// against 15360 keys, half kept, 63.6 -> 55.2 us; whole items that fill every unit take up to 0.59 us a step (H2 S15360 all blocks, 240 items: 284 us whole,
// 236 and a merge in two parts).  On tile lists parts store half as much and a step is as long; dQ that recomputes S
// and dP is like forward, dQ from dS two products instead of six; a dK/dV slab takes 0.9 us with 128 keys (128 KiB a part) and
// 0.6 us with 64 (64 KiB).
//
// L is on the device: the host says from which lengths on which numbers of parts pay, up to the longest possible lists, and the kernel
// looks at the lists (a load of 16 cache lines, 0.3 to 0.5 us a launch).  Forward + backward, parts for lists that hold 60 % / for the
// lists there are, 128-token blocks, 10 and 80 % kept: H1 S12800 138 / 98 and 327 / 328 us, H4 S1920 62.7 / 51.9 and 81.5 / 83.6, H2
// S4096 74.2 / 65.5 and 110.0 / 108.8, H2 S1536 50.7 / 49.3 and 64.0 / 66.4.  Behind a whole round: H24 S3072, 10 and 30 % kept, 160 / 140 and 240 / 230
// us, H12 S3072 15 % 112.4 / 114.3 (lists just short of the line, of which the longest would have been worth cutting).
//
// Lists that differ: whole items of a single round take as long as the longest list, parts about as long as a list that is 0.6 of the mean
// and 0.4 of the longest.  So the line for one round is drawn where  slope(1) longest - slope(parts) (0.6 mean + 0.4 longest)  reaches
// what the parts cost besides.  Forward, decided by the mean / so: H1 S20480, 128-token blocks, Bernoulli masks of 10 % 56.5 / 45.8 us,
// densities that rise ninefold along the sequence 74.1 / 50.9, causal H5 S4352 68.2 / 50.6.  So that such masks can be cut, launches of
// up to half a round are planned too where lists of one length would have to hold more than 60 %, if lists that fall to nothing
// gain well; lists of one length there pay 2 us for the look and a merge with nothing to do (H5 S4352, a quarter kept 22.1 -> 24.0 us;
// always cut they took 30.8).  Tile lists of 128 rows differ more than the halves that are worked on, so only half of what the longest
// is above the mean counts there (H2 S8192, 64-token blocks, 31 % kept, lists of 67 chunks and up to 73 for halves of 40 each).  dQ from
// dS is not judged by the longest list: it is bound by memory, which the short lists leave to the long ones (H3 S10240, 30 % kept,
// backward 182 -> 195 us).
//
// More than half a round is cut as well, in launches of less than one round, where work-groups end together: dK/dV of 136 tiles (H1
// S17408), 30, 50 and 100 % kept, backward 227 -> 213, 350 -> 301 and 566 -> 496 us.  In a second round only where all the launch's lists
// are nearly full and so nearly alike: with items in falling order of length the long ones make way for the short ones by themselves,
// and a chip that is not full runs faster.  420 tiles (H3 S17920), 30, 70 and 100 % kept, whole / cut 474 / 503, 995 / 1001 and 1387 /
// 1340 us; 680 tiles (H8 S10880), more than two rounds, 40 % kept 579 / 599.  Nor on tile lists, where a part scans its lists twice: H8/4
// S13824, 64 x 384 blocks, 44 % kept, dK/dV 401 -> 456 us.
//
// A part on a tile list scans the whole list before it takes its own steps: H5 S1536, 16 x 64 blocks, a third kept, dK/dV of 120 half
// tiles of 27 steps 25.4 us whole, 22.4 us and a merge of 5.0 in two parts.
constexpr double kMergeCost = 60;   // the launch
constexpr double kScanCost = 40;    // and, on tile lists, the scans
constexpr int64_t kNoteBytes = 16;  // behind the parts' results
constexpr float kNever = 3e38f;     // entries
SplitPlan plan_split(int num_items, int wgs_per_cu, int max_steps, StepCost step, int64_t slot_bytes, void* ws, int64_t ws_bytes,
                     const ListLengths& lengths) {
  SplitPlan plan{};
  plan.first = num_items;
  plan.parts = 1;
  if (ws == nullptr || num_items <= 0) return plan;
  int slots = compute_units() * wgs_per_cu;
  if (slots > kSplitMaxSlots) slots = kSplitMaxSlots;
  const int rest = num_items % slots;
  if (rest == 0 || (2 * rest > slots && (num_items >= 2 * slots || step.scans))) return plan;
  // cost(n) = slope(n) steps + parts and, where there are any, the launch that merges them.  From how long a list on is a number of
  // parts the cheapest: the slope falls from one candidate to the next, and one that is never the cheapest gives way.
  auto slope = [&](int n) {
    const int wgs = rest * n, alone = slots / wgs_per_cu;
    if (n == 1 && wgs <= alone && num_items >= 2 * slots) return step.few;  // items of the round before are still there
    if (n == 1 && wgs <= alone) return step.alone * (1 + 0.15 * std::max(0, 2 * wgs - alone) / alone);  // a full chip runs at a lower clock: 240 items 0.59 us a step
    if (wgs <= alone) return step.alone / n;
    if (wgs <= slots) return (step.few + (step.full - step.few) * (wgs - alone) / (slots - alone)) / n;
    return step.full * ((wgs + slots - 1) / slots) / n;
  };
  struct Candidate { int parts; double slope, fixed, least; } hull[kMostParts] = {{1, slope(1), 0., 0.}};
  int n_hull = 1;
  for (int n = 2; n <= kMostParts && (int64_t)rest * n * slot_bytes + kNoteBytes <= ws_bytes; ++n) {
    if (num_items > slots && rest * n > slots && 2 * rest <= slots) break;  // a last round that fills up while others end gains nothing from another
    Candidate next{n, slope(n), (double)rest * n + kMergeCost + (step.scans ? kScanCost : 0), 0.};
    if (wgs_per_cu == 1 && 2 * rest > slots && next.slope > 0.75 * slope(1)) continue;  // 0.8 of a round in five parts: H2 S29440 1055 -> 1095 us
    while (n_hull > 0 && next.slope < hull[n_hull - 1].slope) {
      next.least = (next.fixed - hull[n_hull - 1].fixed) / (hull[n_hull - 1].slope - next.slope);
      if (n_hull == 1 || next.least > hull[n_hull - 1].least) {
        hull[n_hull++] = next;
        break;
      }
      --n_hull;
    }
  }
  if (n_hull == 1) return plan;
  const bool device = lengths.cnt != nullptr || lengths.mask != nullptr, one_round = device && num_items < slots && step.own_pace;
  const double least = hull[1].least * (hull[0].slope - hull[1].slope);
  const bool uneven = one_round && 2 * rest <= slots && max_steps * (hull[0].slope - 0.5 * hull[1].slope) >= 2.5 * least;
  if (hull[1].least > 0.6 * max_steps && !uneven) return plan;  // lists of usual density stay whole
  const bool second = num_items > slots && 2 * rest > slots;
  if (second) hull[1].least = std::max(hull[1].least, 0.9 * max_steps);
  // Behind two rounds and more parts start as the items in front of them end, so lists fuller than usual are not cut finer for it (forward of
  // H24 S11520, all blocks, 112 items in 2 / 4 parts 1441 / 1449 us; H24 S30720, 128 items 10115 / 10123).
  const double longest = device && num_items < 2 * slots ? max_steps : 0.6 * max_steps;
  while (n_hull > 2 && hull[n_hull - 1].least > longest) --n_hull;
  plan.parts = hull[n_hull - 1].parts;
  plan.items = rest;
  plan.first = num_items - rest;
  plan.note = reinterpret_cast<int32_t*>(static_cast<char*>(ws) + (int64_t)rest * plan.parts * slot_bytes);
  plan.ws = static_cast<float*>(ws);
  if (!device) return plan;

  // The lists of the items that are split, or all of the launch's in second rounds more than half full (dK/dV), which have to be alike.
  ListLook& look = plan.look;
  const int64_t rows = (int64_t)num_items * lengths.tile_rows / lengths.list_rows, from = second ? 0 : (int64_t)plan.first * lengths.tile_rows / lengths.list_rows;
  const int64_t span = lengths.shared ? std::min<int64_t>(rows - from, lengths.rows_per_head) : rows - from;
  look.cnt = lengths.cnt;
  look.mask = lengths.mask;
  look.blocks = lengths.blocks;
  look.first = (int)(lengths.shared ? lengths.rows_per_head - span : from);
  look.row_tiles = std::max(lengths.list_rows / lengths.tile_rows, 1);
  look.shared = lengths.shared;
  look.group = lengths.shared ? 1 : lengths.group;
  look.rows_per_head = lengths.rows_per_head;
  look.stride = (int)(std::max<int64_t>(span - 4, 0) / 15);
  look.last = (int)(span - 1);
  look.step = (float)lengths.steps * lengths.group / (look.group > 1 ? 4 : 1);
  look.spread = !one_round ? 0.f : step.scans ? 0.5f : 1.f;
  look.whole = (float)hull[0].slope * look.step;
  look.cut = (float)hull[1].slope * look.step;
  look.least = (float)(hull[1].least * (hull[0].slope - hull[1].slope));
  look.fewest = hull[1].parts;
  for (float& n : look.more) n = kNever;
  for (int i = 2; i < n_hull; ++i)
    for (int n = hull[i - 1].parts + 1; n <= hull[i].parts; ++n) look.more[n - look.fewest - 1] = (float)(hull[i].least / look.step);
  return plan;
}

// Forward and dQ launches of less than a round.  With parts that follow each other an XCD reads 1 / gcd(parts, 8) of what all items read; more than its L2
// holds (4 MiB) comes from the memory-side cache as often as there are items that select it, which bounds such launches: 144 tiles of 24 heads on 6 kv heads of
// 30720 keys in three parts copy 0.9 GB.  Parts in turn / grouped (keys and values of one kv head in MiB x kv heads, parts): forward H24/6, 768 rows against
// 30720 keys (15 x 6, three) 144 / 129 us, H4 2304 against 46080 (22 x 4, three) 152 / 130, H24 1280 against 20480 (10 x 24, two) 147 / 139, H12 the same (10 x 12,
// four) 100.6 / 96.3; steps H12 1536 against 15360 380 / 349, H8 768 against 7680 (3.75 x 8, three) 150 / 138.  Where an L2 holds it, the work-groups of an XCD
// then all wait for the same few lines: steps H4 S3840 (1.9 x 4, four parts) 114.0 / 116.9, H2 S6144 140.6 / 143.4.  Behind a whole round: H12 S3456 155.4 / 156.8.
void group_parts(SplitPlan& plan, int tiles, int64_t bytes) {
  constexpr int64_t kL2Bytes = 4 << 20;
  if (plan.ws == nullptr || plan.first > 0) return;
  plan.share = tiles;
  const int64_t all = (plan.items + tiles - 1) / tiles * bytes;
  for (int n = 2; n <= plan.parts; ++n)
    if (all > kL2Bytes * (n % 8 == 0 ? 8 : n % 4 == 0 ? 4 : n % 2 == 0 ? 2 : 1)) plan.grouped |= 1u << n;
}

namespace {

constexpr int kQueueBytes = 256;
constexpr int kRankItems = 64;      // items a block of the ordering launch places
constexpr int kMostOrdered = 2048;  // items of a launch that is ordered at all: eight rounds

// Backward statistics, one pass over O and dO: stats[r] = lse[r] * log2(e) and stats[rows + r] = -delta[r] =
// -sum_c dO[r, c] * O[r, c] in fp32 (reference: bwd_attend_prep_ker, flex_block_attn_h100.cu:375-379).  The backward
// kernels exponentiate in base 2, hence the pre-scaled LSE; they start the dP accumulators from the second plane, so that
// the matrix instructions themselves form dP - delta (the reference preloads its accumulator the same way,
// flex_block_attn_h100.cu:445-467), hence the sign.  16 lanes per row (16 bytes of each operand per lane); 256 threads to a block.
//
// Bound by memory: 524 bytes of a row, each once.  With a row to 16 lanes the blocks ended as soon as their two loads had come back, so that
// starting them set the pace; launches that fill the GPU with four rows to 16 lanes request all eight loads first (262144 rows 30.1 -> 22.1 us,
// 6.2 TB/s; 552960 rows 64.2 -> 55.7 us, 5.2 TB/s).
//
// kFill: dO has fewer rows to a head than O (lengths that are no whole tiles) and is copied on the way, with rows of zeros for what fills up the last
// tile: a launch of 6.2 us less at B2 H8 S3136.
constexpr int kStatsRows = 16, kStatsDeep = 4;
constexpr int64_t kStatsMany = 131072;  // rows: eight blocks of 64 rows for each of 256 compute units
__host__ __device__ inline bool stats_deep(const BwdStats& s) { return s.rows >= kStatsMany; }
template <int kDeep, bool kFill>
FBA_DEVICE void stats_rows_of(const BwdStats& s, int block, int blocks) {
  const int sub = threadIdx.x & 15;
  for (int64_t r0 = (int64_t)block * (kStatsRows * kDeep) + (threadIdx.x >> 4); r0 < s.rows; r0 += (int64_t)blocks * (kStatsRows * kDeep)) {
    bf16x8 a[kDeep], b[kDeep];
    float lse[kDeep];
#pragma unroll
    for (int d = 0; d < kDeep; ++d) {
      const int64_t r = r0 + d * kStatsRows < s.rows ? r0 + d * kStatsRows : r0;
      a[d] = *reinterpret_cast<const bf16x8*>(s.o + r * kHeadDim + sub * 8);
      lse[d] = s.lse[r];
      if constexpr (kFill) {
        const uint32_t head = (uint32_t)r / (uint32_t)s.head_rows;
        const int at = (int)((uint32_t)r - head * (uint32_t)s.head_rows);
        bf16x8 x = {};
        if (at < s.given_rows) x = *reinterpret_cast<const bf16x8*>(s.d_o + ((int64_t)head * s.given_rows + at) * kHeadDim + sub * 8);
        b[d] = x;
      } else {
        b[d] = *reinterpret_cast<const bf16x8*>(s.d_o + r * kHeadDim + sub * 8);
      }
    }
#pragma unroll
    for (int d = 0; d < kDeep; ++d) {
      const int64_t r = r0 + d * kStatsRows;
      if constexpr (kFill)
        if (r < s.rows) *reinterpret_cast<bf16x8*>(s.filled + r * kHeadDim + sub * 8) = b[d];
      float acc = 0.f;
#pragma unroll
      for (int t = 0; t < 8; ++t) acc += (float)a[d][t] * (float)b[d][t];
      acc += __shfl_xor(acc, 8);
      acc += __shfl_xor(acc, 4);
      acc += __shfl_xor(acc, 2);
      acc += __shfl_xor(acc, 1);
      if (sub == 0 && r < s.rows) {
        s.stats[r] = lse[d] * 1.4426950408889634f;
        s.stats[s.rows + r] = -acc;
      }
    }
  }
}
FBA_DEVICE void stats_rows(const BwdStats& s, int block, int blocks) {
  if (s.filled != nullptr) {
    if (stats_deep(s)) stats_rows_of<kStatsDeep, true>(s, block, blocks);
    else stats_rows_of<1, true>(s, block, blocks);
  } else {
    if (stats_deep(s)) stats_rows_of<kStatsDeep, false>(s, block, blocks);
    else stats_rows_of<1, false>(s, block, blocks);
  }
}
int stats_blocks(const BwdStats& s) {
  const int rows = kStatsRows * (stats_deep(s) ? kStatsDeep : 1);
  return (int)std::min<int64_t>((s.rows + rows - 1) / rows, 65536);
}

__global__ __attribute__((amdgpu_flat_work_group_size(256, 256))) void bwd_stats_kernel(const BwdStats s) { stats_rows(s, blockIdx.x, gridDim.x); }

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
// spans * ceil(longest run / 64) blocks.
struct ItemOrder {
  int blocks, spans, segment;
  int32_t* order;
};
FBA_DEVICE void order_items(const BwdParams& p, const ItemOrder& make, int block, int* lens) {
  const int tid = threadIdx.x, spans = make.spans, segment = make.segment;
  const int span = block % spans, i0 = block / spans * kRankItems;
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
  if ((tid & 3) == 0 && i0 + (tid >> 2) < count) make.order[(int64_t)(lo + before) * spans + span] = start + i;
}

// Lists of very different length (a sink block that every query selects, windows shifted in at a border): while other compute units are done, the
// longest list goes on.  Then the items are cut to about equal pieces instead, and the pieces start in falling order of length.
//
// What decides: with the whole chip at work a slab takes a work-group 1.0 us (two slabs in 2.0), with most of it idle 0.75, since the
// clock rises; so lists up to 1.3 times what an even share would be lose nothing by it, and cutting costs the partial results and their
// merge, about 20 us.  (H1 S30720, 60 % kept at random, lists of 37 to 59 blocks on 240 compute units: 45 an even share, dK/dV 552 us whole; as
// much when the longest were cut.)
// Steps, whole lists / pieces (with the launches as they were before there were any; median of nine): score-driven masks with a sink block, 128-row query
// and 384-row key blocks, top-12, H1 S24192 753 / 377 us, H2 947 / 636, top-16 H2 S69120 4196 / 2170; 3 x 3 x 3 windows over 3 x 4 x 5 tiles, H1 825 / 639, H2
// 1495 / 1095; video latents H4 S73728 11906 / 9275.  What pieces alone are worth there: 714, 902, 4100, 822, 1473 and 11800 us without them.
// Launches of less than a round: the smallest piece with which there is one for every compute unit at most.  Others: an even share;
// what is longer than 1.5 of them is cut.
struct PieceMaker {
  int32_t* header;
  Piece* list;
  CutItem* cut;
  int slots, max_slots, most;  // compute units, partial results the workspace has room for, pieces the launch has work-groups for
  int parts;                   // that the host has planned for all items alike
};
constexpr int kFrontThreads = 256, kFrontWaves = kFrontThreads / 64;
constexpr int kBins = 256;
constexpr float kSlabAlone = 0.75f, kSlabFull = 1.f, kPiecesCost = 20.f;  // us

// Sum over (or largest of) the block's threads, the same in all of them.  `scratch`: kFrontWaves ints.
template <bool kMax>
FBA_DEVICE int over_block(int x, int* scratch) {
  const int w = kMax ? wave_max(x) : wave_sum(x);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) scratch[threadIdx.x >> 6] = w;
  __syncthreads();
  int all = scratch[0];
#pragma unroll
  for (int i = 1; i < kFrontWaves; ++i) all = kMax ? max(all, scratch[i]) : all + scratch[i];
  return all;
}
// Sum over the threads in front of this one, and over all.
FBA_DEVICE int before_thread(int x, int* scratch, int& all) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int sum = x;
#pragma unroll
  for (int d = 1; d < 64; d *= 2) {
    const int y = __shfl_up(sum, d);
    sum += lane >= d ? y : 0;
  }
  __syncthreads();
  if (lane == 63) scratch[wave] = sum;
  __syncthreads();
  int before = sum - x;
  all = 0;
#pragma unroll
  for (int i = 0; i < kFrontWaves; ++i) {
    before += i < wave ? scratch[i] : 0;
    all += scratch[i];
  }
  return before;
}

FBA_DEVICE int list_entries(const BwdParams& p, int item) {  // of a key tile of 128 rows, over the query heads of its group
  const int tiles_per_head = p.Skv / 128, group = p.Hq / p.Hkv;
  const int bhk = item / tiles_per_head, kblk = (item - bhk * tiles_per_head) * 128 / p.k_block;
  if (p.mask_bh == 1) return p.k_cnt[kblk] * group;
  const int64_t row = (int64_t)bhk * group * p.nK + kblk;  // query heads of a kv head are consecutive
  int n = 0;
  for (int g = 0; g < group; ++g) n += p.k_cnt[row + (int64_t)g * p.nK];
  return n;
}

FBA_DEVICE void plan_pieces(const BwdParams& p, const PieceMaker& make, int* lens) {
  __shared__ int scratch[kFrontWaves], bins[kBins];
  const int tid = threadIdx.x, items = p.num_items;
  const int each = (items + kFrontThreads - 1) / kFrontThreads, first = min(tid * each, items), last = min(first + each, items);  // this thread's
  int longest = 0, sum = 0;
  for (int j = tid; j < items; j += kFrontThreads) {
    const int n = list_entries(p, j) * (p.q_block / 32);
    lens[j] = n;
    longest = max(longest, n);
    sum += n;
  }
  longest = over_block<true>(longest, scratch);
  const float share = (float)over_block<false>(sum, scratch) / (float)make.slots;  // (items times the longest possible list is below 2^31)
  float whole = (float)longest;  // how long the longest list makes the launch, in slabs
  int size = max(64, ((int)share + 4) & ~3), most = size + size / 2;  // of a piece; what is longer is cut
  if (items <= make.slots) {
    for (int n = 2; n <= make.parts; ++n)  // parts of all items alike, where the host has planned them
      whole = fminf(whole, n * items <= make.slots ? (float)longest / n : fmaxf((float)longest / n, share + 0.5f * (float)longest / n));
    int low = min(size, longest), high = max(longest, 4);  // the smallest size that makes no more pieces than there are compute units
    while (high - low > max(4, high / 32)) {
      const int middle = (low + high) / 2;
      const float per = 1.f / (float)middle;
      int n = 0;
      for (int j = first; j < last; ++j) n += max(1, (int)__builtin_ceilf((float)lens[j] * per));
      if (over_block<false>(n, scratch) <= make.slots) high = middle; else low = middle + 1;
    }
    size = most = (high + 7) & ~3;
  }
  const float per_size = 1.f / (float)size;
  auto pieces_of = [&](int n) { return n <= most ? 1 : (int)__builtin_ceilf((float)n * per_size); };
  const float cut_time = 1.05f * fmaxf(kSlabAlone * (float)most, kSlabFull * share) + kPiecesCost;
  int n_cut = 0, n_slots = 0, cut_at = 0, slot_at = 0;
  bool cuts = fmaxf(kSlabAlone * whole, kSlabFull * share) > 1.05f * cut_time;
  if (cuts) {
    int packed = 0;  // items that are cut << 16 | their pieces: an even share or more each, so some thousands at most
    for (int j = first; j < last; ++j) {
      const int n = pieces_of(lens[j]);
      packed += n > 1 ? 1 << 16 | n : 0;
    }
    int all;
    const int before = before_thread(packed, scratch, all);
    n_cut = all >> 16;
    n_slots = all & 0xffff;
    cut_at = before >> 16;
    slot_at = before & 0xffff;
    cuts = n_cut > 0 && n_slots <= make.max_slots && items + n_slots - n_cut <= make.most;
  }
  if (tid == 0) {
    make.header[0] = cuts ? items + n_slots - n_cut : 0;
    make.header[1] = n_cut;
  }
  if (!cuts) return;

  // long pieces first: counted by length, then dealt out (which of two as long as each other comes first makes no difference to any result)
  bins[tid] = 0;
  __syncthreads();
  const float per_slab = (float)(kBins - 1) / (float)most;
  auto bin_of = [&](int slabs) { return kBins - 1 - min((int)((float)slabs * per_slab), kBins - 1); };
  for (int j = first; j < last; ++j) {
    const int n = pieces_of(lens[j]);
    atomicAdd(&bins[bin_of(lens[j] / n)], n);
  }
  __syncthreads();
  int unused;
  const int in_front = before_thread(bins[tid], scratch, unused);
  bins[tid] = in_front;
  __syncthreads();
  for (int j = first; j < last; ++j) {
    const int n = pieces_of(lens[j]), quads = lens[j] / 4;  // boundaries on multiples of four slabs
    const int at = atomicAdd(&bins[bin_of(lens[j] / n)], n);
    for (int q = 0; q < n; ++q) {
      const int from = (int)((int64_t)quads * q / n), to = (int)((int64_t)quads * (q + 1) / n);
      make.list[at + q] = {j, 4 * from, 4 * (to - from), n > 1 ? slot_at + q : -1};
    }
    if (n > 1) {
      make.cut[cut_at++] = {j, slot_at, n, 0};
      slot_at += n;
    }
  }
}
static_assert(kBins == kFrontThreads);

// What runs in front of a dK/dV kernel, side by side in one launch: the plan of its pieces, the order of its items, its claim counters, the
// statistics.  In launches of their own the order or the counters took 5 to 6 us and a gap beside 5 us of statistics at S24192; now all of it takes 6 to
// 8.5 us (H4 S8192, 32 of 64 kept, step 309 -> 298 us; H8 S9216 1369 -> 1334).
__global__ __attribute__((amdgpu_flat_work_group_size(256, 256))) void bwd_front_kernel(const BwdParams p, const ItemOrder make,
                                                                                        const PieceMaker pieces) {
  __shared__ int lens[kMostOrdered];
  const int planner = pieces.header != nullptr ? 1 : 0;  // the first block
  const int block = (int)blockIdx.x - planner;
  if (p.queue != nullptr && blockIdx.x == 0 && threadIdx.x < kQueueBytes / 4) p.queue[threadIdx.x] = 0;
  if (block < 0) plan_pieces(p, pieces, lens);
  else if (block < make.blocks) order_items(p, make, block, lens);
  else if (p.make.stats != nullptr) stats_rows(p.make, block - make.blocks, gridDim.x - planner - make.blocks);
}

}  // namespace

hipError_t launch_bwd_stats(const BwdStats& s, hipStream_t stream) {
  if (s.rows <= 0) return hipSuccess;
  hipLaunchKernelGGL(bwd_stats_kernel, dim3(stats_blocks(s)), dim3(256), 0, stream, s);
  return hipGetLastError();
}

// One work-group per compute unit.
void plan_bwd_dkdv(BwdParams& p, const KeyTiles& tiles) {
  p.num_items = p.B * p.Hkv * (p.Skv / tiles.rows);
  const int group = p.Hq / p.Hkv;
  const ListLengths lengths{p.tiled ? nullptr : p.k_cnt, p.mask_bh == 1, tiles.rows, p.k_block, p.nK, group, p.q_block / 32};  // tile lists: the host decides
  p.split = plan_split(p.num_items, 1, group * (p.Sq / 32), StepCost{tiles.step, tiles.step, tiles.step, p.tiled != 0}, tiles.slot_bytes, p.split.ws, p.split_ws_bytes,
                       lengths);
}

namespace {

// A dK/dV launch as it is planned: work-groups, and what has to run in front of it.
struct KeyTileLaunch {
  int grid = 0;
  ItemOrder make{};
  PieceMaker maker{};
};

KeyTileLaunch place_key_tiles(BwdParams& p, const KeyTiles& tiles, bool takes_pieces) {
  KeyTileLaunch launch;
  auto& [grid, make, maker] = launch;
  const int slots = compute_units();
  const int heads = p.B * p.Hkv;
  char* const ws = reinterpret_cast<char*>(p.split.ws);  // whether or not anything is split
  plan_bwd_dkdv(p, tiles);
  plan_xcd_mapping(heads, p.split.first, p.items_per_xcd, p.split.main_wgs);
  const int parts = (p.num_items - p.split.first) * p.split.parts;
  p.queue = nullptr;
  p.order = nullptr;

  // What else lives in the workspace, from its end: the claim counters, then the order of the items.
  int64_t top = ws == nullptr ? 0 : (p.split_ws_bytes - kQueueBytes) & ~(int64_t)15;
  const int64_t bottom = parts * tiles.slot_bytes + kNoteBytes;
  p.results_end = (bottom + 15) & ~(int64_t)15;
  int* const queue = ws != nullptr && top >= bottom ? reinterpret_cast<int*>(ws + top) : nullptr;
  top = (top - (int64_t)p.num_items * 4) & ~(int64_t)15;
  const int64_t order_at = top;
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
  const bool ordered = !p.tiled && queue != nullptr && order_at >= bottom && p.num_items > slots && p.num_items <= std::min(8 * slots, kMostOrdered) &&
                       longest >= (p.split.first + parts >= 4 * slots ? 128 : 192);
  if (ordered) p.split.main_wgs = p.split.first;

  // Room for pieces, where lists can be so long that cutting them pays (plan_pieces) and there are not so many that the longest cannot
  // count.  A launch that needs none pays for work-groups that exit at once, one to a compute unit, and for a merge that finds nothing to do (5 us in
  // a trace): steps with / without pieces in the library, B2 H16/4 S8192 1033 / 1031 us, H8 S8192 290 / 288, H4 S16384 5 % kept 163 / 161, H1 S32768 10 % 268 / 267,
  // H2 S32768 30 % 1276 / 1274.  The planning hides behind the statistics, so a dK/dV kernel called by itself goes without.
  const int most_pieces = p.num_items <= slots ? slots : p.num_items + slots;
  const int64_t piece_bytes = 64 + most_pieces * (int64_t)sizeof(Piece) + slots * (int64_t)sizeof(CutItem);
  top = (top - piece_bytes) & ~(int64_t)63;
  p.pieces = {};
  if (takes_pieces && p.make.stats != nullptr && !p.tiled && queue != nullptr && p.num_items <= kMostOrdered && longest >= (p.num_items > slots ? 256 : 512) && (int64_t)p.num_items * longest < 0x7fffffffLL &&
      top >= std::max(bottom, 2 * slots * tiles.slot_bytes)) {
    maker = {reinterpret_cast<int32_t*>(ws + top), reinterpret_cast<Piece*>(ws + top + 64), reinterpret_cast<CutItem*>(ws + top + 64) + most_pieces, slots,
             2 * slots, most_pieces, p.split.items == p.num_items ? p.split.parts : 1};
    p.pieces = {maker.header, maker.list, maker.cut};
    p.split.ws = reinterpret_cast<float*>(ws);
    // The device may decide against pieces, and then makes the parts that the host has planned: whichever end later.
    p.results_end = std::max(p.results_end, 2 * slots * tiles.slot_bytes);
  }
  p.kept_from = maker.header != nullptr ? top : ordered ? order_at : queue != nullptr ? reinterpret_cast<char*>(queue) - ws : p.split_ws_bytes;

  // Launches of four rounds and more let the work-groups claim their grid indices, with some more work-groups than indices,
  // so that an XCD that is through early takes over from the others (claim_work; either mapping deals grid index i to XCD
  // i % 8, which is all a claim relies on).  FBA_CLAIM_WORK=0 switches claiming off, for measurements.
  p.total_work = p.split.main_wgs + parts;
  if (p.pieces.header != nullptr) p.total_work = std::max(p.total_work, most_pieces);
  grid = p.total_work;
  const char* claim = getenv("FBA_CLAIM_WORK");
  if (queue != nullptr && !(claim != nullptr && claim[0] == '0') && p.split.main_wgs + parts >= 4 * slots) {
    p.queue = queue;
    grid += (p.total_work / 8 + 7) / 8 * 8;  // an eighth more work-groups, a whole number per XCD
  }
  if (ordered) {
    const int tiles_per_head = p.Skv / tiles.rows;
    make.spans = heads >= 8 ? 8 : 1;
    const int two_rounds = 2 * slots / make.spans;
    make.segment = (two_rounds + tiles_per_head - 1) / tiles_per_head * tiles_per_head;
    make.blocks = make.spans * (((p.num_items + make.spans - 1) / make.spans + kRankItems - 1) / kRankItems);
    make.order = reinterpret_cast<int32_t*>(ws + order_at);
    p.order = make.order;
    if (2 * p.split.items <= slots) p.split.look.order = p.order;
  }
  return launch;
}

}  // namespace

hipError_t plan_key_tiles(BwdParams& p, const KeyTiles& tiles, int& grid, hipStream_t stream, bool takes_pieces) {
  const auto [work_groups, make, maker] = place_key_tiles(p, tiles, takes_pieces);
  grid = work_groups;
  const int front = (maker.header != nullptr) + make.blocks + (p.make.stats != nullptr ? stats_blocks(p.make) : p.queue != nullptr ? 1 : 0);
  if (front > 0) hipLaunchKernelGGL(bwd_front_kernel, dim3(front), dim3(kFrontThreads), 0, stream, p, make, maker);
  return hipGetLastError();
}

bool put_behind(SplitPlan& split, int64_t slot_bytes, const Merge& before) {
  if (split.items == 0) return true;
  const int64_t end = before.results_end + split.items * split.parts * slot_bytes + (int64_t)sizeof(int32_t);
  if (end > before.kept_from) return false;
  split.ws += before.results_end / 4;
  split.note += before.results_end / 4;
  return true;
}

SplitRegions plan_split_regions(BwdParams p, bool from_ds) {
  SplitRegions r{0, 0, -1, -1, p.split_ws_bytes};
  float* const ws = p.split.ws;
  BwdParams dq = p;
  const KeyTiles& tiles = p.tiled ? kKeyTiles64 : kKeyTiles128;
  place_key_tiles(p, tiles, /*takes_pieces=*/!p.tiled);
  Merge before;
  if (p.split.items > 0) r.parts_end = p.split.items * p.split.parts * tiles.slot_bytes + (int64_t)sizeof(int32_t);
  if (p.pieces.header != nullptr) r.pieces_end = 2 * compute_units() * tiles.slot_bytes;
  if (r.parts_end > 0 || r.pieces_end > 0) {
    before.wgs = 1;
    before.results_end = p.results_end;
    r.kept_from = before.kept_from = p.kept_from;
  }
  int rows = 128;
  if (from_ds) rows = 32 * plan_bwd_dq_from_ds(dq);
  else plan_bwd_dq(dq);
  const int64_t slot_bytes = rows * kHeadDim * 4;
  if (dq.split.items > 0 && before.wgs > 0 && put_behind(dq.split, slot_bytes, before)) {
    r.dq_from = reinterpret_cast<char*>(dq.split.ws) - reinterpret_cast<char*>(ws);
    r.dq_end = std::max(r.dq_from + dq.split.items * dq.split.parts * slot_bytes, reinterpret_cast<char*>(dq.split.note + 1) - reinterpret_cast<char*>(ws));
  }
  return r;
}

}  // namespace fba
