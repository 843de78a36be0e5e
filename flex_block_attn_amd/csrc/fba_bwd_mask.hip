// Backward straight from the block mask, for problems too small to fill the GPU: no lists, no statistics pass, no dS hand-over, no
// parts, one launch: gfx950, head_dim 128, bf16 in / fp32 accumulate / bf16 out, no atomics.
//
// Work-groups of eight waves in two kinds, side by side in one grid; every wave of both takes every eighth of the selected 32-row
// slabs, brings it in on its own (16 KiB of LDS per wave, no barrier in the loop), and the eight meet in LDS at the end.
//   key tiles: 32 keys of a kv head against the query slabs that select them (all query heads of the group): dV, dK
//     S = Q K^T, dP = dO V^T             A = Q / dO slab rows from LDS, B = K / V rows from LDS (shared by the waves), lane = key
//     dV^T += dO^T P,  dK^T += Q^T dS    A through transposing LDS fetches, B = P / dS packed to bf16
//     delta = rowsum(dO o O) of a slab's rows is formed on the way, O in 16-byte pieces of rows, dO from LDS
//   query tiles: 32 query rows against the key slabs they select: dQ; S and dP are formed again
//     S^T = K Q^T, dP^T = V dO^T         A = K / V slab rows from LDS, B = Q / dO rows in registers, lane = query row
//     dQ^T += K^T dS^T
//
// Like fwd_mask_kernel this is bound by latency: what it replaces is a chain of lists, statistics, dK/dV, merge, dQ, merge, each
// waiting for the one in front, of which the host has to launch every one.  The slab loop has one buffer per operand, whose next
// slab is asked for as soon as the matrix instructions that read it last have their operands.  key_tile needs a few registers more than there are: 4 (14
// with 16-row halves) go to scratch and come back between its two accumulations, behind copies that are on their way.
#include <algorithm>
#include <type_traits>

#include "fba_common.h"
#include "fba_kernels.h"

namespace fba {

namespace {

constexpr int kSlab = 32;
constexpr int kSlabBytes = kSlab * kRowBytes;        // 8 KiB
constexpr int kWaves = 8;
constexpr int kTileBase = kWaves * 2 * kSlabBytes;   // behind the waves' slabs: K rows, V rows of a key tile
constexpr int kStatBase = kTileBase + 2 * kSlabBytes;
constexpr int kStatFloats = 2 * kSlab;               // of a wave: lse * log2(e), -delta
constexpr int kSmemBytes = kStatBase + kWaves * kStatFloats * 4;
constexpr float kLog2e = 1.4426950408889634f;

// The 32-row query slabs of a kv head's query heads, one after the other, that select some key tile.  All lanes of a wave call
// everything together.
template <bool kTwo>
struct ColumnCursor {
  const uint8_t* column;   // mask byte (query block 0, the key tile's block) of the group's first head
  int64_t head_bytes;      // to the next head's (0: one mask for all)
  int nK, q_block, Sq, slabs, total, lane;  // slabs of a head, of all heads
  int base;                         // first of the 64 slabs at hand
  int ahead0, ahead1;               // this lane's mask bytes of the 64 that follow, for the first and the last 16 rows
  unsigned long long m0, m1, left;  // ballots of the 64; those not passed yet, the current one lowest

  FBA_DEVICE void load(int at) {
    ahead0 = ahead1 = 0;
    const int i = at + lane;
    if (i < total) {
      const int g = i / slabs, row = (i - g * slabs) * kSlab;
      const uint8_t* const c = column + g * head_bytes;
      ahead0 = c[(int64_t)(row / q_block) * nK];
      if (kTwo && row + 16 < Sq) ahead1 = c[(int64_t)((row + 16) / q_block) * nK];
    }
  }
  FBA_DEVICE void take() {
    m0 = __builtin_amdgcn_ballot_w64(ahead0 != 0);
    m1 = kTwo ? __builtin_amdgcn_ballot_w64(ahead1 != 0) : m0;
    left = m0 | m1;
    load(base + 64);
  }
  FBA_DEVICE void start() {
    base = 0;
    load(0);
    take();
  }
  // n selected slabs on; false past the last one
  FBA_DEVICE bool skip(int n) {
    for (;;) {
      const int here = __popcll(left);
      if (n < here) {
        for (; n > 0; --n) left &= left - 1;
        return true;
      }
      n -= here;
      base += 64;
      if (base >= total) return false;
      take();
    }
  }
  FBA_DEVICE int slab() const { return base + __builtin_ctzll(left); }
  FBA_DEVICE int halves() const {
    const int b = __builtin_ctzll(left);
    return (int)((m0 >> b) & 1) | (int)((m1 >> b) & 1) << 1;
  }
};

// The compiler knows of no order between the copies and its LDS reads: no read moves up across a fence, and reads of a buffer
// have returned before it is filled again.
FBA_DEVICE void fence() { asm volatile("" ::: "memory"); }
FBA_DEVICE void reads_done() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

FBA_DEVICE float dot8(bf16x8 a, bf16x8 b) {
  float d = 0.f;
#pragma unroll
  for (int t = 0; t < 4; ++t)
    d = __builtin_amdgcn_fdot2_f32_bf16((bf16x2){a[2 * t], a[2 * t + 1]}, (bf16x2){b[2 * t], b[2 * t + 1]}, d, false);
  return d;
}

// Sum over the 16 lanes of a row, in all of them.
FBA_DEVICE float row16_sum(float x) {
  auto turned = [](float y, auto n) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, y), 0x120 + decltype(n)::value, 0xf, 0xf, false));
  };
  x += turned(x, std::integral_constant<int, 8>{});
  x += turned(x, std::integral_constant<int, 4>{});
  x += turned(x, std::integral_constant<int, 2>{});
  x += turned(x, std::integral_constant<int, 1>{});
  return x;
}

// Every wave hands in its 32 x 128 tile (16 KiB in place of its slabs, chunk c of row r at slot c ^ r); thread t stores columns
// 8 (t % 16) .. +7 of row t / 16, if there is one.
FBA_DEVICE void sum_tiles(char* smem, const f32x16 (&acc)[4], float scale, __bf16* out, int rows) {
  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, h = lane >> 5;
  f32x4* dst = reinterpret_cast<f32x4*>(smem + (tid >> 6) * 2 * kSlabBytes) + l32 * 32;
#pragma unroll
  for (int mb = 0; mb < 4; ++mb)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      dst[(8 * mb + 2 * g + h) ^ l32] = (f32x4){acc[mb][4 * g + 0], acc[mb][4 * g + 1], acc[mb][4 * g + 2], acc[mb][4 * g + 3]};
  __syncthreads();
  const int r = tid >> 4, c8 = 2 * (tid & 15);
  f32x4 sum[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
  for (int w = 0; w < kWaves; ++w)
#pragma unroll
    for (int j = 0; j < 2; ++j) sum[j] += reinterpret_cast<const f32x4*>(smem + w * 2 * kSlabBytes)[r * 32 + ((c8 + j) ^ r)];
  if (r < rows)
    *reinterpret_cast<bf16x8*>(out + r * kHeadDim + 4 * c8) =
        pack8(sum[0][0] * scale, sum[0][1] * scale, sum[0][2] * scale, sum[0][3] * scale, sum[1][0] * scale, sum[1][1] * scale, sum[1][2] * scale, sum[1][3] * scale);
}

// What the two kinds of work-groups share: a wave's slab buffers and the copies into them.
struct WaveSlabs {
  char *first, *second;  // Q and dO, or K and V
  uint32_t off[4];       // copy i (0..7) of a slab fills its rows 4 i .. 4 i + 3; the swizzle repeats after 16 rows
  FBA_DEVICE void init(char* smem, int wave, int lane) {
    first = smem + wave * 2 * kSlabBytes;
    second = first + kSlabBytes;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = 4 * i + (lane >> 4);
      off[i] = (uint32_t)(row * kRowBytes + (((lane & 15) ^ swz(row)) << 4));
    }
  }
  // last: bytes from the slab's first row to its last 16
  FBA_DEVICE void copy(char* buf, const char* from, int last = 16 * kRowBytes) const {
    const uint32_t dst = lds_addr(buf);
    // the same in all lanes, which the compiler does not see behind the cursors' loops
    const uint64_t at = reinterpret_cast<uint64_t>(from);
    const char* const src = reinterpret_cast<const char*>((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(at >> 32)) << 32 |
                                                          (uint32_t)__builtin_amdgcn_readfirstlane((int)at));
    last = __builtin_amdgcn_readfirstlane(last);
#pragma unroll
    for (int i = 0; i < 8; ++i) dma16(dst + 4 * i * kRowBytes, src + (i >> 2) * last, off[i & 3]);
  }
};

template <bool kTwo>
FBA_DEVICE void key_tile(const BwdMaskParams& p, int item, char* smem) {
  const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tiles_per_head = p.Skv / kSlab, group = p.Hq / p.Hkv;
  const int bhk = item / tiles_per_head, key0 = (item - bhk * tiles_per_head) * kSlab;
  const int64_t krow0 = (int64_t)bhk * p.Skv + key0, bh0 = (int64_t)bhk * group;

  ColumnCursor<kTwo> cursor;
  cursor.column = p.mask + (p.mask_bh == 1 ? 0 : bh0 * p.nQ * p.nK) + key0 / p.k_block;
  cursor.head_bytes = p.mask_bh == 1 ? 0 : (int64_t)p.nQ * p.nK;
  cursor.nK = p.nK;
  cursor.q_block = p.q_block;
  cursor.Sq = p.Sq;
  cursor.slabs = (p.Sq + kSlab - 1) / kSlab;
  cursor.total = group * cursor.slabs;
  cursor.lane = lane;

  WaveSlabs slabs;
  slabs.init(smem, wave, lane);
  char* const k_lds = smem + kTileBase;
  char* const v_lds = k_lds + kSlabBytes;
  {  // wave w brings in rows 4 w .. 4 w + 3 of K and V
    const int row = 4 * wave + (lane >> 4);
    const uint32_t off = (uint32_t)(row * kRowBytes + (((lane & 15) ^ swz(row)) << 4));
    dma16(lds_addr(k_lds) + wave * 4 * kRowBytes, reinterpret_cast<const char*>(p.k + krow0 * kHeadDim), off);
    dma16(lds_addr(v_lds) + wave * 4 * kRowBytes, reinterpret_cast<const char*>(p.v + krow0 * kHeadDim), off);
  }
  cursor.start();

  RowMajorOffsets rm;
  rm.init(lane);
  TransposedOffsets tr;
  tr.init(lane);
  float* const stat = reinterpret_cast<float*>(smem + kStatBase) + wave * kStatFloats;
  f32x16 acc_k[4], acc_v[4];
#pragma unroll
  for (int mb = 0; mb < 4; ++mb)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc_k[mb][r] = acc_v[mb][r] = 0.f;

  // first query row of the cursor's slab over all heads (of o as well), and the way from it to the last 16 (they may not be there)
  auto first_row = [&](int& last, int64_t& o_row) -> int64_t {
    const int i = cursor.slab(), g = i / cursor.slabs, row = (i - g * cursor.slabs) * kSlab;
    last = kTwo && row + 16 >= p.Sq ? 0 : 16;
    o_row = (bh0 + g) * p.o_rows + row;
    return (bh0 + g) * p.Sq + row;
  };
  bf16x8 o[8];  // rows 4 i + lane / 16, columns 8 (lane % 16) .. +7
  float lse;    // of row lane % 32
  auto request_stats = [&](int64_t row, int64_t o_row, int last) {
    const __bf16* const src = p.o + (o_row + (lane >> 4)) * kHeadDim + (lane & 15) * 8;
#pragma unroll
    for (int i = 0; i < 8; ++i) o[i] = *reinterpret_cast<const bf16x8*>(src + (4 * (i & 3) + (i >> 2) * last) * kHeadDim);
    lse = p.lse[row + (lane & 15) + ((lane >> 4) & 1) * last];
  };

  bool more = cursor.skip(wave);
  int last = 16;
  int64_t row = 0, o_row = 0;
  if (more) {
    row = first_row(last, o_row);
    slabs.copy(slabs.first, reinterpret_cast<const char*>(p.q + row * kHeadDim), last * kRowBytes);
    slabs.copy(slabs.second, reinterpret_cast<const char*>(p.d_o + row * kHeadDim), last * kRowBytes);
    request_stats(row, o_row, last);
  }
  wait_vmem<0>();
  __syncthreads();  // K and V are there
  while (more) {
    const int halves = cursor.halves();
    const bool on0 = !kTwo || (halves & 1) != 0, on1 = !kTwo || (halves & 2) != 0;
    more = cursor.skip(kWaves);
    if (more) row = first_row(last, o_row);
    wait_vmem<0>();
    fence();
    // -delta and lse of the slab's rows
    float minus_delta = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float d = row16_sum(dot8(o[i], lds_read_b128(slabs.second, tile_off(4 * i + (lane >> 4), lane & 15))));
      minus_delta = (lane & 15) == i ? -d : minus_delta;
    }
    if (lane < 32) stat[lane] = lse * kLog2e;
    if ((lane & 15) < 8) stat[kSlab + 4 * (lane & 15) + (lane >> 4)] = minus_delta;
    fence();
    // accumulator element 4g + e of half-wave h is query row 8g + 4h + e of the slab
    f32x16 s, dp;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const f32x4 d4 = *reinterpret_cast<const f32x4*>(stat + kSlab + 8 * g + 4 * h);
#pragma unroll
      for (int e = 0; e < 4; ++e) { s[4 * g + e] = 0.f; dp[4 * g + e] = d4[e]; }
    }
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
      s = mfma32(lds_read_b128(slabs.first, rm.rd[ks]), lds_read_b128(k_lds, rm.rd[ks]), s);
      dp = mfma32(lds_read_b128(slabs.second, rm.rd[ks]), lds_read_b128(v_lds, rm.rd[ks]), dp);
    }
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const f32x4 l4 = *reinterpret_cast<const f32x4*>(stat + 8 * g + 4 * h);
      const bool on = g < 2 ? on0 : on1;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float pv = fast_exp2(__builtin_fmaf(s[4 * g + e], p.scale_log2e, -l4[e]));
        const float ds = pv * dp[4 * g + e];
        s[4 * g + e] = on ? pv : 0.f;  // selects: inf or NaN of a masked row's P and dS is discarded (not of its Q and dO, which meet these zeros)
        dp[4 * g + e] = on ? ds : 0.f;
      }
    }
    bf16x8 pk[2], dsk[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      pk[j] = pack8(s[8 * j + 0], s[8 * j + 1], s[8 * j + 2], s[8 * j + 3], s[8 * j + 4], s[8 * j + 5], s[8 * j + 6], s[8 * j + 7]);
      dsk[j] = pack8(dp[8 * j + 0], dp[8 * j + 1], dp[8 * j + 2], dp[8 * j + 3], dp[8 * j + 4], dp[8 * j + 5], dp[8 * j + 6], dp[8 * j + 7]);
    }
    auto add = [&](f32x16(&acc)[4], const char* buf, const bf16x8(&b)[2]) {
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int mb = 0; mb < 4; ++mb) {
          const int roff = 16 * j * kRowBytes;
          acc[mb] = mfma32(cat(lds_read_tr(buf, tr.rd[mb][0] + roff), lds_read_tr(buf, tr.rd[mb][1] + roff)), b[j], acc[mb]);
        }
#pragma unroll
      for (int mb = 0; mb < 4; ++mb) pin(acc[mb]);
    };
    add(acc_v, slabs.second, pk);
    reads_done();
    if (more) {
      slabs.copy(slabs.second, reinterpret_cast<const char*>(p.d_o + row * kHeadDim), last * kRowBytes);
      request_stats(row, o_row, last);
    }
    add(acc_k, slabs.first, dsk);
    reads_done();
    if (more) slabs.copy(slabs.first, reinterpret_cast<const char*>(p.q + row * kHeadDim), last * kRowBytes);
  }
  sum_tiles(smem, acc_v, 1.f, p.dv + krow0 * kHeadDim, kSlab);
  __syncthreads();
  sum_tiles(smem, acc_k, p.scale, p.dk + krow0 * kHeadDim, kSlab);
}

template <bool kTwo>
FBA_DEVICE void query_tile(const BwdMaskParams& p, int item, char* smem) {
  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tiles_per_head = (p.Sq + kSlab - 1) / kSlab;
  const int bh = item / tiles_per_head;
  const int row0 = (item - bh * tiles_per_head) * kSlab;
  const int64_t qrow0 = (int64_t)bh * p.Sq + row0;
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

  WaveSlabs slabs;
  slabs.init(smem, wave, lane);
  // Q and dO as B operands: lane holds row l32 (rows past the end: copies of the last one, not stored), d = 16 ks + 8 h .. +7
  bf16x8 qreg[8], doreg[8];
  float minus_delta, lse2;
  {
    const int64_t my_row = (int64_t)bh * p.Sq + min(row0 + l32, p.Sq - 1);
    const int64_t at = my_row * kHeadDim + 8 * h;
    const int64_t o_at = ((int64_t)bh * p.o_rows + min(row0 + l32, p.Sq - 1)) * kHeadDim + 8 * h;
    bf16x8 o[8];
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
      qreg[ks] = *reinterpret_cast<const bf16x8*>(p.q + at + 16 * ks);
      doreg[ks] = *reinterpret_cast<const bf16x8*>(p.d_o + at + 16 * ks);
      o[ks] = *reinterpret_cast<const bf16x8*>(p.o + o_at + 16 * ks);
    }
    lse2 = p.lse[my_row] * kLog2e;
    float d = 0.f;
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) d += dot8(doreg[ks], o[ks]);
    minus_delta = -sum_halves(d);
  }
  RowMajorOffsets rm;
  rm.init(lane);
  TransposedOffsets tr;
  tr.init(lane);
  f32x16 acc[4];
#pragma unroll
  for (int mb = 0; mb < 4; ++mb)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[mb][r] = 0.f;

  bool more = cursor.skip(wave);
  if (more) {
    const int64_t off = (int64_t)cursor.slab() * kSlabBytes;
    slabs.copy(slabs.second, vp + off);
    slabs.copy(slabs.first, kp + off);
  }
  while (more) {
    const int halves = cursor.halves();
    more = cursor.skip(kWaves);
    const int64_t off = more ? (int64_t)cursor.slab() * kSlabBytes : 0;
    const bool active = !kTwo || ((halves >> (l32 >> 4)) & 1) != 0;
    wait_vmem<0>();
    fence();
    f32x16 s, dp;
#pragma unroll
    for (int r = 0; r < 16; ++r) { s[r] = 0.f; dp[r] = minus_delta; }
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
      dp = mfma32(lds_read_b128(slabs.second, rm.rd[ks]), doreg[ks], dp);
      s = mfma32(lds_read_b128(slabs.first, rm.rd[ks]), qreg[ks], s);
    }
    pin(s);
    pin(dp);
    reads_done();
    if (more) slabs.copy(slabs.second, vp + off);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float ds = fast_exp2(__builtin_fmaf(s[r], p.scale_log2e, -lse2)) * dp[r];
      dp[r] = active ? ds : 0.f;  // a select: inf or NaN of a masked row's P and dS is discarded (not of the keys it does not select)
    }
    bf16x8 dsk[2];
#pragma unroll
    for (int j = 0; j < 2; ++j)
      dsk[j] = pack8(dp[8 * j + 0], dp[8 * j + 1], dp[8 * j + 2], dp[8 * j + 3], dp[8 * j + 4], dp[8 * j + 5], dp[8 * j + 6], dp[8 * j + 7]);
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int mb = 0; mb < 4; ++mb) {
        const int roff = 16 * j * kRowBytes;
        acc[mb] = mfma32(cat(lds_read_tr(slabs.first, tr.rd[mb][0] + roff), lds_read_tr(slabs.first, tr.rd[mb][1] + roff)), dsk[j], acc[mb]);
      }
#pragma unroll
    for (int mb = 0; mb < 4; ++mb) pin(acc[mb]);
    reads_done();
    if (more) slabs.copy(slabs.first, kp + off);
  }
  sum_tiles(smem, acc, p.scale, p.dq + qrow0 * kHeadDim, p.Sq - row0);
}

}  // namespace

template <bool kTwo>  // q_block is an odd multiple of 16: the two 16-row halves of a slab have mask rows of their own
__global__ __attribute__((amdgpu_flat_work_group_size(64 * kWaves, 64 * kWaves), amdgpu_waves_per_eu(2, 2))) void bwd_mask_kernel(const BwdMaskParams p) {
  extern __shared__ __attribute__((aligned(16))) char smem[];  // [wave](Q | dO or K | V slab), K rows, V rows, statistics
  if ((int)blockIdx.x < p.key_wgs) {
    const int item = xcd_remap(blockIdx.x, p.key_per_xcd);
    if (item < p.key_items) key_tile<kTwo>(p, item, smem);
  } else {
    const int item = xcd_remap(blockIdx.x - p.key_wgs, p.query_per_xcd);
    if (item < p.query_items) query_tile<kTwo>(p, item, smem);
  }
}

// Is a problem small enough for bwd_mask_kernel?  A round of work-groups takes 14 us and 0.33 us for every listed slab (S2048, 90 % kept:
// 35 us of backward; H2 S4096 102 us, in two rounds, against 81 on lists).  Whole steps as replayed graphs, lists / mask, 128-token blocks unless noted, 10, 40
// and 90 % kept: H1 S768 51 / 23, 53 / 30, 55 / 30 us; H2 S1536, 384-token blocks 68 / 34, 74 / 39, 72 / 42; H3 S1728, 192-token blocks 74 / 37,
// 87 / 48, 91 / 57; H4 S2048 70 / 44, 82 / 56, 90 / 74; H8/2 S1024 61 / 36, 68 / 48, 75 / 68; H1 S4096, 128 slabs, 71 / 37, 81 / 56, 96 / 78.
// So the line is drawn at 160 slabs in a round, which is where 90 % kept would lose and half of it still gains.
bool bwd_takes_mask(int64_t heads, int64_t kv_heads, int64_t q_len, int64_t kv_len) {
  if (heads <= 0 || kv_heads <= 0) return false;
  const int64_t key_slabs = heads / kv_heads * ((q_len + kSlab - 1) / kSlab), query_slabs = kv_len / kSlab;  // of a tile, at most
  const int64_t key_tiles = kv_heads * (kv_len / kSlab), query_tiles = heads * ((q_len + kSlab - 1) / kSlab);
  const int64_t units = device_compute_units();
  return key_tiles + query_tiles <= 2 * units && std::max(key_slabs, query_slabs) <= 160 && key_tiles * key_slabs + query_tiles * query_slabs <= 160 * units;
}

hipError_t launch_bwd_mask(BwdMaskParams p, hipStream_t stream) {
  void (*fn)(const BwdMaskParams) = p.q_block % 32 != 0 ? &bwd_mask_kernel<true> : &bwd_mask_kernel<false>;
  p.key_items = p.B * p.Hkv * (p.Skv / kSlab);
  p.query_items = p.B * p.Hq * ((p.Sq + kSlab - 1) / kSlab);
  int query_wgs;
  plan_xcd_mapping(p.B * p.Hkv, p.key_items, p.key_per_xcd, p.key_wgs);
  plan_xcd_mapping(p.B * p.Hq, p.query_items, p.query_per_xcd, query_wgs);
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, kSmemBytes);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(fn, dim3(p.key_wgs + query_wgs), dim3(64 * kWaves), kSmemBytes, stream, p);
  return hipGetLastError();
}

}  // namespace fba
