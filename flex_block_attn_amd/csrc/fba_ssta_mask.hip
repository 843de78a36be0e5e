// Score-driven block masks ("SSTA" style): every query block attends to a diagonal band of key blocks, to the first key
// blocks of the sequence, and to the top-k key blocks ranked by <mean of the query block's rows, mean of the key block's
// rows>.  Three HBM-bound kernels: block means of Q and K, then scores + top-k + union into the bool block mask the
// compaction kernel consumes, and the (un)permutation of a video latent grid into contiguous tiles.
#include "fba_common.h"
#include "fba_kernels.h"

namespace fba {

namespace {

constexpr int kD = 128;

__device__ __forceinline__ float bf16_lo(uint32_t u) { return __uint_as_float(u << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t u) { return __uint_as_float(u & 0xffff0000u); }

// out[g, :] = mean over rows [g*block, (g+1)*block) of x, x [n_blocks*block, 128] bf16, out fp32; of one tensor or two (q and k of a mask
// in one launch).  One work-group per block: 16 lanes cover one 256-byte row, the 16 row groups of the work-group stride through the
// block, then add up through LDS in a fixed order (the result does not depend on scheduling).
struct MeanJobs {
  const __bf16* x[2];
  float* out[2];
  int block[2];
  float inv_block[2];
  unsigned second;  // first block of the second tensor (past the end: there is none)
};
__global__ __attribute__((amdgpu_flat_work_group_size(256, 256))) void block_mean_kernel(const MeanJobs jobs) {
  __shared__ float red[16][kD + 4];
  const int tid = threadIdx.x, c = tid & 15, r0 = tid >> 4;
  const int which = blockIdx.x >= jobs.second ? 1 : 0, block = jobs.block[which];
  const unsigned g0 = blockIdx.x - (which ? jobs.second : 0);
  const uint4* src = reinterpret_cast<const uint4*>(jobs.x[which] + (size_t)g0 * block * kD);
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  int r = r0;
  for (; r + 48 < block; r += 64) {
    uint4 u[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) u[i] = src[(size_t)(r + 16 * i) * 16 + c];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      acc[0] += bf16_lo(u[i].x); acc[1] += bf16_hi(u[i].x); acc[2] += bf16_lo(u[i].y); acc[3] += bf16_hi(u[i].y);
      acc[4] += bf16_lo(u[i].z); acc[5] += bf16_hi(u[i].z); acc[6] += bf16_lo(u[i].w); acc[7] += bf16_hi(u[i].w);
    }
  }
  for (; r < block; r += 16) {
    const uint4 u = src[(size_t)r * 16 + c];
    acc[0] += bf16_lo(u.x); acc[1] += bf16_hi(u.x); acc[2] += bf16_lo(u.y); acc[3] += bf16_hi(u.y);
    acc[4] += bf16_lo(u.z); acc[5] += bf16_hi(u.z); acc[6] += bf16_lo(u.w); acc[7] += bf16_hi(u.w);
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) red[r0][c * 8 + e] = acc[e];
  __syncthreads();
  if (tid < kD) {
    float s = 0.f;
#pragma unroll
    for (int g = 0; g < 16; ++g) s += red[g][tid];
    jobs.out[which][(size_t)g0 * kD + tid] = s * jobs.inv_block[which];
  }
}

constexpr int kQPerWave = 2;
constexpr int kQPerGroup = 8;       // query blocks per work-group (4 waves x 2)
constexpr int kChunk = 64;          // key blocks per LDS chunk: one per lane
constexpr int kMostChunks = 64;     // nK <= 4096
constexpr int kRowStride = kD + 4;  // floats; 16 lanes read 16 bytes of a row each from 64 different banks

// Four floats of a mean.  Callers hand in means at the address of any float, and so much alignment is all that the loads may be told of.
typedef f32x4 f32x4_any __attribute__((aligned(4)));

// A score as an unsigned number in the same order; 0 for what is never picked (NaN, -inf, no key block).  -0 becomes +0 as an integer:
// -ffast-math knows no signed zeros and would drop an addition of +0.
__device__ __forceinline__ uint32_t rank_key(float x) {
  const uint32_t bits = __float_as_uint(x), u = bits == 0x80000000u ? 0u : bits;
  return x > -__builtin_inff() ? u ^ ((uint32_t)((int32_t)u >> 31) | 0x80000000u) : 0u;
}

// mask[bh, i, j] = (j among the topk largest <q_mean[bh,i], k_mean[kv(bh),j]>, ties to the lower j)
//                  || |j - (i*q_block)/k_block| <= band || j < sink || base[i, j]   (base: optional [nQ, nK] mask)
//                  || j in the sliding window of i (window: optional, blocks as tiles of a 3-D grid, see TileWindow).
// A wave ranks two query blocks; lane l holds the scores of key blocks l, l+64, ... (kMaxChunks of them) in registers: 128 of them with 64 chunks, and
// no more than 256 registers altogether, so that two waves share a SIMD.  (In scratch, where HIP's float4 kept the compiler from unrolling the
// chunks, and with one wave to a SIMD: see the last two figures.)
//
// Bound by latency.  The k-th largest score is found bit by bit, from how many scores reach a candidate (a ballot and a population count per
// 64 of them), both query blocks side by side; picking the largest topk times over, with a maximum over the wave each time, took
// most of the time.  Key means come in as 16 bytes a lane, a chunk ahead.  Before / now, launch included: 189 x 63 blocks, top-12, 28.8 / 9.9 us;
// 24 heads of 540 x 180, top-16, 106 / 39; 8 of 300 x 300 60 / 31; 50 x 1000, top-40, 154 / 58; 30 x 2000, top-5, 194 / 163 (182 in scratch, 160 with one
// wave); 8 heads of 1000 x 4000, top-16, 1370 / 533 (605, 925).
template <int kMaxChunks>
__global__ __attribute__((amdgpu_flat_work_group_size(256, 256), amdgpu_waves_per_eu(kMaxChunks > 16 ? 2 : 1))) void ssta_mask_kernel(
    const float* __restrict__ q_mean, const float* __restrict__ k_mean, const uint8_t* __restrict__ base,
    uint8_t* __restrict__ mask, int Hq, int Hkv, int nQ, int nK, int q_block, int k_block, int topk, int band, int sink, const TileWindow window) {
  __shared__ __attribute__((aligned(16))) float k_lds[kChunk * kRowStride];
  __shared__ __attribute__((aligned(16))) float q_lds[kQPerGroup * kD];
  constexpr int kLoads = kChunk * kD / 4 / 256;  // of 16 bytes, per thread and chunk
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t bh = blockIdx.y;
  const int64_t kv_seq = (bh / Hq) * Hkv + (bh % Hq) / (Hq / Hkv);
  const int i0 = blockIdx.x * kQPerGroup;
  const int n_chunks = (nK + kChunk - 1) / kChunk;
  const f32x4_any* const k_rows = reinterpret_cast<const f32x4_any*>(k_mean) + kv_seq * nK * (kD / 4);
  f32x4 ahead[kLoads];
  auto load = [&](int chunk) {
#pragma unroll
    for (int x = 0; x < kLoads; ++x) {
      const int j = chunk * kChunk + (tid >> 5) + 8 * x;
      ahead[x] = j < nK ? (f32x4)k_rows[(size_t)j * (kD / 4) + (tid & 31)] : (f32x4){0.f, 0.f, 0.f, 0.f};
    }
  };
  load(0);
  {
    const int i = i0 + (tid >> 5);
    reinterpret_cast<f32x4*>(q_lds)[tid] =
        i < nQ ? (f32x4)reinterpret_cast<const f32x4_any*>(q_mean)[((size_t)bh * nQ + i) * (kD / 4) + (tid & 31)] : (f32x4){0.f, 0.f, 0.f, 0.f};
  }
  uint32_t key[kQPerWave][kMaxChunks];
#pragma unroll
  for (int t = 0; t < kMaxChunks; ++t) {
    key[0][t] = key[1][t] = 0;
    if (t < n_chunks) {  // uniform over the work-group
      __syncthreads();
#pragma unroll
      for (int x = 0; x < kLoads; ++x) *reinterpret_cast<f32x4*>(k_lds + ((tid >> 5) + 8 * x) * kRowStride + 4 * (tid & 31)) = ahead[x];
      __syncthreads();
      if (t + 1 < n_chunks) load(t + 1);
      float s0 = 0.f, s1 = 0.f;
      const f32x4* kr = reinterpret_cast<const f32x4*>(k_lds + lane * kRowStride);
      const f32x4* q0 = reinterpret_cast<const f32x4*>(q_lds + (wave * kQPerWave) * kD);
#pragma unroll 8
      for (int d = 0; d < kD / 4; ++d) {
        const f32x4 kv = kr[d], a = q0[d], b = q0[kD / 4 + d];
        s0 = __builtin_fmaf(a.x, kv.x, s0); s1 = __builtin_fmaf(b.x, kv.x, s1);
        s0 = __builtin_fmaf(a.y, kv.y, s0); s1 = __builtin_fmaf(b.y, kv.y, s1);
        s0 = __builtin_fmaf(a.z, kv.z, s0); s1 = __builtin_fmaf(b.z, kv.z, s1);
        s0 = __builtin_fmaf(a.w, kv.w, s0); s1 = __builtin_fmaf(b.w, kv.w, s1);
      }
      if (t * kChunk + lane < nK) {
        key[0][t] = rank_key(s0);
        key[1][t] = rank_key(s1);
      }
    }
  }
  // how many keys of a query block reach `least`, over the wave
  auto reach = [&](int qq, uint32_t least) {
    int n = 0;
#pragma unroll
    for (int t = 0; t < kMaxChunks; ++t)
      if (t < n_chunks) n += __popcll(__builtin_amdgcn_ballot_w64(key[qq][t] >= least));
    return n;
  };
  uint32_t line[kQPerWave];  // the topk-th largest key, or one that exactly topk keys reach
  int above[kQPerWave];      // keys beyond it, where it is the topk-th largest and keys equal to it have to be picked from; -1: all that reach it
  bool open[kQPerWave];
#pragma unroll
  for (int qq = 0; qq < kQPerWave; ++qq) {
    open[qq] = topk > 0 && reach(qq, 1u) > topk;
    line[qq] = topk <= 0 ? 0xffffffffu : open[qq] ? 0u : 1u;  // (no key is all ones: that would be a NaN)
    above[qq] = -1;
  }
  for (int bit = 31; bit >= 0 && (open[0] || open[1]); --bit) {
#pragma unroll
    for (int qq = 0; qq < kQPerWave; ++qq) {
      const uint32_t least = line[qq] | 1u << bit;
      const int n = open[qq] ? reach(qq, least) : 0;
      if (n >= topk) line[qq] = least;
      if (n == topk) open[qq] = false;
    }
  }
#pragma unroll
  for (int qq = 0; qq < kQPerWave; ++qq)
    if (open[qq]) above[qq] = reach(qq, line[qq] + 1);

#pragma unroll
  for (int qq = 0; qq < kQPerWave; ++qq) {
    const int i = i0 + wave * kQPerWave + qq;
    if (i >= nQ) break;  // uniform over the wave
    uint64_t sel = 0;
    int room = above[qq] < 0 ? 0x7fffffff : topk - above[qq];  // for keys on the line, those of lower j first
#pragma unroll
    for (int t = 0; t < kMaxChunks; ++t)
      if (t < n_chunks) {
        const bool on = key[qq][t] == line[qq];
        const unsigned long long tie = __builtin_amdgcn_ballot_w64(on);
        const int rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(tie >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)tie, 0));
        if (key[qq][t] > line[qq] || (on && rank < room)) sel |= 1ull << t;
        room -= above[qq] < 0 ? 0 : __popcll(tie);
      }
    const int diag = (int)(((int64_t)i * q_block) / k_block);
    uint8_t* row = mask + (size_t)(bh * nQ + i) * nK;
#pragma unroll
    for (int t = 0; t < kMaxChunks; ++t) {
      const int j = t * kChunk + lane;
      if (j < nK) {
        const int dist = j > diag ? j - diag : diag - j;
        const uint32_t keep = base ? (base[(size_t)i * nK + j] != 0) : window.n[0] > 0 ? window.holds(i, j) : 0u;
        row[j] = (uint8_t)((uint32_t)((sel >> t) & 1u) | (dist <= band) | (j < sink) | keep);
      }
    }
  }
}

// Token rows of up to three tensors between raster and tile order (see tile_permute_kernel), a work-group per tile, and on the way to
// tiles the mean of every tile's rows, in the order in which block_mean_kernel adds them up.  Where a row lies in the grid is worked
// out once per row of a tile and kept in LDS.  Bound by memory like the single steps, which read q and k a second time for their
// means and are a launch each: q, k, v and two means, H24 S69120 3 x 163 + 2 x 89 -> 488 us (5.2 TB/s).  With the window worked out in
// ssta_mask_kernel instead of on the host, H1 S1536 162 -> 64 us a call, H3 S15360 340 -> 287, H24 S69120 13.38 -> 13.15 ms.
constexpr int kMostTileRows = 2048;
struct GatherJobs {
  const uint4* src[3];
  uint4* dst[3];
  float* mean[3];      // null: not wanted
  unsigned first[3];   // first block of each tensor
};
template <bool kToTiles>
__global__ __attribute__((amdgpu_flat_work_group_size(256, 256))) void tile_gather_kernel(const GatherJobs jobs, int T, int H, int W, int tT, int tH, int tW,
                                                                                          float inv_rows) {
  __shared__ int offs[kMostTileRows];  // of a tile's rows from its first one, in raster order
  __shared__ float red[16][kD + 4];
  const int tid = threadIdx.x, c = tid & 15, r0 = tid >> 4;
  const int j = blockIdx.x >= jobs.first[2] ? 2 : blockIdx.x >= jobs.first[1] ? 1 : 0;
  const int tile_sz = tT * tH * tW, nH = H / tH, nW = W / tW;
  const int64_t block = blockIdx.x - jobs.first[j];  // tiles of all sequences in tile order
  const int tiles = T / tT * nH * nW;
  const int64_t seq = block / tiles;
  const int tile = (int)(block - seq * tiles);
  const int bt = tile / (nH * nW), bh = (tile / nW) % nH, bw = tile % nW;
  for (int in = tid; in < tile_sz; in += 256) {
    const int it = in / (tH * tW), rest = in - it * (tH * tW), ih = rest / tW;
    offs[in] = (it * H + ih) * W + rest - ih * tW;
  }
  __syncthreads();
  const int64_t raster0 = (seq * T * H * W + ((int64_t)bt * tT * H + bh * tH) * W + bw * tW) * 16 + c, tile0 = block * tile_sz * 16 + c;
  const uint4* const src = jobs.src[j] + (kToTiles ? raster0 : tile0);
  uint4* const dst = jobs.dst[j] + (kToTiles ? tile0 : raster0);
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  auto add = [&](const uint4& u) {
    acc[0] += bf16_lo(u.x); acc[1] += bf16_hi(u.x); acc[2] += bf16_lo(u.y); acc[3] += bf16_hi(u.y);
    acc[4] += bf16_lo(u.z); acc[5] += bf16_hi(u.z); acc[6] += bf16_lo(u.w); acc[7] += bf16_hi(u.w);
  };
  auto at = [&](int r, bool raster) { return (int64_t)(raster ? offs[r] : r) * 16; };
  int r = r0;
  for (; r + 48 < tile_sz; r += 64) {
    uint4 u[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) u[i] = src[at(r + 16 * i, kToTiles)];
#pragma unroll
    for (int i = 0; i < 4; ++i) dst[at(r + 16 * i, !kToTiles)] = u[i];
    if constexpr (kToTiles) {
#pragma unroll
      for (int i = 0; i < 4; ++i) add(u[i]);
    }
  }
  for (; r < tile_sz; r += 16) {
    const uint4 u = src[at(r, kToTiles)];
    dst[at(r, !kToTiles)] = u;
    if constexpr (kToTiles) add(u);
  }
  if (!kToTiles || jobs.mean[j] == nullptr) return;
#pragma unroll
  for (int e = 0; e < 8; ++e) red[r0][c * 8 + e] = acc[e];
  __syncthreads();
  if (tid < kD) {
    float s = 0.f;
#pragma unroll
    for (int g = 0; g < 16; ++g) s += red[g][tid];
    jobs.mean[j][block * kD + tid] = s * inv_rows;
  }
}

// Gather of 256-byte token rows between the raster order of a (T, H, W) grid and tile order, in which the tT x tH x tW
// tokens of one tile are consecutive (tiles in raster order of the tile grid, tokens in raster order inside the tile).
// to_tiles = 1: out[tile order] = x[raster order]; 0: the inverse.  16 lanes move one row.
__global__ __attribute__((amdgpu_flat_work_group_size(256, 256))) void tile_permute_kernel(
    const uint4* __restrict__ x, uint4* __restrict__ out, int64_t n_seq, int T, int H, int W, int tT, int tH, int tW,
    int to_tiles) {
  const int64_t S = (int64_t)T * H * W;
  const int64_t row = (int64_t)blockIdx.x * 16 + (threadIdx.x >> 4);
  if (row >= n_seq * S) return;
  const int c = threadIdx.x & 15;
  const int64_t seq = row / S;
  int64_t p = row - seq * S;  // position in tile order
  const int tile_sz = tT * tH * tW, nH = H / tH, nW = W / tW;
  const int tile = (int)(p / tile_sz), in = (int)(p - (int64_t)tile * tile_sz);
  const int bt = tile / (nH * nW), bh = (tile / nW) % nH, bw = tile % nW;
  const int it = in / (tH * tW), ih = (in / tW) % tH, iw = in % tW;
  const int64_t raster = ((int64_t)(bt * tT + it) * H + (bh * tH + ih)) * W + (bw * tW + iw);
  const int64_t a = (seq * S + raster) * 16 + c, b = row * 16 + c;
  if (to_tiles) out[b] = x[a];
  else out[a] = x[b];
}

// Rows for sequences that are no whole number of 128-row tiles: dst[s, r] = src[s, r] where both have row r, zeros in the rows
// dst has more, for up to three tensors of 256-byte rows in one launch (q, k, v on the way in; their gradients on the way out).
// 16 lanes move a row, every thread four rows.  Bound by memory and launches: one launch in place of a fill and a copy per tensor.  B2
// H8/2 S3136 -> 3200, q16 k64: forward + backward 289 -> 269 us, first pass on new inputs 413 -> 309 us.
struct ResizeJobs {
  const uint4* src[3];
  uint4* dst[3];
  int64_t rows[3];       // of dst, over all sequences
  int src_len[3], dst_len[3];
  unsigned first[3];     // first block of each tensor
};
__global__ __attribute__((amdgpu_flat_work_group_size(256, 256))) void resize_rows_kernel(const ResizeJobs jobs) {
  const int j = blockIdx.x >= jobs.first[2] ? 2 : blockIdx.x >= jobs.first[1] ? 1 : 0;
  const int c = threadIdx.x & 15;
  const int64_t row0 = (int64_t)(blockIdx.x - jobs.first[j]) * 64 + (threadIdx.x >> 4);
  uint4 v[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int64_t row = row0 + 16 * i, seq = row / jobs.dst_len[j], r = row - seq * jobs.dst_len[j];
    v[i] = row < jobs.rows[j] && r < jobs.src_len[j] ? jobs.src[j][(seq * jobs.src_len[j] + r) * 16 + c] : make_uint4(0, 0, 0, 0);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (row0 + 16 * i < jobs.rows[j]) jobs.dst[j][(row0 + 16 * i) * 16 + c] = v[i];
}

// The mask that goes with them: dst [M, dst_q, dst_k], zero where src [M, src_q, src_k] has no block.
__global__ __attribute__((amdgpu_flat_work_group_size(256, 256))) void resize_mask_kernel(const uint8_t* __restrict__ src, uint8_t* __restrict__ dst, int64_t n,
                                                                                          int src_q, int src_k, int dst_q, int dst_k) {
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (t >= n) return;
  const int64_t row = t / dst_k, m = row / dst_q;
  const int j = (int)(t - row * dst_k), i = (int)(row - m * dst_q);
  dst[t] = i < src_q && j < src_k ? src[(m * src_q + i) * src_k + j] : 0;
}

}  // namespace

hipError_t launch_resize_rows(int n, const void* const* src, void* const* dst, const int64_t* n_seq, const int32_t* src_len, const int32_t* dst_len,
                              hipStream_t stream) {
  ResizeJobs jobs{};
  int64_t blocks = 0;
  for (int j = 0; j < 3; ++j) {
    jobs.first[j] = (unsigned)blocks;  // a tensor that is not there starts behind the grid's last block
    if (j >= n) continue;
    jobs.src[j] = static_cast<const uint4*>(src[j]);
    jobs.dst[j] = static_cast<uint4*>(dst[j]);
    jobs.src_len[j] = src_len[j];
    jobs.dst_len[j] = dst_len[j];
    jobs.rows[j] = n_seq[j] * dst_len[j];
    blocks += (jobs.rows[j] + 63) / 64;
    if (blocks > 0x7fffffffLL) return hipErrorInvalidValue;
  }
  if (blocks == 0) return hipSuccess;
  hipLaunchKernelGGL(resize_rows_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, jobs);
  return hipGetLastError();
}

hipError_t launch_resize_mask(const uint8_t* src, uint8_t* dst, int64_t M, int src_q, int src_k, int dst_q, int dst_k, hipStream_t stream) {
  const int64_t n = M * dst_q * dst_k, blocks = (n + 255) / 256;
  if (blocks <= 0) return hipSuccess;
  if (blocks > 0x7fffffffLL) return hipErrorInvalidValue;
  hipLaunchKernelGGL(resize_mask_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, src, dst, n, src_q, src_k, dst_q, dst_k);
  return hipGetLastError();
}

hipError_t launch_block_mean(const BlockMeans (&of)[2], hipStream_t stream) {
  const int64_t n = of[0].n_blocks + of[1].n_blocks;
  if (n <= 0) return hipSuccess;
  if (n > 0x7fffffffLL) return hipErrorInvalidValue;
  MeanJobs jobs{};
  for (int i = 0; i < 2; ++i) {
    jobs.x[i] = of[i].x;
    jobs.out[i] = of[i].out;
    jobs.block[i] = of[i].block;
    jobs.inv_block[i] = 1.0f / (float)of[i].block;
  }
  jobs.second = (unsigned)of[0].n_blocks;
  hipLaunchKernelGGL(block_mean_kernel, dim3((unsigned)n), dim3(256), 0, stream, jobs);
  return hipGetLastError();
}

hipError_t launch_ssta_mask(const float* q_mean, const float* k_mean, const uint8_t* base, uint8_t* mask, int64_t BH, int Hq, int Hkv, int nQ,
                            int nK, int q_block, int k_block, int topk, int band, int sink, const TileWindow& window, hipStream_t stream) {
  if (BH <= 0 || BH > 65535 || nK > kChunk * kMostChunks) return hipErrorInvalidValue;
  // score registers per lane and query block: 256, 1024 or 4096 key blocks
  void (*fn)(const float*, const float*, const uint8_t*, uint8_t*, int, int, int, int, int, int, int, int, int, const TileWindow) =
      nK <= kChunk * 4 ? &ssta_mask_kernel<4> : nK <= kChunk * 16 ? &ssta_mask_kernel<16> : &ssta_mask_kernel<kMostChunks>;
  hipLaunchKernelGGL(fn, dim3((unsigned)((nQ + kQPerGroup - 1) / kQPerGroup), (unsigned)BH), dim3(256), 0,
                     stream, q_mean, k_mean, base, mask, Hq, Hkv, nQ, nK, q_block, k_block, topk, band, sink, window);
  return hipGetLastError();
}

hipError_t launch_tile_gather(int n, const void* const* x, void* const* out, float* const* mean, const int64_t* n_seq, int T, int H, int W, int tT,
                              int tH, int tW, int to_tiles, hipStream_t stream) {
  const int64_t tile_sz = (int64_t)tT * tH * tW, tiles = (int64_t)(T / tT) * (H / tH) * (W / tW);
  // tiles of a few rows would leave most of a work-group idle, large ones do not fit the table
  if (tile_sz < 64 || tile_sz > kMostTileRows) {
    for (int j = 0; j < n; ++j) {
      hipError_t e = launch_tile_permute(x[j], out[j], n_seq[j], T, H, W, tT, tH, tW, to_tiles, stream);
      if (e == hipSuccess && to_tiles && mean[j] != nullptr) e = launch_block_mean({{(const __bf16*)out[j], mean[j], n_seq[j] * tiles, (int)tile_sz}, {}}, stream);
      if (e != hipSuccess) return e;
    }
    return hipSuccess;
  }
  GatherJobs jobs{};
  int64_t blocks = 0;
  for (int j = 0; j < 3; ++j) {
    jobs.first[j] = (unsigned)blocks;  // a tensor that is not there starts behind the grid's last block
    if (j >= n) continue;
    jobs.src[j] = static_cast<const uint4*>(x[j]);
    jobs.dst[j] = static_cast<uint4*>(out[j]);
    jobs.mean[j] = to_tiles ? mean[j] : nullptr;
    blocks += n_seq[j] * tiles;
    if (blocks > 0x7fffffffLL) return hipErrorInvalidValue;
  }
  if (blocks == 0) return hipSuccess;
  hipLaunchKernelGGL(to_tiles ? tile_gather_kernel<true> : tile_gather_kernel<false>, dim3((unsigned)blocks), dim3(256), 0, stream, jobs, T, H, W, tT, tH, tW,
                     1.0f / (float)tile_sz);
  return hipGetLastError();
}

hipError_t launch_tile_permute(const void* x, void* out, int64_t n_seq, int T, int H, int W, int tT, int tH, int tW,
                               int to_tiles, hipStream_t stream) {
  const int64_t rows = n_seq * T * H * W;
  const int64_t blocks = (rows + 15) / 16;
  if (blocks <= 0) return hipSuccess;
  if (blocks > 0x7fffffffLL) return hipErrorInvalidValue;
  hipLaunchKernelGGL(tile_permute_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, (const uint4*)x, (uint4*)out, n_seq,
                     T, H, W, tT, tH, tW, to_tiles);
  return hipGetLastError();
}

}  // namespace fba
