// C ABI entry points: argument validation, variant selection, launches.  See include/fba.h for the contract.
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>

#include "../../include/fba.h"
#include "fba_kernels.h"

namespace {

thread_local char g_err[512] = "";

int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

struct Shape {
  int64_t mask_bh;
  int B, Hq, Hkv, Sq, Skv, D, q_block, k_block;
};

// Shape rules of the operator (flex_block_attn_interface.py:18-32, flex_block_attn_h100.cu:833-850).
int check_shape(const Shape& s) {
  if (s.D != 128) return fail(FBA_ERR_INVALID, "head_dim must be 128, got %d", s.D);
  if (s.B <= 0 || s.Hq <= 0 || s.Hkv <= 0 || s.Sq <= 0 || s.Skv <= 0)
    return fail(FBA_ERR_INVALID, "B, Hq, Hkv, Sq, Skv must be positive (got %d %d %d %d %d)", s.B, s.Hq, s.Hkv, s.Sq, s.Skv);
  if (s.Hq % s.Hkv != 0) return fail(FBA_ERR_INVALID, "Hq (%d) must be a multiple of Hkv (%d)", s.Hq, s.Hkv);
  if (s.q_block <= 0 || s.q_block % 16 != 0) return fail(FBA_ERR_INVALID, "q_block (%d) must be a positive multiple of 16", s.q_block);
  if (s.k_block <= 0 || s.k_block % 64 != 0) return fail(FBA_ERR_INVALID, "k_block (%d) must be a positive multiple of 64", s.k_block);
  if (s.k_block % s.q_block != 0 && s.q_block % s.k_block != 0)
    return fail(FBA_ERR_INVALID, "one of q_block (%d), k_block (%d) must divide the other", s.q_block, s.k_block);
  if (s.Sq % s.q_block != 0) return fail(FBA_ERR_INVALID, "Sq (%d) must be a multiple of q_block (%d)", s.Sq, s.q_block);
  if (s.Skv % s.k_block != 0) return fail(FBA_ERR_INVALID, "Skv (%d) must be a multiple of k_block (%d)", s.Skv, s.k_block);
  if (s.mask_bh != 1 && s.mask_bh != (int64_t)s.B * s.Hq)
    return fail(FBA_ERR_INVALID, "mask_bh (%lld) must be 1 or B*Hq (%lld)", (long long)s.mask_bh, (long long)s.B * s.Hq);
  if ((int64_t)s.B * s.Hq * (int64_t)(s.Sq / 128 + 1) > 0x7fffffffLL || (int64_t)s.B * s.Hkv * (int64_t)(s.Skv / 128 + 1) > 0x7fffffffLL)
    return fail(FBA_ERR_INVALID, "problem too large for a 32-bit work-item index");
  return FBA_OK;
}

int check_ptrs(std::initializer_list<std::pair<const char*, const void*>> ps) {
  for (auto& kv : ps) {
    if (kv.second == nullptr) return fail(FBA_ERR_INVALID, "%s is null", kv.first);
    if (!aligned16(kv.second)) return fail(FBA_ERR_INVALID, "%s is not 16-byte aligned", kv.first);
  }
  return FBA_OK;
}

// Which dK/dV kernel runs on block lists: the one with 64 keys per wave (one wave per SIMD) by default.  It is about 9 %
// faster than the one with 32 keys per wave (two waves per SIMD) without the dS hand-over and about 7 % faster with it
// (a wave alone on its SIMD pays for every cycle its dS stores take to issue).  Both do the same arithmetic in the same
// order.  FBA_DKDV_KEYS_PER_WAVE = 32 or 64 overrides the choice (measurement of the two).
hipError_t launch_dkdv_variant(fba::BwdParams& p, hipStream_t stream, fba::Merge* later) {
  const char* env = getenv("FBA_DKDV_KEYS_PER_WAVE");
  const int keys = env ? atoi(env) : 64;
  if (p.tiled) return fba::launch_bwd_dkdv_slab(p, stream, later);
  if (keys == 64) return fba::launch_bwd_dkdv64(p, stream, later);
  return fba::launch_bwd_dkdv(p, stream, later);
}

int hip_fail(hipError_t e, const char* what) { return fail(FBA_ERR_HIP, "%s: %s", what, hipGetErrorString(e)); }

// Optional workspace for tail splitting: null (nothing is split), or 16-byte aligned with a non-negative size.
int check_split_ws(const void* ws, int64_t bytes) {
  if (ws == nullptr) return FBA_OK;
  if (!aligned16(ws)) return fail(FBA_ERR_INVALID, "split_ws is not 16-byte aligned");
  if (bytes < 0) return fail(FBA_ERR_INVALID, "split_ws_bytes must not be negative");
  return FBA_OK;
}

}  // namespace

extern "C" {

int32_t fba_version(void) { return FBA_VERSION; }

const char* fba_last_error(void) { return g_err; }

int64_t fba_split_workspace_bytes(void) { return fba::kSplitWsBytes; }

int32_t fba_mask_compact(const uint8_t* mask, int64_t mask_bh, int32_t nQ, int32_t nK, int32_t* q_cnt, int32_t* q_idx,
                         int32_t* k_cnt, int32_t* k_idx, void* hip_stream) {
  if (mask_bh <= 0 || nQ <= 0 || nK <= 0)
    return fail(FBA_ERR_INVALID, "mask_bh, nQ, nK must be positive (got %lld %d %d)", (long long)mask_bh, nQ, nK);
  if (!mask || !q_cnt || !q_idx || !k_cnt || !k_idx) return fail(FBA_ERR_INVALID, "null pointer argument");
  hipError_t e = fba::launch_mask_compact(mask, mask_bh, nQ, nK, q_cnt, q_idx, k_cnt, k_idx, (hipStream_t)hip_stream);
  return e == hipSuccess ? FBA_OK : hip_fail(e, "mask_compact launch");
}

}  // extern "C"

namespace {

// Which list flavour a shape needs: block lists when both block sizes are multiples of the 128-row kernel tiles, tile
// lists otherwise.  Tile lists need Sq and Skv to be multiples of 128.
int check_lists(const Shape& s, bool tiled, const char* what) {
  const bool aligned = s.q_block % 128 == 0 && s.k_block % 128 == 0;
  if (!tiled && !aligned)
    return fail(FBA_ERR_UNSUPPORTED, "%s: q_block (%d) and k_block (%d) are not both multiples of 128; build tile lists "
                "with fba_tile_lists and call the _tiled entry point", what, s.q_block, s.k_block);
  if (tiled && (s.Sq % 128 != 0 || s.Skv % 128 != 0))
    return fail(FBA_ERR_UNSUPPORTED, "%s: tile lists need Sq (%d) and Skv (%d) to be multiples of 128", what, s.Sq, s.Skv);
  return FBA_OK;
}

int check_tile_list_shape(int32_t nQ, int32_t nK, int32_t q_block, int32_t k_block) {
  if (q_block <= 0 || q_block % 16 != 0) return fail(FBA_ERR_INVALID, "q_block (%d) must be a positive multiple of 16", q_block);
  if (k_block <= 0 || k_block % 64 != 0) return fail(FBA_ERR_INVALID, "k_block (%d) must be a positive multiple of 64", k_block);
  const int64_t Sq = (int64_t)nQ * q_block, Skv = (int64_t)nK * k_block;
  if (Sq % 128 != 0 || Skv % 128 != 0)
    return fail(FBA_ERR_UNSUPPORTED, "tile lists need Sq (%lld) and Skv (%lld) to be multiples of 128", (long long)Sq, (long long)Skv);
  if (Sq / 32 >= (1 << 23) || nK >= (1 << 23)) return fail(FBA_ERR_INVALID, "sequence too long for 24-bit list entries");
  return FBA_OK;
}

int fwd_impl(const void* q, const void* k, const void* v, void* o, float* lse, const int32_t* q_cnt, const int32_t* q_idx, const uint8_t* mask,
             int64_t mask_bh, int32_t B, int32_t Hq, int32_t Hkv, int32_t Sq, int32_t Skv, int32_t head_dim, int32_t q_block,
             int32_t k_block, void* split_ws, int64_t split_ws_bytes, void* hip_stream, bool tiled, decltype(fba::FwdParams::make) make = {}) {
  const Shape s{mask_bh, B, Hq, Hkv, Sq, Skv, head_dim, q_block, k_block};
  if (int rc = check_shape(s)) return rc;
  if (int rc = check_ptrs({{"q", q}, {"k", k}, {"v", v}, {"o", o}})) return rc;
  if (!lse || (!mask && (!q_cnt || !q_idx))) return fail(FBA_ERR_INVALID, "null pointer argument");
  if (int rc = check_lists(s, tiled, "forward")) return rc;
  if (int rc = check_split_ws(split_ws, split_ws_bytes)) return rc;
  fba::FwdParams p{};
  p.q = (const __bf16*)q; p.k = (const __bf16*)k; p.v = (const __bf16*)v; p.o = (__bf16*)o; p.lse = lse;
  p.q_cnt = q_cnt; p.q_idx = q_idx; p.mask = mask; p.make = make; p.mask_bh = mask_bh;
  p.B = B; p.Hq = Hq; p.Hkv = Hkv; p.Sq = Sq; p.Skv = Skv; p.nQ = Sq / q_block; p.nK = Skv / k_block;
  p.q_block = q_block; p.k_block = k_block;
  p.scale_log2e = 1.4426950408889634f / 11.313708498984761f;
  p.tiled = tiled ? 1 : 0;
  p.split.ws = (float*)split_ws; p.split_ws_bytes = split_ws_bytes;
  {
    const char* rows = getenv("FBA_FWD_TILE_ROWS");
    p.variant = rows && atoi(rows) == 384 ? 0 : 1;  // 128-row work-groups unless asked otherwise
  }
  hipError_t e = fba::launch_fwd(p, (hipStream_t)hip_stream);
  return e == hipSuccess ? FBA_OK : hip_fail(e, "forward launch");
}

}  // namespace

extern "C" {

int32_t fba_fwd(const void* q, const void* k, const void* v, void* o, float* lse, const int32_t* q_cnt,
                const int32_t* q_idx, int64_t mask_bh, int32_t B, int32_t Hq, int32_t Hkv, int32_t Sq, int32_t Skv,
                int32_t head_dim, int32_t q_block, int32_t k_block, void* split_ws, int64_t split_ws_bytes, void* hip_stream) {
  return fwd_impl(q, k, v, o, lse, q_cnt, q_idx, nullptr, mask_bh, B, Hq, Hkv, Sq, Skv, head_dim, q_block, k_block, split_ws, split_ws_bytes,
                  hip_stream, false);
}

int32_t fba_fwd_tiled(const void* q, const void* k, const void* v, void* o, float* lse, const int32_t* qt_cnt,
                      const int32_t* qt_ent, int64_t mask_bh, int32_t B, int32_t Hq, int32_t Hkv, int32_t Sq, int32_t Skv,
                      int32_t head_dim, int32_t q_block, int32_t k_block, void* split_ws, int64_t split_ws_bytes,
                      void* hip_stream) {
  return fwd_impl(q, k, v, o, lse, qt_cnt, qt_ent, nullptr, mask_bh, B, Hq, Hkv, Sq, Skv, head_dim, q_block, k_block, split_ws, split_ws_bytes, hip_stream, true);
}

int32_t fba_fwd_blocks(const void* q, const void* k, const void* v, void* o, float* lse, const uint8_t* mask, int32_t* q_cnt, int32_t* q_idx, int32_t* k_cnt,
                       int32_t* k_idx, int64_t mask_bh, int32_t B, int32_t Hq, int32_t Hkv, int32_t Sq, int32_t Skv, int32_t head_dim, int32_t q_block,
                       int32_t k_block, void* split_ws, int64_t split_ws_bytes, void* hip_stream) {
  if (!mask) return fail(FBA_ERR_INVALID, "null pointer argument");
  const bool make = q_cnt || q_idx || k_cnt || k_idx;
  if (make && (!q_cnt || !q_idx || !k_cnt || !k_idx)) return fail(FBA_ERR_INVALID, "forward: all four lists, or none");
  if (make && q_block > 0 && k_block > 0 && mask_bh * ((int64_t)Sq / q_block + Skv / k_block) > fba::kMakeRows)
    return fail(FBA_ERR_UNSUPPORTED, "forward: more than %d rows of lists; build them with fba_mask_compact", fba::kMakeRows);
  if (k_block > 0 && Skv / k_block > fba::kMaskBlocks)
    return fail(FBA_ERR_UNSUPPORTED, "forward: %d key blocks are more than %d; build lists with fba_mask_compact and call fba_fwd", Skv / k_block, fba::kMaskBlocks);
  return fwd_impl(q, k, v, o, lse, nullptr, nullptr, mask, mask_bh, B, Hq, Hkv, Sq, Skv, head_dim, q_block, k_block, split_ws, split_ws_bytes, hip_stream, false,
                  {q_cnt, q_idx, k_cnt, k_idx, 0});
}

int32_t fba_fwd_blocks_use(int64_t mask_bh, int32_t B, int32_t Hq, int32_t Sq, int32_t Skv, int32_t q_block, int32_t k_block) {
  if (mask_bh <= 0 || B <= 0 || Hq <= 0 || Sq <= 0 || Skv <= 0 || q_block <= 0 || k_block <= 0) return 0;
  if (q_block % 128 != 0 || k_block % 128 != 0 || Skv / k_block > fba::kMaskBlocks) return 0;
  const bool lists = mask_bh * ((int64_t)Sq / q_block + Skv / k_block) <= fba::kMakeRows;
  return FBA_BLOCKS_TAKEN | (lists ? FBA_BLOCKS_LISTS : 0) | (fba::fwd_takes_halves((int64_t)B * Hq * Sq, Skv) ? FBA_BLOCKS_HALVES : 0);
}

int32_t fba_fwd_mask_copy(const void* q, const void* k, const void* v, void* o, float* lse, const uint8_t* mask, uint8_t* mask_copy, int32_t o_rows,
                          int64_t mask_bh, int32_t B, int32_t Hq, int32_t Hkv, int32_t Sq, int32_t Skv, int32_t head_dim, int32_t q_block, int32_t k_block, void* hip_stream) {
  const Shape s{mask_bh, B, Hq, Hkv, Sq, Skv, head_dim, q_block, k_block};
  if (int rc = check_shape(s)) return rc;
  if (int rc = check_ptrs({{"q", q}, {"k", k}, {"v", v}, {"o", o}})) return rc;
  if (!lse || !mask) return fail(FBA_ERR_INVALID, "null pointer argument");
  if ((int64_t)B * Hq * Sq >= (1LL << 30)) return fail(FBA_ERR_INVALID, "B*Hq*Sq must be below 2^30");
  fba::FwdMaskParams p{};
  p.q = (const __bf16*)q; p.k = (const __bf16*)k; p.v = (const __bf16*)v; p.o = (__bf16*)o; p.lse = lse;
  if (o_rows < Sq || (int64_t)B * Hq * o_rows > 0x7fffffffLL) return fail(FBA_ERR_INVALID, "o_rows (%d) must be Sq (%d) or more, B*Hq*o_rows below 2^31", o_rows, Sq);
  p.mask = mask; p.mask_copy = mask_copy; p.o_rows = o_rows; p.mask_bh = mask_bh;
  p.B = B; p.Hq = Hq; p.Hkv = Hkv; p.Sq = Sq; p.Skv = Skv; p.nQ = Sq / q_block; p.nK = Skv / k_block;
  p.q_block = q_block; p.k_block = k_block;
  p.scale_log2e = 1.4426950408889634f / 11.313708498984761f;
  hipError_t e = fba::launch_fwd_mask(p, (hipStream_t)hip_stream);
  return e == hipSuccess ? FBA_OK : hip_fail(e, "forward (from the mask) launch");
}

int32_t fba_fwd_mask(const void* q, const void* k, const void* v, void* o, float* lse, const uint8_t* mask, int64_t mask_bh, int32_t B, int32_t Hq,
                     int32_t Hkv, int32_t Sq, int32_t Skv, int32_t head_dim, int32_t q_block, int32_t k_block, void* hip_stream) {
  return fba_fwd_mask_copy(q, k, v, o, lse, mask, nullptr, Sq, mask_bh, B, Hq, Hkv, Sq, Skv, head_dim, q_block, k_block, hip_stream);
}

int32_t fba_fwd_takes_mask(int64_t rows, int32_t Skv) { return fba::fwd_takes_mask(rows, Skv) ? 1 : 0; }

int32_t fba_bwd_mask(const void* q, const void* k, const void* v, const void* o, const void* d_o, const float* lse, const uint8_t* mask, int32_t o_rows,
                     int64_t mask_bh, void* dq, void* dk, void* dv, int32_t B, int32_t Hq, int32_t Hkv, int32_t Sq, int32_t Skv, int32_t head_dim, int32_t q_block,
                     int32_t k_block, void* hip_stream) {
  const Shape s{mask_bh, B, Hq, Hkv, Sq, Skv, head_dim, q_block, k_block};
  if (int rc = check_shape(s)) return rc;
  if (int rc = check_ptrs({{"q", q}, {"k", k}, {"v", v}, {"o", o}, {"d_o", d_o}, {"dq", dq}, {"dk", dk}, {"dv", dv}})) return rc;
  if (!lse || !mask) return fail(FBA_ERR_INVALID, "null pointer argument");
  if ((int64_t)B * Hq * Sq >= (1LL << 30) || (int64_t)B * Hkv * Skv >= (1LL << 30)) return fail(FBA_ERR_INVALID, "B*Hq*Sq and B*Hkv*Skv must be below 2^30");
  if (o_rows < Sq || (int64_t)B * Hq * o_rows > 0x7fffffffLL) return fail(FBA_ERR_INVALID, "o_rows (%d) must be Sq (%d) or more, B*Hq*o_rows below 2^31", o_rows, Sq);
  fba::BwdMaskParams p{};
  p.o_rows = o_rows;
  p.q = (const __bf16*)q; p.k = (const __bf16*)k; p.v = (const __bf16*)v; p.o = (const __bf16*)o; p.d_o = (const __bf16*)d_o; p.lse = lse;
  p.dq = (__bf16*)dq; p.dk = (__bf16*)dk; p.dv = (__bf16*)dv;
  p.mask = mask; p.mask_bh = mask_bh;
  p.B = B; p.Hq = Hq; p.Hkv = Hkv; p.Sq = Sq; p.Skv = Skv; p.nQ = Sq / q_block; p.nK = Skv / k_block;
  p.q_block = q_block; p.k_block = k_block;
  p.scale = 1.f / 11.313708498984761f;
  p.scale_log2e = 1.4426950408889634f / 11.313708498984761f;
  hipError_t e = fba::launch_bwd_mask(p, (hipStream_t)hip_stream);
  return e == hipSuccess ? FBA_OK : hip_fail(e, "backward (from the mask) launch");
}

int32_t fba_bwd_takes_mask(int32_t B, int32_t Hq, int32_t Hkv, int32_t Sq, int32_t Skv) {
  return fba::bwd_takes_mask((int64_t)B * Hq, (int64_t)B * Hkv, Sq, Skv) ? 1 : 0;
}

static int check_means(const void* x, const float* out, int64_t n_seq, int32_t S, int32_t block) {
  if (n_seq <= 0 || S <= 0) return fail(FBA_ERR_INVALID, "n_seq and S must be positive (got %lld %d)", (long long)n_seq, S);
  if (block <= 0 || block % 16 != 0 || S % block != 0)
    return fail(FBA_ERR_INVALID, "block (%d) must be a positive multiple of 16 that divides S (%d)", block, S);
  if (!out) return fail(FBA_ERR_INVALID, "out is null");
  return check_ptrs({{"x", x}});
}

int32_t fba_block_mean(const void* x, float* out, int64_t n_seq, int32_t S, int32_t block, int32_t head_dim, void* hip_stream) {
  if (head_dim != 128) return fail(FBA_ERR_INVALID, "head_dim must be 128, got %d", head_dim);
  if (int rc = check_means(x, out, n_seq, S, block)) return rc;
  hipError_t e = fba::launch_block_mean({{(const __bf16*)x, out, n_seq * (S / block), block}, {}}, (hipStream_t)hip_stream);
  return e == hipSuccess ? FBA_OK : hip_fail(e, "block_mean launch");
}

int32_t fba_block_mean_pair(const void* x, float* out, int64_t n_seq, int32_t S, int32_t block, const void* x2, float* out2, int64_t n_seq2, int32_t S2,
                            int32_t block2, int32_t head_dim, void* hip_stream) {
  if (head_dim != 128) return fail(FBA_ERR_INVALID, "head_dim must be 128, got %d", head_dim);
  if (int rc = check_means(x, out, n_seq, S, block)) return rc;
  if (int rc = check_means(x2, out2, n_seq2, S2, block2)) return rc;
  hipError_t e = fba::launch_block_mean({{(const __bf16*)x, out, n_seq * (S / block), block}, {(const __bf16*)x2, out2, n_seq2 * (S2 / block2), block2}},
                                        (hipStream_t)hip_stream);
  return e == hipSuccess ? FBA_OK : hip_fail(e, "block_mean launch");
}

int32_t fba_ssta_mask(const float* q_mean, const float* k_mean, const uint8_t* base, uint8_t* mask, int32_t B, int32_t Hq, int32_t Hkv, int32_t nQ,
                      int32_t nK, int32_t q_block, int32_t k_block, int32_t topk, int32_t band, int32_t sink,
                      void* hip_stream) {
  if (B <= 0 || Hq <= 0 || Hkv <= 0 || nQ <= 0 || nK <= 0)
    return fail(FBA_ERR_INVALID, "B, Hq, Hkv, nQ, nK must be positive (got %d %d %d %d %d)", B, Hq, Hkv, nQ, nK);
  if (Hq % Hkv != 0) return fail(FBA_ERR_INVALID, "Hq (%d) must be a multiple of Hkv (%d)", Hq, Hkv);
  if (q_block <= 0 || k_block <= 0) return fail(FBA_ERR_INVALID, "q_block and k_block must be positive");
  if (topk < 0 || band < -1 || sink < 0) return fail(FBA_ERR_INVALID, "topk, sink must be >= 0 and band >= -1 (got %d %d %d)", topk, sink, band);
  if (!q_mean || !k_mean || !mask) return fail(FBA_ERR_INVALID, "null pointer argument");
  if (nK > 4096) return fail(FBA_ERR_UNSUPPORTED, "at most 4096 key blocks are ranked per query block (got %d)", nK);
  if ((int64_t)B * Hq > 65535) return fail(FBA_ERR_UNSUPPORTED, "B*Hq (%lld) must be at most 65535", (long long)B * Hq);
  hipError_t e = fba::launch_ssta_mask(q_mean, k_mean, base, mask, (int64_t)B * Hq, Hq, Hkv, nQ, nK, q_block, k_block, topk, band,
                                       sink, fba::TileWindow{}, (hipStream_t)hip_stream);
  return e == hipSuccess ? FBA_OK : hip_fail(e, "ssta_mask launch");
}

int32_t fba_ssta_mask_3d(const float* q_mean, const float* k_mean, uint8_t* mask, int32_t B, int32_t Hq, int32_t Hkv, int32_t nT, int32_t nH,
                         int32_t nW, int32_t half_t, int32_t half_h, int32_t half_w, int32_t topk, int32_t sink, void* hip_stream) {
  if (B <= 0 || Hq <= 0 || Hkv <= 0 || nT <= 0 || nH <= 0 || nW <= 0)
    return fail(FBA_ERR_INVALID, "B, Hq, Hkv and the grid of tiles must be positive (got %d %d %d, %d x %d x %d)", B, Hq, Hkv, nT, nH, nW);
  if (Hq % Hkv != 0) return fail(FBA_ERR_INVALID, "Hq (%d) must be a multiple of Hkv (%d)", Hq, Hkv);
  if (topk < 0 || sink < 0) return fail(FBA_ERR_INVALID, "topk, sink must be >= 0 (got %d %d)", topk, sink);
  if (!q_mean || !k_mean || !mask) return fail(FBA_ERR_INVALID, "null pointer argument");
  const int64_t tiles = (int64_t)nT * nH * nW;
  if (tiles > 4096) return fail(FBA_ERR_UNSUPPORTED, "at most 4096 key blocks are ranked per query block (got %lld)", (long long)tiles);
  if ((int64_t)B * Hq > 65535) return fail(FBA_ERR_UNSUPPORTED, "B*Hq (%lld) must be at most 65535", (long long)B * Hq);
  fba::TileWindow w{{nT, nH, nW}, {half_t, half_h, half_w}, {}, {}};
  for (int x = 0; x < 3; ++x) {  // the window of a border tile is shifted inwards
    w.low[x] = w.half[x] < w.n[x] - 1 ? w.half[x] : w.n[x] - 1;
    w.high[x] = w.n[x] - 1 - w.half[x] > 0 ? w.n[x] - 1 - w.half[x] : 0;
  }
  hipError_t e = fba::launch_ssta_mask(q_mean, k_mean, nullptr, mask, (int64_t)B * Hq, Hq, Hkv, (int)tiles, (int)tiles, 1, 1, topk, -1, sink, w,
                                       (hipStream_t)hip_stream);
  return e == hipSuccess ? FBA_OK : hip_fail(e, "ssta_mask (3-D) launch");
}

int32_t fba_tile_permute(const void* x, void* out, int64_t n_seq, int32_t T, int32_t H, int32_t W, int32_t tile_t,
                         int32_t tile_h, int32_t tile_w, int32_t head_dim, int32_t to_tiles, void* hip_stream) {
  if (head_dim != 128) return fail(FBA_ERR_INVALID, "head_dim must be 128, got %d", head_dim);
  if (n_seq <= 0 || T <= 0 || H <= 0 || W <= 0 || tile_t <= 0 || tile_h <= 0 || tile_w <= 0)
    return fail(FBA_ERR_INVALID, "n_seq, grid and tile extents must be positive");
  if (T % tile_t != 0 || H % tile_h != 0 || W % tile_w != 0)
    return fail(FBA_ERR_INVALID, "tile (%d, %d, %d) must divide the grid (%d, %d, %d)", tile_t, tile_h, tile_w, T, H, W);
  if ((int64_t)T * H * W > 0x7fffffffLL) return fail(FBA_ERR_INVALID, "grid too large");
  if (x == out) return fail(FBA_ERR_INVALID, "x and out must not alias");
  if (int rc = check_ptrs({{"x", x}, {"out", out}})) return rc;
  hipError_t e = fba::launch_tile_permute(x, out, n_seq, T, H, W, tile_t, tile_h, tile_w, to_tiles ? 1 : 0, (hipStream_t)hip_stream);
  return e == hipSuccess ? FBA_OK : hip_fail(e, "tile_permute launch");
}

int32_t fba_tile_gather(int32_t n, const void* const* x, void* const* out, float* const* mean, const int64_t* n_seq, int32_t T, int32_t H, int32_t W,
                        int32_t tile_t, int32_t tile_h, int32_t tile_w, int32_t head_dim, int32_t to_tiles, void* hip_stream) {
  if (head_dim != 128) return fail(FBA_ERR_INVALID, "head_dim must be 128, got %d", head_dim);
  if (n < 1 || n > 3) return fail(FBA_ERR_INVALID, "tile_gather takes one to three tensors (got %d)", n);
  if (!x || !out || !mean || !n_seq) return fail(FBA_ERR_INVALID, "null pointer argument");
  if (T <= 0 || H <= 0 || W <= 0 || tile_t <= 0 || tile_h <= 0 || tile_w <= 0) return fail(FBA_ERR_INVALID, "grid and tile extents must be positive");
  if (T % tile_t != 0 || H % tile_h != 0 || W % tile_w != 0)
    return fail(FBA_ERR_INVALID, "tile (%d, %d, %d) must divide the grid (%d, %d, %d)", tile_t, tile_h, tile_w, T, H, W);
  if ((int64_t)T * H * W > 0x7fffffffLL) return fail(FBA_ERR_INVALID, "grid too large");
  const int64_t tile_rows = (int64_t)tile_t * tile_h * tile_w;
  for (int j = 0; j < n; ++j) {
    if (int rc = check_ptrs({{"x", x[j]}, {"out", out[j]}})) return rc;
    if (x[j] == out[j]) return fail(FBA_ERR_INVALID, "x and out must not alias");
    if (n_seq[j] <= 0) return fail(FBA_ERR_INVALID, "n_seq must be positive");
    if (to_tiles && mean[j] && tile_rows % 16 != 0) return fail(FBA_ERR_INVALID, "means need tiles of a multiple of 16 tokens (got %lld)", (long long)tile_rows);
  }
  hipError_t e = fba::launch_tile_gather(n, x, out, mean, n_seq, T, H, W, tile_t, tile_h, tile_w, to_tiles ? 1 : 0, (hipStream_t)hip_stream);
  return e == hipSuccess ? FBA_OK : hip_fail(e, "tile_gather launch");
}

int32_t fba_tile_lists(const uint8_t* mask, int64_t mask_bh, int32_t nQ, int32_t nK, int32_t q_block, int32_t k_block,
                       int32_t* qt_cnt, int32_t* qt_ent, int32_t* kt_cnt, int32_t* kt_ent, void* hip_stream) {
  if (mask_bh <= 0 || nQ <= 0 || nK <= 0)
    return fail(FBA_ERR_INVALID, "mask_bh, nQ, nK must be positive (got %lld %d %d)", (long long)mask_bh, nQ, nK);
  if (int rc = check_tile_list_shape(nQ, nK, q_block, k_block)) return rc;
  const int64_t Sq = (int64_t)nQ * q_block, Skv = (int64_t)nK * k_block;
  if (!mask || !qt_cnt || !qt_ent || !kt_cnt || !kt_ent) return fail(FBA_ERR_INVALID, "null pointer argument");
  hipError_t e = fba::launch_tile_lists(mask, mask_bh, nQ, nK, nK, q_block, k_block, (int)(Sq / 128), (int)(Skv / 128), (int)(Sq / 32),
                                        qt_cnt, qt_ent, kt_cnt, kt_ent, (hipStream_t)hip_stream);
  return e == hipSuccess ? FBA_OK : hip_fail(e, "tile_lists launch");
}

static int fill_bwd(fba::BwdParams& p, const Shape& s) {
  p.mask_bh = s.mask_bh;
  p.B = s.B; p.Hq = s.Hq; p.Hkv = s.Hkv; p.Sq = s.Sq; p.Skv = s.Skv; p.nQ = s.Sq / s.q_block; p.nK = s.Skv / s.k_block;
  p.q_block = s.q_block; p.k_block = s.k_block;
  p.out_q = s.Sq; p.out_kv = s.Skv;
  p.scale = 1.f / 11.313708498984761f;
  p.scale_log2e = 1.4426950408889634f / 11.313708498984761f;
  return FBA_OK;
}

int32_t fba_split_plan(int32_t launch, int64_t mask_bh, int32_t B, int32_t Hq, int32_t Hkv, int32_t Sq, int32_t Skv, int32_t head_dim, int32_t q_block,
                       int32_t k_block, int64_t split_ws_bytes, int64_t* plan) {
  const Shape s{mask_bh, B, Hq, Hkv, Sq, Skv, head_dim, q_block, k_block};
  if (int rc = check_shape(s)) return rc;
  if (plan == nullptr || split_ws_bytes < 0) return fail(FBA_ERR_INVALID, "null plan or negative split_ws_bytes");
  const bool tiled = q_block % 128 != 0 || k_block % 128 != 0;
  if (int rc = check_lists(s, tiled, "split_plan")) return rc;
  // addresses that are only compared with null and subtracted from each other
  float* const ws = split_ws_bytes > 0 ? reinterpret_cast<float*>(16) : nullptr;
  const int32_t* const cnt = reinterpret_cast<const int32_t*>(16);
  fba::BwdParams b{};
  fill_bwd(b, s);
  b.tiled = tiled ? 1 : 0;
  b.q_cnt = b.k_cnt = cnt;
  b.split.ws = ws; b.split_ws_bytes = split_ws_bytes;
  switch (launch) {
    case 4:
      if (fba_fwd_blocks_use(mask_bh, B, Hq, Sq, Skv, q_block, k_block) == 0) return fail(FBA_ERR_UNSUPPORTED, "split_plan: fba_fwd_blocks does not take such sizes");
      [[fallthrough]];
    case 0: {
      fba::FwdParams f{};
      f.mask_bh = mask_bh;
      f.B = B; f.Hq = Hq; f.Hkv = Hkv; f.Sq = Sq; f.Skv = Skv; f.nQ = b.nQ; f.nK = b.nK;
      f.q_block = q_block; f.k_block = k_block;
      if (launch == 0) f.q_cnt = cnt;
      else f.mask = reinterpret_cast<const uint8_t*>(cnt);
      f.tiled = b.tiled; f.variant = 1;
      f.split = b.split; f.split_ws_bytes = split_ws_bytes;
      fba::plan_fwd(f);
      b.num_items = f.num_items;
      b.split = f.split;
      break;
    }
    case 1: fba::plan_bwd_dkdv(b, tiled ? fba::kKeyTiles64 : fba::kKeyTiles128); break;
    case 2: fba::plan_bwd_dq(b); break;
    case 3: fba::plan_bwd_dq_from_ds(b); break;
    default: return fail(FBA_ERR_INVALID, "launch must be 0 to 4, got %d", launch);
  }
  const fba::SplitPlan& sp = b.split;
  const bool split = sp.first < b.num_items;
  plan[0] = b.num_items;
  plan[1] = sp.first;
  plan[2] = sp.parts;
  const fba::ListLook& l = sp.look;
  const bool looks = split && (l.cnt != nullptr || l.mask != nullptr);
  plan[3] = looks;
  plan[4] = looks ? reinterpret_cast<const char*>(sp.note) - reinterpret_cast<const char*>(ws) : 0;
  const float cost[4] = {l.spread, l.whole / l.step, l.cut / l.step, l.least};
  for (int j = 0; j < 4; ++j) plan[5 + j] = looks ? (int64_t)(1000 * cost[j]) : 0;
  plan[9] = looks ? l.fewest : 0;
  for (int j = 0; j < fba::kMostParts - 2; ++j) plan[10 + j] = looks && l.more[j] < 1e9f ? (int64_t)std::ceil(l.more[j] * l.step) : 0x7fffffff;
  return FBA_OK;
}

int32_t fba_split_regions(int32_t units, int32_t from_ds, int64_t mask_bh, int32_t B, int32_t Hq, int32_t Hkv, int32_t Sq, int32_t Skv, int32_t head_dim,
                          int32_t q_block, int32_t k_block, int64_t split_ws_bytes, int64_t* regions) {
  const Shape s{mask_bh, B, Hq, Hkv, Sq, Skv, head_dim, q_block, k_block};
  if (int rc = check_shape(s)) return rc;
  if (regions == nullptr || split_ws_bytes <= 0 || units < 0) return fail(FBA_ERR_INVALID, "null regions, no workspace or negative units");
  const bool tiled = q_block % 128 != 0 || k_block % 128 != 0;
  if (int rc = check_lists(s, tiled, "split_regions")) return rc;
  const fba::AssumedUnits assumed(units);
  fba::BwdParams b{};
  fill_bwd(b, s);
  b.tiled = tiled ? 1 : 0;
  b.q_cnt = b.k_cnt = reinterpret_cast<const int32_t*>(16);  // addresses that are only compared with null and subtracted from each other
  b.split.ws = reinterpret_cast<float*>(16); b.split_ws_bytes = split_ws_bytes;
  b.make.stats = reinterpret_cast<float*>(16);
  const fba::SplitRegions r = fba::plan_split_regions(b, from_ds != 0);
  regions[0] = r.parts_end; regions[1] = r.pieces_end; regions[2] = r.dq_from; regions[3] = r.dq_end; regions[4] = r.kept_from;
  return FBA_OK;
}

int32_t fba_bwd_stats(const void* o, const void* d_o, const float* lse, float* stats, int64_t rows, int32_t head_dim,
                      void* hip_stream) {
  if (head_dim != 128) return fail(FBA_ERR_INVALID, "head_dim must be 128, got %d", head_dim);
  if (rows < 0 || rows >= (1LL << 30)) return fail(FBA_ERR_INVALID, "rows must be in [0, 2^30)");
  if (int rc = check_ptrs({{"o", o}, {"d_o", d_o}})) return rc;
  if (!lse || !stats) return fail(FBA_ERR_INVALID, "null pointer argument");
  hipError_t e = fba::launch_bwd_stats({(const __bf16*)o, (const __bf16*)d_o, lse, stats, rows}, (hipStream_t)hip_stream);
  return e == hipSuccess ? FBA_OK : hip_fail(e, "stats launch");
}

static int dq_impl(const void* q, const void* k, const void* v, const void* d_o, const float* stats, void* dq,
                   const int32_t* q_cnt, const int32_t* q_idx, int64_t mask_bh, int32_t B, int32_t Hq, int32_t Hkv,
                   int32_t Sq, int32_t Skv, int32_t head_dim, int32_t q_block, int32_t k_block, void* split_ws, int64_t split_ws_bytes,
                   void* hip_stream, bool tiled, const fba::Merge& before) {
  const Shape s{mask_bh, B, Hq, Hkv, Sq, Skv, head_dim, q_block, k_block};
  if (int rc = check_shape(s)) return rc;
  if (int rc = check_ptrs({{"q", q}, {"k", k}, {"v", v}, {"d_o", d_o}, {"dq", dq}})) return rc;
  if (!stats || !q_cnt || !q_idx) return fail(FBA_ERR_INVALID, "null pointer argument");
  if (int rc = check_lists(s, tiled, "dq")) return rc;
  if (int rc = check_split_ws(split_ws, split_ws_bytes)) return rc;
  fba::BwdParams p{};
  fill_bwd(p, s);
  p.tiled = tiled ? 1 : 0;
  p.q = (const __bf16*)q; p.k = (const __bf16*)k; p.v = (const __bf16*)v; p.d_o = (const __bf16*)d_o;
  p.stats = stats; p.dq = (__bf16*)dq; p.q_cnt = q_cnt; p.q_idx = q_idx;
  p.split.ws = (float*)split_ws; p.split_ws_bytes = split_ws_bytes;
  hipError_t e = fba::launch_bwd_dq(p, (hipStream_t)hip_stream, before);
  return e == hipSuccess ? FBA_OK : hip_fail(e, "dq launch");
}

static int dkdv_impl(const void* q, const void* k, const void* v, const void* d_o, const float* stats, void* dk, void* dv,
                     const int32_t* k_cnt, const int32_t* k_idx, int64_t mask_bh, int32_t B, int32_t Hq, int32_t Hkv,
                     int32_t Sq, int32_t Skv, int32_t head_dim, int32_t q_block, int32_t k_block, void* split_ws, int64_t split_ws_bytes,
                     void* hip_stream, bool tiled, const fba::BwdStats& make, fba::Merge* later) {
  const Shape s{mask_bh, B, Hq, Hkv, Sq, Skv, head_dim, q_block, k_block};
  if (int rc = check_shape(s)) return rc;
  if (int rc = check_ptrs({{"q", q}, {"k", k}, {"v", v}, {"d_o", d_o}, {"dk", dk}, {"dv", dv}})) return rc;
  if (!stats || !k_cnt || !k_idx) return fail(FBA_ERR_INVALID, "null pointer argument");
  if (int rc = check_lists(s, tiled, "dkdv")) return rc;
  if (int rc = check_split_ws(split_ws, split_ws_bytes)) return rc;
  if ((int64_t)B * Hq * Sq >= (1LL << 30)) return fail(FBA_ERR_INVALID, "B*Hq*Sq must be below 2^30");
  fba::BwdParams p{};
  fill_bwd(p, s);
  p.tiled = tiled ? 1 : 0;
  p.q = (const __bf16*)q; p.k = (const __bf16*)k; p.v = (const __bf16*)v; p.d_o = (const __bf16*)d_o;
  p.stats = stats; p.make = make; p.dk = (__bf16*)dk; p.dv = (__bf16*)dv; p.k_cnt = k_cnt; p.k_idx = k_idx;
  p.split.ws = (float*)split_ws; p.split_ws_bytes = split_ws_bytes;
  hipError_t e = launch_dkdv_variant(p, (hipStream_t)hip_stream, later);
  return e == hipSuccess ? FBA_OK : hip_fail(e, "dkdv launch");
}

static int bwd_impl(const void* q, const void* k, const void* v, const void* o, const void* d_o, const float* lse,
                    float* stats, void* dq, void* dk, void* dv, const int32_t* q_cnt, const int32_t* q_idx,
                    const int32_t* k_cnt, const int32_t* k_idx, int64_t mask_bh, int32_t B, int32_t Hq, int32_t Hkv,
                    int32_t Sq, int32_t Skv, int32_t head_dim, int32_t q_block, int32_t k_block, void* split_ws, int64_t split_ws_bytes,
                    void* hip_stream, bool tiled) {
  const Shape s{mask_bh, B, Hq, Hkv, Sq, Skv, head_dim, q_block, k_block};
  if (int rc = check_shape(s)) return rc;
  if (int rc = check_lists(s, tiled, "backward")) return rc;
  if (int rc = check_split_ws(split_ws, split_ws_bytes)) return rc;
  // everything is validated before the first launch, so that a rejected call leaves nothing on the stream
  if (int rc = check_ptrs({{"q", q}, {"k", k}, {"v", v}, {"o", o}, {"d_o", d_o}, {"dq", dq}, {"dk", dk}, {"dv", dv}})) return rc;
  if (!lse || !stats || !q_cnt || !q_idx || !k_cnt || !k_idx) return fail(FBA_ERR_INVALID, "null pointer argument");
  if ((int64_t)B * Hq * Sq >= (1LL << 30)) return fail(FBA_ERR_INVALID, "B*Hq*Sq must be below 2^30");
  fba::Merge merge;
  if (int rc = dkdv_impl(q, k, v, d_o, stats, dk, dv, k_cnt, k_idx, mask_bh, B, Hq, Hkv, Sq, Skv, head_dim, q_block, k_block,
                         split_ws, split_ws_bytes, hip_stream, tiled, {(const __bf16*)o, (const __bf16*)d_o, lse, stats, (int64_t)B * Hq * Sq}, &merge))
    return rc;
  return dq_impl(q, k, v, d_o, stats, dq, q_cnt, q_idx, mask_bh, B, Hq, Hkv, Sq, Skv, head_dim, q_block, k_block, split_ws, split_ws_bytes,
                 hip_stream, tiled, merge);
}

int32_t fba_bwd_dq(const void* q, const void* k, const void* v, const void* d_o, const float* stats, void* dq,
                   const int32_t* q_cnt, const int32_t* q_idx, int64_t mask_bh, int32_t B, int32_t Hq, int32_t Hkv,
                   int32_t Sq, int32_t Skv, int32_t head_dim, int32_t q_block, int32_t k_block, void* split_ws, int64_t split_ws_bytes,
                   void* hip_stream) {
  return dq_impl(q, k, v, d_o, stats, dq, q_cnt, q_idx, mask_bh, B, Hq, Hkv, Sq, Skv, head_dim, q_block, k_block, split_ws, split_ws_bytes,
                 hip_stream, false, {});
}

int32_t fba_bwd_dkdv(const void* q, const void* k, const void* v, const void* d_o, const float* stats, void* dk, void* dv,
                     const int32_t* k_cnt, const int32_t* k_idx, int64_t mask_bh, int32_t B, int32_t Hq, int32_t Hkv,
                     int32_t Sq, int32_t Skv, int32_t head_dim, int32_t q_block, int32_t k_block, void* split_ws, int64_t split_ws_bytes,
                     void* hip_stream) {
  return dkdv_impl(q, k, v, d_o, stats, dk, dv, k_cnt, k_idx, mask_bh, B, Hq, Hkv, Sq, Skv, head_dim, q_block, k_block, split_ws,
                   split_ws_bytes, hip_stream, false, {}, nullptr);
}

int32_t fba_bwd(const void* q, const void* k, const void* v, const void* o, const void* d_o, const float* lse,
                float* stats, void* dq, void* dk, void* dv, const int32_t* q_cnt, const int32_t* q_idx,
                const int32_t* k_cnt, const int32_t* k_idx, int64_t mask_bh, int32_t B, int32_t Hq, int32_t Hkv,
                int32_t Sq, int32_t Skv, int32_t head_dim, int32_t q_block, int32_t k_block, void* split_ws, int64_t split_ws_bytes,
                void* hip_stream) {
  return bwd_impl(q, k, v, o, d_o, lse, stats, dq, dk, dv, q_cnt, q_idx, k_cnt, k_idx, mask_bh, B, Hq, Hkv, Sq, Skv, head_dim,
                  q_block, k_block, split_ws, split_ws_bytes, hip_stream, false);
}

int32_t fba_probe_mfma(const float* src, float* sink, int32_t work_groups, int32_t iters, void* hip_stream) {
  if (work_groups <= 0 || iters <= 0) return fail(FBA_ERR_INVALID, "work_groups and iters must be positive (got %d %d)", work_groups, iters);
  if (!sink) return fail(FBA_ERR_INVALID, "sink is null");
  hipError_t e = fba::launch_probe_mfma(src, sink, work_groups, iters, (hipStream_t)hip_stream);
  return e == hipSuccess ? FBA_OK : hip_fail(e, "probe launch");
}

int32_t fba_probe_read(const void* src, int64_t bytes, uint32_t* sink, int32_t work_groups, void* hip_stream) {
  if (work_groups <= 0 || bytes <= 0 || bytes % 32768 != 0)
    return fail(FBA_ERR_INVALID, "work_groups must be positive and bytes a positive multiple of 32768 (got %d %lld)", work_groups, (long long)bytes);
  if (!src || !sink) return fail(FBA_ERR_INVALID, "src or sink is null");
  hipError_t e = fba::launch_probe_read(src, bytes, sink, work_groups, (hipStream_t)hip_stream);
  return e == hipSuccess ? FBA_OK : hip_fail(e, "probe launch");
}

int32_t fba_pair_slots_bounds(const int32_t* q_cnt, const int32_t* q_idx, const int32_t* k_cnt, const int32_t* k_idx, int64_t mask_bh,
                       int32_t nQ, int32_t nK, int32_t* pair_base, int32_t* q_slot, int32_t* bounds, void* hip_stream) {
  if (mask_bh <= 0 || nQ <= 0 || nK <= 0)
    return fail(FBA_ERR_INVALID, "mask_bh, nQ, nK must be positive (got %lld %d %d)", (long long)mask_bh, nQ, nK);
  if (mask_bh * (int64_t)nQ * nK > 0x7fffffffLL) return fail(FBA_ERR_INVALID, "more than 2^31 mask entries");
  if (!q_cnt || !q_idx || !k_cnt || !k_idx || !pair_base || !q_slot) return fail(FBA_ERR_INVALID, "null pointer argument");
  hipError_t e = fba::launch_pair_slots(q_cnt, q_idx, k_cnt, k_idx, mask_bh, nQ, nK, pair_base, q_slot, bounds, (hipStream_t)hip_stream);
  return e == hipSuccess ? FBA_OK : hip_fail(e, "pair_slots launch");
}

int32_t fba_pair_slots(const int32_t* q_cnt, const int32_t* q_idx, const int32_t* k_cnt, const int32_t* k_idx, int64_t mask_bh,
                       int32_t nQ, int32_t nK, int32_t* pair_base, int32_t* q_slot, void* hip_stream) {
  return fba_pair_slots_bounds(q_cnt, q_idx, k_cnt, k_idx, mask_bh, nQ, nK, pair_base, q_slot, nullptr, hip_stream);
}

// Arguments of the dS hand-over, checked once for all three entry points that take them.
static int check_handover(const Shape& s, const void* ds_ws, int64_t ds_ws_bytes, const int32_t* pair_base, int64_t n_pairs, const char* what) {
  if (s.q_block % 128 != 0 || s.k_block % 128 != 0)
    return fail(FBA_ERR_UNSUPPORTED, "%s: the dS hand-over needs q_block (%d) and k_block (%d) to be multiples of 128", what, s.q_block, s.k_block);
  if (!pair_base) return fail(FBA_ERR_INVALID, "pair_base is null");
  if (int rc = check_ptrs({{"ds_ws", ds_ws}})) return rc;
  if (n_pairs < 0) return fail(FBA_ERR_INVALID, "n_pairs must not be negative");
  const int64_t need = n_pairs * (int64_t)s.q_block * s.k_block * 2;
  if (ds_ws_bytes < need)
    return fail(FBA_ERR_INVALID, "%s: ds_ws holds %lld bytes, %lld pairs of %d x %d need %lld", what, (long long)ds_ws_bytes,
                (long long)n_pairs, s.q_block, s.k_block, (long long)need);
  return FBA_OK;
}

static int dkdv_handover_impl(const void* q, const void* k, const void* v, const void* d_o, const float* stats, void* dk, void* dv,
                              void* ds_ws, int64_t ds_ws_bytes, const int32_t* k_cnt, const int32_t* k_idx, const int32_t* pair_base,
                              int64_t n_pairs, int64_t mask_bh, int32_t B, int32_t Hq, int32_t Hkv, int32_t Sq, int32_t Skv,
                              int32_t head_dim, int32_t q_block, int32_t k_block, void* split_ws, int64_t split_ws_bytes,
                              void* hip_stream, const fba::BwdStats& make, fba::Merge* later) {
  const Shape s{mask_bh, B, Hq, Hkv, Sq, Skv, head_dim, q_block, k_block};
  if (int rc = check_shape(s)) return rc;
  if (int rc = check_handover(s, ds_ws, ds_ws_bytes, pair_base, n_pairs, "dkdv")) return rc;
  if (int rc = check_split_ws(split_ws, split_ws_bytes)) return rc;
  if (int rc = check_ptrs({{"q", q}, {"k", k}, {"v", v}, {"d_o", d_o}, {"dk", dk}, {"dv", dv}})) return rc;
  if (!stats || !k_cnt || !k_idx) return fail(FBA_ERR_INVALID, "null pointer argument");
  if ((int64_t)B * Hq * Sq >= (1LL << 30)) return fail(FBA_ERR_INVALID, "B*Hq*Sq must be below 2^30");
  fba::BwdParams p{};
  fill_bwd(p, s);
  p.q = (const __bf16*)q; p.k = (const __bf16*)k; p.v = (const __bf16*)v; p.d_o = (const __bf16*)d_o;
  p.stats = stats; p.make = make; p.dk = (__bf16*)dk; p.dv = (__bf16*)dv; p.k_cnt = k_cnt; p.k_idx = k_idx;
  p.ds_ws = (__bf16*)ds_ws; p.pair_base = pair_base;
  p.ws_pairs = ds_ws_bytes / ((int64_t)q_block * k_block * 2);
  p.split.ws = (float*)split_ws; p.split_ws_bytes = split_ws_bytes;
  hipError_t e = launch_dkdv_variant(p, (hipStream_t)hip_stream, later);
  return e == hipSuccess ? FBA_OK : hip_fail(e, "dkdv (hand-over) launch");
}

int32_t fba_bwd_dkdv_handover(const void* q, const void* k, const void* v, const void* d_o, const float* stats, void* dk, void* dv,
                              void* ds_ws, int64_t ds_ws_bytes, const int32_t* k_cnt, const int32_t* k_idx, const int32_t* pair_base,
                              int64_t n_pairs, int64_t mask_bh, int32_t B, int32_t Hq, int32_t Hkv, int32_t Sq, int32_t Skv,
                              int32_t head_dim, int32_t q_block, int32_t k_block, void* split_ws, int64_t split_ws_bytes,
                              void* hip_stream) {
  return dkdv_handover_impl(q, k, v, d_o, stats, dk, dv, ds_ws, ds_ws_bytes, k_cnt, k_idx, pair_base, n_pairs, mask_bh, B, Hq, Hkv, Sq, Skv, head_dim,
                            q_block, k_block, split_ws, split_ws_bytes, hip_stream, {}, nullptr);
}

static int dq_from_ds_impl(const void* k, const void* ds_ws, int64_t ds_ws_bytes, void* dq, const int32_t* q_cnt, const int32_t* q_idx,
                           const int32_t* q_slot, const int32_t* pair_base, int64_t n_pairs, int64_t mask_bh, int32_t B, int32_t Hq,
                           int32_t Hkv, int32_t Sq, int32_t Skv, int32_t head_dim, int32_t q_block, int32_t k_block, void* split_ws,
                           int64_t split_ws_bytes, void* hip_stream, const fba::Merge& before) {
  const Shape s{mask_bh, B, Hq, Hkv, Sq, Skv, head_dim, q_block, k_block};
  if (int rc = check_shape(s)) return rc;
  if (int rc = check_handover(s, ds_ws, ds_ws_bytes, pair_base, n_pairs, "dq")) return rc;
  if (int rc = check_split_ws(split_ws, split_ws_bytes)) return rc;
  if (int rc = check_ptrs({{"k", k}, {"dq", dq}})) return rc;
  if (!q_cnt || !q_idx || !q_slot) return fail(FBA_ERR_INVALID, "null pointer argument");
  fba::BwdParams p{};
  fill_bwd(p, s);
  p.k = (const __bf16*)k; p.dq = (__bf16*)dq; p.q_cnt = q_cnt; p.q_idx = q_idx;
  p.ds_ws = (__bf16*)const_cast<void*>(ds_ws); p.pair_base = pair_base; p.q_slot = q_slot;
  p.ws_pairs = ds_ws_bytes / ((int64_t)q_block * k_block * 2);
  p.split.ws = (float*)split_ws; p.split_ws_bytes = split_ws_bytes;
  hipError_t e = fba::launch_bwd_dq_from_ds(p, (hipStream_t)hip_stream, before);
  return e == hipSuccess ? FBA_OK : hip_fail(e, "dq (from dS) launch");
}

int32_t fba_bwd_dq_from_ds(const void* k, const void* ds_ws, int64_t ds_ws_bytes, void* dq, const int32_t* q_cnt, const int32_t* q_idx,
                           const int32_t* q_slot, const int32_t* pair_base, int64_t n_pairs, int64_t mask_bh, int32_t B, int32_t Hq,
                           int32_t Hkv, int32_t Sq, int32_t Skv, int32_t head_dim, int32_t q_block, int32_t k_block, void* split_ws,
                           int64_t split_ws_bytes, void* hip_stream) {
  return dq_from_ds_impl(k, ds_ws, ds_ws_bytes, dq, q_cnt, q_idx, q_slot, pair_base, n_pairs, mask_bh, B, Hq, Hkv, Sq, Skv, head_dim, q_block, k_block, split_ws,
                         split_ws_bytes, hip_stream, {});
}

int32_t fba_bwd_handover(const void* q, const void* k, const void* v, const void* o, const void* d_o, const float* lse, float* stats,
                         void* ds_ws, int64_t ds_ws_bytes, void* dq, void* dk, void* dv, const int32_t* q_cnt, const int32_t* q_idx,
                         const int32_t* k_cnt, const int32_t* k_idx, const int32_t* pair_base, const int32_t* q_slot, int64_t n_pairs,
                         int64_t mask_bh, int32_t B, int32_t Hq, int32_t Hkv, int32_t Sq, int32_t Skv, int32_t head_dim,
                         int32_t q_block, int32_t k_block, void* split_ws, int64_t split_ws_bytes, void* hip_stream) {
  const Shape s{mask_bh, B, Hq, Hkv, Sq, Skv, head_dim, q_block, k_block};
  if (int rc = check_shape(s)) return rc;
  // everything is validated before the first launch, so that a rejected call leaves nothing on the stream
  if (int rc = check_handover(s, ds_ws, ds_ws_bytes, pair_base, n_pairs, "backward")) return rc;
  if (int rc = check_split_ws(split_ws, split_ws_bytes)) return rc;
  if (int rc = check_ptrs({{"q", q}, {"k", k}, {"v", v}, {"o", o}, {"d_o", d_o}, {"dq", dq}, {"dk", dk}, {"dv", dv}})) return rc;
  if (!lse || !stats || !q_cnt || !q_idx || !k_cnt || !k_idx || !q_slot) return fail(FBA_ERR_INVALID, "null pointer argument");
  if ((int64_t)B * Hq * Sq >= (1LL << 30)) return fail(FBA_ERR_INVALID, "B*Hq*Sq must be below 2^30");
  fba::Merge merge;
  if (int rc = dkdv_handover_impl(q, k, v, d_o, stats, dk, dv, ds_ws, ds_ws_bytes, k_cnt, k_idx, pair_base, n_pairs, mask_bh, B, Hq, Hkv, Sq, Skv, head_dim,
                                  q_block, k_block, split_ws, split_ws_bytes, hip_stream, {(const __bf16*)o, (const __bf16*)d_o, lse, stats, (int64_t)B * Hq * Sq}, &merge))
    return rc;
  return dq_from_ds_impl(k, ds_ws, ds_ws_bytes, dq, q_cnt, q_idx, q_slot, pair_base, n_pairs, mask_bh, B, Hq, Hkv, Sq, Skv, head_dim,
                         q_block, k_block, split_ws, split_ws_bytes, hip_stream, merge);
}

int32_t fba_tile_slots_bounds(const int32_t* kt_cnt, const int32_t* kt_ent, int64_t mask_bh, int32_t n_qt, int32_t n_kt, int32_t* pair_base,
                       int32_t* kt_slot, int32_t* slot_table, int32_t* bounds, void* hip_stream) {
  if (mask_bh <= 0 || n_qt <= 0 || n_kt <= 0)
    return fail(FBA_ERR_INVALID, "mask_bh, n_qt, n_kt must be positive (got %lld %d %d)", (long long)mask_bh, n_qt, n_kt);
  if (mask_bh * (int64_t)n_kt * n_qt * 4 > 0x7fffffffLL) return fail(FBA_ERR_INVALID, "more than 2^31 tile-list entries");
  if (!kt_cnt || !kt_ent || !pair_base || !kt_slot || !slot_table) return fail(FBA_ERR_INVALID, "null pointer argument");
  hipError_t e = fba::launch_tile_slots(kt_cnt, kt_ent, mask_bh, n_qt, n_kt, 4 * n_qt, pair_base, kt_slot, slot_table, bounds, (hipStream_t)hip_stream);
  return e == hipSuccess ? FBA_OK : hip_fail(e, "tile_slots launch");
}

int32_t fba_tile_slots(const int32_t* kt_cnt, const int32_t* kt_ent, int64_t mask_bh, int32_t n_qt, int32_t n_kt, int32_t* pair_base,
                       int32_t* kt_slot, int32_t* slot_table, void* hip_stream) {
  return fba_tile_slots_bounds(kt_cnt, kt_ent, mask_bh, n_qt, n_kt, pair_base, kt_slot, slot_table, nullptr, hip_stream);
}

static int bwd_tiled_impl(const void* q, const void* k, const void* v, const void* o, const void* d_o, void* d_o_ws, const float* lse, float* stats, void* ds_ws,
                          int64_t ds_ws_bytes, void* dq, void* dk, void* dv, const int32_t* qt_cnt, const int32_t* qt_ent, const int32_t* kt_cnt,
                          const int32_t* kt_ent, const int32_t* pair_base, const int32_t* kt_slot, const int32_t* slot_table, int64_t n_pairs, int64_t mask_bh,
                          int32_t B, int32_t Hq, int32_t Hkv, int32_t Sq, int32_t Skv, int32_t out_q, int32_t out_kv, int32_t head_dim, int32_t q_block,
                          int32_t k_block, void* split_ws, int64_t split_ws_bytes, void* hip_stream, bool numbered) {
  const Shape s{mask_bh, B, Hq, Hkv, Sq, Skv, head_dim, q_block, k_block};
  if (int rc = check_shape(s)) return rc;
  if (int rc = check_lists(s, true, "backward")) return rc;
  if (int rc = check_split_ws(split_ws, split_ws_bytes)) return rc;
  // everything is validated before the first launch, so that a rejected call leaves nothing on the stream
  if (int rc = check_ptrs({{"q", q}, {"k", k}, {"v", v}, {"o", o}, {"d_o", d_o}, {"dq", dq}, {"dk", dk}, {"dv", dv}})) return rc;
  if (d_o_ws != nullptr)
    if (int rc = check_ptrs({{"d_o_ws", d_o_ws}})) return rc;
  if (numbered || ds_ws != nullptr)
    if (int rc = check_ptrs({{"ds_ws", ds_ws}})) return rc;
  if (!lse || !stats || !qt_cnt || !qt_ent || !kt_cnt || !kt_ent || (numbered && (!pair_base || !kt_slot || !slot_table))) return fail(FBA_ERR_INVALID, "null pointer argument");
  if ((int64_t)B * Hq * Sq >= (1LL << 30)) return fail(FBA_ERR_INVALID, "B*Hq*Sq must be below 2^30");
  if (out_q <= 0 || out_q > Sq || out_kv <= 0 || out_kv > Skv)
    return fail(FBA_ERR_INVALID, "out_q (%d) and out_kv (%d) must be positive and Sq, Skv (%d, %d) at most", out_q, out_kv, Sq, Skv);
  if (ds_ws != nullptr) {
    if (n_pairs < 0) return fail(FBA_ERR_INVALID, "n_pairs must not be negative");
    const int64_t pairs = numbered ? n_pairs : (int64_t)B * Hq * (Sq / 128) * (Skv / 128), need = pairs * 128 * 128 * 2;
    if (ds_ws_bytes < need)
      return fail(FBA_ERR_INVALID, "backward: ds_ws holds %lld bytes, %lld tile pairs of 128 x 128 need %lld", (long long)ds_ws_bytes, (long long)pairs,
                  (long long)need);
  }
  fba::BwdParams p{};
  fill_bwd(p, s);
  p.make = {(const __bf16*)o, (const __bf16*)d_o, lse, stats, (int64_t)B * Hq * Sq, (__bf16*)d_o_ws, Sq, out_q};
  p.tiled = 1;
  p.out_q = out_q; p.out_kv = out_kv;
  p.q = (const __bf16*)q; p.k = (const __bf16*)k; p.v = (const __bf16*)v; p.d_o = (const __bf16*)(d_o_ws != nullptr ? d_o_ws : d_o);
  p.stats = stats; p.dq = (__bf16*)dq; p.dk = (__bf16*)dk; p.dv = (__bf16*)dv;
  p.q_cnt = qt_cnt; p.q_idx = qt_ent; p.k_cnt = kt_cnt; p.k_idx = kt_ent;
  p.ds_ws = (__bf16*)ds_ws;
  if (numbered) {
    p.pair_base = pair_base; p.k_slot = kt_slot; p.q_slot = slot_table;
    p.ws_pairs = ds_ws_bytes / (128 * 128 * 2);
  }
  p.split.ws = (float*)split_ws; p.split_ws_bytes = split_ws_bytes;
  fba::Merge merge;
  hipError_t e = fba::launch_bwd_dkdv_slab(p, (hipStream_t)hip_stream, &merge);
  if (e != hipSuccess) return hip_fail(e, "dkdv (tile lists) launch");
  e = ds_ws != nullptr ? fba::launch_bwd_dq_from_ds(p, (hipStream_t)hip_stream, merge) : fba::launch_bwd_dq(p, (hipStream_t)hip_stream, merge);
  return e == hipSuccess ? FBA_OK : hip_fail(e, "dq (tile lists) launch");
}

int32_t fba_bwd_tiled_cut(const void* q, const void* k, const void* v, const void* o, const void* d_o, void* d_o_ws, const float* lse, float* stats, void* ds_ws,
                          int64_t ds_ws_bytes, void* dq, void* dk, void* dv, const int32_t* qt_cnt, const int32_t* qt_ent, const int32_t* kt_cnt,
                          const int32_t* kt_ent, const int32_t* pair_base, const int32_t* kt_slot, const int32_t* slot_table, int64_t n_pairs, int64_t mask_bh,
                          int32_t B, int32_t Hq, int32_t Hkv, int32_t Sq, int32_t Skv, int32_t out_q, int32_t out_kv, int32_t head_dim, int32_t q_block,
                          int32_t k_block, void* split_ws, int64_t split_ws_bytes, void* hip_stream) {
  return bwd_tiled_impl(q, k, v, o, d_o, d_o_ws, lse, stats, ds_ws, ds_ws_bytes, dq, dk, dv, qt_cnt, qt_ent, kt_cnt, kt_ent, pair_base, kt_slot, slot_table, n_pairs,
                        mask_bh, B, Hq, Hkv, Sq, Skv, out_q, out_kv, head_dim, q_block, k_block, split_ws, split_ws_bytes, hip_stream, ds_ws != nullptr && pair_base != nullptr);
}

int32_t fba_bwd_tiled_handover(const void* q, const void* k, const void* v, const void* o, const void* d_o, const float* lse, float* stats,
                               void* ds_ws, int64_t ds_ws_bytes, void* dq, void* dk, void* dv, const int32_t* qt_cnt,
                               const int32_t* qt_ent, const int32_t* kt_cnt, const int32_t* kt_ent, const int32_t* pair_base,
                               const int32_t* kt_slot, const int32_t* slot_table, int64_t n_pairs, int64_t mask_bh, int32_t B,
                               int32_t Hq, int32_t Hkv, int32_t Sq, int32_t Skv, int32_t head_dim, int32_t q_block, int32_t k_block,
                               void* split_ws, int64_t split_ws_bytes, void* hip_stream) {
  return bwd_tiled_impl(q, k, v, o, d_o, nullptr, lse, stats, ds_ws, ds_ws_bytes, dq, dk, dv, qt_cnt, qt_ent, kt_cnt, kt_ent, pair_base, kt_slot, slot_table, n_pairs,
                        mask_bh, B, Hq, Hkv, Sq, Skv, Sq, Skv, head_dim, q_block, k_block, split_ws, split_ws_bytes, hip_stream, true);
}

}  // extern "C"

namespace {

// Workspace of fba_bwd_noalloc: the two statistics planes of backward (lse * log2(e), -delta) for up to kScratchRows
// query rows, 32 MiB, held by every GPU the library is loaded on until the process ends.  In host code the array's name
// is only a handle for hipGetSymbolAddress; kernels get the device address looked up below.
constexpr int64_t kScratchRows = 1LL << 22;
constexpr int kMaxDevices = 64;
static __device__ __align__(256) float scratch[2 * kScratchRows];
float* g_scratch_addr[kMaxDevices] = {};
std::mutex g_scratch_mutex;

// Device address of `scratch` on the current device (each GPU has its own copy at its own address); looked up on the
// first call on that device.
int scratch_address(float** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return hip_fail(e, "hipGetDevice");
  if (dev < 0 || dev >= kMaxDevices) return fail(FBA_ERR_UNSUPPORTED, "device ordinal %d is beyond the %d devices supported", dev, kMaxDevices);
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (g_scratch_addr[dev] == nullptr) {
    void* ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return hip_fail(e, "hipGetSymbolAddress(scratch)");
    if (ptr == nullptr) return fail(FBA_ERR_HIP, "hipGetSymbolAddress(scratch) returned a null address");
    g_scratch_addr[dev] = static_cast<float*>(ptr);
  }
  *out = g_scratch_addr[dev];
  return FBA_OK;
}

}  // namespace

extern "C" {

int32_t fba_lists_cut(const uint8_t* mask, int64_t mask_bh, int32_t nQ, int32_t nK, int32_t mask_q, int32_t mask_k, int32_t q_block, int32_t k_block,
                      int32_t* q_cnt, int32_t* q_idx, int32_t* k_cnt, int32_t* k_idx, void* hip_stream) {
  const bool both = k_cnt != nullptr && k_idx != nullptr;
  if (!both && (k_cnt != nullptr || k_idx != nullptr)) return fail(FBA_ERR_INVALID, "k_cnt and k_idx must both be given or both be null");
  if (mask_bh <= 0 || nQ <= 0 || nK <= 0)
    return fail(FBA_ERR_INVALID, "mask_bh, nQ, nK must be positive (got %lld %d %d)", (long long)mask_bh, nQ, nK);
  if (mask_q <= 0 || mask_q > nQ || mask_k <= 0 || mask_k > nK)
    return fail(FBA_ERR_INVALID, "the mask's rows and columns (%d, %d) must be positive and nQ, nK (%d, %d) at most", mask_q, mask_k, nQ, nK);
  if (!mask || !q_cnt || !q_idx) return fail(FBA_ERR_INVALID, "null pointer argument");
  hipError_t e;
  if (q_block % 128 == 0 && k_block % 128 == 0) {
    if (mask_q != nQ || mask_k != nK) return fail(FBA_ERR_INVALID, "block lists are of whole masks (got %d, %d of %d, %d)", mask_q, mask_k, nQ, nK);
    e = fba::launch_mask_compact(mask, mask_bh, nQ, nK, q_cnt, q_idx, k_cnt, k_idx, (hipStream_t)hip_stream);
  } else {
    if (int rc = check_tile_list_shape(nQ, nK, q_block, k_block)) return rc;
    const int64_t Sq = (int64_t)nQ * q_block, Skv = (int64_t)nK * k_block;
    e = fba::launch_tile_lists(mask, mask_bh, mask_q, mask_k, nK, q_block, k_block, (int)(Sq / 128), both ? (int)(Skv / 128) : 0, (int)(Sq / 32), q_cnt, q_idx,
                               k_cnt, k_idx, (hipStream_t)hip_stream);
  }
  return e == hipSuccess ? FBA_OK : hip_fail(e, "list launch");
}

int32_t fba_lists(const uint8_t* mask, int64_t mask_bh, int32_t nQ, int32_t nK, int32_t q_block, int32_t k_block, int32_t* q_cnt,
                  int32_t* q_idx, int32_t* k_cnt, int32_t* k_idx, void* hip_stream) {
  return fba_lists_cut(mask, mask_bh, nQ, nK, nQ, nK, q_block, k_block, q_cnt, q_idx, k_cnt, k_idx, hip_stream);
}

int32_t fba_resize_rows(int32_t n, const void* const* src, void* const* dst, const int64_t* n_seq, const int32_t* src_len, const int32_t* dst_len,
                        void* hip_stream) {
  if (n < 1 || n > 3) return fail(FBA_ERR_INVALID, "resize_rows takes one to three tensors (got %d)", n);
  if (!src || !dst || !n_seq || !src_len || !dst_len) return fail(FBA_ERR_INVALID, "null pointer argument");
  for (int j = 0; j < n; ++j) {
    if (int rc = check_ptrs({{"src", src[j]}, {"dst", dst[j]}})) return rc;
    if (n_seq[j] <= 0 || src_len[j] <= 0 || dst_len[j] <= 0)
      return fail(FBA_ERR_INVALID, "sequences and lengths must be positive (got %lld %d %d)", (long long)n_seq[j], src_len[j], dst_len[j]);
    if (n_seq[j] >= (1LL << 31)) return fail(FBA_ERR_INVALID, "too many sequences (%lld)", (long long)n_seq[j]);
  }
  hipError_t e = fba::launch_resize_rows(n, src, dst, n_seq, src_len, dst_len, (hipStream_t)hip_stream);
  return e == hipSuccess ? FBA_OK : hip_fail(e, "resize_rows launch");
}

int32_t fba_resize_mask(const uint8_t* src, uint8_t* dst, int64_t mask_bh, int32_t src_q, int32_t src_k, int32_t dst_q, int32_t dst_k, void* hip_stream) {
  if (mask_bh <= 0 || src_q <= 0 || src_k <= 0 || dst_q <= 0 || dst_k <= 0)
    return fail(FBA_ERR_INVALID, "mask_bh and the numbers of blocks must be positive (got %lld %d %d %d %d)", (long long)mask_bh, src_q, src_k, dst_q, dst_k);
  if (mask_bh >= (1LL << 31)) return fail(FBA_ERR_INVALID, "too many masks (%lld)", (long long)mask_bh);
  if (!src || !dst) return fail(FBA_ERR_INVALID, "null pointer argument");
  hipError_t e = fba::launch_resize_mask(src, dst, mask_bh, src_q, src_k, dst_q, dst_k, (hipStream_t)hip_stream);
  return e == hipSuccess ? FBA_OK : hip_fail(e, "resize_mask launch");
}

// For problems that take less time than it costs to number their pairs and to wait for the count: B1 H2 S1536, 384-token
// blocks, forward + backward 304 -> 224 us against numbered pairs (four launches, a pinned copy and a wait less); B2 H8/2
// S3136 q16 k64 430 -> 332 us.  The price is a workspace of all pairs instead of the selected ones, so the caller draws the
// line where its memory limit does.
int32_t fba_bwd_dense(const void* q, const void* k, const void* v, const void* o, const void* d_o, const float* lse, float* stats,
                      void* ds_ws, int64_t ds_ws_bytes, void* dq, void* dk, void* dv, const int32_t* q_cnt, const int32_t* q_idx,
                      const int32_t* k_cnt, const int32_t* k_idx, int64_t mask_bh, int32_t B, int32_t Hq, int32_t Hkv, int32_t Sq,
                      int32_t Skv, int32_t head_dim, int32_t q_block, int32_t k_block, void* split_ws, int64_t split_ws_bytes,
                      void* hip_stream) {
  const Shape s{mask_bh, B, Hq, Hkv, Sq, Skv, head_dim, q_block, k_block};
  if (int rc = check_shape(s)) return rc;
  const bool tiled = q_block % 128 != 0 || k_block % 128 != 0;
  if (int rc = check_lists(s, tiled, "backward")) return rc;
  if (int rc = check_split_ws(split_ws, split_ws_bytes)) return rc;
  // everything is validated before the first launch, so that a rejected call leaves nothing on the stream
  if (int rc = check_ptrs({{"q", q}, {"k", k}, {"v", v}, {"o", o}, {"d_o", d_o}, {"dq", dq}, {"dk", dk}, {"dv", dv}, {"ds_ws", ds_ws}})) return rc;
  if (!lse || !stats || !q_cnt || !q_idx || !k_cnt || !k_idx) return fail(FBA_ERR_INVALID, "null pointer argument");
  if ((int64_t)B * Hq * Sq >= (1LL << 30)) return fail(FBA_ERR_INVALID, "B*Hq*Sq must be below 2^30");
  const int64_t need = (int64_t)B * Hq * Sq * Skv * 2;
  if (ds_ws_bytes < need)
    return fail(FBA_ERR_INVALID, "backward: ds_ws holds %lld bytes, all pairs of %d heads, %d x %d, need %lld", (long long)ds_ws_bytes, B * Hq, Sq,
                Skv, (long long)need);
  fba::BwdParams p{};
  fill_bwd(p, s);
  p.make = {(const __bf16*)o, (const __bf16*)d_o, lse, stats, (int64_t)B * Hq * Sq};
  p.tiled = tiled ? 1 : 0;
  p.q = (const __bf16*)q; p.k = (const __bf16*)k; p.v = (const __bf16*)v; p.d_o = (const __bf16*)d_o;
  p.stats = stats; p.dq = (__bf16*)dq; p.dk = (__bf16*)dk; p.dv = (__bf16*)dv;
  p.q_cnt = q_cnt; p.q_idx = q_idx; p.k_cnt = k_cnt; p.k_idx = k_idx;
  p.ds_ws = (__bf16*)ds_ws;  // pair_base stays null: dense numbering
  p.split.ws = (float*)split_ws; p.split_ws_bytes = split_ws_bytes;
  fba::Merge merge;
  hipError_t e = launch_dkdv_variant(p, (hipStream_t)hip_stream, &merge);
  if (e != hipSuccess) return hip_fail(e, "dkdv (dense hand-over) launch");
  e = fba::launch_bwd_dq_from_ds(p, (hipStream_t)hip_stream, merge);
  return e == hipSuccess ? FBA_OK : hip_fail(e, "dq (from dS, dense) launch");
}

int32_t fba_bwd_noalloc(const void* q, const void* k, const void* v, const void* o, const void* d_o, const float* lse,
                        void* dq, void* dk, void* dv, const int32_t* q_cnt, const int32_t* q_idx, const int32_t* k_cnt,
                        const int32_t* k_idx, int64_t mask_bh, int32_t B, int32_t Hq, int32_t Hkv, int32_t Sq, int32_t Skv,
                        int32_t head_dim, int32_t q_block, int32_t k_block, void* hip_stream) {
  const int64_t rows = (int64_t)B * Hq * Sq;
  if (B > 0 && Hq > 0 && Sq > 0 && rows > kScratchRows)
    return fail(FBA_ERR_UNSUPPORTED, "fba_bwd_noalloc: B*Hq*Sq = %lld query rows exceed the built-in workspace of %lld rows; "
                "call fba_bwd with a caller-owned stats buffer", (long long)rows, (long long)kScratchRows);
  float* stats = nullptr;
  if (int rc = scratch_address(&stats)) return rc;
  return bwd_impl(q, k, v, o, d_o, lse, stats, dq, dk, dv, q_cnt, q_idx, k_cnt, k_idx, mask_bh, B, Hq, Hkv, Sq, Skv, head_dim,
                  q_block, k_block, nullptr, 0, hip_stream, false);
}

int32_t fba_bwd_tiled(const void* q, const void* k, const void* v, const void* o, const void* d_o, const float* lse,
                      float* stats, void* dq, void* dk, void* dv, const int32_t* qt_cnt, const int32_t* qt_ent,
                      const int32_t* kt_cnt, const int32_t* kt_ent, int64_t mask_bh, int32_t B, int32_t Hq, int32_t Hkv,
                      int32_t Sq, int32_t Skv, int32_t head_dim, int32_t q_block, int32_t k_block,
                      void* split_ws, int64_t split_ws_bytes, void* hip_stream) {
  return bwd_impl(q, k, v, o, d_o, lse, stats, dq, dk, dv, qt_cnt, qt_ent, kt_cnt, kt_ent, mask_bh, B, Hq, Hkv, Sq, Skv, head_dim,
                  q_block, k_block, split_ws, split_ws_bytes, hip_stream, true);
}

}  // extern "C"
