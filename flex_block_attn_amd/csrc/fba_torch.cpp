// Host side of the operator in native code: what runs between a call of flex_block_attn_func and the kernels of
// libfba_gfx950.so, and the autograd node that carries it.  Everything here is host work around the C ABI of include/fba.h:
// checks, allocations from torch's caching allocator, the plan of the backward pass, launches.
//
// Why native: on small problems the kernels take a few tens of microseconds, and the same steps in Python took several times
// that.  Per call, Python / native: B1 H1 S768, 128-token blocks, forward 45 / 16 us; B1 H2 S1536, 384-token blocks, forward +
// backward 224 / 88 us; large problems the same.
//
// The library is not linked but bound by path (bind), so that FBA_LIBRARY can name another build of it.
#include <dlfcn.h>

#include <cstdlib>
#include <numeric>

#include <ATen/ATen.h>
#include <ATen/core/CachingHostAllocator.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/Event.h>
#include <c10/core/impl/VirtualGuardImpl.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/custom_class.h>
#include <torch/extension.h>

#include "../../include/fba.h"

// Which torch this was compiled against.  The loader looks for this text in the file before it loads it (another torch's ABI may
// differ without a symbol that does not resolve), so it has to stay in the image.
extern "C" __attribute__((used, visibility("default"))) const char fba_torch_built_for[] = "fba_torch built for torch " FBA_TORCH_BUILD ";";

namespace {

constexpr int64_t kHeadDim = 128;
constexpr int64_t kXcds = 8;

// ---------------------------------------------------------------------------------------------------------------------
// the C ABI, bound at run time
// ---------------------------------------------------------------------------------------------------------------------
#define FBA_FUNCTIONS(X)                                                                                                \
  X(fba_version) X(fba_last_error) X(fba_split_workspace_bytes) X(fba_lists_cut) X(fba_pair_slots_bounds) X(fba_tile_slots_bounds)        \
  X(fba_fwd) X(fba_fwd_tiled) X(fba_fwd_blocks) X(fba_fwd_blocks_use) X(fba_fwd_mask_copy) X(fba_fwd_takes_mask) X(fba_bwd_mask) X(fba_bwd_takes_mask) X(fba_bwd) X(fba_bwd_handover) X(fba_bwd_tiled_cut) X(fba_bwd_dense) \
  X(fba_resize_rows) X(fba_resize_mask)

struct Library {
#define DECLARE(f) decltype(&::f) f = nullptr;
  FBA_FUNCTIONS(DECLARE)
#undef DECLARE
} lib;

// Everything is resolved before anything is replaced: a library that is refused leaves the one in use bound.
void bind(const std::string& path) {
  void* handle = dlopen(path.c_str(), RTLD_NOW | RTLD_LOCAL);
  TORCH_CHECK(handle != nullptr, "cannot load ", path, ": ", dlerror());
  Library found;
#define RESOLVE(f)                                                    \
  found.f = reinterpret_cast<decltype(&::f)>(dlsym(handle, #f));      \
  TORCH_CHECK(found.f != nullptr, path, " does not export ", #f);
  FBA_FUNCTIONS(RESOLVE)
#undef RESOLVE
  // the argument lists of this module are those of the header it was compiled with
  if (found.fba_version() != FBA_VERSION)
    throw pybind11::import_error(path + " reports version " + std::to_string(found.fba_version()) + ", the host module was built for version " +
                                 std::to_string(FBA_VERSION) + ": rebuild both with `python -m flex_block_attn_amd.build`");
  lib = found;
}

// A failed C ABI call raises _lib.FbaError.  It is set as a Python error here, and not translated where a call returns to
// Python, because a failure in backward travels through the autograd engine, which hands on Python errors as they are and
// makes a plain RuntimeError of any other exception.
[[noreturn]] void raise_call_error(int code) {
  const std::string message = lib.fba_last_error();  // of this thread
  pybind11::gil_scoped_acquire gil;
  const pybind11::object type = pybind11::module_::import("flex_block_attn_amd._lib").attr("FbaError");
  PyErr_SetObject(type.ptr(), type(code, message).ptr());
  python_error error;
  error.persist();
  throw error;
}
void check(int code) {
  if (code != FBA_OK) raise_call_error(code);
}

void* current_stream(const at::Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

// ---------------------------------------------------------------------------------------------------------------------
// shapes and lists
// ---------------------------------------------------------------------------------------------------------------------
struct Problem {
  int64_t B, Hq, Hkv, Sq, Skv, q_block, k_block, mask_bh;
  bool tiled() const { return q_block % 128 != 0 || k_block % 128 != 0; }
  int64_t nQ() const { return Sq / q_block; }
  int64_t nK() const { return Skv / k_block; }
  int64_t pair_bytes() const { return (tiled() ? 128 * 128 : q_block * k_block) * 2; }
  int64_t dense_bytes() const { return B * Hq * Sq * Skv * 2; }
};

// What the kernels read: query-major and key-major lists (block lists or tile lists) and, once the pairs are numbered, their
// numbers (see include/fba.h).
struct Lists {
  int32_t *q_cnt = nullptr, *q_idx = nullptr, *k_cnt = nullptr, *k_idx = nullptr;
  int32_t *pair_base = nullptr, *q_slot = nullptr, *k_slot = nullptr;
  int64_t q_rows, q_len, k_rows, k_len, slot_len;  // per head of the mask
  explicit Lists(const Problem& p) {
    q_rows = p.tiled() ? p.Sq / 128 : p.nQ();
    q_len = p.nK();
    k_rows = p.tiled() ? p.Skv / 128 : p.nK();
    k_len = p.tiled() ? p.Sq / 32 : p.nQ();
    slot_len = p.tiled() ? p.Skv / 128 : p.nK();  // entries of a q_slot row
  }
};

// Largest dS workspace backward allocates on its own: at most `limit` bytes, and at most `factor` times the bytes of the
// call's own tensors (q, o, dO, dq and k, v, dk, dv in bf16).
int64_t ds_limit(const Problem& p, double limit, double factor) {
  const double own = 2.0 * kHeadDim * (5.0 * p.B * p.Hq * p.Sq + 4.0 * p.B * p.Hkv * p.Skv);
  return (int64_t)std::min(limit, factor * own);
}

// Is backward to hand dS over in a workspace with a place for every pair?  It takes a constant off a step, two launches, a pinned
// copy and a wait (17-36 us), and costs memory that grows with all pairs instead of the selected ones.  So the line is drawn
// where the constant is 2 to 5 % of a step, and the memory stays under 1 % of the card's.  Steps with pairs numbered / dense,
// 10 % and 40 % kept, 128-token blocks: H4 S4096 (128 MiB) 110 / 84 and 136 / 114 us; H24 S3072 (432 MiB) 165 / 145 and 279 / 261;
// H24 S4096 (768 MiB) 187 / 170 and 369 / 352; H24 S5120 (1.2 GiB) 252 / 235 and 570 / 550; H24 S6784 (2.1 GiB) 378 / 362 and
// 927 / 910; B2 H22 S3584, 64 x 128 blocks, 57 % kept (1.05 GiB) 830 / 794.
// Steps recorded into a graph use it as far as the limit allows: the wait for the pair count cannot be captured.
constexpr int64_t kDenseMost = 2LL << 30;
bool dense_fits(int64_t bytes, int64_t limit) {
  if (bytes > limit) return false;
  if (bytes <= kDenseMost) return true;
  pybind11::gil_scoped_acquire gil;
  return pybind11::module_::import("torch").attr("cuda").attr("is_current_stream_capturing")().cast<bool>();
}

// Listed pairs of every (batch, kv head) unit, from the pair numbers at the head boundaries of the mask: the heads of a GQA group
// share their kv head's launch.
std::vector<int64_t> unit_pairs(const std::vector<int64_t>& bounds, int64_t units, int64_t group) {
  std::vector<int64_t> pairs(units);
  const bool shared = bounds.size() == 2;  // one mask for all heads
  for (int64_t u = 0; u < units; ++u) pairs[u] = shared ? bounds[1] * group : bounds[(u + 1) * group] - bounds[u * group];
  return pairs;
}

using Chunk = std::tuple<int64_t, int64_t, int64_t>;  // first unit, end unit, pairs

// Cuts the (batch, kv head) units into consecutive chunks of equal length whose dS fits `limit` bytes: as few chunks as the
// total needs, shortened while some chunk is still too large, and then, if a chunk holds more than one unit per XCD,
// shortened to a multiple of the XCD count (twelve heads per chunk cost dK/dV 3 % against eight).  Nothing when a single
// unit does not fit.
c10::optional<std::vector<Chunk>> plan_head_chunks(const std::vector<int64_t>& unit_pairs, int64_t pair_bytes, int64_t limit) {
  const int64_t n = (int64_t)unit_pairs.size();
  int64_t total = 0;
  for (int64_t u : unit_pairs) total += u;
  total *= pair_bytes;
  if (total == 0) return std::vector<Chunk>{{0, n, 0}};
  auto cut = [&](int64_t per) {
    std::vector<Chunk> chunks;
    for (int64_t u = 0; u < n; u += per) {
      int64_t pairs = 0;
      for (int64_t i = u; i < std::min(n, u + per); ++i) pairs += unit_pairs[i];
      chunks.emplace_back(u, std::min(n, u + per), pairs);
    }
    return chunks;
  };
  auto fits = [&](int64_t per) {
    for (const Chunk& c : cut(per))
      if (std::get<2>(c) * pair_bytes > limit) return false;
    return true;
  };
  if (limit <= 0) return c10::nullopt;
  const int64_t want = (total + limit - 1) / limit;
  int64_t per = (n + want - 1) / want;
  while (per >= 1 && !fits(per)) --per;
  if (per < 1) return c10::nullopt;
  if (per < n && per > kXcds && per % kXcds != 0 && fits(per - per % kXcds)) per -= per % kXcds;
  return cut(per);
}

struct SplitWorkspace {  // see "Tail splitting" in include/fba.h
  at::Tensor buffer;
  int64_t bytes;
  SplitWorkspace(const at::Tensor& like, int64_t n) : bytes(n) {
    if (n > 0) buffer = at::empty({n}, like.options().dtype(at::kByte));
  }
  void* ptr() const { return bytes > 0 ? buffer.data_ptr() : nullptr; }
};

// ---------------------------------------------------------------------------------------------------------------------
// forward and backward on lists
// ---------------------------------------------------------------------------------------------------------------------
std::pair<at::Tensor, at::Tensor> run_forward(const Problem& p, const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const Lists& l,
                                              int64_t split_bytes) {
  at::Tensor o = at::empty_like(q);
  at::Tensor lse = at::empty({p.B, p.Hq, p.Sq, 1}, q.options().dtype(at::kFloat));
  SplitWorkspace split(q, split_bytes);
  check((p.tiled() ? lib.fba_fwd_tiled : lib.fba_fwd)(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), lse.data_ptr<float>(), l.q_cnt, l.q_idx,
                                                      p.mask_bh, p.B, p.Hq, p.Hkv, p.Sq, p.Skv, kHeadDim, p.q_block, p.k_block, split.ptr(),
                                                      split.bytes, current_stream(q)));
  return {o, lse};
}

// The same on the block mask, where fba_fwd_blocks takes it.  The 384-row work-groups that FBA_FWD_TILE_ROWS asks for read lists.
int blocks_use(const Problem& p) {
  const int use = lib.fba_fwd_blocks_use(p.mask_bh, p.B, p.Hq, p.Sq, p.Skv, p.q_block, p.k_block);
  const char* const rows = use != 0 && p.q_block % 384 == 0 ? std::getenv("FBA_FWD_TILE_ROWS") : nullptr;
  return rows == nullptr || std::atoi(rows) != 384 ? use : 0;
}
std::pair<at::Tensor, at::Tensor> run_forward_on_blocks(const Problem& p, const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const at::Tensor& mask,
                                                        const Lists& make, int64_t split_bytes) {
  at::Tensor o = at::empty_like(q);
  at::Tensor lse = at::empty({p.B, p.Hq, p.Sq, 1}, q.options().dtype(at::kFloat));
  SplitWorkspace split(q, split_bytes);
  check(lib.fba_fwd_blocks(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), lse.data_ptr<float>(), static_cast<const uint8_t*>(mask.data_ptr()), make.q_cnt, make.q_idx,
                           make.k_cnt, make.k_idx, p.mask_bh, p.B, p.Hq, p.Hkv, p.Sq, p.Skv, kHeadDim, p.q_block, p.k_block, split.ptr(), split.bytes,
                           current_stream(q)));
  return {o, lse};
}

// Does forward read the block mask itself?  (Decided on the padded lengths, whether or not the call pads.)
bool takes_mask(const Problem& p) { return lib.fba_fwd_takes_mask(p.B * p.Hq * p.Sq, p.Skv) != 0; }

// Does backward, too?  Then neither pass builds lists, and nothing is padded.
bool backward_takes_mask(const Problem& p) { return takes_mask(p) && lib.fba_bwd_takes_mask(p.B, p.Hq, p.Hkv, p.Sq, p.Skv) != 0; }

// Forward from the mask; q, k, v as the caller has them (lengths need not be whole tiles).  mask_copy: null, or where a copy of the mask
// goes.  o_rows: rows of a head of o, as many as q has or more.
std::pair<at::Tensor, at::Tensor> run_forward_on_mask(const Problem& p, const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const at::Tensor& mask,
                                                      void* mask_copy = nullptr, int64_t o_rows = 0) {
  o_rows = std::max(o_rows, q.size(2));
  at::Tensor o = at::empty({p.B, p.Hq, o_rows, kHeadDim}, q.options());
  at::Tensor lse = at::empty({p.B, p.Hq, q.size(2), 1}, q.options().dtype(at::kFloat));
  check(lib.fba_fwd_mask_copy(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), lse.data_ptr<float>(), static_cast<const uint8_t*>(mask.data_ptr()),
                              static_cast<uint8_t*>(mask_copy), o_rows, p.mask_bh, p.B, p.Hq, p.Hkv, q.size(2), k.size(2), kHeadDim, p.q_block, p.k_block,
                              current_stream(q)));
  return {o, lse};
}

// Backward from the mask; p as forward had it.
std::vector<at::Tensor> run_backward_on_mask(const Problem& p, const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const at::Tensor& o,
                                             const at::Tensor& lse, const at::Tensor& d_o, const at::Tensor& mask) {
  at::Tensor dq = at::empty_like(q), dk = at::empty_like(k), dv = at::empty_like(v);
  check(lib.fba_bwd_mask(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), d_o.data_ptr(), lse.data_ptr<float>(),
                         static_cast<const uint8_t*>(mask.data_ptr()), o.size(2), p.mask_bh, dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), p.B, p.Hq, p.Hkv, q.size(2),
                         k.size(2), kHeadDim, p.q_block, p.k_block, current_stream(q)));
  return {dq, dk, dv};
}

enum class HandOver { kNever, kAuto, kWhole };  // dQ recomputes; as the limits allow; all heads at once whatever the size

// bounds: pair numbers at the head boundaries of the mask (mask_bh + 1 of them); empty: pairs not numbered.  out_q, out_kv: rows of a head of dq
// and of dk, dv (0: as many as q and k have; fewer on tile lists only); d_o has out_q as well.
std::vector<at::Tensor> run_backward(const Problem& p, const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const at::Tensor& o,
                                     const at::Tensor& lse, const at::Tensor& d_o, const Lists& l, const std::vector<int64_t>& bounds, HandOver mode,
                                     bool dense, int64_t limit, int64_t split_bytes, int64_t out_q = 0, int64_t out_kv = 0) {
  if (out_q == 0) out_q = p.Sq;
  if (out_kv == 0) out_kv = p.Skv;
  at::Tensor dq = at::empty({p.B, p.Hq, out_q, kHeadDim}, q.options()), dk = at::empty({p.B, p.Hkv, out_kv, kHeadDim}, k.options()), dv = at::empty_like(dk);
  const at::Tensor d_o_ws = out_q != p.Sq ? at::empty_like(q) : at::Tensor();  // (dO filled up to whole tiles)
  void* const stream = current_stream(q);
  const int64_t group = p.Hq / p.Hkv, units = p.B * p.Hkv;
  auto workspace = [&](int64_t bytes) {
    at::Tensor ws;
    try {
      ws = at::empty({bytes}, q.options().dtype(at::kByte));
    } catch (const c10::OutOfMemoryError&) {
      if (mode == HandOver::kWhole) throw;
    }
    return ws;
  };
  at::Tensor ds;
  c10::optional<std::vector<Chunk>> chunks;
  if (dense) {
    ds = workspace(p.dense_bytes());
  } else if (mode != HandOver::kNever && !bounds.empty()) {
    const std::vector<int64_t> pairs = unit_pairs(bounds, units, group);
    int64_t total = std::accumulate(pairs.begin(), pairs.end(), int64_t{0}), most = 0;
    if (total > 0) {
      if (mode == HandOver::kWhole) chunks = std::vector<Chunk>{{0, units, total}};
      else chunks = plan_head_chunks(pairs, p.pair_bytes(), limit);
    }
    if (chunks) {
      for (const Chunk& c : *chunks) most = std::max(most, std::get<2>(c));
      ds = workspace(most * p.pair_bytes());
    }
  }
  SplitWorkspace split(q, split_bytes);
  const auto f32 = q.options().dtype(at::kFloat);
  if (!ds.defined() || dense) {
    at::Tensor stats = at::empty({2, p.B, p.Hq, p.Sq}, f32);
    if (p.tiled())
      check(lib.fba_bwd_tiled_cut(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), d_o.data_ptr(), d_o_ws.defined() ? d_o_ws.data_ptr() : nullptr,
                                  lse.data_ptr<float>(), stats.data_ptr<float>(),
                                  ds.defined() ? ds.data_ptr() : nullptr, ds.defined() ? ds.numel() : 0, dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), l.q_cnt,
                                  l.q_idx, l.k_cnt, l.k_idx, nullptr, nullptr, nullptr, 0, p.mask_bh, p.B, p.Hq, p.Hkv, p.Sq, p.Skv, out_q, out_kv, kHeadDim,
                                  p.q_block, p.k_block, split.ptr(), split.bytes, stream));
    else if (ds.defined())
      check(lib.fba_bwd_dense(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), d_o.data_ptr(), lse.data_ptr<float>(), stats.data_ptr<float>(),
                              ds.data_ptr(), ds.numel(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), l.q_cnt, l.q_idx, l.k_cnt, l.k_idx, p.mask_bh,
                              p.B, p.Hq, p.Hkv, p.Sq, p.Skv, kHeadDim, p.q_block, p.k_block, split.ptr(), split.bytes, stream));
    else
      check(lib.fba_bwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), d_o.data_ptr(), lse.data_ptr<float>(), stats.data_ptr<float>(), dq.data_ptr(),
                        dk.data_ptr(), dv.data_ptr(), l.q_cnt, l.q_idx, l.k_cnt, l.k_idx, p.mask_bh, p.B, p.Hq, p.Hkv, p.Sq, p.Skv, kHeadDim, p.q_block,
                        p.k_block, split.ptr(), split.bytes, stream));
    return {dq, dk, dv};
  }
  // One launch sequence per chunk of kv heads [u0, u1): every pointer moves to the chunk's first head, the chunk is described
  // as a batch of one, and the workspace pointer is moved back by the pairs of the heads in front of the chunk, so that the
  // absolute pair numbers of the lists land inside the workspace.
  int64_t longest = 0;
  for (const Chunk& c : *chunks) longest = std::max(longest, std::get<1>(c) - std::get<0>(c));
  at::Tensor stats = at::empty({2, longest * group * p.Sq}, f32);
  auto bf16_at = [](const at::Tensor& t, int64_t elements) { return static_cast<char*>(t.data_ptr()) + 2 * elements; };
  for (const auto& [u0, u1, pairs] : *chunks) {
    const int64_t h0 = u0 * group, nh = (u1 - u0) * group, nu = u1 - u0;
    const int64_t m0 = p.mask_bh > 1 ? h0 : 0;  // first head of the list tensors
    const int64_t qo = h0 * p.Sq * kHeadDim, ko = u0 * p.Skv * kHeadDim;
    char* const ws = static_cast<char*>(ds.data_ptr()) - (p.mask_bh > 1 ? bounds[h0] * p.pair_bytes() : 0);
    const int64_t mask_bh = p.mask_bh > 1 ? nh : 1;
    const float* lse0 = lse.data_ptr<float>() + h0 * p.Sq;
    const int32_t *q_cnt = l.q_cnt + m0 * l.q_rows, *q_idx = l.q_idx + m0 * l.q_rows * l.q_len;
    const int32_t *k_cnt = l.k_cnt + m0 * l.k_rows, *k_idx = l.k_idx + m0 * l.k_rows * l.k_len;
    const int32_t *base = l.pair_base + m0 * l.k_rows, *q_slot = l.q_slot + m0 * l.q_rows * l.slot_len;
    if (p.tiled())
      check(lib.fba_bwd_tiled_cut(bf16_at(q, qo), bf16_at(k, ko), bf16_at(v, ko), bf16_at(o, qo), bf16_at(d_o, h0 * out_q * kHeadDim),
                                  d_o_ws.defined() ? bf16_at(d_o_ws, qo) : nullptr, lse0, stats.data_ptr<float>(), ws,
                                  pairs * p.pair_bytes(), bf16_at(dq, h0 * out_q * kHeadDim), bf16_at(dk, u0 * out_kv * kHeadDim),
                                  bf16_at(dv, u0 * out_kv * kHeadDim), q_cnt, q_idx, k_cnt, k_idx, base, l.k_slot + m0 * l.k_rows * l.k_len, q_slot, pairs,
                                  mask_bh, 1, nh, nu, p.Sq, p.Skv, out_q, out_kv, kHeadDim, p.q_block, p.k_block, split.ptr(), split.bytes, stream));
    else
      check(lib.fba_bwd_handover(bf16_at(q, qo), bf16_at(k, ko), bf16_at(v, ko), bf16_at(o, qo), bf16_at(d_o, qo), lse0, stats.data_ptr<float>(), ws,
                                 pairs * p.pair_bytes(), bf16_at(dq, qo), bf16_at(dk, ko), bf16_at(dv, ko), q_cnt, q_idx, k_cnt, k_idx, base, q_slot,
                                 pairs, mask_bh, 1, nh, nu, p.Sq, p.Skv, kHeadDim, p.q_block, p.k_block, split.ptr(), split.bytes, stream));
  }
  return {dq, dk, dv};
}

// ---------------------------------------------------------------------------------------------------------------------
// the whole operator
// ---------------------------------------------------------------------------------------------------------------------
// What backward needs besides tensors autograd saves: the lists (one allocation), the host copy of the pair numbers at the
// head boundaries when the pairs are numbered, and the settings of the call.
struct Saved : torch::CustomClassHolder {
  Problem p;
  Lists lists;
  at::Tensor list_buffer, host_bounds;
  bool from_mask = false;  // there are no lists: list_buffer holds a copy of the mask
  int64_t o_rows = 0;      // and o has as many rows to a head as if there were
  bool ragged_q = false, ragged_kv = false;  // lengths that lists would have been padded for
  c10::Event copied{c10::DeviceType::CUDA};
  bool dense = false;
  int64_t limit = 0, split_bytes;
  int64_t q_len, kv_len;  // of the caller's tensors; p describes the padded ones
  bool padded() const { return q_len != p.Sq || kv_len != p.Skv; }
  explicit Saved(const Problem& problem) : p(problem), lists(problem) {}
};

// The lists of `mask` in one buffer; key-major half and (numbered) pair numbers only where backward will read them.  The mask is the
// caller's: blocks that fill up the last tiles are in the lists' extents only.
void build_lists(Saved& s, const at::Tensor& mask, bool backward, bool numbered, bool launch = true) {
  const Problem& p = s.p;
  Lists& l = s.lists;
  const int64_t M = p.mask_bh;
  int64_t used = 0;
  auto take = [&](int64_t n) {
    const int64_t at = used;
    used += (n + 63) / 64 * 64;
    return at;
  };
  const int64_t q_cnt = take(M * l.q_rows), q_idx = take(M * l.q_rows * l.q_len);
  int64_t k_cnt = 0, k_idx = 0, base = 0, q_slot = 0, k_slot = 0;
  if (backward) {
    k_cnt = take(M * l.k_rows);
    k_idx = take(M * l.k_rows * l.k_len);
  }
  if (numbered) {
    base = take(M * l.k_rows + 1);
    q_slot = take(M * l.q_rows * l.slot_len);
    if (p.tiled()) k_slot = take(M * l.k_rows * l.k_len);
  }
  s.list_buffer = at::empty({used}, mask.options().dtype(at::kInt));
  int32_t* const b = s.list_buffer.data_ptr<int32_t>();
  void* const stream = current_stream(mask);
  l.q_cnt = b + q_cnt;
  l.q_idx = b + q_idx;
  if (backward) {
    l.k_cnt = b + k_cnt;
    l.k_idx = b + k_idx;
  }
  if (!launch) return;  // room for them only: forward makes them
  check(lib.fba_lists_cut(static_cast<const uint8_t*>(mask.data_ptr()), M, p.nQ(), p.nK(), s.q_len / p.q_block, s.kv_len / p.k_block, p.q_block, p.k_block,
                          l.q_cnt, l.q_idx, l.k_cnt, l.k_idx, stream));
  if (!numbered) return;
  l.pair_base = b + base;
  l.q_slot = b + q_slot;
  // The host's copy of the numbers at the head boundaries is written by the kernel that forms them.
  s.host_bounds = at::empty({M + 1}, at::TensorOptions().dtype(at::kInt).pinned_memory(true));
  int32_t* const bounds = s.host_bounds.data_ptr<int32_t>();
  if (p.tiled()) {
    l.k_slot = b + k_slot;
    check(lib.fba_tile_slots_bounds(l.k_cnt, l.k_idx, M, l.q_rows, l.k_rows, l.pair_base, l.k_slot, l.q_slot, bounds, stream));
  } else {
    check(lib.fba_pair_slots_bounds(l.q_cnt, l.q_idx, l.k_cnt, l.k_idx, M, p.nQ(), p.nK(), l.pair_base, l.q_slot, bounds, stream));
  }
  // This is ordered before whatever the caller enqueues next: backward waits for it alone, not for the forward kernel.  The memory is
  // given back to others only when this stream is through with it, also where nobody ever asks for gradients.
  const c10::Stream on = c10::impl::VirtualGuardImpl(c10::DeviceType::CUDA).getStream(mask.device());
  at::getHostAllocator(at::kCUDA)->record_event(bounds, s.host_bounds.storage().data_ptr().get_context(), on);
  s.copied.record(on);
}

// Sequences that are no whole number of 128-row tiles: copies cut or padded with zeros to `len` rows, all in one launch.  A
// tensor that has the length already is returned as it is unless `always`.
std::vector<at::Tensor> resized(const std::vector<std::pair<at::Tensor, int64_t>>& tensors, bool always = false) {
  std::vector<at::Tensor> out;
  const void* src[3];
  void* dst[3];
  int64_t n_seq[3];
  int32_t src_len[3], dst_len[3], n = 0;
  for (const auto& [t, len] : tensors) {
    const bool as_is = t.size(2) == len && !always;
    out.push_back(as_is ? t : at::empty({t.size(0), t.size(1), len, kHeadDim}, t.options()));
    if (as_is) continue;
    src[n] = t.data_ptr();
    dst[n] = out.back().data_ptr();
    n_seq[n] = t.size(0) * t.size(1);
    src_len[n] = t.size(2);
    dst_len[n++] = len;
  }
  if (n > 0) check(lib.fba_resize_rows(n, src, dst, n_seq, src_len, dst_len, current_stream(tensors[0].first)));
  return out;
}

// Inputs of a call as the kernels take them.  No block selects the rows that are appended.  The mask is for a forward pass that reads
// it itself; lists are made of the caller's, which saves a launch of 5 us (the fill of the last tiles) at B2 H8/2 S3136.
struct Inputs {
  at::Tensor q, k, v, mask;
  Inputs(const at::Tensor& q_, const at::Tensor& k_, const at::Tensor& v_, const at::Tensor& mask_, const Saved& s) : q(q_), k(k_), v(v_), mask(mask_) {
    if (!s.padded()) return;
    const Problem& p = s.p;
    auto r = resized({{q, p.Sq}, {k, p.Skv}, {v, p.Skv}});
    q = r[0];
    k = r[1];
    v = r[2];
    if (!takes_mask(p)) return;
    mask = at::empty({p.mask_bh, p.nQ(), p.nK()}, mask_.options());
    check(lib.fba_resize_mask(static_cast<const uint8_t*>(mask_.data_ptr()), static_cast<uint8_t*>(mask.data_ptr()), p.mask_bh, s.q_len / p.q_block,
                              s.kv_len / p.k_block, p.nQ(), p.nK(), current_stream(q)));
  }
};

// What autograd hands back in backward is whatever a saved-tensor hook made of it (another type, shape or layout), and the
// kernels read it by raw pointer: the same contract as for the inputs of a call.  `o` and `lse` may be strided, q, k, v not.
at::Tensor unpacked(const Saved& s, const char* name, const at::Tensor& t, at::IntArrayRef shape, at::ScalarType type, bool strided) {
  TORCH_CHECK_VALUE(t.defined() && t.device() == s.list_buffer.device(), "saved ", name, " must come back as a tensor on ", s.list_buffer.device());
  TORCH_CHECK_TYPE(t.scalar_type() == type, "saved ", name, " must come back as ", type, ", got ", t.scalar_type());
  TORCH_CHECK_VALUE(t.sizes() == shape, "saved ", name, " must come back with shape ", shape, ", got ", t.sizes());
  TORCH_CHECK_VALUE(strided || t.is_contiguous(), "saved ", name, " must come back contiguous");
  return t.contiguous();
}

struct Attention : torch::autograd::Function<Attention> {
  static at::Tensor forward(torch::autograd::AutogradContext* ctx, const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const at::Tensor& mask,
                            c10::intrusive_ptr<Saved> s) {
    if (s->from_mask) {  // (the caller may write to the mask before backward comes)
      s->list_buffer = at::empty({mask.numel()}, mask.options().dtype(at::kByte));
      // Where lists would have padded the queries, o has the strides it has there.
      const int64_t q_len = s->q_len;
      auto [o, lse] = run_forward_on_mask(s->p, q, k, v, mask, s->list_buffer.data_ptr(), s->o_rows);
      const bool cut = s->o_rows != q_len;
      // As with lists, inputs of lengths that are no whole tiles may be written to before backward comes: copies are saved (2.4 us of a
      // replayed step of 77, B2 H2 S1984).
      std::vector<std::pair<at::Tensor, int64_t>> copies;
      if (s->ragged_q) copies.emplace_back(q, q_len);
      if (s->ragged_kv) copies.insert(copies.end(), {{k, s->kv_len}, {v, s->kv_len}});
      const std::vector<at::Tensor> own = resized(copies, /*always=*/true);
      const at::Tensor* const own_kv = own.data() + (s->ragged_q ? 1 : 0);
      ctx->save_for_backward({s->ragged_q ? own[0] : q, s->ragged_kv ? own_kv[0] : k, s->ragged_kv ? own_kv[1] : v, o, lse});
      ctx->saved_data["s"] = c10::IValue::make_capsule(std::move(s));
      return cut ? o.narrow(2, 0, q_len).detach() : o;
    }
    const Inputs in(q, k, v, mask, *s);
    // Forward makes the lists of a step on the way where it can.  Steps that number their pairs need them before forward is through (the host waits for the
    // count); with many rows the lists would hold up the launch, whose last work-groups make them.
    // Lists that are there anyway: from the mask only where forward takes 64-row work-groups on it.  Otherwise it has nothing
    // to gain from the mask (B1 H8/2 128 x 17920, 128-token blocks, 102 of 140 kept: forward 33.8 us on lists, 34.9 on the mask).
    const bool on_mask = takes_mask(s->p);
    const int use = on_mask ? 0 : blocks_use(s->p);
    const bool with_lists = s->dense && (use & FBA_BLOCKS_LISTS) != 0, on_blocks = with_lists || (use & FBA_BLOCKS_HALVES) != 0;
    build_lists(*s, mask, /*backward=*/true, /*numbered=*/!s->dense, /*launch=*/!with_lists);
    auto [o, lse] = on_mask     ? run_forward_on_mask(s->p, in.q, in.k, in.v, in.mask)
                    : on_blocks ? run_forward_on_blocks(s->p, in.q, in.k, in.v, in.mask, with_lists ? s->lists : Lists(s->p), s->split_bytes)
                                : run_forward(s->p, in.q, in.k, in.v, s->lists, s->split_bytes);
    ctx->save_for_backward({in.q, in.k, in.v, o, lse});
    // The rows that were appended are cut off here and not behind this function, where autograd would give back gradients for them in
    // two launches of its own, a fill and a copy (13 of 280 us at B2 H8/2 S3136).  What is handed out shares its version with
    // the saved tensor, so that a change in place is noticed.
    const bool cut = s->q_len != s->p.Sq;
    const int64_t q_len = s->q_len;
    ctx->saved_data["s"] = c10::IValue::make_capsule(std::move(s));
    return cut ? o.narrow(2, 0, q_len).detach() : o;
  }
  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx, torch::autograd::variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const auto capsule = ctx->saved_data["s"].toCapsule();
    Saved& s = *static_cast<Saved*>(capsule.get());
    const c10::DeviceGuard guard(s.list_buffer.device());
    const Problem& p = s.p;
    const int64_t q_shape[4] = {p.B, p.Hq, p.Sq, kHeadDim}, o_shape[4] = {p.B, p.Hq, s.from_mask ? s.o_rows : p.Sq, kHeadDim},
                  kv_shape[4] = {p.B, p.Hkv, p.Skv, kHeadDim}, lse_shape[4] = {p.B, p.Hq, p.Sq, 1};
    const at::Tensor q = unpacked(s, "q", saved[0], q_shape, at::kBFloat16, false), k = unpacked(s, "k", saved[1], kv_shape, at::kBFloat16, false),
                     v = unpacked(s, "v", saved[2], kv_shape, at::kBFloat16, false), o = unpacked(s, "o", saved[3], o_shape, at::kBFloat16, true),
                     lse = unpacked(s, "lse", saved[4], lse_shape, at::kFloat, true);
    at::Tensor d_o = grads[0].to(at::kBFloat16).contiguous();
    if (s.from_mask) {
      if (s.o_rows != p.Sq && (reinterpret_cast<uintptr_t>(d_o.data_ptr()) & 15) != 0) d_o = d_o.clone();  // as below
      const auto g = run_backward_on_mask(p, q, k, v, o, lse, d_o, s.list_buffer);
      return {g[0], g[1], g[2], at::Tensor(), at::Tensor()};
    }
    if (s.q_len != p.Sq && (reinterpret_cast<uintptr_t>(d_o.data_ptr()) & 15) != 0) d_o = d_o.clone();  // it is filled up 16 bytes at a time
    std::vector<int64_t> bounds;
    if (!s.dense) {
      s.copied.synchronize();
      const int32_t* h = s.host_bounds.data_ptr<int32_t>();
      bounds.assign(h, h + p.mask_bh + 1);
    }
    const auto g = run_backward(p, q, k, v, o, lse, d_o, s.lists, bounds, HandOver::kAuto, s.dense, s.limit, s.split_bytes, s.q_len, s.kv_len);
    return {g[0], g[1], g[2], at::Tensor(), at::Tensor()};
  }
};

// flex_block_attn_func for arguments that need no preparation but padding to whole tiles; nothing for all others (wrong types or
// shapes, strided tensors), which Python then reports or prepares.
c10::optional<at::Tensor> attention(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, int64_t q_block, int64_t k_block, const at::Tensor& mask,
                                    double limit, double factor, int64_t split_bytes) {
  // a traced call has to appear in the trace, forward-mode differentiation and function transforms have to be refused: all go
  // through the Python autograd function, which does that
  if (torch::jit::tracer::isTracing()) return c10::nullopt;
  if (c10::impl::tls_local_dispatch_key_set().included_.has(c10::DispatchKey::FuncTorchDynamicLayerFrontMode)) return c10::nullopt;
  for (const at::Tensor* t : {&q, &k, &v})
    if (t->_fw_grad(0).defined()) return c10::nullopt;
  for (const at::Tensor* t : {&q, &k, &v})
    if (!t->is_cuda() || t->scalar_type() != at::kBFloat16 || t->dim() != 4 || !t->is_contiguous() || t->size(3) != kHeadDim ||
        t->device() != q.device() || (reinterpret_cast<uintptr_t>(t->data_ptr()) & 15) != 0)
      return c10::nullopt;
  if (mask.device() != q.device() || mask.scalar_type() != at::kBool || (mask.dim() != 2 && mask.dim() != 4) || !mask.is_contiguous()) return c10::nullopt;
  Problem p{q.size(0), q.size(1), k.size(1), q.size(2), k.size(2), q_block, k_block, mask.dim() == 2 ? 1 : q.size(0) * q.size(1)};
  const int64_t md = mask.dim();
  if (q.numel() == 0 || k.numel() == 0 || k.size(0) != p.B || v.sizes() != k.sizes() || p.Hq % p.Hkv != 0) return c10::nullopt;
  if (q_block <= 0 || k_block <= 0 || q_block % 16 != 0 || k_block % 64 != 0 || (k_block % q_block != 0 && q_block % k_block != 0)) return c10::nullopt;
  if (p.Sq % q_block != 0 || p.Skv % k_block != 0 || mask.size(md - 2) != p.nQ() || mask.size(md - 1) != p.nK()) return c10::nullopt;
  if (md == 4 && (mask.size(0) != p.B || mask.size(1) != p.Hq)) return c10::nullopt;
  const int64_t q_len = p.Sq, kv_len = p.Skv;
  if (p.tiled()) {  // whole blocks are appended until the tiles are whole as well
    auto whole = [](int64_t len, int64_t block) { return len % 128 == 0 ? len : (len + std::lcm(block, 128L) - 1) / std::lcm(block, 128L) * std::lcm(block, 128L); };
    p.Sq = whole(q_len, q_block);
    p.Skv = whole(kv_len, k_block);
  }
  if (p.B * p.Hq * p.Sq >= (1LL << 30) || p.B * p.Hkv * p.Skv >= (1LL << 30) || p.mask_bh * p.nQ() * p.nK() > 0x7fffffffLL ||
      p.mask_bh * (p.Sq / 32 + 1) * (p.Skv / 128 + 1) > 0x7fffffffLL)
    return c10::nullopt;
  const c10::DeviceGuard guard(q.device());
  if (split_bytes < 0) split_bytes = lib.fba_split_workspace_bytes();
  auto s = c10::make_intrusive<Saved>(p);
  s->split_bytes = split_bytes;
  s->q_len = q_len;
  s->kv_len = kv_len;
  const bool backward = at::GradMode::is_enabled() && (q.requires_grad() || k.requires_grad() || v.requires_grad());
  if (!backward) {
    if (takes_mask(p)) return run_forward_on_mask(p, q, k, v, mask).first;
    if (blocks_use(p) != 0) return run_forward_on_blocks(p, q, k, v, mask, Lists(p), split_bytes).first;
    const Inputs in(q, k, v, mask, *s);
    build_lists(*s, mask, false, false);
    const at::Tensor o = run_forward(p, in.q, in.k, in.v, s->lists, split_bytes).first;
    return s->padded() ? o.narrow(2, 0, q_len) : o;
  }
  if (backward_takes_mask(p)) {
    s->from_mask = true;
    s->o_rows = p.Sq;
    s->ragged_q = p.Sq != q_len;
    s->ragged_kv = p.Skv != kv_len;
    s->p.Sq = q_len;
    s->p.Skv = kv_len;
  } else {
    s->limit = ds_limit(p, limit, factor);
    s->dense = dense_fits(p.dense_bytes(), s->limit);
  }
  return Attention::apply(q, k, v, mask, std::move(s));
}

// The same for whatever a Python caller passes: nothing for objects that are no tensors, for tensor subclasses (their results are
// of their type, which Python sees to) and for block sizes that are no ints of 32 bits.
c10::optional<at::Tensor> attention_of(pybind11::handle q, pybind11::handle k, pybind11::handle v, pybind11::handle q_block, pybind11::handle k_block,
                                       pybind11::handle mask, double limit, double factor, int64_t split_bytes) {
  for (pybind11::handle t : {q, k, v, mask})
    if (!THPVariable_CheckTypeExact(Py_TYPE(t.ptr()))) return c10::nullopt;
  int64_t blocks[2];
  for (int i = 0; i < 2; ++i) {
    PyObject* const size = (i ? k_block : q_block).ptr();
    int overflow = 0;
    if (!PyLong_CheckExact(size)) return c10::nullopt;
    blocks[i] = PyLong_AsLongLongAndOverflow(size, &overflow);
    if (overflow != 0 || blocks[i] > 0x7fffffffLL) return c10::nullopt;
  }
  const at::Tensor qt = THPVariable_Unpack(q.ptr()), kt = THPVariable_Unpack(k.ptr()), vt = THPVariable_Unpack(v.ptr()), mt = THPVariable_Unpack(mask.ptr());
  pybind11::gil_scoped_release no_gil;
  return attention(qt, kt, vt, blocks[0], blocks[1], mt, limit, factor, split_bytes);
}

// ---------------------------------------------------------------------------------------------------------------------
// entry points on lists (checked by the caller)
// ---------------------------------------------------------------------------------------------------------------------
int32_t* ints(const c10::optional<at::Tensor>& t) { return t ? t->data_ptr<int32_t>() : nullptr; }

Problem problem_of(const at::Tensor& q, const at::Tensor& k, int64_t q_block, int64_t k_block, int64_t mask_bh) {
  return {q.size(0), q.size(1), k.size(1), q.size(2), k.size(2), q_block, k_block, mask_bh};
}

std::pair<at::Tensor, at::Tensor> forward_on_lists(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, int64_t q_block, int64_t k_block,
                                                   int64_t mask_bh, const at::Tensor& q_cnt, const at::Tensor& q_idx, int64_t split_bytes) {
  const c10::DeviceGuard guard(q.device());
  const Problem p = problem_of(q, k, q_block, k_block, mask_bh);
  Lists l(p);
  l.q_cnt = q_cnt.data_ptr<int32_t>();
  l.q_idx = q_idx.data_ptr<int32_t>();
  return run_forward(p, q, k, v, l, split_bytes);
}

// Nothing where forward takes lists.  `mask` is a contiguous bool tensor.
c10::optional<std::pair<at::Tensor, at::Tensor>> forward_on_mask(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, int64_t q_block, int64_t k_block,
                                                                 const at::Tensor& mask) {
  const c10::DeviceGuard guard(q.device());
  const Problem p = problem_of(q, k, q_block, k_block, mask.dim() == 2 ? 1 : q.size(0) * q.size(1));
  if (!takes_mask(p)) return c10::nullopt;
  return run_forward_on_mask(p, q, k, v, mask);
}

// For the Python autograd function: is backward to take the mask, too?  If so, forward_on_mask comes before it.
bool backward_takes_mask_of(const at::Tensor& q, const at::Tensor& k, int64_t q_block, int64_t k_block) {
  const c10::DeviceGuard guard(q.device());
  return backward_takes_mask(problem_of(q, k, q_block, k_block, 1));
}
std::vector<at::Tensor> backward_on_mask(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const at::Tensor& o, const at::Tensor& lse,
                                         const at::Tensor& d_o, int64_t q_block, int64_t k_block, const at::Tensor& mask) {
  const c10::DeviceGuard guard(q.device());
  return run_backward_on_mask(problem_of(q, k, q_block, k_block, mask.dim() == 2 ? 1 : q.size(0) * q.size(1)), q, k, v, o, lse, d_o, mask);
}

std::vector<at::Tensor> backward_on_lists(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const at::Tensor& o, const at::Tensor& lse,
                                          const at::Tensor& d_o, int64_t q_block, int64_t k_block, int64_t mask_bh, const at::Tensor& q_cnt,
                                          const at::Tensor& q_idx, const at::Tensor& k_cnt, const at::Tensor& k_idx,
                                          const c10::optional<at::Tensor>& pair_base, const c10::optional<at::Tensor>& q_slot,
                                          const c10::optional<at::Tensor>& k_slot, const std::vector<int64_t>& bounds, c10::optional<bool> hand_over,
                                          bool dense, int64_t limit, int64_t split_bytes) {
  const c10::DeviceGuard guard(q.device());
  const Problem p = problem_of(q, k, q_block, k_block, mask_bh);
  Lists l(p);
  l.q_cnt = q_cnt.data_ptr<int32_t>();
  l.q_idx = q_idx.data_ptr<int32_t>();
  l.k_cnt = k_cnt.data_ptr<int32_t>();
  l.k_idx = k_idx.data_ptr<int32_t>();
  l.pair_base = ints(pair_base);
  l.q_slot = ints(q_slot);
  l.k_slot = ints(k_slot);
  const HandOver mode = !hand_over ? HandOver::kAuto : *hand_over ? HandOver::kWhole : HandOver::kNever;
  return run_backward(p, q, k, v, o, lse, d_o, l, bounds, mode, dense, limit, split_bytes);
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("bind", &bind);
  m.def("unit_pairs", &unit_pairs);
  m.def("plan_head_chunks", &plan_head_chunks);
  m.def("dense_fits", &dense_fits);
  m.def("attention", &attention_of);
  m.def("forward", &forward_on_lists, pybind11::call_guard<pybind11::gil_scoped_release>());
  m.def("forward_on_mask", &forward_on_mask, pybind11::call_guard<pybind11::gil_scoped_release>());
  m.def("backward_takes_mask", &backward_takes_mask_of);
  m.def("backward_on_mask", &backward_on_mask, pybind11::call_guard<pybind11::gil_scoped_release>());
  m.def("backward", &backward_on_lists, pybind11::call_guard<pybind11::gil_scoped_release>());
}
