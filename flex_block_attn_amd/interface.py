"""Operator surface of flex-block-attn on MI355X.

Same names, argument order and return arity as the reference's flex_block_attn/flex_block_attn_interface.py
(`flex_block_attn_func` :91-106, `FlexBlockAttnFunc` :14-89, `_flex_block_attn_forward` :6-8,
`_flex_block_attn_backward` :10-12).  The kernels live in libfba_gfx950.so; the host work around them (allocations, the plan
of the backward pass, launches, the autograd node) is native code in the module fba_torch.  This file holds the checks and
their messages, and the calls on precompacted lists.

What differs from the reference, deliberately:
  * the bool block mask is turned into index lists once, on the GPU (`compact_block_mask`), at its true
    (q_block x kv_block) granularity; the coarse / fine mask pair of flex_block_attn_interface.py:38-66 is not needed;
  * backward reuses the key-major lists emitted by the same compaction instead of transposing the masks
    (flex_block_attn_interface.py:85-86);
  * dq, dk, dv come back in the dtype of q (bf16) rather than fp32 (flex_block_attn_h100.cu:1077-1088);
  * `lse` is the natural-log softmax denominator, shape (B, H, Sq, 1); the reference's value at that position is
    -sqrt(128) times it (flex_block_attn_h100.cu:303-307) and is only ever consumed by its own backward.
"""
import ctypes
import math
import os
from dataclasses import dataclass
from typing import Optional

import torch

from . import _lib

HEAD_DIM = 128


@dataclass
class BlockLists:
    """Active-block index lists of one block mask (see include/fba.h, fba_mask_compact).

    With `tiled` set the four tensors are tile lists instead (fba_tile_lists: qt_cnt, qt_ent, kt_cnt, kt_ent), which the
    kernels need when a block size is not a multiple of 128."""

    q_cnt: torch.Tensor  # [mask_bh, nQ] int32
    q_idx: torch.Tensor  # [mask_bh, nQ, nK] int32, ascending, -1 padded
    k_cnt: torch.Tensor  # [mask_bh, nK] int32
    k_idx: torch.Tensor  # [mask_bh, nK, nQ] int32, ascending, -1 padded
    mask_bh: int
    nQ: int
    nK: int
    tiled: bool = False
    # pair numbering for the dS hand-over of backward, filled by `number_pairs`.  Block lists (fba_pair_slots):
    # pair_base [mask_bh * nK + 1], q_slot [mask_bh, nQ, nK].  Tile lists (fba_tile_slots): pair_base
    # [mask_bh * Skv/128 + 1], q_slot [mask_bh, Sq/128, Skv/128] (the slot table), k_slot [mask_bh, Skv/128, Sq/32].
    pair_base: Optional[torch.Tensor] = None  # int32; the last entry is the number of listed pairs
    q_slot: Optional[torch.Tensor] = None     # int32
    k_slot: Optional[torch.Tensor] = None     # int32, tile lists only
    _count: Optional[tuple] = None            # (pinned host copy of pair_base at head boundaries, event after the copy)

    def pair_bounds(self):
        """pair_base at the head boundaries of the mask ([mask_bh + 1] ints, first 0, last = number of listed pairs), read
        from the host copy that `number_pairs` requested; waits for that copy only, not for work enqueued after it."""
        host, event = self._count
        event.synchronize()
        return host.tolist()

    def listed_pairs(self):
        """Number of pairs in the lists (sum of k_cnt)."""
        return int(self.pair_bounds()[-1])

    def transposed(self):
        """Lists of the transposed mask (query and key roles swapped); no device work.  Block lists only."""
        if self.tiled:
            raise ValueError("tile lists cannot be transposed")
        return BlockLists(self.k_cnt, self.k_idx, self.q_cnt, self.q_idx, self.mask_bh, self.nK, self.nQ)


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def _stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def _require_device(t, name):
    if not t.is_cuda:
        raise ValueError(f"{name} must be a GPU tensor (the HIP kernels have no CPU fallback)")


def compact_block_mask(block_mask, with_pair_numbers=False):
    """bool block mask [nQ, nK] or [B, H, nQ, nK] (GPU) -> BlockLists, via the compaction kernel.  `with_pair_numbers`
    also numbers the pairs right away (what the dS hand-over of backward needs; see `number_pairs`)."""
    if block_mask.dtype != torch.bool:
        raise TypeError(f"block_mask must be a bool tensor, got {block_mask.dtype}")
    if block_mask.dim() not in (2, 4):
        raise ValueError(f"block_mask must have 2 or 4 dimensions, got {block_mask.dim()}")
    _require_device(block_mask, "block_mask")
    m = block_mask.contiguous()
    nQ, nK = m.shape[-2], m.shape[-1]
    mask_bh = 1 if m.dim() == 2 else m.shape[0] * m.shape[1]
    dev = m.device
    q_cnt = torch.empty((mask_bh, nQ), dtype=torch.int32, device=dev)
    q_idx = torch.empty((mask_bh, nQ, nK), dtype=torch.int32, device=dev)
    k_cnt = torch.empty((mask_bh, nK), dtype=torch.int32, device=dev)
    k_idx = torch.empty((mask_bh, nK, nQ), dtype=torch.int32, device=dev)
    with torch.cuda.device(dev):
        _lib.call("fba_mask_compact", _ptr(m), mask_bh, nQ, nK, _ptr(q_cnt), _ptr(q_idx), _ptr(k_cnt), _ptr(k_idx), _stream())
    lists = BlockLists(q_cnt, q_idx, k_cnt, k_idx, mask_bh, nQ, nK)
    # numbered right away when a backward pass will follow: the host copy of the pair count is then ordered before
    # whatever the caller enqueues next, and backward finds it without waiting for the forward kernel
    return number_pairs(lists) if with_pair_numbers else lists


def needs_tile_lists(q_block_size, kv_block_size):
    """The kernels work on 128-row tiles: block sizes that are not multiples of 128 go through tile lists."""
    return q_block_size % 128 != 0 or kv_block_size % 128 != 0


def tile_block_mask(block_mask, q_block_size, kv_block_size, with_pair_numbers=False):
    """bool block mask -> tile lists (a BlockLists with `tiled` set), via fba_tile_lists.  `with_pair_numbers` also
    numbers the tile pairs right away (see `number_pairs`)."""
    if block_mask.dtype != torch.bool:
        raise TypeError(f"block_mask must be a bool tensor, got {block_mask.dtype}")
    if block_mask.dim() not in (2, 4):
        raise ValueError(f"block_mask must have 2 or 4 dimensions, got {block_mask.dim()}")
    _require_device(block_mask, "block_mask")
    m = block_mask.contiguous()
    nQ, nK = m.shape[-2], m.shape[-1]
    Sq, Skv = nQ * q_block_size, nK * kv_block_size
    if Sq % 128 or Skv % 128:
        raise _lib.FbaError(_lib.FBA_ERR_UNSUPPORTED, f"tile lists need sequence lengths that are multiples of 128, got {Sq} and {Skv}")
    mask_bh = 1 if m.dim() == 2 else m.shape[0] * m.shape[1]
    i32 = dict(dtype=torch.int32, device=m.device)
    qt_cnt = torch.empty((mask_bh, Sq // 128), **i32)
    qt_ent = torch.empty((mask_bh, Sq // 128, nK), **i32)
    kt_cnt = torch.empty((mask_bh, Skv // 128), **i32)
    kt_ent = torch.empty((mask_bh, Skv // 128, Sq // 32), **i32)
    with torch.cuda.device(m.device):
        _lib.call("fba_tile_lists", _ptr(m), mask_bh, nQ, nK, q_block_size, kv_block_size, _ptr(qt_cnt), _ptr(qt_ent),
                  _ptr(kt_cnt), _ptr(kt_ent), _stream())
    lists = BlockLists(qt_cnt, qt_ent, kt_cnt, kt_ent, mask_bh, nQ, nK, tiled=True)
    return number_pairs(lists) if with_pair_numbers else lists


def lists_for(block_mask, q_block_size, kv_block_size, with_pair_numbers=False):
    """The list flavour the kernels need for these block sizes."""
    if needs_tile_lists(q_block_size, kv_block_size):
        return tile_block_mask(block_mask, q_block_size, kv_block_size, with_pair_numbers)
    return compact_block_mask(block_mask, with_pair_numbers)


def _check_qkv(q, k, v):
    """Tensor contract of the extension (flex_block_attn_h100.cu:820-858)."""
    for name, t in (("q", q), ("k", k), ("v", v)):
        _require_device(t, name)
        if t.dtype != torch.bfloat16:
            raise TypeError(f"{name} must be bfloat16, got {t.dtype}")
        if t.dim() != 4:
            raise ValueError(f"{name} must have shape (batch, heads, seq, head_dim)")
        if not t.is_contiguous():
            raise ValueError(f"{name} must be contiguous")
    B, Hq, Sq, D = q.shape
    Bk, Hkv, Skv, Dk = k.shape
    if D != HEAD_DIM or Dk != HEAD_DIM or v.shape[3] != HEAD_DIM:
        raise ValueError("head_dim must be 128")
    if Bk != B or v.shape[0] != B:
        raise ValueError("q, k, v batch dimensions must match")
    if v.shape[1] != Hkv or v.shape[2] != Skv:
        raise ValueError("k and v must have the same shape")
    if Hq % Hkv != 0:
        raise ValueError("q heads must be a multiple of kv heads")
    return B, Hq, Hkv, Sq, Skv


def _check_blocks(q, k, q_block_size, kv_block_size, block_mask):
    """Block-size and mask-shape rules (flex_block_attn_interface.py:18-32)."""
    assert q_block_size % 16 == 0, f"q_block_size ({q_block_size}) must be divisible by 16"
    assert kv_block_size % 64 == 0, f"kv_block_size ({kv_block_size}) must be divisible by 64"
    assert kv_block_size % q_block_size == 0 or q_block_size % kv_block_size == 0, (
        f"kv_block_size ({kv_block_size}) must be divisible by q_block_size ({q_block_size}), or vice versa."
    )
    q_seq_len, kv_seq_len = q.shape[2], k.shape[2]
    assert q_seq_len % q_block_size == 0, f"q_seq_len ({q_seq_len}) must be divisible by q_block_size ({q_block_size})"
    assert kv_seq_len % kv_block_size == 0, f"kv_seq_len ({kv_seq_len}) must be divisible by kv_block_size ({kv_block_size})"
    if block_mask.dim() not in (2, 4):
        raise ValueError(f"block_mask must have 2 or 4 dimensions, got {block_mask.dim()}")
    q_block_num, kv_block_num = block_mask.shape[-2], block_mask.shape[-1]
    assert q_block_size * q_block_num == q_seq_len, (
        f"q_block_size ({q_block_size}) * q_block_num ({q_block_num}) must equal q_seq_len ({q_seq_len})"
    )
    assert kv_block_size * kv_block_num == kv_seq_len, (
        f"kv_block_size ({kv_block_size}) * kv_block_num ({kv_block_num}) must equal kv_seq_len ({kv_seq_len})"
    )
    if block_mask.dim() == 4 and tuple(block_mask.shape[:2]) != (q.shape[0], q.shape[1]):
        raise ValueError(
            f"4-D block_mask must be [batch, heads, q_blocks, kv_blocks] = [{q.shape[0]}, {q.shape[1]}, ...], "
            f"got {tuple(block_mask.shape)}"
        )


def _check_lists(lists, q, B, Hq, Sq, Skv, q_block_size, kv_block_size):
    """The kernels index the list tensors by raw pointer: metadata, dtype, device, layout and exact shapes must fit."""
    if lists.nQ * q_block_size != Sq or lists.nK * kv_block_size != Skv:
        raise ValueError("block lists do not match the sequence lengths and block sizes")
    if lists.tiled != needs_tile_lists(q_block_size, kv_block_size):
        raise ValueError("wrong list flavour for these block sizes (see lists_for)")
    if lists.mask_bh not in (1, B * Hq):
        raise ValueError("block lists do not match batch * heads")
    M = lists.mask_bh
    if lists.tiled:
        shapes = ((M, Sq // 128), (M, Sq // 128, lists.nK), (M, Skv // 128), (M, Skv // 128, Sq // 32))
    else:
        shapes = ((M, lists.nQ), (M, lists.nQ, lists.nK), (M, lists.nK), (M, lists.nK, lists.nQ))
    names, tensors = ["q_cnt", "q_idx", "k_cnt", "k_idx"], [lists.q_cnt, lists.q_idx, lists.k_cnt, lists.k_idx]
    if lists.pair_base is not None and lists.tiled:
        names += ["pair_base", "q_slot", "k_slot"]
        tensors += [lists.pair_base, lists.q_slot, lists.k_slot]
        shapes += ((M * (Skv // 128) + 1,), (M, Sq // 128, Skv // 128), (M, Skv // 128, Sq // 32))
    elif lists.pair_base is not None:
        names += ["pair_base", "q_slot"]
        tensors += [lists.pair_base, lists.q_slot]
        shapes += ((M * lists.nK + 1,), (M, lists.nQ, lists.nK))
    for name, t, shape in zip(names, tensors, shapes):
        if t.dtype != torch.int32 or t.device != q.device or not t.is_contiguous() or tuple(t.shape) != shape:
            raise ValueError(f"block lists: {name} must be a contiguous int32 tensor of shape {shape} on {q.device}, "
                             f"got {tuple(t.shape)} {t.dtype} on {t.device}")


# Workspace for tail splitting (see include/fba.h), allocated per call from torch's caching allocator; MiB, 0 or less switches
# splitting off, unset: what the library's planner can use at most.
SPLIT_WORKSPACE_MIB = os.environ.get("FBA_SPLIT_WORKSPACE_MIB")


def _split_bytes():
    return _lib.load().fba_split_workspace_bytes() if SPLIT_WORKSPACE_MIB is None else max(0, int(float(SPLIT_WORKSPACE_MIB) * 2 ** 20))


def _split_workspace(device):
    """(tensor or None, pointer, bytes) of a fresh tail-splitting workspace on `device`."""
    n = _split_bytes()
    if n <= 0:
        return None, None, 0
    ws = torch.empty((n,), dtype=torch.uint8, device=device)
    return ws, _ptr(ws), n


# Types that torch.empty_like turns into a plain tensor.  Results for any other tensor type have the type empty_like gives them, so
# that a subclass goes through the operator as through torch's own.
_PLAIN = (torch.Tensor, torch.nn.Parameter)


def _typed_like(result, t):
    return result if type(t) in _PLAIN else torch.empty_like(t).copy_(result)


def forward_with_lists(q, k, v, q_block_size, kv_block_size, lists):
    """Forward on compacted lists -> (o [B,H,Sq,128] bf16, lse [B,H,Sq,1] fp32)."""
    B, Hq, Hkv, Sq, Skv = _check_qkv(q, k, v)
    _check_lists(lists, q, B, Hq, Sq, Skv, q_block_size, kv_block_size)
    o, lse = _lib.host().forward(q, k, v, q_block_size, kv_block_size, lists.mask_bh, lists.q_cnt, lists.q_idx, _split_bytes())
    return _typed_like(o, q), lse


def _forward(q, k, v, q_block_size, kv_block_size, block_mask, lists):
    """Forward with the kernel the native call takes: problems too small to fill the GPU read the mask itself."""
    B, Hq, Hkv, Sq, Skv = _check_qkv(q, k, v)
    _check_lists(lists, q, B, Hq, Sq, Skv, q_block_size, kv_block_size)
    got = _lib.host().forward_on_mask(q, k, v, q_block_size, kv_block_size, block_mask.contiguous())
    return forward_with_lists(q, k, v, q_block_size, kv_block_size, lists) if got is None else (_typed_like(got[0], q), got[1])


def _backward_takes_mask(q, k, v, q_block_size, kv_block_size, block_mask):
    """Whether neither pass needs lists (small problems, as the native call decides).  What lists could not be made of is left to them, so that it is
    refused with gradients as without: other masks, and lengths that are no whole tiles (flex_block_attn_func pads them)."""
    if block_mask.dtype != torch.bool or not block_mask.is_cuda or block_mask.device != q.device or block_mask.numel() == 0:
        return False
    if q.shape[2] % 128 or k.shape[2] % 128:
        return False
    _check_qkv(q, k, v)
    return q.numel() > 0 and k.numel() > 0 and _lib.host().backward_takes_mask(q, k, q_block_size, kv_block_size)


def _backward_inputs(q, o, lse, do):
    """o, lse and dO of a backward pass as the kernels take them."""
    if do.dtype != torch.bfloat16:
        do = do.to(torch.bfloat16)
    do = do.contiguous()
    o = o.contiguous()
    if o.shape != q.shape or do.shape != q.shape:
        raise ValueError("o and do must have the shape of q")
    if lse.dtype != torch.float32 or lse.numel() != q.shape[0] * q.shape[1] * q.shape[2]:
        raise ValueError("lse must be float32 with B*H*Sq elements")
    return o, lse.contiguous(), do


def _backward_on_mask(q, k, v, o, lse, do, q_block_size, kv_block_size, mask):
    _check_qkv(q, k, v)
    o, lse, do = _backward_inputs(q, o, lse, do)
    grads = _lib.host().backward_on_mask(q, k, v, o, lse, do, q_block_size, kv_block_size, mask)
    return tuple(_typed_like(g, t) for g, t in zip(grads, (q, k, v)))


def number_pairs(lists):
    """Pair numbering for the dS hand-over, kept on `lists`: block pairs of block lists (fba_pair_slots), pairs of
    128-row tiles of tile lists (fba_tile_slots).  The number of listed pairs, which sizes the workspace, is copied to
    pinned host memory asynchronously; `lists.listed_pairs()` waits for that copy alone."""
    if lists.pair_base is None:
        dev = lists.k_cnt.device
        i32 = dict(dtype=torch.int32, device=dev)
        host = torch.empty((lists.mask_bh + 1,), dtype=torch.int32, pin_memory=True)
        k_slot = None
        with torch.cuda.device(dev):
            if lists.tiled:
                n_qt, n_kt = lists.q_cnt.shape[1], lists.k_cnt.shape[1]
                pair_base = torch.empty((lists.mask_bh * n_kt + 1,), **i32)
                q_slot = torch.empty((lists.mask_bh, n_qt, n_kt), **i32)
                k_slot = torch.empty((lists.mask_bh, n_kt, 4 * n_qt), **i32)
                _lib.call("fba_tile_slots", _ptr(lists.k_cnt), _ptr(lists.k_idx), lists.mask_bh, n_qt, n_kt, _ptr(pair_base),
                          _ptr(k_slot), _ptr(q_slot), _stream())
            else:
                pair_base = torch.empty((lists.mask_bh * lists.nK + 1,), **i32)
                q_slot = torch.empty((lists.mask_bh, lists.nQ, lists.nK), **i32)
                _lib.call("fba_pair_slots", _ptr(lists.q_cnt), _ptr(lists.q_idx), _ptr(lists.k_cnt), _ptr(lists.k_idx), lists.mask_bh,
                          lists.nQ, lists.nK, _ptr(pair_base), _ptr(q_slot), _stream())
            host.copy_(pair_base[:: lists.k_cnt.shape[1]], non_blocking=True)  # one entry per head of the mask, and the total
            event = torch.cuda.Event()
            event.record()
        lists.pair_base, lists.q_slot, lists.k_slot, lists._count = pair_base, q_slot, k_slot, (host, event)
    return lists


# Largest dS workspace backward allocates on its own: at most DS_WORKSPACE_LIMIT_GIB, and at most DS_WORKSPACE_FACTOR
# times the bytes of the call's own tensors (q, k, v, o, dO, dq, dk, dv), so that backward memory stays proportional to
# the sequence length like the reference's.  A backward pass whose selected pairs need more is run in chunks of heads
# through a workspace within the limit (every head's dS is independent); when not even one kv head fits, or the
# allocation fails, backward recomputes S and dP in the dQ kernel instead (fba_bwd), which needs no workspace.  The
# default of 20 GiB lets the benchmark shapes with 24 heads run in chunks of at least 8 heads, one per XCD (chunks of
# fewer heads are slower per head); FBA_DS_WORKSPACE_LIMIT_GIB=8 costs them up to 9 % of backward.
# (The limit deliberately reads no allocator or driver state: hipMemGetInfo takes milliseconds, and torch's memory
# counters build a dictionary of a few hundred entries per call, enough to trigger a full pass of Python's cyclic garbage
# collector, 40 ms in a process that has torch loaded, every few dozen calls.)
DS_WORKSPACE_LIMIT_GIB = float(os.environ.get("FBA_DS_WORKSPACE_LIMIT_GIB", "20"))
DS_WORKSPACE_FACTOR = float(os.environ.get("FBA_DS_WORKSPACE_FACTOR", "6"))


def ds_workspace_limit(q, k):
    """Bytes of dS workspace the default backward may allocate for these q and k/v shapes."""
    own = (5 * q.numel() + 4 * k.numel()) * 2  # q, o, dO, dq and k, v, dk, dv (bf16)
    return int(min(DS_WORKSPACE_LIMIT_GIB * 2 ** 30, DS_WORKSPACE_FACTOR * own))


def _unit_pairs(lists, B, Hq, Hkv):
    """(listed pairs of every (batch, kv head), pair numbers at the head boundaries), as backward counts them."""
    bounds = number_pairs(lists).pair_bounds()
    return _lib.host().unit_pairs(bounds, B * Hkv, Hq // Hkv), bounds


def ds_workspace_bytes(lists, B, Hq, q_block_size, kv_block_size):
    """(pairs over all heads, bytes of dS workspace) the hand-over backward needs for all heads of these lists at once."""
    listed = number_pairs(lists).listed_pairs()
    pairs = listed * (B * Hq if lists.mask_bh == 1 else 1)
    return pairs, pairs * (128 * 128 if lists.tiled else q_block_size * kv_block_size) * 2


def dense_ds_bytes(q, k):
    """Bytes of a dS workspace with a place for every (query row, key) pair of every head (fba_bwd_dense)."""
    return q.shape[0] * q.shape[1] * q.shape[2] * k.shape[2] * 2


def dense_ds_fits(q, k):
    """Whether backward hands dS over without numbering the selected pairs: true for small problems, where the numbering
    launches and the wait for the pair count would be a good part of the time (all pairs of all heads in at most 2 GiB and
    within the limit above), and within the limit alone while the current stream is captured."""
    with torch.cuda.device_of(q):
        return _lib.host().dense_fits(dense_ds_bytes(q, k), ds_workspace_limit(q, k))


def plan_head_chunks(unit_pairs, pair_bytes, limit_bytes):
    """Cuts the (batch, kv head) units into consecutive chunks of equal length whose dS fits `limit_bytes`: as few chunks
    as the total needs, shortened while some chunk is still too large, and then, if a chunk holds more than one unit per
    XCD, shortened to a multiple of the XCD count (twelve heads per chunk cost dK/dV 3 % against eight).  Returns
    [(first unit, end unit, pairs)], or None when a single unit does not fit."""
    return _lib.host().plan_head_chunks(list(unit_pairs), pair_bytes, int(limit_bytes))


def backward_with_lists(q, k, v, o, lse, do, q_block_size, kv_block_size, lists, hand_over=None):
    """Backward on compacted lists -> (dq, dk, dv), bf16, shaped like q, k, v.

    hand_over=None (default): the key-major kernel stores dS once and dQ is formed from it (ten products per block
    pair instead of fourteen), in chunks of heads through a workspace of at most `ds_workspace_limit(q, k)` bytes; if not
    even one kv head fits, as False.  Small problems whose pairs are not numbered yet use a workspace with a place for every
    pair (fba_bwd_dense).  True: the same with one workspace for all heads, whatever its size (fba_bwd_handover /
    fba_bwd_tiled_handover in one call).  False: dQ recomputes S and dP (fba_bwd or fba_bwd_tiled, no workspace)."""
    B, Hq, Hkv, Sq, Skv = _check_qkv(q, k, v)
    _check_lists(lists, q, B, Hq, Sq, Skv, q_block_size, kv_block_size)
    o, lse, do = _backward_inputs(q, o, lse, do)
    dense = hand_over is None and lists.pair_base is None and dense_ds_fits(q, k)
    bounds = [] if dense or hand_over is False else number_pairs(lists).pair_bounds()
    grads = _lib.host().backward(q, k, v, o, lse, do, q_block_size, kv_block_size, lists.mask_bh, lists.q_cnt, lists.q_idx, lists.k_cnt, lists.k_idx,
                                 lists.pair_base, lists.q_slot, lists.k_slot, bounds, hand_over, dense, ds_workspace_limit(q, k), _split_bytes())
    return tuple(_typed_like(g, t) for g, t in zip(grads, (q, k, v)))


def _flex_block_attn_forward(q, k, v, q_block_size, kv_block_size, block_mask, small_block_mask, use_small_block_mode):
    """Drop-in for flex_block_attn_interface.py:6-8.  `small_block_mask` is the mask at (q_block x kv_block)
    granularity (it equals `block_mask` when the two block sizes agree); `block_mask`, the max-pooled copy the
    reference's kernel needs, is accepted and ignored."""
    fine = small_block_mask if use_small_block_mode else block_mask
    _check_blocks(q, k, q_block_size, kv_block_size, fine)
    lists = lists_for(fine, q_block_size, kv_block_size)
    return forward_with_lists(q, k, v, q_block_size, kv_block_size, lists)


def _flex_block_attn_backward(q, k, v, o, lse, do, q_block_size, kv_block_size, block_mask, small_block_mask, use_small_block_mode):
    """Drop-in for flex_block_attn_interface.py:10-12.  As in the reference, both masks arrive TRANSPOSED
    ([..., kv_blocks, q_blocks], flex_block_attn_interface.py:85-86)."""
    fine_t = small_block_mask if use_small_block_mode else block_mask
    if fine_t.dim() not in (2, 4):
        raise ValueError(f"block_mask must have 2 or 4 dimensions, got {fine_t.dim()}")
    if needs_tile_lists(q_block_size, kv_block_size):
        lists = tile_block_mask(fine_t.transpose(-1, -2).contiguous(), q_block_size, kv_block_size)
    else:
        lists = compact_block_mask(fine_t).transposed()
    return backward_with_lists(q, k, v, o, lse, do, q_block_size, kv_block_size, lists)


class FlexBlockAttnFunc(torch.autograd.Function):
    """autograd wrapper, same signature as flex_block_attn_interface.py:14-89."""

    @staticmethod
    def forward(ctx, q, k, v, q_block_size, kv_block_size, block_mask, is_grad_enabled):
        _check_blocks(q, k, q_block_size, kv_block_size, block_mask)
        is_grad = is_grad_enabled and any(x.requires_grad for x in [q, k, v])
        if is_grad and _backward_takes_mask(q, k, v, q_block_size, kv_block_size, block_mask):
            mask = block_mask.contiguous().clone()  # the caller may write to theirs before backward comes
            o, lse = _lib.host().forward_on_mask(q, k, v, q_block_size, kv_block_size, mask)
            o = _typed_like(o, q)
            ctx.save_for_backward(q, k, v, o, lse)
            ctx.q_block_size = q_block_size
            ctx.kv_block_size = kv_block_size
            ctx.lists, ctx.mask = None, mask
            return o
        lists = lists_for(block_mask, q_block_size, kv_block_size, with_pair_numbers=is_grad and not dense_ds_fits(q, k))
        o, lse = _forward(q, k, v, q_block_size, kv_block_size, block_mask, lists)
        if is_grad:
            ctx.save_for_backward(q, k, v, o, lse)
            ctx.q_block_size = q_block_size
            ctx.kv_block_size = kv_block_size
            ctx.lists = lists  # integer index tensors built here, no part of the autograd graph
        return o

    @staticmethod
    def backward(ctx, dout, *args):
        q, k, v, o, lse = ctx.saved_tensors
        if ctx.lists is None:
            return *_backward_on_mask(q, k, v, o, lse, dout, ctx.q_block_size, ctx.kv_block_size, ctx.mask), None, None, None, None
        dq, dk, dv = backward_with_lists(q, k, v, o, lse, dout, ctx.q_block_size, ctx.kv_block_size, ctx.lists)
        return dq, dk, dv, None, None, None, None


def flex_block_attn_func(q, k, v, q_block_size, kv_block_size, block_mask):
    """Block-sparse attention: softmax(q k^T / sqrt(128)) v restricted, per query block, to the key blocks that
    `block_mask` selects.

    q: (batch, heads, q_seq_len, 128) bf16; k, v: (batch, kv_heads, kv_seq_len, 128) bf16; block_mask: bool
    [q_seq_len / q_block_size, kv_seq_len / kv_block_size] or [batch, heads, ...]. Returns o shaped like q.
    """
    split = -1 if SPLIT_WORKSPACE_MIB is None else _split_bytes()
    o = _lib.host().attention(q, k, v, q_block_size, kv_block_size, block_mask, DS_WORKSPACE_LIMIT_GIB * 2 ** 30, DS_WORKSPACE_FACTOR, split)
    if o is not None:
        return o
    # arguments that need preparation (a mask that is not contiguous, strided tensors whose lengths are no whole tiles), calls
    # that are traced, tensor subclasses, and everything that is going to be reported
    pad_q = _pad_rows(q.shape[2], q_block_size, kv_block_size)
    pad_k = _pad_rows(k.shape[2], kv_block_size, q_block_size)
    if pad_q == 0 and pad_k == 0:
        return FlexBlockAttnFunc.apply(q, k, v, q_block_size, kv_block_size, block_mask, torch.is_grad_enabled())
    # The kernels work on 128-row tiles.  A sequence that is not a multiple of 128 (possible only with block sizes that
    # are not) is padded with rows that no block selects; the padded query rows come back as zeros and are cut off.
    _check_blocks(q, k, q_block_size, kv_block_size, block_mask)
    F = torch.nn.functional
    qp = F.pad(q, (0, 0, 0, pad_q))
    kp, vp = F.pad(k, (0, 0, 0, pad_k)), F.pad(v, (0, 0, 0, pad_k))
    mp = F.pad(block_mask, (0, pad_k // kv_block_size, 0, pad_q // q_block_size), value=False)
    o = FlexBlockAttnFunc.apply(qp, kp, vp, q_block_size, kv_block_size, mp, torch.is_grad_enabled())
    return o[:, :, : q.shape[2]]


def _pad_rows(seq_len, block, other_block):
    """Rows to append so that a sequence cut into `block`-row blocks becomes a whole number of 128-row tiles (0 when
    both block sizes are multiples of 128: the kernels then never see a partial tile)."""
    if not needs_tile_lists(block, other_block) or seq_len % 128 == 0:
        return 0
    unit = block * 128 // math.gcd(block, 128)
    return -seq_len % unit
