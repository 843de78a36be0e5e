"""Caller-side steps of the operator in video models, on the GPU: score-driven ("SSTA" style) block masks and the tile
permutation of a latent grid.

The reference names these (create_sta_3d_mask, create_ssta_3d_mask, create_moba_3d_mask, ssta_3d_attention) but has
not released them (flex_block_attn/__init__.py:7-12, README.md:54-55); the definitions below are this package's own and
are stated in include/fba.h.  The static sliding-tile mask is `masks.sta_3d_block_mask`.
"""
import ctypes
import numbers

import torch

from . import _lib
from .interface import HEAD_DIM, _ptr, _require_device, _stream


def _check_seq(x, name):
    _require_device(x, name)
    if x.dtype != torch.bfloat16 or x.dim() != 4 or x.shape[-1] != HEAD_DIM:
        raise ValueError(f"{name} must be a (batch, heads, seq, {HEAD_DIM}) bfloat16 tensor, got {tuple(x.shape)} {x.dtype}")
    return x.contiguous()


def _means_of(x, block_size):
    """(x as the kernels take it, an empty tensor for the means of its blocks)"""
    x = _check_seq(x, "x")
    B, H, S, _ = x.shape
    if block_size <= 0 or S % block_size:
        raise ValueError(f"seq_len ({S}) must be divisible by block_size ({block_size})")
    return x, torch.empty((B, H, S // block_size, HEAD_DIM), dtype=torch.float32, device=x.device)


def block_mean(x, block_size):
    """(B, H, S, 128) bf16 -> (B, H, S / block_size, 128) fp32: the mean of every block of `block_size` rows."""
    x, out = _means_of(x, block_size)
    B, H, S, _ = x.shape
    with torch.cuda.device(x.device):
        _lib.call("fba_block_mean", _ptr(x), _ptr(out), B * H, S, block_size, HEAD_DIM, _stream())
    return out


def _block_means(q, k, q_block_size, kv_block_size):
    """`block_mean` of both, in one launch where they are on one device."""
    (q, q_mean), (k, k_mean) = _means_of(q, q_block_size), _means_of(k, kv_block_size)
    if q.device != k.device or q.numel() == 0 or k.numel() == 0:
        return block_mean(q, q_block_size), block_mean(k, kv_block_size)
    with torch.cuda.device(q.device):
        _lib.call("fba_block_mean_pair", _ptr(q), _ptr(q_mean), q.shape[0] * q.shape[1], q.shape[2], q_block_size, _ptr(k), _ptr(k_mean),
                  k.shape[0] * k.shape[1], k.shape[2], kv_block_size, HEAD_DIM, _stream())
    return q_mean, k_mean


def ssta_mask_from_means(q_mean, k_mean, q_block_size, kv_block_size, topk=16, band=1, sink_blocks=1, base_mask=None):
    """Block means (B, Hq, nQ, 128), (B, Hkv, nK, 128) fp32 -> bool mask (B, Hq, nQ, nK)."""
    _require_device(q_mean, "q_mean")
    _require_device(k_mean, "k_mean")
    if q_mean.dtype != torch.float32 or k_mean.dtype != torch.float32 or q_mean.dim() != 4 or k_mean.dim() != 4:
        raise ValueError("q_mean and k_mean must be 4-D float32 tensors")
    if q_mean.shape[-1] != HEAD_DIM or k_mean.shape[-1] != HEAD_DIM or q_mean.shape[0] != k_mean.shape[0]:
        raise ValueError("q_mean and k_mean must be (B, H, blocks, 128) with equal batch")
    q_mean, k_mean = q_mean.contiguous(), k_mean.contiguous()
    B, Hq, nQ, _ = q_mean.shape
    Hkv, nK = k_mean.shape[1], k_mean.shape[2]
    if base_mask is not None:
        _require_device(base_mask, "base_mask")
        if base_mask.dtype != torch.bool or tuple(base_mask.shape) != (nQ, nK):
            raise ValueError(f"base_mask must be a bool tensor of shape ({nQ}, {nK})")
        base_mask = base_mask.contiguous()
    mask = torch.empty((B, Hq, nQ, nK), dtype=torch.bool, device=q_mean.device)
    with torch.cuda.device(q_mean.device):
        _lib.call("fba_ssta_mask", _ptr(q_mean), _ptr(k_mean), _ptr(base_mask) if base_mask is not None else None, _ptr(mask), B, Hq, Hkv, nQ, nK, q_block_size, kv_block_size,
                  topk, band, sink_blocks, _stream())
    return mask


def create_ssta_mask(q, k, q_block_size, kv_block_size, topk=16, band=1, sink_blocks=1, base_mask=None):
    """Block mask (B, Hq, nQ, nK), bool, for `flex_block_attn_func(q, k, v, q_block_size, kv_block_size, mask)`:
    query block i keeps the key block that holds its first row and its `band` neighbours on either side, the first
    `sink_blocks` key blocks, the `topk` key blocks with the largest <mean(q block i), mean(k block j)>, and whatever
    the optional 2-D `base_mask` (nQ, nK) selects (band=-1 switches the band off)."""
    return ssta_mask_from_means(*_block_means(q, k, q_block_size, kv_block_size), q_block_size, kv_block_size, topk, band, sink_blocks, base_mask)


def create_moba_mask(q, k, q_block_size, kv_block_size, topk):
    """Top-k block selection alone (no band, no sink), plus the query block's own key block."""
    return create_ssta_mask(q, k, q_block_size, kv_block_size, topk=topk, band=0, sink_blocks=0)


def _permute(x, grid, tile, to_tiles):
    x = _check_seq(x, "x")
    B, H, S, _ = x.shape
    T, Hh, W = grid
    if T * Hh * W != S:
        raise ValueError(f"grid {tuple(grid)} does not have seq_len ({S}) tokens")
    out = torch.empty_like(x)
    with torch.cuda.device(x.device):
        _lib.call("fba_tile_permute", _ptr(x), _ptr(out), B * H, T, Hh, W, tile[0], tile[1], tile[2], HEAD_DIM, int(to_tiles), _stream())
    return out


class _TilePermute(torch.autograd.Function):
    """A permutation of token rows: the gradient is the inverse permutation of the incoming gradient."""

    @staticmethod
    def forward(ctx, x, grid, tile, to_tiles):
        ctx.args = (tuple(grid), tuple(tile), to_tiles)
        return _permute(x, grid, tile, to_tiles)

    @staticmethod
    def backward(ctx, g):
        grid, tile, to_tiles = ctx.args
        return _permute(g.to(torch.bfloat16), grid, tile, not to_tiles), None, None, None


def _gather(xs, grid, tile, to_tiles, means=()):
    """`_permute` of up to three tensors on one device in one launch -> (permuted tensors, means of the tiles of those numbered
    in `means`, (B, H, tiles, 128) fp32)."""
    xs = [_check_seq(x, "x") for x in xs]
    T, Hh, W = grid
    for x in xs:
        if T * Hh * W != x.shape[2]:
            raise ValueError(f"grid {tuple(grid)} does not have seq_len ({x.shape[2]}) tokens")
    outs = [torch.empty_like(x) for x in xs]
    tiles = T * Hh * W // (tile[0] * tile[1] * tile[2])
    mean = {j: torch.empty((*xs[j].shape[:2], tiles, HEAD_DIM), dtype=torch.float32, device=xs[j].device) for j in means}
    n = len(xs)
    pointers = ctypes.c_void_p * n
    with torch.cuda.device(xs[0].device):
        _lib.call("fba_tile_gather", n, pointers(*(x.data_ptr() for x in xs)), pointers(*(o.data_ptr() for o in outs)),
                  pointers(*(mean[j].data_ptr() if j in mean else None for j in range(n))), (ctypes.c_int64 * n)(*(x.shape[0] * x.shape[1] for x in xs)),
                  T, Hh, W, tile[0], tile[1], tile[2], HEAD_DIM, int(to_tiles), _stream())
    return outs, [mean[j] for j in means]


class _TilePermuteAll(torch.autograd.Function):
    """q, k, v from raster to tile order in one launch, with the tile means of q and k (constants of the backward pass)."""

    @staticmethod
    def forward(ctx, q, k, v, grid, tile):
        ctx.args = (tuple(grid), tuple(tile))
        ctx.set_materialize_grads(False)  # autograd would fill two tensors of zeros for the means
        outs, means = _gather((q, k, v), grid, tile, True, means=(0, 1))
        ctx.mark_non_differentiable(*means)
        return (*outs, *means)

    @staticmethod
    def backward(ctx, gq, gk, gv, *_):
        given = (gq, gk, gv)
        wanted = [j for j in range(3) if ctx.needs_input_grad[j] and given[j] is not None]
        grads = [None] * 5
        if not wanted:
            return tuple(grads)
        outs, _ = _gather([given[j].to(torch.bfloat16) for j in wanted], *ctx.args, False)
        for j, g in zip(wanted, outs):
            grads[j] = g
        return tuple(grads)


def tile_tokens(x, grid, tile=(6, 8, 8)):
    """(B, H, T*Hh*W, 128) in raster order of the latent grid -> tile order: the tokens of each `tile` become one
    contiguous block (384 tokens for 6x8x8), tiles in raster order of the tile grid."""
    return _TilePermute.apply(x, grid, tile, True)


def untile_tokens(x, grid, tile=(6, 8, 8)):
    """Inverse of `tile_tokens`."""
    return _TilePermute.apply(x, grid, tile, False)


def create_sta_3d_mask(tiles, window, device=None, clamp=True):
    """Static sliding-tile mask over a (t, h, w) grid of tiles: `masks.sta_3d_block_mask`, moved to `device`."""
    from . import masks

    m = masks.sta_3d_block_mask(tiles, window, clamp=clamp)
    return m if device is None else m.to(device)


def create_ssta_3d_mask(q, k, grid, tile=(6, 8, 8), window=(3, 3, 3), topk=16, sink_blocks=1):
    """Sliding-tile window united with score-selected tiles, for q, k already in tile order: bool (B, H, n, n) with
    n = number of tiles."""
    block = tile[0] * tile[1] * tile[2]
    return _ssta_3d_mask_from_means(*_block_means(q, k, block, block), grid, tile, window, topk, sink_blocks)


def _ssta_3d_mask_from_means(q_mean, k_mean, grid, tile, window, topk, sink_blocks):
    """`ssta_mask_from_means` with the sliding window over the grid of tiles, which the kernel works out by itself."""
    nT, nH, nW = (g // t for g, t in zip(grid, tile))
    extents = tuple(window)
    B, Hq, nQ, _ = q_mean.shape
    Hkv, nK = k_mean.shape[1], k_mean.shape[2]
    # The kernel takes three extents that a 32-bit integer holds; anything else is worked out, or refused, where the mask is made of tensors.
    plain = len(extents) == 3 and all(isinstance(w, numbers.Integral) and 0 <= w < 2**31 for w in extents)
    if not plain or nT * nH * nW != nQ or nQ != nK or q_mean.shape[0] != k_mean.shape[0] or q_mean.device != k_mean.device:
        base = create_sta_3d_mask((nT, nH, nW), extents, device=q_mean.device)
        return ssta_mask_from_means(q_mean, k_mean, 1, 1, topk, -1, sink_blocks, base)
    half = [int(w) // 2 for w in extents]
    mask = torch.empty((B, Hq, nQ, nK), dtype=torch.bool, device=q_mean.device)
    with torch.cuda.device(q_mean.device):
        _lib.call("fba_ssta_mask_3d", _ptr(q_mean), _ptr(k_mean), _ptr(mask), B, Hq, Hkv, nT, nH, nW, *half, topk, sink_blocks, _stream())
    return mask


def create_moba_3d_mask(q, k, grid, tile=(6, 8, 8), topk=16):
    """Score-selected tiles plus the query tile itself, for q, k in tile order."""
    block = tile[0] * tile[1] * tile[2]
    return create_moba_mask(q, k, block, block, topk)


def ssta_3d_attention(q, k, v, grid, tile=(6, 8, 8), window=(3, 3, 3), topk=16, sink_blocks=1):
    """Attention over a video latent in raster order: tokens go to tile order, every query tile attends to its
    sliding-tile window, to the sink tiles and to its top-k tiles by mean scores, and the output returns to raster
    order.  Differentiable in q, k, v; the mask is a constant of the backward pass."""
    from .interface import flex_block_attn_func

    block = tile[0] * tile[1] * tile[2]
    if block > 0 and block % 16 == 0 and q.device == k.device == v.device:
        qt, kt, vt, q_mean, k_mean = _TilePermuteAll.apply(q, k, v, grid, tile)
        with torch.no_grad():
            mask = _ssta_3d_mask_from_means(q_mean, k_mean, grid, tile, window, topk, sink_blocks)
    else:
        qt, kt, vt = (tile_tokens(x, grid, tile) for x in (q, k, v))
        with torch.no_grad():
            mask = create_ssta_3d_mask(qt.detach(), kt.detach(), grid, tile, window, topk, sink_blocks)
    return untile_tokens(flex_block_attn_func(qt, kt, vt, block, block, mask), grid, tile)
