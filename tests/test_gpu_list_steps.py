"""Lists of masks around the edges of a scan's step (both flavours; tile lists take four steps of 64 entries at a time), and tile lists of a
mask that ends inside the last tile (fba_lists_cut) against those of the mask filled up with unselected blocks.  Exact.  Gradients that leave
out the rows of the fill (fba_bwd_tiled_cut), from dO with and without them: the bits of the calls that write them."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


def _ptr(t):
    return ctypes.c_void_p(0 if t is None else t.data_ptr())


def _stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def _lists(m, nQ, nK, qbs, kbs, both=True):
    from flex_block_attn_amd import _lib

    M, rows, cols = m.shape
    tiled = qbs % 128 != 0 or kbs % 128 != 0
    n_q, n_k, k_len = (nQ * qbs // 128, nK * kbs // 128, nQ * qbs // 32) if tiled else (nQ, nK, nQ)
    i32 = dict(dtype=torch.int32, device=m.device)
    out = [torch.full(s, -7, **i32) for s in ((M, n_q), (M, n_q, nK), (M, n_k), (M, n_k, k_len))]
    given = out if both else out[:2] + [None, None]
    _lib.call("fba_lists_cut", _ptr(m), M, nQ, nK, rows, cols, qbs, kbs, *map(_ptr, given), _stream())
    return out


@pytest.mark.parametrize("nQ,nK", [(1, 1), (63, 257), (64, 256), (255, 65), (256, 64), (257, 320), (520, 513)])
def test_compaction_of_long_rows(gpu, nQ, nK):
    g = torch.Generator().manual_seed(nQ + nK)
    m = torch.rand((2, nQ, nK), generator=g) < 0.4
    q_cnt, q_idx, k_cnt, k_idx = (t.cpu() for t in _lists(m.to(gpu), nQ, nK, 128, 128))
    for x, cnt, idx in ((m, q_cnt, q_idx), (m.transpose(1, 2), k_cnt, k_idx)):
        n = x.shape[-1]
        want = torch.where(x, torch.arange(n).expand_as(x), n).sort(-1).values
        assert torch.equal(cnt.long(), x.sum(-1)) and torch.equal(idx.long(), torch.where(want == n, -1, want))


@pytest.mark.parametrize("rows,cols,nQ,nK,qbs,kbs", [
    (1, 1, 8, 2, 16, 64),          # one block of each
    (196, 49, 200, 50, 16, 64),    # 24.5 tiles
    (5, 3, 6, 4, 64, 64),
    (3, 7, 4, 8, 64, 192),         # key blocks that straddle tiles
    (513, 255, 514, 256, 64, 64),  # rows around a step of 256 entries
    (260, 259, 264, 260, 16, 64),
    (4, 258, 4, 258, 64, 64),      # whole tiles
])
@pytest.mark.parametrize("both", [True, False])
def test_lists_of_a_mask_that_ends_inside_a_tile(gpu, rows, cols, nQ, nK, qbs, kbs, both):
    g = torch.Generator().manual_seed(rows * cols + qbs)
    m = torch.rand((3, rows, cols), generator=g) < 0.5
    m[1] = True
    whole = torch.zeros((3, nQ, nK), dtype=torch.bool)
    whole[:, :rows, :cols] = m
    got, want = _lists(m.to(gpu), nQ, nK, qbs, kbs, both), _lists(whole.to(gpu), nQ, nK, qbs, kbs)
    for a, b in zip(got[: 4 if both else 2], want):
        assert torch.equal(a, b)
    # every 128-row tile lists the key blocks that one of its rows selects
    touched = whole.repeat_interleave(qbs, 1).reshape(3, nQ * qbs // 128, 128, nK).any(2)
    assert torch.equal(want[0].cpu().long(), touched.sum(-1))


@pytest.mark.parametrize("B,Hq,Hkv,rows,cols,nQ,nK,qbs,kbs", [
    (1, 1, 1, 1, 1, 8, 2, 16, 64),          # a tile of which 16 rows and half of the keys are left
    (2, 4, 2, 49, 13, 56, 14, 16, 64),      # grouped heads, whole 64-key halves left out
    (1, 2, 2, 5, 130, 6, 132, 64, 64),      # few query tiles, long lists
    (1, 1, 1, 131, 3, 132, 4, 64, 64),      # few key tiles, whose lists are cut into parts
    (1, 3, 1, 7, 3, 8, 4, 64, 192),         # key blocks that straddle tiles
    (1, 2, 1, 6, 4, 6, 4, 64, 64),          # nothing left out
])
@pytest.mark.parametrize("fill", [True, False])
def test_gradients_without_the_fill(gpu, fill, B, Hq, Hkv, rows, cols, nQ, nK, qbs, kbs):
    from flex_block_attn_amd import _lib

    g = torch.Generator().manual_seed(rows * cols + qbs)
    Sq, Skv, out_q, out_kv = nQ * qbs, nK * kbs, rows * qbs, cols * kbs
    m = (torch.rand((B * Hq, rows, cols), generator=g) < 0.6).to(gpu)
    lists = _lists(m, nQ, nK, qbs, kbs)

    def padded(heads, length, used):
        t = torch.zeros((B, heads, length, 128), dtype=torch.bfloat16)
        t[:, :, :used] = torch.randn((B, heads, used, 128), generator=g)
        return t.to(gpu)

    q, do = padded(Hq, Sq, out_q), padded(Hq, Sq, out_q)
    k, v = padded(Hkv, Skv, out_kv), padded(Hkv, Skv, out_kv)
    split = torch.empty(_lib.load().fba_split_workspace_bytes(), dtype=torch.uint8, device=gpu)
    ws = (_ptr(split), split.numel(), _stream())
    shape = (B, Hq, Hkv, Sq, Skv)
    o, lse, stats = torch.empty_like(q), torch.empty((B, Hq, Sq, 1), device=gpu), torch.empty((2, B, Hq, Sq), device=gpu)
    _lib.call("fba_fwd_tiled", *map(_ptr, (q, k, v, o, lse, *lists[:2])), B * Hq, *shape, 128, qbs, kbs, *ws)
    i32 = dict(dtype=torch.int32, device=gpu)
    M, n_qt, n_kt = B * Hq, Sq // 128, Skv // 128
    base, slot, table = torch.empty((M * n_kt + 1,), **i32), torch.empty((M, n_kt, Sq // 32), **i32), torch.empty((M, n_qt, n_kt), **i32)
    _lib.call("fba_tile_slots", *map(_ptr, lists[2:]), M, n_qt, n_kt, *map(_ptr, (base, slot, table)), _stream())
    pairs = int(base[-1])
    ins = [_ptr(t) for t in (q, k, v, o, do, lse, stats)]
    l4 = [_ptr(t) for t in lists]

    def outs(n_q, n_kv):
        return [torch.full((B, h, n, 128), 7, dtype=torch.bfloat16, device=gpu) for h, n in ((Hq, n_q), (Hkv, n_kv), (Hkv, n_kv))]

    for kind in ("recompute", "dense", "numbered"):
        ds = torch.empty((max(1, M * n_qt * n_kt if kind == "dense" else pairs) * 32768,), dtype=torch.uint8, device=gpu)
        want, got = outs(Sq, Skv), outs(out_q, out_kv)
        tail = (M, *shape, 128, qbs, kbs, *ws)
        if kind == "recompute":
            _lib.call("fba_bwd_tiled", *ins, *map(_ptr, want), *l4, *tail)
        elif kind == "dense":
            _lib.call("fba_bwd_dense", *ins, _ptr(ds), ds.numel(), *map(_ptr, want), *l4, *tail)
        else:
            _lib.call("fba_bwd_tiled_handover", *ins, _ptr(ds), ds.numel(), *map(_ptr, want), *l4, *map(_ptr, (base, slot, table)), pairs, *tail)
        numbers = (base, slot, table) if kind == "numbered" else (None,) * 3
        given, filled = do[:, :, :out_q].contiguous(), torch.full_like(do, 7)
        _lib.call("fba_bwd_tiled_cut", *ins[:4], *map(_ptr, (given, filled) if fill else (do, None)), *ins[5:], _ptr(None if kind == "recompute" else ds), ds.numel(), *map(_ptr, got), *l4, *map(_ptr, numbers),
                  pairs if kind == "numbered" else 0, M, *shape, out_q, out_kv, 128, qbs, kbs, *ws)
        for a, b in zip(got, want):
            assert torch.equal(a, b[:, :, : a.shape[2]]), kind
            assert bool((b[:, :, a.shape[2] :] == 0).all()), kind
        assert torch.equal(filled, do if fill else torch.full_like(do, 7)), kind
