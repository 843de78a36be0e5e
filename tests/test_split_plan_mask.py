"""fba_split_plan of forward on the block mask: 64-row tiles that are not cut, 128-row tiles cut as on lists, sizes that fba_fwd_blocks refuses; and
that the device leaves its decision where the plan says, the one it comes to on lists of that length."""
import ctypes

import pytest
import torch

LISTS, MASK = 0, 4


def plan(launch, B, Hq, Hkv, Sq, Skv, qbs, kbs):
    from flex_block_attn_amd import _lib

    out = (ctypes.c_int64 * 16)()
    _lib.call("fba_split_plan", launch, B * Hq, B, Hq, Hkv, Sq, Skv, 128, qbs, kbs, _lib.load().fba_split_workspace_bytes(), out)
    return list(out)


def test_plans():
    from flex_block_attn_amd import _lib

    small = (1, 6, 3, 1408, 1408, 128, 128)
    assert plan(LISTS, *small)[:2] == [66, 0] and plan(MASK, *small)[:4] == [132, 132, 1, 0]
    for sizes in ((1, 24, 6, 768, 30720, 128, 128), (1, 66, 66, 1024, 3072, 128, 128), (1, 3, 3, 4992, 30 * 384, 384, 384)):
        assert plan(MASK, *sizes) == plan(LISTS, *sizes) and plan(MASK, *sizes)[3] == 1
    for sizes in ((1, 24, 6, 768, 128 * 257, 128, 128), (1, 24, 6, 768, 3072, 64, 64)):
        with pytest.raises(_lib.FbaError, match="does not take"):
            plan(MASK, *sizes)


@pytest.mark.gpu
@pytest.mark.parametrize("keep", [1, 24, 96, 240])
def test_the_device_leaves_its_decision_there(gpu, keep):
    import flex_block_attn_amd as fba
    from flex_block_attn_amd import _lib
    from flex_block_attn_amd.interface import _ptr, _stream

    B, Hq, Hkv, Sq, Skv = 1, 24, 6, 768, 30720
    g = torch.Generator(device=gpu).manual_seed(keep)
    score = torch.rand((B, Hq, Sq // 128, Skv // 128), generator=g, device=gpu)
    m = torch.zeros(score.shape, dtype=torch.bool, device=gpu).scatter_(-1, score.topk(keep, -1).indices, True)
    q, k, v = (torch.randn((B, H, S, 128), generator=g, device=gpu).to(torch.bfloat16) for H, S in ((Hq, Sq), (Hkv, Skv), (Hkv, Skv)))
    o, lse = torch.empty_like(q), torch.empty((B, Hq, Sq, 1), device=gpu)
    lists = fba.lists_for(m, 128, 128)
    ws = torch.zeros(_lib.load().fba_split_workspace_bytes() // 4, dtype=torch.int32, device=gpu)
    tail = (lists.mask_bh, B, Hq, Hkv, Sq, Skv, 128, 128, 128, _ptr(ws), ws.numel() * 4, _stream())
    notes = []
    for launch in (LISTS, MASK):
        ws.zero_()
        if launch == LISTS:
            _lib.call("fba_fwd", *map(_ptr, (q, k, v, o, lse, lists.q_cnt, lists.q_idx)), *tail)
        else:
            _lib.call("fba_fwd_blocks", *map(_ptr, (q, k, v, o, lse, m)), None, None, None, None, *tail)
        pl = plan(launch, B, Hq, Hkv, Sq, Skv, 128, 128)
        notes.append(int(ws[pl[4] // 4]))
        assert 1 <= notes[-1] <= pl[2]
    assert notes[0] == notes[1] and (keep != 240 or notes[0] > 1)
