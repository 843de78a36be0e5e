"""What a backward pass keeps in the split workspace while the parts of dK/dV are still to be summed: those parts (or pieces of key tiles) and the note behind
them, the parts and the note of dQ, which is launched with that sum, and the order, the counters and the plan of the pieces at the end.  On the host, over sizes of
the workspace and numbers of compute units; and one such call on the GPU."""
import ctypes

import pytest
import torch


def regions(units, from_ds, B, Hq, Hkv, Sq, Skv, qbs, kbs, mib):
    from flex_block_attn_amd import _lib

    out = (ctypes.c_int64 * 5)()
    _lib.call("fba_split_regions", units, from_ds, B * Hq, B, Hq, Hkv, Sq, Skv, 128, qbs, kbs, mib << 20, out)
    return list(out)


@pytest.mark.parametrize("units", [32, 64, 128, 256])
@pytest.mark.parametrize("mib", [13, 30, 65, 96, 128, 256])
def test_dq_keeps_clear_of_what_is_still_to_be_summed(units, mib):
    beside = 0
    for from_ds in (0, 1):
        for B, Hq, Hkv in ((1, 1, 1), (1, 2, 2), (1, 3, 3), (1, 4, 1), (2, 4, 2), (1, 24, 24)):
            for qbs, kbs in ((128, 128), (384, 128), (384, 384), (64, 64), (16, 128)):
                unit = max(qbs, kbs)
                for q_len in (2048, 16384, 17408, 61440):
                    for kv_len in (1024, 3072, 5504, 17408, 30720):
                        Sq, Skv = q_len // unit * unit, kv_len // unit * unit
                        Sq += Sq % 128 and unit
                        Skv += Skv % 128 and unit
                        parts, pieces, dq, dq_end, kept = regions(units, from_ds, B, Hq, Hkv, Sq, Skv, qbs, kbs, mib)
                        what = (B, Hq, Hkv, Sq, Skv, qbs, kbs, from_ds, parts, pieces, dq, dq_end, kept)
                        assert max(parts, pieces) <= kept <= mib << 20, what
                        if dq >= 0:
                            beside += 1
                            assert max(parts, pieces) <= dq < dq_end <= kept, what
    assert beside > 0 or mib < 30


def test_more_parts_than_pieces():
    """136 key tiles in five parts each, more than the 512 places of pieces: dQ's parts begin behind them."""
    parts, pieces, dq, dq_end, kept = regions(256, 0, 1, 1, 1, 17408, 17408, 128, 128, 128)
    assert parts > pieces > 0 and dq >= parts


@pytest.mark.gpu
@pytest.mark.parametrize("B,Hq,Hkv,Sq,Skv,qbs,kbs,density,ws_mib", [
    (1, 1, 1, 17408, 17408, 128, 128, 0.8, 128),  # pieces possible, not made: 136 key tiles in parts, dQ's parts behind them
    (1, 1, 1, 17408, 17408, 128, 128, 0.8, 96),   # dQ's do not fit there
    (1, 1, 1, 30720, 30720, 384, 384, 0.6, 256),
])
def test_whole_pass_as_launch_by_launch(gpu, B, Hq, Hkv, Sq, Skv, qbs, kbs, density, ws_mib):
    """The same bits as from the entry points that do one launch and its sum, where those cut alike (lists of equal length: no pieces)."""
    import flex_block_attn_amd as fba
    from flex_block_attn_amd import _lib
    from flex_block_attn_amd.interface import _ptr, _stream

    print(f"regions H{Hq} S{Sq} q{qbs} {density} {ws_mib} MiB", flush=True)
    g = torch.Generator(device=gpu).manual_seed(Sq + ws_mib)
    nQ, nK = Sq // qbs, Skv // kbs
    # a band that wraps around: all lists of rows and of columns are equally long
    m = ((torch.arange(nK, device=gpu) - torch.arange(nQ, device=gpu)[:, None]) % nK < round(density * nK)).expand(B, Hq, nQ, nK).contiguous()
    q, do = (torch.randn((B, Hq, Sq, 128), generator=g, device=gpu).to(torch.bfloat16) for _ in range(2))
    k, v = (torch.randn((B, Hkv, Skv, 128), generator=g, device=gpu).to(torch.bfloat16) for _ in range(2))
    lists = fba.lists_for(m, qbs, kbs)
    o, lse = fba.forward_with_lists(q, k, v, qbs, kbs, lists)
    shape = (lists.mask_bh, B, Hq, Hkv, Sq, Skv, 128, qbs, kbs)
    ws = torch.empty(ws_mib << 18, device=gpu)

    def fresh():
        ws.fill_(float("nan"))
        return _ptr(ws), ws.numel() * 4, _stream()

    stats = torch.empty((2, B, Hq, Sq), device=gpu)
    dq, dk, dv, dq1, dk1, dv1 = (torch.empty_like(t) for t in (q, k, v) * 2)
    _lib.call("fba_bwd_stats", *map(_ptr, (o, do, lse, stats)), B * Hq * Sq, 128, _stream())
    _lib.call("fba_bwd_dkdv", *map(_ptr, (q, k, v, do, stats, dk1, dv1, lists.k_cnt, lists.k_idx)), *shape, *fresh())
    _lib.call("fba_bwd_dq", *map(_ptr, (q, k, v, do, stats, dq1, lists.q_cnt, lists.q_idx)), *shape, *fresh())
    for _ in range(3):
        _lib.call("fba_bwd", *map(_ptr, (q, k, v, o, do, lse, stats, dq, dk, dv, lists.q_cnt, lists.q_idx, lists.k_cnt, lists.k_idx)), *shape, *fresh())
        for name, a, b in (("dq", dq, dq1), ("dk", dk, dk1), ("dv", dv, dv1)):
            assert torch.equal(a, b), name
