"""How many parts the device makes, read from the note it leaves in the workspace: by the lengths of the lists that are cut, or of all of the
launch's where tiles are taken in order of length.  Lists that differ along the sequence and from head to head, grouped heads, a shared mask, block and
tile lists; lengths well off the lines of the plan, so that no choice of sample decides.  Launches cut in parts agree with whole ones to the
rounding of bf16 results (fp32 sums in another order), bit for bit where one part is made."""
import ctypes

import pytest
import torch

FWD, DKDV, DQ = 0, 1, 2
HEAD = 128


def plan(launch, B, Hq, Hkv, Sq, Skv, qbs, kbs, dims, ws_bytes=None):
    from flex_block_attn_amd import _lib

    out = (ctypes.c_int64 * 16)()
    n = _lib.load().fba_split_workspace_bytes() if ws_bytes is None else ws_bytes
    _lib.call("fba_split_plan", launch, 1 if dims == 2 else B * Hq, B, Hq, Hkv, Sq, Skv, HEAD, qbs, kbs, n, out)
    return dict(zip(("items", "first", "parts", "device", "note", "spread", "whole", "cut", "least", "fewest"), out), more=list(out)[10:])


def decision(pl, length):
    """(parts, how far off the line between one part and more, what the number of parts goes by) for lists of these lengths."""
    mean, longest = float(length.double().mean()), float(length.max())
    whole = mean + pl["spread"] / 1000 * (longest - mean)
    cut = mean + 0.4 * (whole - mean)
    gain = pl["whole"] * whole - pl["cut"] * cut
    return pl["fewest"] + sum(cut >= n for n in pl["more"]) if gain >= pl["least"] else 1, gain / pl["least"] - 1, cut


def looked_at(pl, length, ordered):
    """The lists that are cut, the shortest in dK/dV launches of more than a round with long lists; all lists of a second round more than half full."""
    if pl["first"] and 2 * (pl["items"] - pl["first"]) > 256 and pl["items"] < 512:
        return length
    return (length.sort(descending=True).values if ordered else length)[pl["first"]:]


def is_ordered(launch, pl, Hq, Hkv, Sq):
    return launch == DKDV and 256 < pl["items"] <= 512 and Hq // Hkv * Sq // 32 >= 192


def mask_of(kind, B, Hq, Sq, Skv, qbs, kbs, dims, g):
    nQ, nK = Sq // qbs, Skv // kbs
    m = torch.rand((B, Hq, nQ, nK) if dims == 4 else (nQ, nK), generator=g)
    if kind == "causal":
        at = torch.arange(nQ)[:, None] / nQ >= torch.arange(nK)[None, :] / nK
        return at.expand(m.shape).contiguous()
    if kind == "last head":  # all of it in the last head, sparse in the others
        return m < torch.where(torch.arange(Hq) == Hq - 1, 1.0, 0.2)[None, :, None, None]
    return m < kind


def steps(launch, m, B, Hq, Hkv, Sq, Skv, qbs, kbs):
    """List length of every tile of the launch, in steps (fine masks: 128-row tiles list what some of their rows select)."""
    m = m.expand(B, Hq, *m.shape[-2:])
    tiled = qbs % 128 or kbs % 128
    if launch == DKDV:
        per_key = m.sum(2) * (qbs // 32)  # [B, Hq, nK]
        per_key = per_key.view(B, Hkv, Hq // Hkv, -1).sum(2)
        return per_key.repeat_interleave(kbs // 128, -1).flatten()
    if tiled:
        union = m.repeat_interleave(qbs, 2).view(B, Hq, Sq // 128, 128, -1).any(3).sum(-1) * (kbs // 64)
        return union.repeat_interleave(2, -1).flatten()  # two 64-row halves read one list
    return (m.sum(-1) * (kbs // 32)).repeat_interleave(qbs // 128, -1).flatten()


CASES = [
    # launch, B, Hq, Hkv, Sq, Skv, qbs, kbs, dims, mask
    (DKDV, 1, 3, 3, 8192, 17920, 256, 128, 4, "causal"),      # more than one round: nearly full lists only
    (DKDV, 1, 3, 3, 8192, 17920, 256, 128, 4, "last head"),
    (DKDV, 1, 3, 3, 8192, 17920, 256, 128, 4, 1.0),
    (DKDV, 1, 3, 3, 8192, 17920, 256, 128, 4, 0.6),
    (DKDV, 1, 5, 5, 8192, 7680, 256, 128, 4, "last head"),    # 44 beyond a round, in order of length: the shortest
    (DKDV, 1, 2, 2, 8192, 18432, 256, 128, 4, "causal"),
    (DKDV, 1, 2, 2, 8192, 18432, 256, 256, 2, "causal"),
    (DKDV, 1, 9, 3, 2048, 12288, 128, 128, 4, "causal"),
    (DKDV, 1, 16, 8, 1024, 8704, 128, 128, 4, "last head"),   # 32 beyond two rounds, in index order: the last kv head's
    (DKDV, 1, 1, 1, 8192, 17408, 128, 128, 2, "causal"),
    (DKDV, 1, 1, 1, 8192, 17408, 128, 128, 2, 0.04),
    (DKDV, 1, 8, 1, 2048, 17408, 128, 128, 4, 0.5),       # lists over eight heads
    (DKDV, 1, 8, 1, 2048, 17408, 128, 128, 4, "last head"),
    (FWD, 1, 3, 3, 8192, 17920, 256, 128, 4, 0.1),
    (FWD, 1, 3, 3, 8192, 17920, 256, 128, 4, 0.5),
    (FWD, 1, 5, 5, 4352, 30720, 128, 384, 4, 0.5),        # 170 tiles
    (FWD, 1, 2, 1, 8192, 16384, 64, 64, 4, 0.4),          # tile lists, half a round of 64-row halves
    (FWD, 1, 1, 1, 12800, 16384, 64, 64, 4, 0.4),         # tile lists, 200 halves
    (FWD, 1, 1, 1, 12800, 16384, 64, 64, 2, 0.03),
    (FWD, 1, 3, 3, 8192, 17920, 8192, 128, 4, 0.6),              # three lists in all
    (FWD, 1, 3, 3, 8192, 17920, 4096, 128, 2, 0.6),              # two
    (DKDV, 1, 5, 1, 4096, 17408, 256, 17408, 4, 1.0),            # one list of five heads' each
    (FWD, 1, 2, 2, 1536, 1536, 128, 128, 2, 0.2),                # 24 tiles
    (FWD, 1, 6, 6, 384, 12288, 128, 128, 4, 0.9),
    (DKDV, 1, 1, 1, 12800, 12800, 128, 128, 4, 0.05),            # 100 tiles
    (DKDV, 1, 1, 1, 12800, 12800, 128, 128, 4, 0.7),
    (DQ, 1, 1, 1, 12800, 12800, 128, 128, 2, "causal"),
    # lists of one round that differ: cut for the longest where the mean would not be
    (FWD, 1, 1, 1, 20480, 20480, 128, 128, 4, 0.1),
    (FWD, 1, 5, 5, 4352, 4352, 128, 128, 4, "causal"),
    (FWD, 1, 5, 5, 4352, 4352, 128, 128, 2, 0.05),
    (FWD, 1, 1, 1, 16384, 8192, 64, 64, 4, "causal"),
    (DKDV, 1, 1, 1, 6144, 17408, 128, 128, 4, "causal"),
    (DKDV, 1, 8, 1, 2048, 17408, 128, 128, 2, "causal"),
    (DQ, 1, 5, 5, 4352, 4352, 128, 128, 4, "causal"),
    (DQ, 1, 3, 3, 8192, 17920, 256, 128, 4, 0.1),
    (DQ, 1, 3, 3, 8192, 17920, 256, 128, 4, 0.5),
]


@pytest.mark.gpu
@pytest.mark.parametrize("launch,B,Hq,Hkv,Sq,Skv,qbs,kbs,dims,kind", CASES)
def test_the_device_decides_by_the_lists_it_cuts(gpu, launch, B, Hq, Hkv, Sq, Skv, qbs, kbs, dims, kind):
    import flex_block_attn_amd as fba
    from flex_block_attn_amd import _lib
    from flex_block_attn_amd.interface import _ptr, _stream

    g = torch.Generator().manual_seed(Sq + Skv)
    m = mask_of(kind, B, Hq, Sq, Skv, qbs, kbs, dims, g)
    pl = plan(launch, B, Hq, Hkv, Sq, Skv, qbs, kbs, dims)
    length = steps(launch, m, B, Hq, Hkv, Sq, Skv, qbs, kbs)
    assert length.numel() == pl["items"]
    want, _, mean = decision(pl, looked_at(pl, length, is_ordered(launch, pl, Hq, Hkv, Sq)))
    print(f"parts launch {launch} B{B} Hq{Hq} Hkv{Hkv} Sq{Sq} Skv{Skv} q{qbs} k{kbs} {kind}: {pl} mean {mean:.0f} -> {want}", flush=True)
    q, do = (torch.randn((B, Hq, Sq, HEAD), generator=g).to(torch.bfloat16).to(gpu) for _ in range(2))
    k, v = (torch.randn((B, Hkv, Skv, HEAD), generator=g).to(torch.bfloat16).to(gpu) for _ in range(2))
    lists = fba.lists_for(m.to(gpu), qbs, kbs)
    stats = torch.stack([torch.full((B, Hq, Sq), 6.0), torch.zeros((B, Hq, Sq))]).to(gpu)  # finite and alike for both runs
    shape = (lists.mask_bh, B, Hq, Hkv, Sq, Skv, HEAD, qbs, kbs)

    def run(ws, n):
        tail = (_ptr(ws) if ws is not None else None, n, _stream())
        if launch == FWD:
            outs = torch.empty_like(q), torch.empty((B, Hq, Sq, 1), device=gpu)
            _lib.call("fba_fwd_tiled" if lists.tiled else "fba_fwd", *map(_ptr, (q, k, v, *outs, lists.q_cnt, lists.q_idx)), *shape, *tail)
        elif launch == DQ:
            outs = (torch.empty_like(q),)
            _lib.call("fba_bwd_dq", *map(_ptr, (q, k, v, do, stats, *outs, lists.q_cnt, lists.q_idx)), *shape, *tail)
        else:
            outs = torch.empty_like(k), torch.empty_like(v)
            _lib.call("fba_bwd_dkdv", *map(_ptr, (q, k, v, do, stats, *outs, lists.k_cnt, lists.k_idx)), *shape, *tail)
        return outs

    n = _lib.load().fba_split_workspace_bytes()
    ws = torch.full((n,), 0x5A, dtype=torch.uint8, device=gpu)
    cut, whole = run(ws, n), run(None, 0)
    made = int(ws[pl["note"]:pl["note"] + 4].view(torch.int32)) if pl["device"] else pl["parts"]
    assert made == want
    for a, b in zip(cut, whole):
        a, b = a.float(), b.float()
        fin = torch.isfinite(b)
        assert torch.equal(torch.isfinite(a), fin)
        assert ((a - b)[fin].norm() <= 2.0 ** -8 * b[fin].norm()).item()  # each side rounds to bf16 once
        assert torch.equal(a, b) == (want == 1)


@pytest.mark.parametrize("launch,B,Hq,Hkv,Sq,Skv,qbs,kbs,dims,kind", CASES)
def test_the_cases_say_what_they_claim(launch, B, Hq, Hkv, Sq, Skv, qbs, kbs, dims, kind):
    """The device decides, and the mean length lies well off every line."""
    pl = plan(launch, B, Hq, Hkv, Sq, Skv, qbs, kbs, dims)
    assert pl["device"] == 1 and pl["parts"] >= 2
    m = mask_of(kind, B, Hq, Sq, Skv, qbs, kbs, dims, torch.Generator().manual_seed(Sq + Skv))
    length = steps(launch, m, B, Hq, Hkv, Sq, Skv, qbs, kbs)
    want, off, mean = decision(pl, looked_at(pl, length, is_ordered(launch, pl, Hq, Hkv, Sq)))
    assert abs(off) > 0.1, (off, mean, pl)
    assert want == 1 or all(not 0.85 * mean < n < 1.15 * mean for n in pl["more"]), (mean, pl)


@pytest.mark.parametrize("launch,B,Hq,Hkv,Sq,Skv,qbs,kbs", [(FWD, 1, 5, 5, 4352, 4352, 128, 128), (FWD, 1, 1, 1, 16384, 8192, 64, 64), (DKDV, 1, 1, 1, 6144, 17408, 128, 128),
                                                             (DKDV, 1, 8, 1, 2048, 17408, 128, 128), (DQ, 1, 5, 5, 4352, 4352, 128, 128)])
def test_the_longest_list_of_a_round_decides(launch, B, Hq, Hkv, Sq, Skv, qbs, kbs):
    """Lists that fall to nothing are cut where lists of one length, as long as their mean, are not."""
    pl = plan(launch, B, Hq, Hkv, Sq, Skv, qbs, kbs, 4)
    most = Hq // Hkv * Sq // 32 if launch == DKDV else Skv // (64 if qbs < 128 else 32)
    at = next(n for n in range(most) if (pl["whole"] - pl["cut"]) * n >= pl["least"])  # equal lists are cut from here on
    falling = torch.linspace(0, min(most, 1.9 * at), 129)
    assert float(falling.mean()) < at and decision(pl, falling)[0] > 1
    assert decision(pl, falling * 0 + at - 1)[0] == 1 and decision(pl, falling * 0 + at)[0] > 1


@pytest.mark.parametrize("launch,H,S,parts", [(FWD, 24, 11520, 2), (FWD, 16, 8704, 4), (FWD, 24, 3072, 4), (DKDV, 8, 9216, 4)])
def test_full_lists_behind_two_rounds_are_cut_like_usual_ones(launch, H, S, parts):
    pl = plan(launch, 1, H, H, S, S, 128, 128, 4)
    steps = torch.full((1,), S // 32)
    assert decision(pl, steps)[0] == pl["parts"] == parts
    assert pl["items"] < 1024 or decision(pl, (0.6 * steps).int())[0] == parts


def test_second_rounds_are_cut_where_lists_are_nearly_full():
    for Sq, Hkv in ((8192, 3), (17920, 3), (8192, 1)):
        pl = plan(DKDV, 1, 3, Hkv, Sq, 17920 * 3 // Hkv, 256, 128, 4)
        assert pl["items"] == 420 and pl["first"] == 256 and pl["parts"] == 3
        assert pl["spread"] == 0 and 0.89 <= pl["least"] / (pl["whole"] - pl["cut"]) / ((3 // Hkv) * Sq / 32) <= 0.91


@pytest.mark.gpu
def test_a_replayed_graph_decides_by_the_lists_of_that_replay(gpu):
    import flex_block_attn_amd as fba

    H, S = 1, 20480
    assert plan(FWD, 1, H, H, S, S, 128, 128, 4)["device"] == 1
    g = torch.Generator().manual_seed(5)
    q, k, v = (torch.randn((1, H, S, HEAD), generator=g).to(torch.bfloat16).to(gpu) for _ in range(3))
    masks = [(torch.rand((1, H, S // 128, S // 128), generator=g) < d).to(gpu) for d in (0.02, 0.5, 0.02)]
    m = masks[0].clone()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        fba.flex_block_attn_func(q, k, v, 128, 128, m)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        o = fba.flex_block_attn_func(q, k, v, 128, 128, m)
    for mask in masks:
        m.copy_(mask)
        graph.replay()
        torch.cuda.synchronize()
        got = o.clone()
        assert torch.equal(got, fba.flex_block_attn_func(q, k, v, 128, 128, mask))
