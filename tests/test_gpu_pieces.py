"""dK/dV launches whose lists differ so much that the device cuts the long ones into pieces (plan_pieces): a block that every query selects,
a few such blocks, all but one list empty.  Less than a round of key tiles, more than one, more than four (where work-groups claim their
items), grouped heads, one mask for all heads, with dS handed over through numbered and through dense pairs and without.  Against the same
call without a workspace, where nothing is cut: each side rounds the same fp32 sums, taken in another order, to bf16 once.  The lists that
are cut show it (other bits).  Nothing else changes a bit where the host plans no parts, so that masks without a long list show none at all there; a repeat
gives the same bits, and a graph follows the lists of its replay."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

HEAD = 128


def _mask(kind, B, Hq, nQ, nK, dims, g):
    shape = ((B, Hq) if dims == 4 else ()) + (nQ, nK)
    m = torch.rand(shape, generator=g) < {"one": 0.0, "even": 0.4}.get(kind, 0.05)
    long = {"sink": [0], "few": [1, nK // 2, nK - 1], "one": [nK // 3], "even": []}[kind]
    for j in long:
        m[..., j] = True
    return m, long


def _backward(fba, q, k, v, o, lse, do, qbs, kbs, lists, hand_over):
    return fba.backward_with_lists(q, k, v, o, lse, do, qbs, kbs, lists, hand_over=hand_over)


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Skv,qbs,kbs,dims,kind", [
    (1, 1, 1, 16384, 16384, 128, 128, 4, "sink"),     # 128 key tiles
    (1, 1, 1, 16384, 16384, 128, 128, 4, "even"),     # the same without a long list: parts of all lists alike, as the host has planned
    (1, 1, 1, 16384, 30720, 128, 128, 4, "even"),     # 240, none planned: left alone, the longest list being a third above the mean
    (1, 2, 2, 8192, 32768, 128, 128, 4, "even"),      # 512: two rounds, left alone
    (1, 1, 1, 16640, 24192, 128, 384, 4, "few"),      # 189, three to a block
    (1, 3, 3, 8192, 17920, 256, 128, 4, "sink"),      # 420: more than a round
    (1, 3, 3, 8192, 17920, 256, 128, 2, "few"),
    (1, 8, 2, 4096, 16640, 128, 128, 4, "one"),       # lists over four heads
    (2, 2, 2, 8192, 32768, 512, 128, 4, "few"),       # 1024: four rounds
])
@pytest.mark.parametrize("hand_over", [None, True, False])
def test_long_lists_in_pieces(gpu, monkeypatch, B, Hq, Hkv, Sq, Skv, qbs, kbs, dims, kind, hand_over):
    import flex_block_attn_amd as fba
    from flex_block_attn_amd import _lib, interface

    g = torch.Generator().manual_seed(Sq + Skv)
    m, long = _mask(kind, B, Hq, Sq // qbs, Skv // kbs, dims, g)
    q, do = (torch.randn((B, Hq, Sq, HEAD), generator=g).to(torch.bfloat16).to(gpu) for _ in range(2))
    k, v = (torch.randn((B, Hkv, Skv, HEAD), generator=g).to(torch.bfloat16).to(gpu) for _ in range(2))
    print(f"pieces B{B} Hq{Hq} Hkv{Hkv} Sq{Sq} Skv{Skv} q{qbs} k{kbs} {kind} {hand_over}", flush=True)
    lists = fba.lists_for(m.to(gpu), qbs, kbs)
    o, lse = fba.forward_with_lists(q, k, v, qbs, kbs, lists)
    run = lambda: _backward(fba, q, k, v, o, lse, do, qbs, kbs, lists, hand_over)
    cut, again = run(), run()
    monkeypatch.setattr(interface, "SPLIT_WORKSPACE_MIB", "0")
    whole = run()
    assert all(torch.equal(a, b) for a, b in zip(cut, again))
    for name, a, b in zip(("dq", "dk", "dv"), cut, whole):
        assert bool(torch.isfinite(a).all()) and ((a.float() - b.float()).norm() <= 2.0 ** -8 * b.float().norm()).item(), name
    plan = (ctypes.c_int64 * 16)()  # of the dK/dV launch: [2] parts
    _lib.call("fba_split_plan", 1, 1 if dims == 2 else B * Hq, B, Hq, Hkv, Sq, Skv, HEAD, qbs, kbs, _lib.load().fba_split_workspace_bytes(), plan)
    for a, b in zip(cut[1:], whole[1:]):
        differs = (a != b).view(B, Hkv, Skv // kbs, -1).any(-1)
        assert bool(differs[..., long].all())  # cut, in every head
        if kind == "one" or plan[2] == 1:
            differs[..., long] = False
            assert not bool(differs.any())
    empty = ~(m if dims == 4 else m.expand(B, Hq, -1, -1)).any(-2).view(B, Hkv, Hq // Hkv, -1).any(2)
    for t in cut[1:]:
        assert bool((t.view(B, Hkv, Skv // kbs, -1)[empty.to(gpu)] == 0).all())


def test_a_graph_follows_the_lists_of_its_replay(gpu):
    import flex_block_attn_amd as fba

    S, g = 16384, torch.Generator().manual_seed(2)
    q, k, v, do = (torch.randn((1, 1, S, HEAD), generator=g).to(torch.bfloat16).to(gpu) for _ in range(4))
    masks = [_mask(kind, 1, 1, S // 128, S // 128, 4, g)[0].to(gpu) for kind in ("sink", "even", "few", "one")]
    m = masks[0].clone()

    def step(mask):
        lists = fba.lists_for(mask, 128, 128)
        return _backward(fba, q, k, v, *fba.forward_with_lists(q, k, v, 128, 128, lists), do, 128, 128, lists, False)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step(m)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = step(m)
    for mask in masks + masks[:1]:
        m.copy_(mask)
        graph.replay()
        torch.cuda.synchronize()
        taken = [t.clone() for t in got]
        want = step(mask)
        for a, b in zip(taken, want):
            assert torch.equal(a, b)
