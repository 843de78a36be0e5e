"""Backward on tile lists whose query blocks are odd multiples of 16 rows: dK/dV puts the 16-row groups that select a key block side by
side, two to a slab, and stores the dS of each by itself.  Odd numbers of groups, one group, lists that end at and go past what a
work-group's list in LDS holds (1024 groups), groups of several query heads, key blocks of 64 and of whole tiles, parts of split
items, ragged lengths.  Against the oracle's explicit dense formula (fp32) with the operator's parity bar for N(0,1) inputs."""
import pytest
import torch

pytestmark = pytest.mark.gpu

MAX_ABS, REL_L2 = 2e-2, 1e-2


def _inputs(g, gpu, B, Hq, Hkv, Sq, Skv):
    q, do = (torch.randn((B, Hq, Sq, 128), generator=g).to(torch.bfloat16).to(gpu) for _ in range(2))
    k, v = (torch.randn((B, Hkv, Skv, 128), generator=g).to(torch.bfloat16).to(gpu) for _ in range(2))
    return q, k, v, do


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Skv,qbs,kbs,density", [
    (1, 1, 1, 128, 128, 16, 64, 0.3),
    (1, 1, 1, 128, 256, 16, 128, 1.0),
    (2, 4, 2, 384, 384, 48, 192, 0.4),
    (1, 3, 1, 640, 1280, 80, 320, 0.5),
    (1, 1, 1, 128 * 129, 128, 16, 64, 0.99),   # 1032 groups in the tile, 1010 to 1032 in a half
    (1, 2, 1, 128 * 130, 256, 16, 128, 1.0),   # 1040 groups a head
    (1, 1, 1, 128 * 128, 128, 16, 64, 1.0),    # 1024
    (1, 6, 6, 128 * 24, 128 * 24, 16, 64, 0.25),
    (1, 2, 2, 1040, 832, 16, 64, 0.5),         # no whole tiles
])
def test_row_groups(oracle, gpu, B, Hq, Hkv, Sq, Skv, qbs, kbs, density):
    import flex_block_attn_amd as fba

    print(f"row groups B{B} Hq{Hq} Hkv{Hkv} Sq{Sq} Skv{Skv} q{qbs} k{kbs} {density}", flush=True)
    g = torch.Generator().manual_seed(Sq + Skv + qbs)
    m = torch.rand((B, Hq, Sq // qbs, Skv // kbs), generator=g) < density
    m[..., 0, 0] = True
    m = m.to(gpu)
    q, k, v, do = _inputs(g, gpu, B, Hq, Hkv, Sq, Skv)
    o_ref, lse_ref = oracle.dense_attention_explicit(q, k, v, m, qbs, kbs)
    want = oracle.dense_attention_backward_explicit(q, k, v, o_ref, lse_ref, do, m, qbs, kbs)
    ins = [t.clone().requires_grad_(True) for t in (q, k, v)]
    o = fba.flex_block_attn_func(*ins, qbs, kbs, m)
    got = torch.autograd.grad(o, ins, do)
    again = torch.autograd.grad(fba.flex_block_attn_func(*ins, qbs, kbs, m), ins, do)
    for name, a, b, c in zip(("dq", "dk", "dv"), got, want, again):
        mabs, rel = oracle.error_metrics(a.float(), b)
        assert mabs <= MAX_ABS * max(1.0, float(b.abs().max())) and rel <= REL_L2, (name, mabs, rel)
        assert torch.equal(a, c), name
    if Sq % 128 == 0:  # numbered pairs and recomputing: the same dK and dV
        lists = fba.lists_for(m, qbs, kbs)
        o, lse = fba.forward_with_lists(q, k, v, qbs, kbs, lists)
        grads = [fba.backward_with_lists(q, k, v, o, lse, do, qbs, kbs, lists, hand_over=ho) for ho in (False, True)]
        assert torch.equal(grads[0][1], grads[1][1]) and torch.equal(grads[0][2], grads[1][2])
        mabs, rel = oracle.error_metrics(grads[1][0].float(), want[0])
        assert mabs <= MAX_ABS * max(1.0, float(want[0].abs().max())) and rel <= REL_L2


def test_query_blocks_without_keys_touch_nothing(gpu):
    """NaN and inf in query blocks that select no key: gradients of everything else keep their bits."""
    import flex_block_attn_amd as fba

    g = torch.Generator().manual_seed(5)
    B, H, S, qbs, kbs = 1, 2, 2048, 16, 64
    m = torch.rand((B, H, S // qbs, S // kbs), generator=g) < 0.2
    m[:, :, 1::4] = False
    m = m.to(gpu)
    q, k, v, do = _inputs(g, gpu, B, H, H, S, S)
    off = torch.zeros(S, dtype=torch.bool, device=gpu)
    off.view(-1, qbs)[1::4] = True
    lists = fba.lists_for(m, qbs, kbs)
    grads = []
    for bad in (0.0, float("nan"), float("inf")):
        q2, do2 = q.clone(), do.clone()
        q2[:, :, off] = bad
        do2[:, :, off] = bad
        o, lse = fba.forward_with_lists(q2, k, v, qbs, kbs, lists)
        grads.append(fba.backward_with_lists(q2, k, v, o, lse, do2, qbs, kbs, lists, hand_over=True))
    for other in grads[1:]:
        assert torch.equal(grads[0][0], other[0])
        assert torch.equal(grads[0][1], other[1]) and torch.equal(grads[0][2], other[2])
