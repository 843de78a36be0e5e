"""dK/dV launches whose items are taken in falling order of list length (more than one round of work-groups, at most eight):
every key tile is computed once and lands where it belongs.  Numbers of items that are no multiple of the XCD count, split
items at the end of the order, grouped heads, shared and separate masks, several sorted segments, lists of equal length and
empty ones.  Against the oracle's explicit dense formula (fp32) with the operator's parity bar, and bit-equal on a repeat."""
import pytest
import torch

pytestmark = pytest.mark.gpu

MAX_ABS, REL_L2 = 2e-2, 1e-2


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Skv,qbs,kbs,dims,density", [
    (1, 18, 9, 2048, 3968, 128, 128, 4, 0.3),   # 279 items on eight runs of unequal length, 23 of them split
    (1, 1, 1, 4096, 32896, 128, 128, 2, 0.2),   # 257 items in one run
    (2, 3, 3, 4096, 12288, 128, 384, 4, 0.3),   # 576 items in one run, 64 of them split, key blocks of three tiles
    (1, 8, 8, 4096, 16384, 128, 128, 4, 0.05),  # 1024 items, one head per XCD, two segments
    (1, 4, 4, 4096, 8320, 128, 128, 4, 1.0),    # 260 lists of one length
    # the same where lists of up to 192 slabs make launches without claim counters ordered as well
    (1, 18, 9, 3072, 3968, 128, 128, 4, 0.3),
    (1, 1, 1, 6144, 32896, 128, 128, 2, 0.2),
    (2, 3, 3, 6144, 12288, 128, 384, 4, 0.3),
    (1, 4, 4, 6144, 8320, 128, 128, 4, 1.0),
    (1, 8, 8, 6144, 32640, 128, 128, 4, 0.05),  # 2040 items, 255 on each run: segments that are no multiple of 64
])
def test_ordered_key_tiles(oracle, gpu, B, Hq, Hkv, Sq, Skv, qbs, kbs, dims, density):
    import flex_block_attn_amd as fba

    g = torch.Generator().manual_seed(Skv + Hq)
    nQ, nK = Sq // qbs, Skv // kbs
    m = torch.rand((nQ, nK) if dims == 2 else (B, Hq, nQ, nK), generator=g) < density * torch.linspace(0.2, 1.8, nK)
    if density < 1:
        m[..., :, 1] = False  # a key block nobody selects
        m[..., 0, 0] = True
    m = torch.ones_like(m).to(gpu) if density == 1.0 else m.to(gpu)
    q, do = (torch.randn((B, Hq, Sq, 128), generator=g).to(torch.bfloat16).to(gpu) for _ in range(2))
    k, v = (torch.randn((B, Hkv, Skv, 128), generator=g).to(torch.bfloat16).to(gpu) for _ in range(2))
    print(f"ordered items B{B} Hq{Hq} Hkv{Hkv} Sq{Sq} Skv{Skv} q{qbs} k{kbs}", flush=True)
    lists = fba.lists_for(m, qbs, kbs)
    o, lse = fba.forward_with_lists(q, k, v, qbs, kbs, lists)
    first, again = ([fba.backward_with_lists(q, k, v, o, lse, do, qbs, kbs, lists, hand_over=ho) for ho in (False, True)] for _ in range(2))
    o_ref, lse_ref = oracle.dense_attention_explicit(q, k, v, m, qbs, kbs)
    want = oracle.dense_attention_backward_explicit(q, k, v, o_ref, lse_ref, do, m, qbs, kbs)
    for a, b in zip(first, again):
        for name, x, y, w in zip(("dq", "dk", "dv"), a, b, want):
            mabs, rel = oracle.error_metrics(x.float(), w)
            assert mabs <= MAX_ABS * max(1.0, float(w.abs().max())) and rel <= REL_L2, (name, mabs, rel)
            assert torch.equal(x, y), name
    assert all(torch.equal(a, b) for a, b in zip(first[0][1:], first[1][1:]))  # dK, dV of both backward paths
