"""dQ from handed-over dS in work-groups of 256 and 384 query rows (query blocks that are multiples of these, launches of two
rounds and more): several tiles to a query block, key blocks of one and of several tiles, lists of one entry and empty ones,
split items, numbered and dense places for dS.  Against the oracle's explicit dense formula (fp32) with the operator's parity bar
for N(0,1) inputs."""
import pytest
import torch

pytestmark = pytest.mark.gpu

MAX_ABS, REL_L2 = 2e-2, 1e-2


@pytest.mark.parametrize("Hq,Hkv,Sq,Skv,qbs,kbs,dims,limit", [
    (16, 4, 12288, 768, 384, 384, 4, 20.0),   # 512 items of 384 rows
    (16, 16, 12672, 1280, 384, 128, 2, 20.0),  # 528: the last sixteen are split; many heads to a mask
    (16, 16, 12288, 768, 768, 384, 4, 20.0),  # two tiles to a query block
    (17, 17, 8192, 1024, 256, 128, 4, 20.0),  # 544 items of 256 rows
    (16, 2, 8192, 1024, 1024, 512, 2, 20.0),
    (16, 16, 12288, 768, 384, 384, 4, 0.25),  # numbered places, several launches below the line
])
def test_wide_query_tiles(oracle, gpu, monkeypatch, Hq, Hkv, Sq, Skv, qbs, kbs, dims, limit):
    import flex_block_attn_amd as fba
    from flex_block_attn_amd import interface

    g = torch.Generator().manual_seed(Sq + Skv + qbs)
    m = torch.rand(((1, Hq) if dims == 4 else ()) + (Sq // qbs, Skv // kbs), generator=g) < 0.5
    m[..., 0, :] = False
    m[..., 1, :] = False
    m[..., 1, -1] = True
    m = m.to(gpu)
    q, do = (torch.randn((1, Hq, Sq, 128), generator=g).to(torch.bfloat16).to(gpu) for _ in range(2))
    k, v = (torch.randn((1, Hkv, Skv, 128), generator=g).to(torch.bfloat16).to(gpu) for _ in range(2))
    print(f"wide query tiles Hq{Hq} Hkv{Hkv} Sq{Sq} Skv{Skv} q{qbs} k{kbs} limit {limit}", flush=True)
    o_ref, lse_ref = oracle.dense_attention_explicit(q, k, v, m, qbs, kbs)
    want = oracle.dense_attention_backward_explicit(q, k, v, o_ref, lse_ref, do, m, qbs, kbs)
    monkeypatch.setattr(interface, "DS_WORKSPACE_LIMIT_GIB", limit)
    ins = [t.clone().requires_grad_(True) for t in (q, k, v)]
    dense = torch.autograd.grad(fba.flex_block_attn_func(*ins, qbs, kbs, m), ins, do)
    lists = fba.lists_for(m, qbs, kbs)
    o, lse = fba.forward_with_lists(q, k, v, qbs, kbs, lists)
    numbered = fba.backward_with_lists(q, k, v, o, lse, do, qbs, kbs, lists, hand_over=True)
    for got in (dense, numbered):
        for name, a, b in zip(("dq", "dk", "dv"), got, want):
            mabs, rel = oracle.error_metrics(a.float(), b)
            assert mabs <= MAX_ABS * max(1.0, float(b.abs().max())) and rel <= REL_L2, (name, mabs, rel)
    assert bool((numbered[0][:, :, :qbs] == 0).all()) and bool((dense[0][:, :, :qbs] == 0).all())
