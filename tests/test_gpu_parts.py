"""How many parts the lists of a launch's last round are cut into is decided on the device, by the lists: the same launches with short
lists (whole items, nothing to merge), middling and full ones (the most parts), with lists that are empty for every second head, more
than half a round and more than a round, grouped heads, a shared mask, block and tile lists.  Against the oracle's explicit dense
formula (fp32) with the operator's parity bar, bit-equal on a repeat, dK and dV the same on both backward paths.  What each launch of a case
cuts is checked against the plans (on the CPU)."""
import ctypes

import pytest
import torch

MAX_ABS, REL_L2 = 2e-2, 1e-2

CASES = {
    # B, Hq, Hkv, Sq, Skv, qbs, kbs, dims: parts of forward, dK/dV, dQ, dQ from dS: "device" decides, the host, or nothing is cut
    (1, 1, 1, 8192, 17408, 128, 128, 2): ("device", "device", "device", "device"),    # dK/dV 136 tiles: more than half a round
    (1, 5, 5, 4352, 4352, 128, 128, 4): ("device", None, "device", None),             # 170 items everywhere
    (1, 12, 3, 2304, 9216, 128, 384, 4): ("device", None, "device", None),            # 216 items everywhere
    (1, 3, 3, 8192, 17920, 256, 128, 4): ("device", "device", "device", "device"),    # dK/dV 420 tiles: a round and more than half
    (1, 8, 1, 2048, 17408, 128, 128, 4): ("device", "device", "device", "device"),    # dK/dV 136 tiles, lists over eight heads
    (1, 3, 3, 2944, 2944, 64, 64, 4): (None, None, None, None),                       # tile lists, 138 items of 64 rows and of 64 keys
    (1, 5, 1, 6528, 8704, 16, 64, 4): (None, None, None, None),                       # 510 of 64 rows, 136 of 64 keys
    (1, 3, 3, 2944, 8192, 64, 64, 4): ("device", "host", None, None),                 # 138 of 64 rows, 384 of 64 keys
    (1, 5, 1, 2560, 6144, 16, 64, 4): ("device", "host", None, None),                 # 200 of 64 rows, 96 of 64 keys, lists over five heads
}


@pytest.mark.parametrize("case", CASES)
def test_what_is_cut(case):
    from flex_block_attn_amd import _lib

    B, Hq, Hkv, Sq, Skv, qbs, kbs, dims = case
    for launch, want in enumerate(CASES[case]):
        plan = (ctypes.c_int64 * 16)()
        _lib.call("fba_split_plan", launch, B * Hq if dims == 4 else 1, B, Hq, Hkv, Sq, Skv, 128, qbs, kbs, _lib.load().fba_split_workspace_bytes(), plan)
        cut = plan[1] < plan[0]
        assert cut == (plan[2] > 1) and (("device" if plan[3] else "host") if cut else None) == want, (launch, list(plan))


@pytest.mark.gpu
@pytest.mark.parametrize("density", [0.03, 0.4, 1.0, "heads"])
@pytest.mark.parametrize("B,Hq,Hkv,Sq,Skv,qbs,kbs,dims", CASES)
def test_parts_by_list_length(oracle, gpu, B, Hq, Hkv, Sq, Skv, qbs, kbs, dims, density):
    import flex_block_attn_amd as fba

    g = torch.Generator().manual_seed(Sq + Skv)
    m = torch.rand(((B, Hq) if dims == 4 else ()) + (Sq // qbs, Skv // kbs), generator=g)
    if density == "heads":
        m = m < 0.5
        if dims == 4:
            m[:, 1::2] = False
    else:
        m = m < density
    m = m.to(gpu)
    q, do = (torch.randn((B, Hq, Sq, 128), generator=g).to(torch.bfloat16).to(gpu) for _ in range(2))
    k, v = (torch.randn((B, Hkv, Skv, 128), generator=g).to(torch.bfloat16).to(gpu) for _ in range(2))
    print(f"parts B{B} Hq{Hq} Hkv{Hkv} Sq{Sq} Skv{Skv} q{qbs} k{kbs} {density}", flush=True)
    lists = fba.lists_for(m, qbs, kbs)
    (o, lse), (o2, lse2) = (fba.forward_with_lists(q, k, v, qbs, kbs, lists) for _ in range(2))
    o_ref, lse_ref = oracle.dense_attention_explicit(q, k, v, m, qbs, kbs)
    mabs, rel = oracle.error_metrics(o.float(), o_ref)
    assert mabs <= MAX_ABS and rel <= REL_L2, (mabs, rel)
    assert torch.equal(torch.isinf(lse).flatten(), torch.isinf(lse_ref).flatten().to(lse.device))
    assert torch.equal(o, o2) and torch.equal(lse, lse2)
    grads = [fba.backward_with_lists(q, k, v, o, lse, do, qbs, kbs, lists, hand_over=ho) for ho in (False, True, True)]
    want = oracle.dense_attention_backward_explicit(q, k, v, o_ref, lse_ref, do, m, qbs, kbs)
    for got in grads[:2]:
        for name, x, w in zip(("dq", "dk", "dv"), got, want):
            mabs, rel = oracle.error_metrics(x.float(), w)
            assert mabs <= MAX_ABS * max(1.0, float(w.abs().max())) and rel <= REL_L2, (name, mabs, rel)
    assert all(torch.equal(x, y) for x, y in zip(grads[1], grads[2]))
    assert torch.equal(grads[0][1], grads[1][1]) and torch.equal(grads[0][2], grads[1][2])
