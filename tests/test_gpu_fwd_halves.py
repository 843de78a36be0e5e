"""Forward on tile lists: work-groups of 64 rows that take the entries naming their half of a 128-row tile from a register of 64
at a time.  List lengths around 64 and its multiples, halves that select
nothing, the first or only the last entries, one chunk in all, key blocks of one and of several chunks, 16-row groups, grouped
heads, shared and separate masks, split launches.  Against the oracle's explicit dense formula (fp32) with the operator's parity
bar for N(0,1) inputs; O, LSE bit-equal on a repeat, and rows without keys exactly 0 and -inf."""
import ctypes

import pytest
import torch

MAX_ABS, REL_L2 = 2e-2, 1e-2


def _mask(kind, shape, g):
    m = torch.rand(shape, generator=g) < 0.4
    nQ, nK = shape[-2:]
    if kind == "all":
        m[:] = True
    elif kind == "one":  # a single key block per query block
        m[:] = False
        m[..., torch.arange(nQ), torch.randint(0, nK, (nQ,), generator=g)] = True
    elif kind == "ends":  # query blocks take turns: nothing, the first block only, the last only, the last 64 or so
        m[:] = False
        m[..., 1::4, 0] = True
        m[..., 2::4, -1] = True
        m[..., 3::4, -min(nK, 65):] = True
    return m


@pytest.mark.parametrize("Skv,cut", [(768, False), (1280, True)])
def test_last_round_of_the_split_case(Skv, cut):
    from flex_block_attn_amd import _lib

    plan = (ctypes.c_int64 * 16)()
    _lib.call("fba_split_plan", 0, 30, 1, 30, 30, 1152, Skv, 128, 16, 64, _lib.load().fba_split_workspace_bytes(), plan)
    assert plan[0] == 540 and plan[1] == (512 if cut else 540) and (plan[2] > 1) == cut


@pytest.mark.gpu
@pytest.mark.parametrize("B,Hq,Hkv,Sq,Skv,qbs,kbs,dims,kind", [
    (1, 1, 1, 128, 128, 64, 64, 2, "all"),
    (1, 1, 1, 128, 128, 16, 128, 2, "one"),
    (1, 2, 2, 256, 4096, 64, 64, 4, "all"),       # 64 entries: one register exactly
    (1, 2, 1, 256, 4224, 64, 64, 4, "all"),       # 66 entries
    (1, 2, 2, 512, 8192, 64, 64, 4, "ends"),      # 128 entries, halves that name few of them
    (2, 3, 3, 512, 16640, 16, 64, 4, "ends"),     # 260 entries, more than one pass of the count
    (2, 2, 1, 640, 2048, 32, 64, 4, "random"),
    (1, 3, 3, 768, 1152, 48, 192, 4, "random"),   # row groups that straddle halves, three chunks to a block
    (1, 2, 2, 1152, 1152, 192, 384, 2, "random"),
    (1, 1, 1, 640, 640, 320, 64, 4, "one"),
    (1, 3, 1, 384, 1152, 128, 64, 4, "random"),   # halves that agree
    (1, 2, 2, 768, 1152, 384, 192, 2, "ends"),
    (2, 24, 24, 1536, 1536, 64, 64, 4, "random"),  # more items than slots
    (1, 30, 30, 1152, 768, 16, 64, 4, "random"),   # a round and 28 items, whole
    (1, 30, 30, 1152, 1280, 16, 64, 4, "random"),  # the last round of 28 items is split
])
def test_fwd_halves(oracle, gpu, B, Hq, Hkv, Sq, Skv, qbs, kbs, dims, kind):
    import flex_block_attn_amd as fba

    g = torch.Generator().manual_seed(Sq + Skv + qbs)
    m = _mask(kind, ((B, Hq) if dims == 4 else ()) + (Sq // qbs, Skv // kbs), g).to(gpu)
    q = torch.randn((B, Hq, Sq, 128), generator=g).to(torch.bfloat16).to(gpu)
    k, v = (torch.randn((B, Hkv, Skv, 128), generator=g).to(torch.bfloat16).to(gpu) for _ in range(2))
    print(f"fwd halves B{B} Hq{Hq} Hkv{Hkv} Sq{Sq} Skv{Skv} q{qbs} k{kbs} {kind}", flush=True)
    lists = fba.lists_for(m, qbs, kbs)
    (o, lse), (o2, lse2) = (fba.forward_with_lists(q, k, v, qbs, kbs, lists) for _ in range(2))
    want, lse_want = oracle.dense_attention_explicit(q, k, v, m, qbs, kbs)
    mabs, rel = oracle.error_metrics(o.float(), want)
    assert mabs <= MAX_ABS and rel <= REL_L2, (mabs, rel)
    lse_want = lse_want.reshape(lse.shape).to(lse.device)
    empty = torch.isinf(lse_want)
    assert torch.equal(torch.isinf(lse), empty) and bool((o[empty[..., 0]] == 0).all())
    assert float((lse - lse_want)[~empty].abs().max()) <= 2e-2  # the denominator sums bf16-rounded P
    assert torch.equal(o, o2) and torch.equal(lse, lse2)


@pytest.mark.gpu
@pytest.mark.parametrize("qbs,kbs,Skv", [(64, 64, 384), (64, 128, 384), (16, 64, 384), (192, 64, 384), (64, 64, 16384)])
def test_fwd_scores_of_minus_infinity(gpu, qbs, kbs, Skv):
    """Keys whose scores are -inf count for nothing, also where they fill the first slabs a wave meets, all of one wave's slabs, or
    (last case) a whole part of a split list."""
    import flex_block_attn_amd as fba

    Sq = 384
    g = torch.Generator().manual_seed(Skv + qbs)
    q, k, v = (torch.randn((1, 1, s, 128), generator=g).to(torch.bfloat16) for s in (Sq, Skv, Skv))
    q[..., 0] = q[..., 0].abs() + 0.125
    out = torch.rand((Skv,), generator=g) < 0.3
    out[:96] = True                        # the first chunk and the first half of the second
    out[torch.arange(Skv) % 64 >= 32] = True  # everything of one of the two waves of a row group
    out[Skv // 2: Skv // 2 + Skv // 4] = True
    k[0, 0, out, 0] = -float("inf")
    mask = torch.ones((Sq // qbs, Skv // kbs), dtype=torch.bool)
    print(f"-inf scores Skv{Skv} q{qbs} k{kbs}", flush=True)
    o, lse = fba.forward_with_lists(q.to(gpu), k.to(gpu), v.to(gpu), qbs, kbs, fba.lists_for(mask.to(gpu), qbs, kbs))
    s = (q[0, 0].double() @ k[0, 0].double().T) / 128 ** 0.5
    want = s.softmax(-1) @ v[0, 0].double()
    got = o[0, 0].double().cpu()
    assert float((got - want).abs().max()) <= MAX_ABS and float((got - want).norm() / want.norm()) <= REL_L2
    assert float((lse.reshape(-1).double().cpu() - s.logsumexp(-1)).abs().max()) <= 2e-2
