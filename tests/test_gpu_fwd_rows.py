"""Forward on tile lists in launches that go to the kernel with 16-row waves: 16-row groups that select nothing, the first or only the last
key blocks, all of them; lists of 64 chunks and around, of several registers of 64; key blocks of one and of several chunks; 32-row
blocks; parts of the last items; grouped heads, shared masks.  Against the oracle's explicit dense formula (fp32) with the operator's
parity bar for N(0,1) inputs; bit-equal on a repeat, and rows without keys exactly 0 and -inf."""
import pytest
import torch

pytestmark = pytest.mark.gpu

MAX_ABS, REL_L2 = 2e-2, 1e-2


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Skv,qbs,kbs,dims,kind", [
    (1, 40, 8, 1024, 128, 16, 64, 4, 0.5),        # two chunks
    (1, 40, 40, 1024, 64 * 64, 16, 64, 4, "all"),
    (2, 20, 10, 1024, 64 * 66, 16, 64, 4, "ends"),
    (1, 320, 320, 128, 64 * 130, 16, 64, 2, 0.9),
    (1, 28, 28, 1536, 2304, 48, 192, 4, 0.4),
    (1, 40, 20, 1280, 1280, 80, 320, 2, 0.3),
    (1, 17, 17, 4096, 4096, 16, 128, 4, "one"),   # 544 tiles: 32 of a second round
    (1, 68, 68, 1024, 8192, 16, 64, 4, 0.6),      # the same with lists long enough for parts
    (1, 64, 64, 2048, 1024, 32, 64, 4, 0.3),
])
def test_fwd_rows(oracle, gpu, B, Hq, Hkv, Sq, Skv, qbs, kbs, dims, kind):
    import flex_block_attn_amd as fba

    print(f"rows B{B} Hq{Hq} Hkv{Hkv} Sq{Sq} Skv{Skv} q{qbs} k{kbs} {kind}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(Sq + Skv + qbs)
    shape = ((B, Hq) if dims == 4 else ()) + (Sq // qbs, Skv // kbs)
    nQ, nK = shape[-2:]
    m = torch.rand(shape, generator=g, device=gpu) < (kind if isinstance(kind, float) else 1.0)
    if kind == "ends":  # nothing, the first block, the last, the last 65
        m[:] = False
        m[..., 1::4, 0] = True
        m[..., 2::4, -1] = True
        m[..., 3::4, -65:] = True
    elif kind == "one":
        m[:] = False
        m[..., torch.arange(nQ), torch.randint(0, nK, (nQ,))] = True
    q = torch.randn((B, Hq, Sq, 128), generator=g, device=gpu).to(torch.bfloat16)
    k, v = (torch.randn((B, Hkv, Skv, 128), generator=g, device=gpu).to(torch.bfloat16) for _ in range(2))
    lists = fba.lists_for(m, qbs, kbs)
    o, lse = fba.forward_with_lists(q, k, v, qbs, kbs, lists)
    again = fba.forward_with_lists(q, k, v, qbs, kbs, lists)
    assert torch.equal(o, again[0]) and torch.equal(lse, again[1])
    empty = ~m.any(-1).expand(B, Hq, nQ).repeat_interleave(qbs, -1)
    assert bool((o[empty] == 0).all()) and bool((lse.view(B, Hq, Sq)[empty] == -float("inf")).all())
    step = max(1, 2 ** 28 // (Sq * Skv)) * (Hq // Hkv)  # heads at a time
    for b in range(B):
        for h in range(0, Hq, step):
            hs, ks = slice(h, h + step), slice(h * Hkv // Hq, (h + step) * Hkv // Hq)
            md = m if dims == 2 else m[b:b + 1, hs]
            o_ref, lse_ref = oracle.dense_attention_explicit(q[b:b + 1, hs], k[b:b + 1, ks], v[b:b + 1, ks], md, qbs, kbs)
            mabs, rel = oracle.error_metrics(o[b:b + 1, hs].float(), o_ref)
            assert mabs <= MAX_ABS and rel <= REL_L2, (b, h, mabs, rel)
            some = ~empty[b:b + 1, hs]
            assert float((lse.view(B, Hq, Sq)[b:b + 1, hs] - lse_ref.view(1, -1, Sq))[some].abs().max()) <= 2e-3


def test_scores_that_rise_and_scores_of_minus_infinity(oracle, gpu):
    """Later keys with larger scores, so that the reference rises time and again; keys whose scores are -inf count for nothing."""
    import flex_block_attn_amd as fba

    g = torch.Generator(device=gpu).manual_seed(3)
    B, H, S, qbs, kbs = 1, 20, 2048, 16, 64
    m = torch.rand((B, H, S // qbs, S // kbs), generator=g, device=gpu) < 0.4
    m[..., 0] = True
    q = torch.randn((B, H, S, 128), generator=g, device=gpu).abs().to(torch.bfloat16)
    k = torch.randn((B, H, S, 128), generator=g, device=gpu)
    k = (k + torch.arange(S, device=gpu).view(1, 1, S, 1) * (8.0 / S)).to(torch.bfloat16)
    v = torch.randn((B, H, S, 128), generator=g, device=gpu).to(torch.bfloat16)
    lists = fba.lists_for(m, qbs, kbs)
    for masked in (False, True):
        if masked:
            q[..., 0] = 1  # (0 times -inf is no score)
            k[:, :, 64:128, 0] = -float("inf")
        o, lse = fba.forward_with_lists(q, k, v, qbs, kbs, lists)
        o_ref, lse_ref = oracle.dense_attention_explicit(q, k, v, m, qbs, kbs)
        mabs, rel = oracle.error_metrics(o.float(), o_ref)
        assert mabs <= MAX_ABS * max(1.0, float(o_ref.abs().max())) and rel <= REL_L2, (masked, mabs, rel)
