"""dK/dV on tile lists at the sizes where its list handling can go wrong: lists longer than one LDS chapter, fewer slabs than
the four of a step, remainders, halves of a 128-key tile with different (or no) slabs, 16-row halves, split launches.  Against
the oracle's explicit dense formula (fp32), with the operator's parity bar for N(0,1) inputs."""
import pytest
import torch

pytestmark = pytest.mark.gpu

MAX_ABS, REL_L2 = 2e-2, 1e-2


def _mask(kind, B, Hq, nQ, nK, g):
    m = torch.rand((B, Hq, nQ, nK), generator=g) < 0.5
    if kind == "all":
        m[:] = True
    elif kind == "one":  # every key block is selected by a single query block
        m[:] = False
        m[..., torch.randint(0, nQ, (nK,), generator=g), torch.arange(nK)] = True
    elif kind == "half":  # every second key block by nobody
        m[..., 1::2] = False
    return m


@pytest.mark.parametrize("Hq,Hkv,Sq,Skv,qbs,kbs,kind", [
    (4, 1, 10240, 128, 64, 64, "all"),      # 1280 slabs per key half: more than a chapter, over four query heads
    (1, 1, 34816, 128, 64, 64, "random"),   # one head, several rounds of the scan
    (2, 2, 640, 640, 32, 64, "random"),     # lists of any length modulo four
    (2, 1, 384, 256, 32, 64, "one"),        # one slab per head, fewer than a step holds and than there are parts
    (2, 2, 512, 512, 16, 64, "random"),     # 16-row halves
    (1, 1, 512, 512, 16, 64, "one"),
    (2, 2, 768, 768, 64, 64, "half"),       # key halves without any slab
    (3, 3, 384, 384, 64, 192, "random"),    # key blocks that straddle key tiles
    (24, 24, 1536, 1536, 64, 64, "random"),  # more key halves than compute units
])
def test_slab_kernel_list_edges(oracle, gpu, Hq, Hkv, Sq, Skv, qbs, kbs, kind):
    import flex_block_attn_amd as fba

    g = torch.Generator().manual_seed(Sq + Skv + qbs)
    m = _mask(kind, 1, Hq, Sq // qbs, Skv // kbs, g).to(gpu)
    q, do = (torch.randn((1, Hq, Sq, 128), generator=g).to(torch.bfloat16).to(gpu) for _ in range(2))
    k, v = (torch.randn((1, Hkv, Skv, 128), generator=g).to(torch.bfloat16).to(gpu) for _ in range(2))
    print(f"tile lists Hq{Hq} Hkv{Hkv} Sq{Sq} Skv{Skv} q{qbs} k{kbs} {kind}", flush=True)
    o_ref, lse_ref = oracle.dense_attention_explicit(q, k, v, m, qbs, kbs)
    want = oracle.dense_attention_backward_explicit(q, k, v, o_ref, lse_ref, do, m, qbs, kbs)
    lists = fba.lists_for(m, qbs, kbs)
    o, lse = fba.forward_with_lists(q, k, v, qbs, kbs, lists)
    grads = [fba.backward_with_lists(q, k, v, o, lse, do, qbs, kbs, lists, hand_over=ho) for ho in (False, True)]
    for got in grads:
        for name, a, b in zip(("dq", "dk", "dv"), got, want):
            mabs, rel = oracle.error_metrics(a.float(), b)
            # gradients beyond unit scale (long columns): bf16 rounding alone is 2^-9 of the value
            assert mabs <= MAX_ABS * max(1.0, float(b.abs().max())) and rel <= REL_L2, (name, mabs, rel)
    assert all(torch.equal(a, b) for a, b in zip(grads[0][1:], grads[1][1:]))
