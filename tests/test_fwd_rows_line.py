"""From how many tiles on forward on tile lists of 16-row blocks goes to the kernel with 16-row waves (128-row tiles, the other has 64): more of them where lists can be long.
The plan on the host; launches on either side of the line against the oracle's explicit dense formula (fp32), with the operator's parity bar for N(0,1) inputs."""
import ctypes

import pytest
import torch

MAX_ABS, REL_L2 = 2e-2, 1e-2


def takes_rows(heads, q_len, kv_len):
    """For 256 compute units."""
    from flex_block_attn_amd import _lib

    plan = (ctypes.c_int64 * 16)()
    _lib.call("fba_split_plan", 0, heads, 1, heads, heads, q_len, kv_len, 128, 16, 64, 65 << 20, plan)
    assert plan[0] in (heads * q_len // 128, heads * q_len // 64)
    return plan[0] == heads * q_len // 128


@pytest.mark.parametrize("kv_len,tiles", [(128, 320), (2048, 320), (3072, 328), (4096, 336), (5120, 344), (30720, 344)])
def test_the_line_rises_with_the_keys(kv_len, tiles):
    assert takes_rows(tiles, 128, kv_len) and not takes_rows(tiles - 1, 128, kv_len)


@pytest.mark.gpu
@pytest.mark.parametrize("Hq,Hkv,Sq,Skv,kind", [
    (40, 8, 1024, 2048, 0.5),       # the line itself, and 64 rows behind it with longer lists
    (40, 40, 1024, 4096, 0.5),
    (44, 11, 1024, 64 * 64, "all"),
    (44, 44, 1024, 64 * 66, "ends"),
    (352, 352, 128, 64 * 130, 0.9),
    (17, 17, 4096, 4096, "one"),
])
def test_either_side_of_the_line(oracle, gpu, Hq, Hkv, Sq, Skv, kind):
    import flex_block_attn_amd as fba

    print(f"rows line Hq{Hq} Hkv{Hkv} Sq{Sq} Skv{Skv} {kind}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(Sq + Skv)
    nQ, nK = Sq // 16, Skv // 64
    m = torch.rand((1, Hq, nQ, nK), generator=g, device=gpu) < (kind if isinstance(kind, float) else 1.0)
    if kind == "ends":  # nothing, the first block, the last, the last 65
        m[:] = False
        m[..., 1::4, 0] = True
        m[..., 2::4, -1] = True
        m[..., 3::4, -65:] = True
    elif kind == "one":
        m = torch.zeros_like(m).scatter_(-1, torch.randint(0, nK, (1, Hq, nQ, 1), generator=g, device=gpu), True)
    q = torch.randn((1, Hq, Sq, 128), generator=g, device=gpu).to(torch.bfloat16)
    k, v = (torch.randn((1, Hkv, Skv, 128), generator=g, device=gpu).to(torch.bfloat16) for _ in range(2))
    o, lse = fba.forward_with_lists(q, k, v, 16, 64, fba.lists_for(m, 16, 64))
    empty = ~m.any(-1).repeat_interleave(16, -1)
    assert bool((o[empty] == 0).all()) and bool((lse.view(1, Hq, Sq)[empty] == -float("inf")).all())
    step = max(1, 2 ** 28 // (Sq * Skv)) * (Hq // Hkv)  # heads at a time
    for h in range(0, Hq, step):
        hs, ks = slice(h, h + step), slice(h * Hkv // Hq, (h + step) * Hkv // Hq)
        o_ref, lse_ref = oracle.dense_attention_explicit(q[:, hs], k[:, ks], v[:, ks], m[:, hs], 16, 64)
        mabs, rel = oracle.error_metrics(o[:, hs].float(), o_ref)
        assert mabs <= MAX_ABS and rel <= REL_L2, (h, mabs, rel)
        some = ~empty[:, hs]
        assert float((lse.view(1, Hq, Sq)[:, hs] - lse_ref.view(1, -1, Sq))[some].abs().max()) <= 2e-3
