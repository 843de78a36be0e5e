"""dQ from handed-over dS on tile lists: waves that select nothing, one chunk, every chunk, chunks far apart; more than 64 chunks of either walk;
odd numbers of chunks; 32-row groups of 64-row, 32-row and 16-row query blocks; key blocks of several chunks; tiles behind a whole round cut into
parts; dense and numbered pairs.  Against the oracle's explicit dense formula (fp32) with the operator's parity bar for N(0,1) inputs."""
import pytest
import torch

pytestmark = pytest.mark.gpu

MAX_ABS, REL_L2 = 2e-2, 1e-2


def _mask(kind, shape, g, gpu):
    m = torch.rand(shape, generator=g, device=gpu) < (kind if isinstance(kind, float) else 1.0)
    nQ, nK = shape[-2:]
    if kind == "far":  # the first and the last key block; a single one somewhere; none; all of the second half
        m[:] = False
        m[..., 0::4, 0] = m[..., 0::4, -1] = True
        m[..., 1::4, nK // 2] = True
        m[..., 3::4, nK // 2:] = True
    return m


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Skv,qbs,kbs,kind", [
    (1, 1, 1, 128, 128, 64, 64, "all"),
    (1, 1, 1, 128, 128, 16, 128, "far"),
    (1, 2, 1, 256, 64 * 64, 64, 64, 0.5),
    (1, 2, 2, 256, 128 * 65, 64, 64, "far"),
    (1, 2, 2, 256, 128 * 65, 16, 64, "far"),
    (2, 2, 1, 384, 192 * 26, 32, 64, 0.1),
    (1, 3, 3, 768, 2688, 64, 192, 0.4),
    (1, 1, 1, 512, 16384, 64, 128, "all"),
    (1, 3, 1, 256, 16384, 16, 64, 0.3),
    (1, 20, 20, 3456, 3456, 64, 64, 0.5),    # 540 tiles: 28 behind a whole round, in parts
])
def test_dq_tiles(oracle, gpu, B, Hq, Hkv, Sq, Skv, qbs, kbs, kind):
    import flex_block_attn_amd as fba

    print(f"dq tiles B{B} Hq{Hq} Hkv{Hkv} Sq{Sq} Skv{Skv} q{qbs} k{kbs} {kind}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(Sq + Skv + qbs)
    m = _mask(kind, (B, Hq, Sq // qbs, Skv // kbs), g, gpu)
    q, do = (torch.randn((B, Hq, Sq, 128), generator=g, device=gpu).to(torch.bfloat16) for _ in range(2))
    k, v = (torch.randn((B, Hkv, Skv, 128), generator=g, device=gpu).to(torch.bfloat16) for _ in range(2))
    lists = fba.lists_for(m, qbs, kbs)
    o, lse = fba.forward_with_lists(q, k, v, qbs, kbs, lists)
    dq = fba.backward_with_lists(q, k, v, o, lse, do, qbs, kbs, lists, hand_over=True)[0]
    assert torch.equal(dq, fba.backward_with_lists(q, k, v, o, lse, do, qbs, kbs, lists, hand_over=True)[0])
    ins = [t.clone().requires_grad_(True) for t in (q, k, v)]
    through = torch.autograd.grad(fba.flex_block_attn_func(*ins, qbs, kbs, m), ins, do)[0]
    for b in range(B):
        for kv in range(Hkv):
            hs = slice(kv * Hq // Hkv, (kv + 1) * Hq // Hkv)
            one = [t[b:b + 1] for t in (q[:, hs], k[:, kv:kv + 1], v[:, kv:kv + 1], do[:, hs], m[:, hs])]
            o_ref, lse_ref = oracle.dense_attention_explicit(*one[:3], one[4], qbs, kbs)
            want = oracle.dense_attention_backward_explicit(*one[:3], o_ref, lse_ref, one[3], one[4], qbs, kbs)[0]
            for got in (dq, through):
                mabs, rel = oracle.error_metrics(got[b:b + 1, hs].float(), want)
                assert mabs <= MAX_ABS * max(1.0, float(want.abs().max())) and rel <= REL_L2, (b, kv, mabs, rel)
