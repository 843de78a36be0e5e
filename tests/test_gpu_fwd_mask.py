"""Forward straight from the block mask (fba_fwd_mask): work-groups of 32 rows whose eight waves share out the selected 32-key slabs.
Fewer slabs than waves, rows that are no whole work-group, 16-row halves with mask rows of their own, mask rows of one ballot
exactly, one more and several, rows that select nothing, the first block or only the last ones, key blocks of two to twelve slabs,
grouped heads, batches, shared and separate masks.  O and LSE against the oracle's explicit dense formula (fp32) with the operator's
parity bar for N(0,1) inputs, bit-equal on a repeat and to the operator where its rule takes this kernel; rows without keys exactly 0
and -inf."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

MAX_ABS, REL_L2 = 2e-2, 1e-2


def _mask(kind, shape, g):
    m = torch.rand(shape, generator=g) < 0.4
    nQ, nK = shape[-2:]
    if kind == "all":
        m[:] = True
    elif kind == "ends":  # query blocks take turns: nothing, the first block only, the last only, the last 65 or so
        m[:] = False
        m[..., 1::4, 0] = True
        m[..., 2::4, -1] = True
        m[..., 3::4, -min(nK, 65):] = True
    return m


def _run(q, k, v, qbs, kbs, m):
    from flex_block_attn_amd import _lib

    B, Hq, Sq, _ = q.shape
    o = torch.empty_like(q)
    lse = torch.empty((B, Hq, Sq, 1), dtype=torch.float32, device=q.device)
    ptr = [ctypes.c_void_p(t.data_ptr()) for t in (q, k, v, o, lse, m)]
    _lib.call("fba_fwd_mask", *ptr, 1 if m.dim() == 2 else B * Hq, B, Hq, k.shape[1], Sq, k.shape[2], 128, qbs, kbs,
              ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    return o, lse


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Skv,qbs,kbs,dims,kind", [
    (1, 1, 1, 16, 64, 16, 64, 2, "all"),           # half a work-group, two slabs
    (1, 2, 1, 48, 128, 16, 64, 4, "random"),       # a work-group and a half
    (1, 1, 1, 128, 256, 128, 128, 2, "all"),       # eight slabs: one for every wave
    (2, 3, 3, 144, 1152, 48, 192, 4, "random"),    # halves with mask rows of their own, six slabs to a block
    (1, 2, 2, 256, 4096, 64, 64, 4, "ends"),       # 64 key blocks: one ballot exactly
    (1, 2, 1, 256, 4160, 64, 64, 4, "ends"),       # 65
    (1, 2, 2, 64, 16640, 16, 64, 4, "random"),     # 260, past the rule
    (2, 2, 1, 768, 768, 384, 384, 2, "random"),    # twelve slabs to a block
    (1, 3, 1, 512, 512, 256, 128, 4, "ends"),
    (1, 10, 2, 640, 640, 32, 64, 4, "random"),     # as many heads as XCDs and more
])
def test_fwd_from_the_mask(oracle, gpu, B, Hq, Hkv, Sq, Skv, qbs, kbs, dims, kind):
    import flex_block_attn_amd as fba
    from flex_block_attn_amd import _lib

    g = torch.Generator().manual_seed(Sq + Skv + qbs)
    m = _mask(kind, ((B, Hq) if dims == 4 else ()) + (Sq // qbs, Skv // kbs), g).to(gpu)
    q = torch.randn((B, Hq, Sq, 128), generator=g).to(torch.bfloat16).to(gpu)
    k, v = (torch.randn((B, Hkv, Skv, 128), generator=g).to(torch.bfloat16).to(gpu) for _ in range(2))
    print(f"fwd mask B{B} Hq{Hq} Hkv{Hkv} Sq{Sq} Skv{Skv} q{qbs} k{kbs} {kind}", flush=True)
    (o, lse), (o2, lse2) = (_run(q, k, v, qbs, kbs, m) for _ in range(2))
    want, lse_want = oracle.dense_attention_explicit(q, k, v, m, qbs, kbs)
    mabs, rel = oracle.error_metrics(o.float(), want)
    assert mabs <= MAX_ABS and rel <= REL_L2, (mabs, rel)
    lse_want = lse_want.reshape(lse.shape).to(lse.device)
    empty = torch.isinf(lse_want)
    assert torch.equal(torch.isinf(lse), empty) and bool((o[empty[..., 0]] == 0).all())
    assert (lse - lse_want)[~empty].abs().max().item() <= 1e-3 if bool((~empty).any()) else True
    assert torch.equal(o, o2) and torch.equal(lse, lse2)
    takes = _lib.load().fba_fwd_takes_mask(B * Hq * Sq, Skv)
    assert takes == (Skv <= 1152)  # few rows: at most 120 slabs and a little more
    if takes:
        assert torch.equal(fba.flex_block_attn_func(q, k, v, qbs, kbs, m), o)


def test_scores_of_minus_infinity(gpu):
    """Keys whose scores are -inf count for nothing, also where they are all a wave or a whole row has."""
    g = torch.Generator().manual_seed(9)
    q, k, v = (torch.randn((1, 1, 256, 128), generator=g).to(torch.bfloat16).to(gpu) for _ in range(3))
    q[..., 0] = 1.0
    k[:, :, :96, 0] = float("-inf")  # three of eight slabs
    m = torch.ones((2, 2), dtype=torch.bool, device=gpu)
    m[1, 1] = False
    o, lse = _run(q, k, v, 128, 128, m)
    s = (q.float() @ k.float().transpose(-1, -2)) * 128 ** -0.5
    s[:, :, 128:, 128:] = float("-inf")
    want = torch.softmax(s, -1) @ v.float()
    assert (o.float() - want).abs().max().item() <= MAX_ABS and torch.isfinite(lse).all()
