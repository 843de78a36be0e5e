"""Backward straight from the block mask (fba_bwd_mask): work-groups of 32 keys and of 32 query rows, whose eight waves share out the
selected 32-row slabs.  Fewer slabs than waves, a length that is no whole slab, 16-row halves with mask rows of their own, columns of one
ballot (64 slabs over all heads of a group) exactly, one more and several, rows and columns that select nothing, grouped heads, batches,
shared and separate masks.  dQ, dK, dV against the oracle's closed form (fp32) with the operator's parity bar for N(0,1) inputs, bit-equal
on a repeat and to the operator where its rule takes this kernel; exactly 0 where nothing is selected."""
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
    elif kind == "ends":  # query blocks take turns: nothing, the first block only, the last only
        m[:] = False
        m[..., 1::3, 0] = True
        m[..., 2::3, -1] = True
    elif kind == "corner":  # one pair
        m[:] = False
        m[..., -1, -1] = True
    return m


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def _run(q, k, v, o, do, lse, qbs, kbs, m):
    from flex_block_attn_amd import _lib

    B, Hq, Sq, _ = q.shape
    dq, dk, dv = torch.full_like(q, 7), torch.full_like(k, 7), torch.full_like(v, 7)
    _lib.call("fba_bwd_mask", *map(_ptr, (q, k, v, o, do, lse, m)), Sq, 1 if m.dim() == 2 else B * Hq, *map(_ptr, (dq, dk, dv)), B, Hq, k.shape[1], Sq,
              k.shape[2], 128, qbs, kbs, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    return dq, dk, dv


def _forward(q, k, v, qbs, kbs, m):
    from flex_block_attn_amd import _lib

    B, Hq, Sq, _ = q.shape
    o, lse, copy = torch.empty_like(q), torch.empty((B, Hq, Sq, 1), dtype=torch.float32, device=q.device), torch.zeros_like(m)
    _lib.call("fba_fwd_mask_copy", *map(_ptr, (q, k, v, o, lse, m, copy)), Sq, 1 if m.dim() == 2 else B * Hq, B, Hq, k.shape[1], Sq, k.shape[2], 128, qbs,
              kbs, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert torch.equal(copy, m)
    return o, lse


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Skv,qbs,kbs,dims,kind", [
    (1, 1, 1, 16, 64, 16, 64, 2, "all"),           # half a slab
    (1, 2, 1, 48, 128, 16, 64, 4, "random"),       # a slab and a half, two heads to a kv head
    (2, 3, 3, 144, 1152, 48, 192, 4, "random"),    # halves with mask rows of their own
    (1, 1, 1, 32, 4160, 32, 64, 4, "ends"),        # 65 key blocks
    (1, 2, 1, 1024, 128, 16, 64, 4, "random"),     # 64 query slabs to a key tile: one ballot exactly
    (1, 2, 1, 1040, 128, 16, 64, 4, "random"),     # 66, the 33rd and the last with one half each
    (1, 8, 2, 1536, 192, 64, 64, 4, "ends"),       # 192
    (2, 2, 1, 768, 768, 384, 384, 2, "random"),    # twelve slabs to a block
    (1, 3, 1, 512, 512, 256, 128, 4, "corner"),
    (1, 10, 2, 640, 640, 32, 64, 4, "random"),     # as many heads as XCDs and more
    (1, 8, 8, 1024, 1024, 128, 128, 4, "all"),     # two rounds of work-groups
])
def test_bwd_from_the_mask(oracle, gpu, B, Hq, Hkv, Sq, Skv, qbs, kbs, dims, kind):
    import flex_block_attn_amd as fba
    from flex_block_attn_amd import _lib

    g = torch.Generator().manual_seed(Sq + Skv + qbs)
    m = _mask(kind, ((B, Hq) if dims == 4 else ()) + (Sq // qbs, Skv // kbs), g).to(gpu)
    q, do = (torch.randn((B, Hq, Sq, 128), generator=g).to(torch.bfloat16).to(gpu) for _ in range(2))
    k, v = (torch.randn((B, Hkv, Skv, 128), generator=g).to(torch.bfloat16).to(gpu) for _ in range(2))
    print(f"bwd mask B{B} Hq{Hq} Hkv{Hkv} Sq{Sq} Skv{Skv} q{qbs} k{kbs} {kind}", flush=True)
    o, lse = _forward(q, k, v, qbs, kbs, m)
    got, again = (_run(q, k, v, o, do, lse, qbs, kbs, m) for _ in range(2))
    o_want, lse_want = oracle.dense_attention_explicit(q, k, v, m, qbs, kbs)
    want = oracle.dense_attention_backward_explicit(q, k, v, o_want, lse_want, do, m, qbs, kbs)
    for name, a, b, w in zip(("dq", "dk", "dv"), got, again, want):
        mabs, rel = oracle.error_metrics(a.float(), w)
        assert mabs <= MAX_ABS and rel <= REL_L2, (name, mabs, rel)
        assert torch.equal(a, b), name
        assert bool((a[w.to(a.device) == 0] == 0).all()), name
    takes = _lib.load().fba_fwd_takes_mask(B * Hq * Sq, Skv) and _lib.load().fba_bwd_takes_mask(B, Hq, Hkv, Sq, Skv)
    assert bool(takes) == (Skv != 4160 and Sq // 32 * (Hq // Hkv) <= 160)
    if takes:
        for t in (q, k, v):
            t.requires_grad_(True)
        mask = m.clone()
        out = fba.flex_block_attn_func(q, k, v, qbs, kbs, mask)
        mask.fill_(False)  # the caller's again once the forward pass has been enqueued
        wide = torch.zeros((B, Hq, Sq, 129), dtype=torch.bfloat16, device=gpu)
        wide[..., 1:] = do
        for grad in (do, wide[..., 1:], do.float()):  # contiguous, strided, of another type
            for a, b in zip(torch.autograd.grad(out, (q, k, v), grad.to(out.dtype) if grad.dtype != out.dtype else grad, retain_graph=True), got):
                assert torch.equal(a, b)


def test_what_masked_rows_hold_is_discarded(gpu):
    """Rows of a slab that do not select a key tile count for nothing, whatever comes of their products with it: dP overflows, P is infinite because they
    select nothing at all.  What they hold themselves is finite (0 times an infinity of theirs would be NaN, as it is in the formula and on lists)."""
    g = torch.Generator().manual_seed(3)
    q, k, v, do = (torch.randn((1, 1, 64, 128), generator=g).to(torch.bfloat16).to(gpu) for _ in range(4))
    m = torch.tensor([[True], [False], [True], [True]], device=gpu)
    o, lse = _forward(q, k, v, 16, 64, m)
    want = _run(q, k, v, o, do, lse, 16, 64, m)
    assert torch.isinf(lse[0, 0, 16:32]).all()
    do[0, 0, 16:32] = 3.0e38  # dP of these rows overflows
    got = _run(q, k, v, o, do, lse, 16, 64, m)
    assert torch.equal(got[0], want[0]) and bool((got[0][0, 0, 16:32] == 0).all())
    assert torch.equal(got[1], want[1]) and torch.equal(got[2], want[2])


def test_the_rule_stays_within_one_buffer_of_the_forward_rule():
    """Sizes far beyond a round of work-groups are left to the kernels on lists."""
    from flex_block_attn_amd import _lib

    lib = _lib.load()
    assert lib.fba_bwd_takes_mask(1, 2, 2, 1536, 1536) and not lib.fba_bwd_takes_mask(1, 24, 24, 30720, 30720)
    assert not lib.fba_bwd_takes_mask(1, 2, 2, 4096, 4096) and not lib.fba_bwd_takes_mask(1, 16, 1, 512, 512)


@pytest.mark.parametrize("grad", [False, True])
def test_the_autograd_function_wants_whole_tiles(gpu, grad):
    """Lengths that are no whole tiles are padded in front of it: handed to it directly they are refused, with gradients or without."""
    import flex_block_attn_amd as fba
    from flex_block_attn_amd._lib import FbaError
    from flex_block_attn_amd.interface import FlexBlockAttnFunc

    q, k, v = (torch.randn((1, 1, n, 128), device=gpu).to(torch.bfloat16).requires_grad_(grad) for n in (48, 192, 192))
    m = torch.ones((3, 3), dtype=torch.bool, device=gpu)
    with pytest.raises(FbaError, match="multiples of 128"):
        FlexBlockAttnFunc.apply(q, k, v, 16, 64, m, True)
    assert fba.flex_block_attn_func(q, k, v, 16, 64, m).shape == q.shape
