"""Calls without gradients on whole 128-row blocks read the block mask where lists had at most 256 key blocks: rows of one block to 256, whole words of 64 and around, fewer
than 16; the first and the last block, none, all; parts, and as many as by the lists; a shared mask, grouped heads; mask bytes other than one; 257 blocks, which go through
lists.  Against forward on lists, bit for bit: rows of equal length, so that both decide alike on the parts; in
small launches, which take 64-row work-groups, to what bf16 roundings come to.  And the
lists that a step has it make in the same launch."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _masks(kind, shape, g, gpu):
    nQ, nK = shape[-2:]
    if kind == "all":
        return torch.ones(shape, dtype=torch.bool, device=gpu)
    if kind == "none":
        return torch.zeros(shape, dtype=torch.bool, device=gpu)
    keep = 1 if kind == "one" else max(1, round(kind * nK))
    score = torch.rand(shape, generator=g, device=gpu)
    if kind == "one":  # the first, the last, one in between
        score[..., 0::3, 0] = score[..., 1::3, -1] = 2.0
    return torch.zeros(shape, dtype=torch.bool, device=gpu).scatter_(-1, score.topk(keep, -1).indices, True)


def halves(rows, kv_len):
    """Does forward on a mask take 64-row work-groups?"""
    return rows <= 128 * 128 and kv_len // 32 <= (148 if rows >= 96 * 128 else 112)


@pytest.mark.parametrize("B,Hq,Hkv,Sq,nK,qbs,kbs,dims", [
    (1, 65, 65, 128, 28, 128, 128, 4),    # 65 to 128 tiles: 64-row work-groups
    (1, 6, 3, 1408, 11, 128, 128, 4),
    (1, 3, 3, 4224, 11, 384, 384, 4),
    (2, 8, 4, 1024, 1, 512, 512, 4),
    (1, 4, 4, 3072, 37, 128, 128, 2),
    (1, 2, 2, 8192, 8, 8192, 512, 4),
    (1, 1, 1, 16384, 36, 128, 128, 4),
    (1, 43, 43, 384, 3, 384, 1536, 4),    # 129
    (1, 70, 70, 128, 1, 128, 128, 4),
    (1, 70, 70, 128, 15, 128, 128, 4),
    (1, 9, 3, 1024, 16, 128, 128, 4),
    (1, 9, 3, 1024, 17, 128, 128, 4),
    (2, 10, 5, 512, 63, 256, 128, 4),
    (1, 24, 6, 768, 64, 128, 128, 4),
    (1, 24, 24, 1280, 65, 128, 128, 2),
    (1, 3, 3, 4992, 30, 384, 384, 4),
    (1, 4, 4, 2304, 129, 128, 128, 4),
    (1, 8, 8, 1152, 192, 384, 128, 4),
    (1, 66, 66, 1024, 24, 128, 128, 4),   # behind a whole round
    (1, 4, 2, 2304, 255, 128, 128, 2),
    (1, 2, 2, 4608, 256, 128, 128, 4),
    (1, 2, 2, 4608, 257, 128, 128, 4),
])
@pytest.mark.parametrize("kind", [0.4, "one", "none", "all"])
def test_as_on_lists(gpu, B, Hq, Hkv, Sq, nK, qbs, kbs, dims, kind):
    import flex_block_attn_amd as fba
    from flex_block_attn_amd import _lib

    print(f"blocks B{B} Hq{Hq} Hkv{Hkv} Sq{Sq} {nK} x {kbs} q{qbs} {kind}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(Sq + nK)
    m = _masks(kind, ((B, Hq) if dims == 4 else ()) + (Sq // qbs, nK), g, gpu)
    q = torch.randn((B, Hq, Sq, 128), generator=g, device=gpu).to(torch.bfloat16)
    k, v = (torch.randn((B, Hkv, nK * kbs, 128), generator=g, device=gpu).to(torch.bfloat16) for _ in range(2))
    assert not _lib.load().fba_fwd_takes_mask(B * Hq * Sq, nK * kbs)
    want = fba.forward_with_lists(q, k, v, qbs, kbs, fba.lists_for(m, qbs, kbs))[0]
    got = fba.flex_block_attn_func(q, k, v, qbs, kbs, m)
    if halves(B * Hq * Sq, nK * kbs):
        # another kernel: either result is within 2.4e-3 (2-norm) of the exact one (P and O in bf16), and a block that is missed changes 64 rows by far more
        a, b = (t.float().reshape(-1, 64 * 128) for t in (got, want))
        assert bool(((a - b).norm(dim=1) <= 5e-3 * b.norm(dim=1)).all())
    else:
        assert torch.equal(got, want)
    if kind == "none":
        assert not bool(got.any())


@pytest.mark.parametrize("B,Hq,Hkv,Sq,nK,qbs,kbs,dims", [
    (1, 66, 66, 128, 1, 128, 128, 4),     # a row and a column of one block
    (1, 12, 4, 1536, 37, 128, 128, 4),
    (2, 3, 3, 4608, 12, 384, 384, 4),
    (1, 8, 8, 8192, 192, 128, 128, 2),    # 256 rows, one mask for all heads
    (1, 4, 4, 8192, 192, 128, 128, 4),    # 1024
    (1, 16, 16, 8192, 1, 8192, 8192, 4),
])
def test_lists_on_the_way(gpu, B, Hq, Hkv, Sq, nK, qbs, kbs, dims):
    """Forward and the lists of one launch: those of fba_mask_compact, padding and all; a step through the operator has the gradients of the lists."""
    import flex_block_attn_amd as fba
    from flex_block_attn_amd import _lib
    from flex_block_attn_amd.interface import _ptr, _stream

    g = torch.Generator(device=gpu).manual_seed(Sq + nK)
    m = torch.rand(((B, Hq) if dims == 4 else ()) + (Sq // qbs, nK), generator=g, device=gpu) < 0.4
    q, do = (torch.randn((B, Hq, Sq, 128), generator=g, device=gpu).to(torch.bfloat16) for _ in range(2))
    k, v = (torch.randn((B, Hkv, nK * kbs, 128), generator=g, device=gpu).to(torch.bfloat16) for _ in range(2))
    want = fba.lists_for(m, qbs, kbs)
    made = [torch.full_like(t, 77) for t in (want.q_cnt, want.q_idx, want.k_cnt, want.k_idx)]
    o, lse = torch.empty_like(q), torch.empty((B, Hq, Sq, 1), device=gpu)
    ws = torch.empty(_lib.load().fba_split_workspace_bytes(), dtype=torch.uint8, device=gpu)
    tail = (want.mask_bh, B, Hq, Hkv, Sq, nK * kbs, 128, qbs, kbs, _ptr(ws), ws.numel(), _stream())
    _lib.call("fba_fwd_blocks", *map(_ptr, (q, k, v, o, lse, m, *made)), *tail)
    for a, b in zip(made, (want.q_cnt, want.q_idx, want.k_cnt, want.k_idx)):
        assert torch.equal(a, b)
    none = o.clone(), lse.clone()
    _lib.call("fba_fwd_blocks", *map(_ptr, (q, k, v, o, lse, m)), None, None, None, None, *tail)
    assert torch.equal(o, none[0]) and torch.equal(lse, none[1])
    with pytest.raises(_lib.FbaError, match="all four"):
        _lib.call("fba_fwd_blocks", *map(_ptr, (q, k, v, o, lse, m, *made[:2])), None, None, *tail)
    ins = [t.clone().requires_grad_(True) for t in (q, k, v)]
    out = fba.flex_block_attn_func(*ins, qbs, kbs, m)
    grads = torch.autograd.grad(out, ins, do)
    if not _lib.load().fba_fwd_takes_mask(B * Hq * Sq, nK * kbs):
        assert torch.equal(out, o)  # the operator makes this very call
    for name, a, b in zip(("dq", "dk", "dv"), grads, fba.backward_with_lists(q, k, v, o, lse, do, qbs, kbs, want)):
        assert float((a.float() - b.float()).norm()) <= 1e-2 * float(b.float().norm()), name  # bf16 sums of another order, where the operator takes other kernels


def test_mask_bytes_and_limits(gpu):
    """Any byte but zero selects; more key blocks than the kernel keeps, and blocks that are no whole tiles, are refused."""
    import flex_block_attn_amd as fba
    from flex_block_attn_amd import _lib
    from flex_block_attn_amd.interface import _ptr, _stream

    g = torch.Generator(device=gpu).manual_seed(5)
    B, H, Sq, nK = 1, 12, 1536, 37
    q = torch.randn((B, H, Sq, 128), generator=g, device=gpu).to(torch.bfloat16)
    k, v = (torch.randn((B, H, nK * 128, 128), generator=g, device=gpu).to(torch.bfloat16) for _ in range(2))
    m = torch.zeros((B, H, Sq // 128, nK), dtype=torch.uint8, device=gpu)
    at = torch.rand(m.shape, generator=g, device=gpu).topk(20, -1).indices
    m.scatter_(-1, at, torch.randint(1, 256, at.shape, generator=g, device=gpu).to(torch.uint8))
    want, want_lse = fba.forward_with_lists(q, k, v, 128, 128, fba.lists_for(m != 0, 128, 128))
    o, lse = torch.empty_like(q), torch.empty((B, H, Sq, 1), device=gpu)
    ws = torch.empty(_lib.load().fba_split_workspace_bytes(), dtype=torch.uint8, device=gpu)
    args = (*map(_ptr, (q, k, v, o, lse, m)), None, None, None, None, B * H, B, H, H, Sq, nK * 128, 128)
    _lib.call("fba_fwd_blocks", *args, 128, 128, _ptr(ws), ws.numel(), _stream())
    assert not halves(B * H * Sq, nK * 128) and torch.equal(o, want) and torch.equal(lse.flatten(), want_lse.flatten())
    with pytest.raises(_lib.FbaError):
        _lib.call("fba_fwd_blocks", *args, 64, 64, _ptr(ws), ws.numel(), _stream())
    with pytest.raises(_lib.FbaError, match="257 key blocks"):
        _lib.call("fba_fwd_blocks", *args[:-2], 257 * 128, 128, 128, 128, _ptr(ws), ws.numel(), _stream())
    lists = [torch.empty(1, dtype=torch.int32, device=gpu) for _ in range(4)]  # (refused before anything is written)
    with pytest.raises(_lib.FbaError, match="1024 rows"):
        _lib.call("fba_fwd_blocks", *map(_ptr, (q, k, v, o, lse, m, *lists)), 22 * B * H, 22 * B, H, H, Sq, nK * 128, 128, 128, 128, _ptr(ws), ws.numel(), _stream())


@pytest.mark.parametrize("step", [False, True])
def test_with_384_row_work_groups_asked_for(gpu, monkeypatch, step):
    """FBA_FWD_TILE_ROWS=384 is for 384-row work-groups, which read lists: the same bits as on lists, in a launch that would take 64-row work-groups (others)."""
    import flex_block_attn_amd as fba

    g = torch.Generator(device=gpu).manual_seed(384)
    q, k, v = (torch.randn((1, 6, 1536, 128), generator=g, device=gpu).to(torch.bfloat16) for _ in range(3))
    m = _masks(0.6, (1, 6, 4, 4), g, gpu)
    assert halves(6 * 1536, 1536)
    monkeypatch.setenv("FBA_FWD_TILE_ROWS", "384")
    want, _ = fba.forward_with_lists(q, k, v, 384, 384, fba.lists_for(m, 384, 384))
    got = fba.flex_block_attn_func(q.requires_grad_(step), k, v, 384, 384, m)
    assert torch.equal(got, want)
