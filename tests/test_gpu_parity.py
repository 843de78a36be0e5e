"""GPU parity: the HIP path, called through the C ABI, against the CPU oracle on the same seeded inputs.

Tolerances (stated by the task for floating point): every one of O, dQ, dK, dV within max-abs 2e-2 and relative
L2 1e-2 of the fp32 oracle, which sees exactly the bf16 values the kernels see.  Mask compaction is integer work and
must be bit-exact.  Full-size cases, where the oracle would take minutes, are checked through properties that hold at
any size.
"""
import os

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

MAX_ABS = 2e-2
REL_L2 = 1e-2
GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")


def _check(oracle, got, want, name, res, peaky=False):
    """max-abs 2e-2 and rel-L2 1e-2, flat, for N(0,1) inputs.  Only for the reference test's N(0.1, 10) row magnitudes
    (`peaky`), whose outputs exceed unit scale, is the absolute bound scaled by max|ref|: rounding such a result to bf16
    alone is an error of 2^-9 relative."""
    mabs, rel = oracle.error_metrics(got.float(), want)
    res[name] = (mabs, rel)
    bound = MAX_ABS * max(1.0, float(want.abs().max())) if peaky else MAX_ABS
    assert mabs <= bound, f"{name}: max-abs {mabs} > {bound}"
    assert rel <= REL_L2, f"{name}: rel-L2 {rel} > {REL_L2}"


def _reference_allclose(got, want):
    """The reference's own forward assertion, torch.allclose(o, sdpa, rtol=1e-2, atol=5e-3)
    (test/test_flex_block_attn.py:139), against the fp32 oracle instead of a bf16 SDPA."""
    g, w = got.float().cpu(), want.float()
    excess = ((g - w).abs() - (5e-3 + 1e-2 * w.abs())).max().item()
    assert torch.allclose(g, w, rtol=1e-2, atol=5e-3), f"o fails allclose(rtol=1e-2, atol=5e-3) by {excess}"


def _run_case(oracle, gpu, B, Hq, Hkv, Sq, Skv, qbs, kbs, mask, seed=0, peaky=False, ref_allclose=False):
    import flex_block_attn_amd as fba
    from flex_block_attn_amd import _lib

    q, k, v, do = oracle.seeded_qkv(B, Hq, Hkv, Sq, Skv, seed=seed, peaky=peaky)
    qb, kb, vb, dob = (t.to(torch.bfloat16) for t in (q, k, v, do))
    o_ref, lse_ref = oracle.c_attention_forward(qb, kb, vb, mask, qbs, kbs)
    dq_ref, dk_ref, dv_ref = oracle.c_attention_backward(qb, kb, vb, o_ref, lse_ref, dob, mask, qbs, kbs)
    qg, kg, vg = (t.to(gpu).requires_grad_(True) for t in (qb, kb, vb))
    print(f"case B{B} Hq{Hq} Hkv{Hkv} Sq{Sq} Skv{Skv} q{qbs} k{kbs} seed{seed} peaky{peaky}", flush=True)
    o = fba.flex_block_attn_func(qg, kg, vg, qbs, kbs, mask.to(gpu))
    o.backward(dob.to(gpu))
    torch.cuda.synchronize()
    res = {}
    _check(oracle, o, o_ref, "o", res, peaky)
    if ref_allclose:
        _reference_allclose(o, o_ref)
    if Sq % 128 == 0 and Skv % 128 == 0 and _lib.load().fba_fwd_takes_mask(B * Hq * Sq, Skv):
        # the operator has read the mask itself: the same inputs through the kernels on lists
        with torch.no_grad():
            o_lists, lse = fba.forward_with_lists(qg, kg, vg, qbs, kbs, fba.lists_for(mask.to(gpu), qbs, kbs))
        _check(oracle, o_lists, o_ref, "o on lists", res, peaky)
        if ref_allclose:
            _reference_allclose(o_lists, o_ref)
        lse, want = lse.flatten().cpu(), lse_ref.flatten().float()
        assert torch.equal(torch.isinf(lse), torch.isinf(want))
        # the denominator sums P rounded to bf16 (2^-8 of it at most), the scores are fp32 sums of 128 products
        fin = ~torch.isinf(want)
        assert ((lse - want)[fin].abs() <= 2.0 ** -8 + 128 * 2.0 ** -24 * want[fin].abs()).all()
    _check(oracle, qg.grad, dq_ref, "dq", res, peaky)
    _check(oracle, kg.grad, dk_ref, "dk", res, peaky)
    _check(oracle, vg.grad, dv_ref, "dv", res, peaky)
    print("   ", {n: (f"{a:.2e}", f"{r:.2e}") for n, (a, r) in res.items()}, flush=True)
    return o, qg.grad, kg.grad, vg.grad


def test_mask_compaction_bit_exact(oracle, gpu):
    import flex_block_attn_amd as fba
    from flex_block_attn_amd import masks

    cases = [
        masks.bernoulli_block_mask(4, 4, 0.5, 0),
        masks.bernoulli_block_mask(80, 80, 0.4, 1),
        masks.bernoulli_block_mask(540, 180, 0.1, 2),
        masks.bernoulli_block_mask(1, 1, 1.0, 3),
        masks.bernoulli_block_mask(65, 129, 0.5, 4),
        torch.zeros((7, 9), dtype=torch.bool),
        torch.ones((30, 30), dtype=torch.bool),
        masks.random_block_mask(1, 24, 80, 80, 32, 5),
        masks.random_block_mask(2, 3, 17, 70, 5, 6),
        masks.sta_3d_block_mask((5, 6, 10), (3, 3, 3)),
    ]
    for m in cases:
        lists = fba.compact_block_mask(m.to(gpu))
        ref = oracle.compact_lists(m)
        ref_c = oracle.c_compact_lists(m)
        for got, want, want_c, name in zip((lists.q_cnt, lists.q_idx, lists.k_cnt, lists.k_idx), ref, ref_c, ("q_cnt", "q_idx", "k_cnt", "k_idx")):
            assert (want == want_c).all()
            assert got.dtype == torch.int32
            assert (got.cpu().numpy() == want).all(), f"{name} differs for mask {tuple(m.shape)}"


def test_mask_compaction_full_size_against_nonzero(gpu):
    """Largest configured masks: per-(b,h) 80x80 random and 24 x 540x180; lists against torch.nonzero on the device."""
    import flex_block_attn_amd as fba
    from flex_block_attn_amd import masks

    for m in (masks.random_block_mask(1, 24, 80, 80, 32, 0), torch.rand((1, 24, 540, 180), generator=torch.Generator().manual_seed(1)) < 0.1):
        mg = m.to(gpu)
        lists = fba.compact_block_mask(mg)
        M, nQ, nK = lists.mask_bh, lists.nQ, lists.nK
        m3 = mg.reshape(M, nQ, nK)
        assert torch.equal(lists.q_cnt, m3.sum(-1).to(torch.int32)) and torch.equal(lists.k_cnt, m3.sum(-2).to(torch.int32))
        nz = torch.nonzero(m3)  # ascending (b, i, j)
        valid = torch.arange(nK, device=gpu)[None, None, :] < lists.q_cnt[..., None]
        assert torch.equal(lists.q_idx[valid].long(), nz[:, 2]) and (lists.q_idx[~valid] == -1).all()
        nzt = torch.nonzero(m3.transpose(1, 2))  # ascending (b, j, i)
        validk = torch.arange(nQ, device=gpu)[None, None, :] < lists.k_cnt[..., None]
        assert torch.equal(lists.k_idx[validk].long(), nzt[:, 2]) and (lists.k_idx[~validk] == -1).all()


def test_config1_cpu_reference_shape(oracle, gpu):
    """B=1, H=2, S=1536, block 384 (4x4 Bernoulli(0.5) mask with the diagonal forced on)."""
    from flex_block_attn_amd import masks

    _run_case(oracle, gpu, 1, 2, 2, 1536, 1536, 384, 384, masks.bernoulli_block_mask(4, 4, 0.5, 0))


def test_golden_fixtures(oracle, gpu):
    import flex_block_attn_amd as fba

    for name in sorted(f for f in os.listdir(GOLDEN) if f.endswith(".npz")):
        z = np.load(os.path.join(GOLDEN, name))
        q, k, v, do = (torch.from_numpy(z[n]).view(torch.bfloat16).to(gpu) for n in ("q", "k", "v", "do"))
        m = torch.from_numpy(z["mask"]).to(gpu)
        qbs, kbs = int(z["q_block"]), int(z["kv_block"])
        print("golden", name, flush=True)
        q.requires_grad_(True), k.requires_grad_(True), v.requires_grad_(True)
        o = fba.flex_block_attn_func(q, k, v, qbs, kbs, m)
        o.backward(do)
        res = {}
        for n, got in (("o", o), ("dq", q.grad), ("dk", k.grad), ("dv", v.grad)):
            _check(oracle, got, torch.from_numpy(z[n]), n, res, peaky=name.startswith("peaky"))
        lists = fba.compact_block_mask(m)
        for n, got in (("q_cnt", lists.q_cnt), ("q_idx", lists.q_idx), ("k_cnt", lists.k_cnt), ("k_idx", lists.k_idx)):
            assert np.array_equal(got.cpu().numpy(), z[n]), (name, n)


def _reference_test_mask(nQ, nK):
    """Block pattern of the reference's own test: |j - i| < 2 or j == 4 (test/test_flex_block_attn.py:8-46), with the
    query block index mapped onto the key block grid; every query block keeps at least one key block."""
    i = (torch.arange(nQ)[:, None] * nK) // nQ
    j = torch.arange(nK)[None, :]
    return ((j - i).abs() < 2) | (j == 4)


@pytest.mark.parametrize("seq,heads", [(768, 1), (1536, 2), (3072, 4)])
@pytest.mark.parametrize("qbs,kbs", [(128, 128), (128, 256), (128, 384), (384, 384), (256, 128)])
def test_reference_grid(oracle, gpu, seq, heads, qbs, kbs):
    """Shape grid, input distribution (random direction x N(0.1, 10) magnitude) and mask pattern of
    test/test_flex_block_attn.py:58-85, for the block sizes this build covers, with the mask stacked to [B, H, nQ, nK]."""
    if seq % qbs or seq % kbs:
        pytest.skip("sequence not divisible")
    nQ, nK = seq // qbs, seq // kbs
    m = _reference_test_mask(nQ, nK)[None, None].expand(1, heads, nQ, nK).contiguous()
    _run_case(oracle, gpu, 1, heads, heads, seq, seq, qbs, kbs, m, seed=seq + heads, peaky=True, ref_allclose=True)


def _reference_raw_mask(nQ, nK):
    """The reference test's pattern on raw block indices, |j - i| < 2 or j == 4 (test/test_flex_block_attn.py:16-38):
    with query blocks smaller than key blocks most query blocks beyond the diagonal keep only key block 4, or nothing."""
    i = torch.arange(nQ)[:, None]
    j = torch.arange(nK)[None, :]
    return ((j - i).abs() < 2) | (j == 4)


TILE_LIST_CASES = [
    (16, 64, 24, 6, 0.5), (32, 64, 12, 6, 0.3), (64, 64, 6, 6, 0.5), (64, 128, 8, 4, 0.5), (16, 384, 48, 2, 0.2),
    (48, 192, 8, 2, 0.5), (128, 64, 3, 6, 0.5), (384, 192, 2, 4, 0.6), (256, 64, 1, 4, 0.5), (64, 256, 8, 2, 1.0),
    (32, 128, 16, 4, 0.0),
]


def test_tile_lists_bit_exact(oracle, gpu):
    """fba_tile_lists against the brute-force lists derived from allowed(i, j) alone."""
    import flex_block_attn_amd as fba
    from flex_block_attn_amd import masks

    for n, (qbs, kbs, nQ, nK, p) in enumerate(TILE_LIST_CASES):
        for m in (masks.bernoulli_block_mask(nQ, nK, p, 40 + n), (torch.rand((2, 3, nQ, nK), generator=torch.Generator().manual_seed(n)) < p)):
            got = fba.tile_block_mask(m.to(gpu), qbs, kbs)
            assert got.tiled
            want = oracle.tile_lists(m, qbs, kbs)
            for g, w, name in zip((got.q_cnt, got.q_idx, got.k_cnt, got.k_idx), want, ("qt_cnt", "qt_ent", "kt_cnt", "kt_ent")):
                assert g.dtype == torch.int32 and tuple(g.shape) == w.shape, (name, g.shape, w.shape)
                assert (g.cpu().numpy() == w).all(), f"{name} differs for q{qbs} k{kbs} mask {tuple(m.shape)}"


@pytest.mark.parametrize("seq,heads", [(768, 1), (1536, 2), (3072, 4)])
@pytest.mark.parametrize("kbs", [64, 128, 256, 384])
@pytest.mark.parametrize("qbs", [16, 32, 64])
def test_reference_grid_small_query_blocks(oracle, gpu, seq, heads, qbs, kbs):
    """The block sizes of the reference's own test grid (q_block 16/32/64 x kv_block 64/128/256/384,
    test/test_flex_block_attn.py:70-71), its input distribution and its raw mask pattern."""
    if seq % kbs:
        pytest.skip("sequence not divisible")
    nQ, nK = seq // qbs, seq // kbs
    m = _reference_raw_mask(nQ, nK)[None, None].expand(1, heads, nQ, nK).contiguous()
    _run_case(oracle, gpu, 1, heads, heads, seq, seq, qbs, kbs, m, seed=seq + qbs + kbs, peaky=True, ref_allclose=True)


@pytest.mark.parametrize("qbs,kbs,Sq,Skv", [(128, 64, 512, 384), (384, 192, 768, 768), (64, 192, 256, 384), (48, 192, 384, 384),
                                            (16, 64, 128, 128), (256, 64, 512, 256), (80, 320, 640, 640)])
def test_block_sizes_off_the_tile_grid(oracle, gpu, qbs, kbs, Sq, Skv):
    """Random masks per head, GQA, block edges that fall inside the kernels' 128-row tiles and 32-row slabs."""
    from flex_block_attn_amd import masks

    nQ, nK = Sq // qbs, Skv // kbs
    m = torch.rand((2, 4, nQ, nK), generator=torch.Generator().manual_seed(qbs + kbs)) < 0.5
    m[..., 0, :] = False  # a query block with nothing selected
    m[..., :, nK - 1] = False  # a key block nobody selects
    m[..., nQ - 1, 0] = True
    _run_case(oracle, gpu, 2, 4, 2, Sq, Skv, qbs, kbs, m, seed=qbs * 7 + kbs)


def test_small_block_private_entry_points(oracle, gpu):
    """use_small_block_mode: the fine mask is the one that counts, the pooled one is ignored
    (flex_block_attn_interface.py:38-66, :85-86 for the transposed masks of backward)."""
    import flex_block_attn_amd as fba

    B, H, S, qbs, kbs = 1, 2, 512, 32, 128
    q, k, v, do = oracle.seeded_qkv(B, H, H, S, S, seed=66)
    qb, kb, vb, dob = (t.to(torch.bfloat16) for t in (q, k, v, do))
    fine = torch.rand((S // qbs, S // kbs), generator=torch.Generator().manual_seed(5)) < 0.5
    fine[:, 0] = True
    pooled = fine.reshape(S // kbs, kbs // qbs, S // kbs).any(1)
    o_ref, lse_ref = oracle.c_attention_forward(qb, kb, vb, fine, qbs, kbs)
    g_ref = oracle.c_attention_backward(qb, kb, vb, o_ref, lse_ref, dob, fine, qbs, kbs)
    qg, kg, vg, dog = (t.to(gpu) for t in (qb, kb, vb, dob))
    o, lse = fba._flex_block_attn_forward(qg, kg, vg, qbs, kbs, pooled.to(gpu), fine.to(gpu), True)
    res = {}
    _check(oracle, o, o_ref, "o", res)
    assert oracle.error_metrics(lse.reshape(B, H, S), lse_ref)[0] < 5e-3
    grads = fba._flex_block_attn_backward(qg, kg, vg, o, lse, dog, qbs, kbs, pooled.t().contiguous().to(gpu),
                                          fine.t().contiguous().to(gpu), True)
    for n, got, want in zip(("dq", "dk", "dv"), grads, g_ref):
        _check(oracle, got, want, n, res)


def _random_configs(n, seed):
    """Seeded draw of legal operator configurations: block sizes from the reference's rule (q % 16, kv % 64, one dividing
    the other), GQA groups, cross lengths, 2-D or per-(b,h) masks of varying density, some with empty rows or columns."""
    import random

    rng = random.Random(seed)
    q_sizes = [16, 32, 48, 64, 96, 128, 192, 256, 384]
    k_sizes = [64, 128, 192, 256, 384]
    out = []
    while len(out) < n:
        qbs, kbs = rng.choice(q_sizes), rng.choice(k_sizes)
        if qbs % kbs and kbs % qbs:
            continue
        nQ, nK = rng.randint(1, max(1, 768 // qbs)), rng.randint(1, max(1, 768 // kbs))
        B, Hkv = rng.choice([1, 2]), rng.choice([1, 2])
        Hq = Hkv * rng.choice([1, 2, 3])
        out.append((B, Hq, Hkv, nQ * qbs, nK * kbs, qbs, kbs, rng.choice([2, 4]), rng.choice([0.15, 0.5, 0.9, 1.0]), rng.randrange(1 << 30)))
    return out


@pytest.mark.parametrize("cfg", _random_configs(24, seed=2024), ids=lambda c: "B%d_Hq%d_Hkv%d_Sq%d_Skv%d_q%d_k%d_m%d_p%s_%d" % c)
def test_seeded_random_configurations(oracle, gpu, cfg):
    B, Hq, Hkv, Sq, Skv, qbs, kbs, mdim, density, seed = cfg
    g = torch.Generator().manual_seed(seed)
    shape = (Sq // qbs, Skv // kbs) if mdim == 2 else (B, Hq, Sq // qbs, Skv // kbs)
    m = torch.rand(shape, generator=g) < density
    _run_case(oracle, gpu, B, Hq, Hkv, Sq, Skv, qbs, kbs, m, seed=seed % 1000)


def test_rising_scores_exercise_the_lazy_rescale(oracle, gpu):
    """Keys whose magnitude grows along the sequence: the running softmax reference has to be raised again and again,
    also in the middle of a key block, which N(0,1) inputs never cause."""
    import flex_block_attn_amd as fba

    B, H, S, bs = 1, 2, 1536, 384
    q, k, v, do = oracle.seeded_qkv(B, H, H, S, S, seed=31)
    ramp = torch.linspace(0.5, 40.0, S)[None, None, :, None]
    k = k * ramp * torch.sign(torch.sin(torch.arange(S) * 0.37))[None, None, :, None]
    q = q * 3.0
    qb, kb, vb, dob = (t.to(torch.bfloat16) for t in (q, k, v, do))
    m = torch.ones((4, 4), dtype=torch.bool)
    o_ref, lse_ref = oracle.c_attention_forward(qb, kb, vb, m, bs, bs)
    g_ref = oracle.c_attention_backward(qb, kb, vb, o_ref, lse_ref, dob, m, bs, bs)
    qg, kg, vg = (t.to(gpu).requires_grad_(True) for t in (qb, kb, vb))
    o = fba.flex_block_attn_func(qg, kg, vg, bs, bs, m.to(gpu))
    o.backward(dob.to(gpu))
    res = {}
    _check(oracle, o, o_ref, "o", res)
    # gradients are far above unit scale here (keys up to 40x): the absolute bound applies after dividing by max|ref|
    for n, got, want in zip(("dq", "dk", "dv"), (qg.grad, kg.grad, vg.grad), g_ref):
        _check(oracle, got, want, n, res, peaky=True)
    print("   rising:", res, flush=True)


def test_gqa_and_cross_attention(oracle, gpu):
    from flex_block_attn_amd import masks

    _run_case(oracle, gpu, 2, 4, 2, 256, 512, 128, 128, masks.random_block_mask(2, 4, 2, 4, 2, 21), seed=3)
    _run_case(oracle, gpu, 1, 6, 1, 384, 768, 128, 384, masks.bernoulli_block_mask(3, 2, 0.5, 22), seed=4)


def test_empty_query_block_and_unselected_key_block(oracle, gpu):
    m = torch.tensor([[True, False, True], [False, False, False], [True, False, True]])
    o, dq, dk, dv = _run_case(oracle, gpu, 1, 2, 2, 384, 384, 128, 128, m, seed=5)
    assert o[:, :, 128:256].abs().max().item() == 0.0 and dq[:, :, 128:256].abs().max().item() == 0.0
    assert dk[:, :, 128:256].abs().max().item() == 0.0 and dv[:, :, 128:256].abs().max().item() == 0.0


def test_lse_and_private_entry_points(oracle, gpu):
    """_flex_block_attn_forward / _flex_block_attn_backward: argument order of the reference, transposed masks in
    backward (flex_block_attn_interface.py:6-12, :85-86)."""
    import flex_block_attn_amd as fba
    from flex_block_attn_amd import masks

    B, H, S, bs = 1, 2, 512, 128
    q, k, v, do = oracle.seeded_qkv(B, H, H, S, S, seed=6)
    qb, kb, vb, dob = (t.to(torch.bfloat16) for t in (q, k, v, do))
    m = masks.bernoulli_block_mask(4, 4, 0.5, 7)
    o_ref, lse_ref = oracle.c_attention_forward(qb, kb, vb, m, bs, bs)
    g_ref = oracle.c_attention_backward(qb, kb, vb, o_ref, lse_ref, dob, m, bs, bs)
    mg = m.to(gpu)
    o, lse = fba._flex_block_attn_forward(qb.to(gpu), kb.to(gpu), vb.to(gpu), bs, bs, mg, mg, False)
    assert lse.shape == (B, H, S, 1) and lse.dtype == torch.float32
    assert oracle.error_metrics(lse.reshape(B, H, S), lse_ref)[0] < 5e-3
    mt = mg.t().contiguous()
    grads = fba._flex_block_attn_backward(qb.to(gpu), kb.to(gpu), vb.to(gpu), o, lse, dob.to(gpu), bs, bs, mt, mt, False)
    res = {}
    for n, got, want in zip(("dq", "dk", "dv"), grads, g_ref):
        assert got.dtype == torch.bfloat16
        _check(oracle, got, want, n, res)


@pytest.mark.parametrize("qbs,kbs,Sq,Skv", [(64, 64, 192, 192), (16, 64, 80, 320), (48, 192, 144, 576), (128, 64, 384, 192), (32, 128, 96, 128)])
def test_sequences_that_are_not_whole_tiles(oracle, gpu, qbs, kbs, Sq, Skv):
    """Sequence lengths that are not multiples of 128 (possible with block sizes that are not): the operator pads them
    with rows no block selects; results and gradients equal the oracle's on the unpadded problem."""
    nQ, nK = Sq // qbs, Skv // kbs
    m = torch.rand((1, 2, nQ, nK), generator=torch.Generator().manual_seed(Sq + Skv)) < 0.6
    m[..., 0] = True
    _run_case(oracle, gpu, 1, 2, 2, Sq, Skv, qbs, kbs, m, seed=Sq + 3 * Skv)


def test_unsupported_shapes_fail_loudly(gpu):
    """The C ABI computes whole 128-row tiles only: asked for anything else it reports so (the Python operator pads
    before it calls); nothing falls back silently."""
    import flex_block_attn_amd as fba
    from flex_block_attn_amd import _lib

    q = torch.zeros((1, 1, 192, 128), dtype=torch.bfloat16, device=gpu)
    m = torch.ones((3, 3), dtype=torch.bool, device=gpu)
    with pytest.raises(_lib.FbaError) as ei:
        fba._flex_block_attn_forward(q, q, q, 64, 64, m, m, False)
    assert ei.value.code == _lib.FBA_ERR_UNSUPPORTED


def test_deterministic(gpu):
    import flex_block_attn_amd as fba
    from flex_block_attn_amd import masks

    g = torch.Generator(device="cpu").manual_seed(9)
    q, k, v, do = (torch.randn((1, 3, 1536, 128), generator=g).to(torch.bfloat16).to(gpu) for _ in range(4))
    # block lists, then tile lists (64-row blocks): forward and the dS hand-over of backward write every element once
    for bs, m in ((384, masks.random_block_mask(1, 3, 4, 4, 2, 10)), (64, masks.random_block_mask(1, 3, 24, 24, 9, 11))):
        outs = []
        for _ in range(2):
            qq, kk, vv = (t.clone().requires_grad_(True) for t in (q, k, v))
            o = fba.flex_block_attn_func(qq, kk, vv, bs, bs, m.to(gpu))
            o.backward(do)
            outs.append((o.detach(), qq.grad, kk.grad, vv.grad))
        for a, b in zip(*outs):
            assert torch.equal(a, b)


def _full_size_properties(gpu, q, k, v, do, qbs, kbs, mask, check_permutation=True, hand_over=None):
    """Properties that need no oracle and hold at any size:
      * V = 1 gives O = 1 (softmax rows sum to one, also across lazily rescaled slabs);
      * doubling dO doubles dQ, dK, dV bit for bit (everything downstream of dO is linear; scaling by 2 is exact);
      * sum(q o dq) = sum(k o dk) per head (both are sum_ij dS_ij S_ij);
      * key blocks that no query block selects get exactly zero dK, dV;
      * permuting key blocks together with the mask columns leaves O unchanged up to summation order."""
    import flex_block_attn_amd as fba

    lists = fba.lists_for(mask, qbs, kbs)
    o1, _ = fba.forward_with_lists(q, k, torch.ones_like(v), qbs, kbs, lists)
    assert (o1.float() - 1).abs().max().item() <= 2 ** -7
    del o1
    o, lse = fba.forward_with_lists(q, k, v, qbs, kbs, lists)
    assert torch.isfinite(o).all() and torch.isfinite(lse).all()
    dq, dk, dv = fba.backward_with_lists(q, k, v, o, lse, do, qbs, kbs, lists, hand_over=hand_over)
    dq2, dk2, dv2 = fba.backward_with_lists(q, k, v, o, lse, do * 2, qbs, kbs, lists, hand_over=hand_over)
    for a, b in ((dq, dq2), (dk, dk2), (dv, dv2)):
        assert torch.isfinite(a).all() and torch.equal(a * 2, b)
    del dq2, dk2, dv2
    qdq = q.float() * dq.float()
    lhs, norm = qdq.sum((-1, -2)), qdq.abs().sum((-1, -2))
    del qdq
    rhs = (k.float() * dk.float()).sum((-1, -2))
    assert ((lhs - rhs).abs() / norm).max().item() < 2e-3
    m4 = mask if mask.dim() == 4 else mask[None, None].expand(q.shape[0], q.shape[1], -1, -1)
    unused = ~m4.any(-2)  # [B, H, nK]
    if unused.any():
        dead = unused.repeat_interleave(kbs, dim=-1)
        assert dk[dead].abs().max().item() == 0.0 and dv[dead].abs().max().item() == 0.0
    if check_permutation:
        nK = mask.shape[-1]
        perm = torch.randperm(nK, generator=torch.Generator(device="cpu").manual_seed(5)).to(gpu)
        tok = (perm[:, None] * kbs + torch.arange(kbs, device=gpu)[None, :]).reshape(-1)
        op, lsep = fba.forward_with_lists(q, k[:, :, tok].contiguous(), v[:, :, tok].contiguous(), qbs, kbs,
                                          fba.lists_for(mask[..., perm].contiguous(), qbs, kbs))
        assert (op.float() - o.float()).abs().max().item() <= 2e-2 and (lsep - lse).abs().max().item() <= 1e-3
    return o, lse, dq, dk, dv


def _full_size_inputs(gpu, B, H, S, seed):
    g = torch.Generator(device="cpu").manual_seed(seed)
    return tuple(torch.randn((B, H, S, 128), generator=g).to(torch.bfloat16).to(gpu) for _ in range(4))


def test_full_size_properties(gpu):
    """Dynamic random sparse configuration at full size: B1 H24 S30720 block 384, 32 of 80 key blocks per row, an
    independent mask per head."""
    from flex_block_attn_amd import masks

    B, H, S, bs, nb = 1, 24, 30720, 384, 80
    q, k, v, do = _full_size_inputs(gpu, B, H, S, 11)
    m = masks.random_block_mask(B, H, nb, nb, 32, 12).to(gpu)
    a = _full_size_properties(gpu, q, k, v, do, bs, bs, m, hand_over=True)
    b = _full_size_properties(gpu, q, k, v, do, bs, bs, m, check_permutation=False, hand_over=False)
    assert torch.equal(a[3], b[3]) and torch.equal(a[4], b[4])  # dK, dV: same kernel arithmetic on either path
    assert (a[2].float() - b[2].float()).abs().max().item() <= 2e-2


def test_fine_block_full_size_properties(gpu):
    """Tile lists at full size: B1 H24 S30720 with independent random 64 x 64 blocks, 40 % kept, an independent mask per
    head; the backward that hands dS over in 128 x 128 tile pairs (about 39 GB of workspace) and the recomputing one."""
    B, H, S, bs = 1, 24, 30720, 64
    nb = S // bs
    q, k, v, do = _full_size_inputs(gpu, B, H, S, 21)
    m = torch.rand((B, H, nb, nb), generator=torch.Generator().manual_seed(22)) < 0.4
    m[..., torch.arange(nb), torch.arange(nb)] = True
    m[..., :, 7] = False  # a key block nobody selects
    m = m.to(gpu)
    a = _full_size_properties(gpu, q, k, v, do, bs, bs, m, hand_over=True)
    b = _full_size_properties(gpu, q, k, v, do, bs, bs, m, check_permutation=False, hand_over=False)
    assert torch.equal(a[3], b[3]) and torch.equal(a[4], b[4])
    assert (a[2].float() - b[2].float()).abs().max().item() <= 2e-2


def test_full_attention_full_size_properties(gpu):
    """Full-attention configuration at full size: B1 H24 S11520 block 384, one all-ones 30x30 mask shared by every
    head (the mask_bh == 1 path with 30 key blocks per row).  With every block selected the result must also equal
    what the same kernels give for one 11520-row block pair, i.e. the block walk itself changes nothing."""
    import flex_block_attn_amd as fba
    from flex_block_attn_amd import masks

    B, H, S, bs = 1, 24, 11520, 384
    q, k, v, do = _full_size_inputs(gpu, B, H, S, 13)
    m = masks.full_block_mask(S // bs, S // bs).to(gpu)
    o, lse, dq, dk, dv = _full_size_properties(gpu, q, k, v, do, bs, bs, m)
    one = torch.ones((1, 1), dtype=torch.bool, device=gpu)
    lists1 = fba.compact_block_mask(one)
    o_1, lse_1 = fba.forward_with_lists(q, k, v, S, S, lists1)
    assert torch.equal(o, o_1) and torch.equal(lse, lse_1)
    for a, b in zip((dq, dk, dv), fba.backward_with_lists(q, k, v, o, lse, do, S, S, lists1)):
        assert torch.equal(a, b)


def test_sliding_tile_full_size_properties(gpu):
    """3-D sliding-tile configuration at full size: B1 H24 S115200 = 300 tiles of 6x8x8 = 384 tokens, 3x3x3 tile
    window (clamped: 27 key tiles per query tile), one 2-D mask for all heads."""
    from flex_block_attn_amd import masks

    B, H, S, bs = 1, 24, 115200, 384
    q, k, v, do = _full_size_inputs(gpu, B, H, S, 15)
    m = masks.sta_3d_block_mask((5, 6, 10), (3, 3, 3), clamp=True).to(gpu)
    assert m.shape == (300, 300) and (m.sum(-1) == 27).all()
    _full_size_properties(gpu, q, k, v, do, bs, bs, m)


@pytest.mark.parametrize("tiles,block,window,clamp", [((2, 3, 4), 128, (3, 3, 3), True), ((2, 3, 4), 128, (3, 3, 3), False),
                                                      ((3, 2, 2), 384, (1, 3, 3), True)])
def test_sliding_tile_mask_against_oracle(oracle, gpu, tiles, block, window, clamp):
    """Forward and backward with a sliding-tile mask against the C oracle, the mask taken from the oracle's own loop
    restatement (not from the product's builder), which must also equal the product's."""
    from flex_block_attn_amd import masks

    n = tiles[0] * tiles[1] * tiles[2]
    m = oracle.sta_3d_mask(tiles, window, clamp)
    assert torch.equal(m, masks.sta_3d_block_mask(tiles, window, clamp=clamp))
    _run_case(oracle, gpu, 1, 2, 2, n * block, n * block, block, block, m, seed=n + block)


def test_asymmetric_full_size_properties(gpu):
    """Asymmetric configuration at full size: B1 H24 S69120, q block 128 x k block 384 with the score-driven mask built
    on the GPU; the oracle-free properties, plus agreement of the selected pairs with the mask's own row structure
    (every query block keeps block 0, its diagonal band and 16 more at most)."""
    import flex_block_attn_amd as fba

    B, H, S, qbs, kbs = 1, 24, 69120, 128, 384
    q, k, v, do = _full_size_inputs(gpu, B, H, S, 21)
    m = fba.create_ssta_mask(q, k, qbs, kbs, topk=16, band=1, sink_blocks=1)
    nQ, nK = S // qbs, S // kbs
    assert m.shape == (B, H, nQ, nK) and m[..., 0].all()
    rows = m.sum(-1)
    assert int(rows.min()) >= 16 and int(rows.max()) <= 16 + 3 + 1
    diag = torch.arange(nQ, device=gpu) * qbs // kbs
    assert m[0, :, torch.arange(nQ, device=gpu), diag].all()
    _full_size_properties(gpu, q, k, v, do, qbs, kbs, m)


def test_pair_numbering_bit_exact(oracle, gpu):
    """fba_pair_slots against the oracle's loop restatement: 2-D and per-(b,h) masks, empty rows and columns, the
    benchmark's 80x80 masks."""
    import flex_block_attn_amd as fba
    from flex_block_attn_amd import masks

    cases = [masks.bernoulli_block_mask(4, 4, 0.5, 0), masks.bernoulli_block_mask(65, 129, 0.5, 4), torch.zeros((7, 9), dtype=torch.bool),
             torch.ones((30, 30), dtype=torch.bool), masks.random_block_mask(1, 24, 80, 80, 32, 5), masks.random_block_mask(2, 3, 17, 70, 5, 6),
             masks.sta_3d_block_mask((5, 6, 10), (3, 3, 3)), torch.rand((1, 24, 540, 180), generator=torch.Generator().manual_seed(1)) < 0.1]
    for m in cases:
        lists = fba.compact_block_mask(m.to(gpu))
        lists = fba.number_pairs(lists)
        pair_base, q_slot, listed = lists.pair_base, lists.q_slot, lists.listed_pairs()
        want_base, want_slot = oracle.pair_numbering(*oracle.compact_lists(m))
        assert pair_base.dtype == torch.int32 and q_slot.dtype == torch.int32 and listed == int(m.sum())
        assert np.array_equal(pair_base.cpu().numpy(), want_base), tuple(m.shape)
        assert np.array_equal(q_slot.cpu().numpy(), want_slot), tuple(m.shape)


def test_tile_pair_numbering_bit_exact(oracle, gpu):
    """fba_tile_slots against the oracle's restatement from allowed(i, j) alone, on the tile-list cases (2-D and
    per-(b,h) masks, empty and full masks, blocks that straddle key tiles)."""
    import flex_block_attn_amd as fba
    from flex_block_attn_amd import masks

    for n, (qbs, kbs, nQ, nK, p) in enumerate(TILE_LIST_CASES):
        for m in (masks.bernoulli_block_mask(nQ, nK, p, 40 + n), (torch.rand((2, 3, nQ, nK), generator=torch.Generator().manual_seed(n)) < p)):
            lists = fba.tile_block_mask(m.to(gpu), qbs, kbs, with_pair_numbers=True)
            want_base, want_table, want_slot = oracle.tile_pair_numbering(m, qbs, kbs)
            for g, w, name in zip((lists.pair_base, lists.q_slot, lists.k_slot), (want_base, want_table, want_slot), ("pair_base", "slot_table", "kt_slot")):
                assert g.dtype == torch.int32 and tuple(g.shape) == w.shape, (name, g.shape, w.shape)
                assert np.array_equal(g.cpu().numpy(), w), f"{name} differs for q{qbs} k{kbs} mask {tuple(m.shape)}"
            assert lists.listed_pairs() == int(want_base[-1])


BACKWARD_PATH_CASES = [
    # B, Hq, Hkv, Sq, Skv, q_block, kv_block, mask dims, density
    (1, 2, 2, 1536, 1536, 384, 384, 4, 0.5),
    (1, 3, 3, 768, 768, 128, 128, 2, 0.6),     # one 2-D mask for three heads: per-head offset into the workspace
    (2, 4, 2, 512, 1024, 128, 256, 4, 0.5),    # grouped kv heads, cross lengths, kv block larger than the q block
    (1, 2, 1, 1024, 768, 256, 128, 4, 0.4),    # q block larger than the kv block
    (1, 6, 2, 768, 1152, 384, 128, 2, 0.7),
    (2, 2, 2, 384, 384, 128, 384, 4, 1.0),
    # tile lists: dS travels in 128 x 128 tile pairs, only the 32 x 32 units that some row selects
    (1, 2, 2, 512, 512, 64, 64, 4, 0.5),
    (1, 3, 3, 768, 768, 16, 64, 2, 0.4),       # one 2-D mask for three heads
    (2, 4, 2, 512, 768, 32, 192, 4, 0.5),      # grouped kv heads; key blocks that straddle key tiles
    (1, 2, 1, 1152, 1152, 48, 192, 4, 0.4),
    (1, 2, 2, 768, 768, 128, 64, 4, 0.5),
    (1, 2, 2, 512, 768, 64, 128, 4, 0.3),
    (1, 2, 2, 256, 256, 64, 64, 4, 1.0),
]


@pytest.mark.parametrize("hand_over", [False, True], ids=["recompute", "handover"])
@pytest.mark.parametrize("cfg", BACKWARD_PATH_CASES, ids=lambda c: "B%d_Hq%d_Hkv%d_Sq%d_Skv%d_q%d_k%d_m%d_p%s" % c)
def test_both_backward_paths_against_oracle(oracle, gpu, cfg, hand_over):
    """fba_bwd / fba_bwd_tiled (dQ recomputes S and dP) and fba_bwd_handover / fba_bwd_tiled_handover (dQ from the dS the
    key-major kernel stored), each against the C oracle; masks with an empty query block and an unselected key block."""
    import flex_block_attn_amd as fba

    B, Hq, Hkv, Sq, Skv, qbs, kbs, mdim, density = cfg
    nQ, nK = Sq // qbs, Skv // kbs
    g = torch.Generator().manual_seed(Sq + Skv + qbs)
    m = torch.rand((nQ, nK) if mdim == 2 else (B, Hq, nQ, nK), generator=g) < density
    if density < 1.0 and nQ > 1 and nK > 1:
        m[..., 0, :] = False
        m[..., :, nK - 1] = False
        m[..., nQ - 1, 0] = True
    q, k, v, do = oracle.seeded_qkv(B, Hq, Hkv, Sq, Skv, seed=Sq + kbs)
    qb, kb, vb, dob = (t.to(torch.bfloat16) for t in (q, k, v, do))
    o_ref, lse_ref = oracle.c_attention_forward(qb, kb, vb, m, qbs, kbs)
    g_ref = oracle.c_attention_backward(qb, kb, vb, o_ref, lse_ref, dob, m, qbs, kbs)
    qg, kg, vg, dog = (t.to(gpu) for t in (qb, kb, vb, dob))
    lists = fba.lists_for(m.to(gpu), qbs, kbs)
    o, lse = fba.forward_with_lists(qg, kg, vg, qbs, kbs, lists)
    print(f"backward path hand_over={hand_over} cfg={cfg}", flush=True)
    grads = fba.backward_with_lists(qg, kg, vg, o, lse, dog, qbs, kbs, lists, hand_over=hand_over)
    res = {}
    for n, got, want in zip(("dq", "dk", "dv"), grads, g_ref):
        _check(oracle, got, want, n, res)
    other = fba.backward_with_lists(qg, kg, vg, o, lse, dog, qbs, kbs, lists, hand_over=not hand_over)
    assert torch.equal(grads[1], other[1]) and torch.equal(grads[2], other[2])  # dK, dV do not depend on the path
    assert (grads[0].float() - other[0].float()).abs().max().item() <= 2e-2


def test_backward_falls_back_without_workspace(gpu, monkeypatch):
    """With the workspace limit at zero the automatic choice is the recomputing backward: same bits as hand_over=False,
    and no dS workspace is allocated."""
    import flex_block_attn_amd as fba
    from flex_block_attn_amd import interface, masks

    g = torch.Generator(device="cpu").manual_seed(3)
    q, k, v, do = (torch.randn((1, 2, 768, 128), generator=g).to(torch.bfloat16).to(gpu) for _ in range(4))
    lists = fba.compact_block_mask(masks.bernoulli_block_mask(6, 6, 0.5, 1).to(gpu))
    o, lse = fba.forward_with_lists(q, k, v, 128, 128, lists)
    want = fba.backward_with_lists(q, k, v, o, lse, do, 128, 128, lists, hand_over=False)
    monkeypatch.setattr(interface, "DS_WORKSPACE_LIMIT_GIB", 0.0)
    assert interface.ds_workspace_limit(q, k) == 0
    got = fba.backward_with_lists(q, k, v, o, lse, do, 128, 128, lists)
    for a, b in zip(got, want):
        assert torch.equal(a, b)
    # an empty mask has no pair to hand over: both settings give zero gradients
    empty = fba.compact_block_mask(torch.zeros((6, 6), dtype=torch.bool, device=gpu))
    o0, lse0 = fba.forward_with_lists(q, k, v, 128, 128, empty)
    for t in fba.backward_with_lists(q, k, v, o0, lse0, do, 128, 128, empty, hand_over=True):
        assert t.abs().max().item() == 0.0
    # the same with tile lists
    tl = fba.tile_block_mask(masks.bernoulli_block_mask(12, 12, 0.5, 2).to(gpu), 64, 64)
    o, lse = fba.forward_with_lists(q, k, v, 64, 64, tl)
    want = fba.backward_with_lists(q, k, v, o, lse, do, 64, 64, tl, hand_over=False)
    for a, b in zip(fba.backward_with_lists(q, k, v, o, lse, do, 64, 64, tl), want):
        assert torch.equal(a, b)
    empty = fba.tile_block_mask(torch.zeros((12, 12), dtype=torch.bool, device=gpu), 64, 64)
    o0, lse0 = fba.forward_with_lists(q, k, v, 64, 64, empty)
    for t in fba.backward_with_lists(q, k, v, o0, lse0, do, 64, 64, empty, hand_over=True):
        assert t.abs().max().item() == 0.0


def test_backward_statistics_against_oracle(oracle, gpu):
    """fba_bwd_stats alone: stats[0] = lse * log2(e), stats[1] = -delta = -rowsum(dO o O), against the C oracle's
    oracle_bwd_delta (flex_block_attn_h100.cu:375-379) on the same bf16 values; rows that are not a multiple of the
    kernel's 16-row groups included."""
    import ctypes

    from flex_block_attn_amd import _lib
    from flex_block_attn_amd.interface import _ptr, _stream

    for rows, seed in ((16 * 37 + 5, 1), (1, 2), (70000, 3)):
        g = torch.Generator(device="cpu").manual_seed(seed)
        o = torch.randn((rows, 128), generator=g).to(torch.bfloat16)
        do = torch.randn((rows, 128), generator=g).to(torch.bfloat16)
        lse = torch.randn((rows,), generator=g) * 3 + 5
        lse[0] = float("-inf")
        want = np.empty((rows,), np.float32)
        oa, da = (np.ascontiguousarray(t.float().numpy()) for t in (o, do))
        oracle.c_lib().oracle_bwd_delta(oa.ctypes.data_as(ctypes.c_void_p), da.ctypes.data_as(ctypes.c_void_p), rows, 128, want.ctypes.data_as(ctypes.c_void_p))
        og, dg, lg = o.to(gpu), do.to(gpu), lse.to(gpu)
        stats = torch.full((2, rows), float("nan"), dtype=torch.float32, device=gpu)
        _lib.call("fba_bwd_stats", _ptr(og), _ptr(dg), _ptr(lg), _ptr(stats), rows, 128, _stream())
        got = stats.cpu()
        assert (-got[1] - torch.from_numpy(want)).abs().max().item() <= 1e-4  # fp32 sums of 128 products of N(0,1) pairs
        want_l2 = lse.double() * 1.4426950408889634
        assert got[0, 0].item() == float("-inf")
        if rows > 1:
            assert (got[0, 1:].double() - want_l2[1:]).abs().max().item() <= 2e-6 * float(want_l2[1:].abs().max())


def test_sweep_harness_runs(gpu, tmp_path):
    """The sweep harness on the GPU, all three modes at a tiny size: CSV files and columns of the reference's scripts
    for this operator (benchmark/utils/utils.py:31-59; random_fwd.py / random_bwd.py / random_memory.py)."""
    import csv

    from flex_block_attn_amd import benchmark

    for mode in ("random", "swa", "full"):
        benchmark.main(["--mode", mode, "--seq-lens", "768", "--num-heads", "1", "--sparse-rates", "0.5", "--rep", "2", "--warmup", "1",
                        "--out", str(tmp_path)])
        lead = ["batch_size", "seq_len", "num_heads", "head_dim", "block_size"] + ([] if mode == "full" else ["sparse_rate"])
        for kind, cols in (("fwd", ["ptm_attn_masks", "ptm_attn_executes"]), ("bwd", ["ptm_attn_bwd"]), ("memory", ["ptm_fwd_memory", "ptm_bwd_memory"])):
            rows = list(csv.DictReader(open(tmp_path / f"{mode}_{kind}_results_384.csv")))
            assert len(rows) == 1 and list(rows[0].keys()) == lead + cols
            assert int(rows[0]["seq_len"]) == 768 and all(float(rows[0][c]) > 0 for c in cols)


def test_matrix_pipe_probe(gpu):
    """fba_probe_mfma: zero operands give zero checksums; with operands a[t], b[t] every accumulator element of a wave's
    32x32 tile is a 16-term dot product repeated 4 * iters times, so the checksums are finite and scale with iters."""
    from flex_block_attn_amd import _lib
    from flex_block_attn_amd.interface import _ptr, _stream

    sink = torch.full((4 * 256,), float("nan"), device=gpu)
    _lib.call("fba_probe_mfma", None, _ptr(sink), 4, 10, _stream())
    assert (sink == 0).all()
    src = torch.full((1024,), 0.5, device=gpu)
    _lib.call("fba_probe_mfma", _ptr(src), _ptr(sink), 4, 10, _stream())
    # each MFMA adds 16 * 0.25 = 4 to every element; 10 of them per accumulator, 4 accumulators x 16 elements summed
    assert torch.equal(sink, torch.full_like(sink, 4.0 * 10 * 64))


def test_read_probe_reads_and_leaves_its_sink(gpu):
    """fba_probe_read: reads the buffer and stores nothing: the sink keeps its value, except for data that folds to the
    one word the kernel tests for (a buffer holding that word once and zeros elsewhere)."""
    from flex_block_attn_amd import _lib
    from flex_block_attn_amd.interface import _ptr, _stream

    src = torch.randint(0, 2 ** 31 - 1, (32768 * 4 // 4,), dtype=torch.int32, device=gpu)
    sink = torch.full((1,), 7, dtype=torch.int32, device=gpu)
    _lib.call("fba_probe_read", _ptr(src), src.numel() * 4, _ptr(sink), 3, _stream())
    assert int(sink[0]) == 7
    src.zero_()
    src[12345] = 0x5EED1E55
    _lib.call("fba_probe_read", _ptr(src), src.numel() * 4, _ptr(sink), 3, _stream())
    torch.cuda.synchronize()
    assert int(sink[0]) == 1  # the word was read by the lane that owns it


@pytest.mark.parametrize("block_size", [64, 128, 384])
def test_readme_usage_verbatim(oracle, gpu, block_size):
    """The reference README's usage section (README.md:24-53), run as written: its two imports, a list-of-lists
    `selected_blocks`, `create_sparse_mask`, the call; on a (block_size * 2) x (block_size * 2) problem as there, at the
    block sizes it names.  The result is compared with the oracle under that 2 x 2 mask."""
    from flex_block_attn import flex_block_attn_func
    from benchmark.utils.utils import create_sparse_mask

    g = torch.Generator(device="cpu").manual_seed(block_size)
    q, key, value = (torch.randn((1, 2, block_size * 2, 128), generator=g).to(torch.bfloat16).to(gpu) for _ in range(3))
    query = q
    q_block_size = k_block_size = block_size
    # take a (block_size * 2)*(block_size * 2) as an example
    selected_blocks = [[0, 1], [1, 0]]
    # create block mask with selected blocks
    sparse_mask = create_sparse_mask(q, block_size, selected_blocks)
    block_mask = sparse_mask
    # compute
    output = flex_block_attn_func(query, key, value, q_block_size, k_block_size, block_mask)

    assert sparse_mask.dtype == torch.bool and sparse_mask.cpu().tolist() == [[False, True], [True, False]]
    want, _ = oracle.c_attention_forward(query.cpu(), key.cpu(), value.cpu(), sparse_mask.cpu(), block_size, block_size)
    _check(oracle, output, want, "o", {})


CHUNK_CASES = [
    # B, Hq, Hkv, Sq, Skv, q_block, k_block, mask dims, density
    (1, 6, 6, 768, 768, 128, 128, 4, 0.6),
    (2, 4, 2, 512, 768, 128, 256, 4, 0.5),
    (1, 6, 3, 768, 768, 384, 384, 2, 0.7),
    (2, 2, 2, 512, 512, 64, 64, 4, 0.5),
    (1, 4, 2, 512, 512, 32, 64, 2, 0.6),
]


@pytest.mark.parametrize("cfg", CHUNK_CASES, ids=lambda c: "B%d_Hq%d_Hkv%d_Sq%d_Skv%d_q%d_k%d_m%d_p%s" % c)
def test_backward_in_head_chunks(oracle, gpu, cfg, monkeypatch):
    """The default backward hands dS over in chunks of kv heads through a bounded workspace.  With the limit set so low
    that every kv head is a chunk of its own (and tail splitting off, so that every tile sums in one order), the result
    must equal the one-workspace hand-over bit for bit: per-head and shared masks, grouped kv heads, batches, block and
    tile lists.  With the limit below one head's need the call falls back to the recomputing backward."""
    import flex_block_attn_amd as fba
    from flex_block_attn_amd import interface

    B, Hq, Hkv, Sq, Skv, qbs, kbs, mdim, density = cfg
    nQ, nK = Sq // qbs, Skv // kbs
    g = torch.Generator().manual_seed(Sq + Skv + qbs + Hq)
    m = (torch.rand((nQ, nK) if mdim == 2 else (B, Hq, nQ, nK), generator=g) < density).to(gpu)
    q, k, v, do = (t.to(torch.bfloat16).to(gpu) for t in oracle.seeded_qkv(B, Hq, Hkv, Sq, Skv, seed=Sq + kbs + 1))
    lists = fba.lists_for(m, qbs, kbs)
    o, lse = fba.forward_with_lists(q, k, v, qbs, kbs, lists)
    monkeypatch.setattr(interface, "SPLIT_WORKSPACE_MIB", "0")
    whole = fba.backward_with_lists(q, k, v, o, lse, do, qbs, kbs, lists, hand_over=True)
    unit_pairs, _ = interface._unit_pairs(lists, B, Hq, Hkv)
    pair_bytes = (128 * 128 if lists.tiled else qbs * kbs) * 2
    assert max(unit_pairs) > 0
    monkeypatch.setattr(interface, "DS_WORKSPACE_FACTOR", 1e9)  # only the absolute limit counts here
    monkeypatch.setattr(interface, "DS_WORKSPACE_LIMIT_GIB", max(unit_pairs) * pair_bytes / 2 ** 30)
    chunks = interface.plan_head_chunks(unit_pairs, pair_bytes, max(unit_pairs) * pair_bytes)
    assert len(chunks) == B * Hkv or sum(unit_pairs) == max(unit_pairs) * B * Hkv
    print(f"chunked backward cfg={cfg} chunks={chunks}", flush=True)
    chunked = fba.backward_with_lists(q, k, v, o, lse, do, qbs, kbs, lists)
    for a, b in zip(chunked, whole):
        assert torch.equal(a, b)
    monkeypatch.setattr(interface, "DS_WORKSPACE_LIMIT_GIB", (max(unit_pairs) * pair_bytes - 1) / 2 ** 30)
    recomputed = fba.backward_with_lists(q, k, v, o, lse, do, qbs, kbs, lists)
    for a, b in zip(recomputed, fba.backward_with_lists(q, k, v, o, lse, do, qbs, kbs, lists, hand_over=False)):
        assert torch.equal(a, b)


def test_backward_workspace_stays_within_its_limit(gpu, monkeypatch):
    """B1 H8 S7680 full attention: all heads at once would need 944 MB of dS; with a 0.25 GiB limit the default backward
    runs four chunks of two heads and its peak allocation stays below limit + outputs + statistics + splitting workspace."""
    import flex_block_attn_amd as fba
    from flex_block_attn_amd import _lib, interface, masks

    B, H, S, bs = 1, 8, 7680, 384
    g = torch.Generator(device="cpu").manual_seed(17)
    q, k, v, do = (torch.randn((B, H, S, 128), generator=g).to(torch.bfloat16).to(gpu) for _ in range(4))
    lists = fba.compact_block_mask(masks.full_block_mask(S // bs, S // bs).to(gpu), with_pair_numbers=True)
    o, lse = fba.forward_with_lists(q, k, v, bs, bs, lists)
    want = fba.backward_with_lists(q, k, v, o, lse, do, bs, bs, lists, hand_over=True)
    limit = 0.25
    monkeypatch.setattr(interface, "DS_WORKSPACE_FACTOR", 1e9)
    monkeypatch.setattr(interface, "DS_WORKSPACE_LIMIT_GIB", limit)
    assert interface.ds_workspace_bytes(lists, B, H, bs, bs)[1] > 3 * limit * 2 ** 30
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    got = fba.backward_with_lists(q, k, v, o, lse, do, bs, bs, lists)
    torch.cuda.synchronize()
    peak = torch.cuda.max_memory_allocated() - before
    outputs = 3 * q.numel() * 2 + 2 * B * H * S * 4
    assert peak <= limit * 2 ** 30 + outputs + _lib.load().fba_split_workspace_bytes() + (2 << 20), f"peak {peak} bytes"
    for a, b in zip(got, want):  # launches of two and of eight heads split their last tiles differently: same sums, another order
        assert (a.float() - b.float()).abs().max().item() <= 2e-2


@pytest.mark.parametrize("cfg", [(1, 2, 2, 1536, 1536, 384, 384), (2, 4, 2, 1024, 768, 128, 256), (1, 3, 3, 3072, 3072, 384, 384), (1, 30, 30, 1536, 1536, 384, 384)],
                         ids=lambda c: "B%d_Hq%d_Hkv%d_Sq%d_Skv%d_q%d_k%d" % c)
def test_measurement_variants_give_the_same_bits(gpu, cfg, monkeypatch):
    """The forward variant kept for measurement (FBA_FWD_TILE_ROWS=384: 384-row work-groups) and the two dK/dV kernels
    (FBA_DKDV_KEYS_PER_WAVE=32 / 64: two waves per SIMD with 32 keys each, the default with the dS hand-over, or one wave
    per SIMD with 64 keys, the default without) do the same arithmetic in the same order: O, LSE, dK, dV and the handed-over dS (seen through dQ) must be bit-equal, with and without tail
    splitting, on grouped heads and on launches larger than the GPU."""
    import flex_block_attn_amd as fba
    from flex_block_attn_amd import interface

    B, Hq, Hkv, Sq, Skv, qbs, kbs = cfg
    g = torch.Generator(device="cpu").manual_seed(Sq + Hq)
    q, do = (torch.randn((B, Hq, Sq, 128), generator=g).to(torch.bfloat16).to(gpu) for _ in range(2))
    k, v = (torch.randn((B, Hkv, Skv, 128), generator=g).to(torch.bfloat16).to(gpu) for _ in range(2))
    m = (torch.rand((B, Hq, Sq // qbs, Skv // kbs), generator=g) < 0.6).to(gpu)
    lists = fba.lists_for(m, qbs, kbs)
    for split in (None, "0"):
        monkeypatch.setattr(interface, "SPLIT_WORKSPACE_MIB", split)
        monkeypatch.delenv("FBA_FWD_TILE_ROWS", raising=False)
        monkeypatch.setenv("FBA_DKDV_KEYS_PER_WAVE", "32")
        o, lse = fba.forward_with_lists(q, k, v, qbs, kbs, lists)
        base = [fba.backward_with_lists(q, k, v, o, lse, do, qbs, kbs, lists, hand_over=h) for h in (True, False)]
        if qbs % 384 == 0 and split == "0":  # the 384-row forward does not split its tail
            monkeypatch.setenv("FBA_FWD_TILE_ROWS", "384")
            o2, lse2 = fba.forward_with_lists(q, k, v, qbs, kbs, lists)
            assert torch.equal(o, o2) and torch.equal(lse, lse2)
        monkeypatch.setenv("FBA_DKDV_KEYS_PER_WAVE", "64")
        for h, want in zip((True, False), base):
            print(f"variant test cfg={cfg} split={split} hand_over={h}", flush=True)
            got = fba.backward_with_lists(q, k, v, o, lse, do, qbs, kbs, lists, hand_over=h)
            for a, b in zip(got, want):
                assert torch.equal(a, b)


def test_tile_list_forward_splits_its_tail(oracle, gpu, monkeypatch):
    """Forward on tile lists with and without the splitting workspace: a launch smaller than the GPU (every tile cut into
    parts) against the oracle, and a launch of 4.5 rounds (the last half round cut into parts) against itself without
    splitting; entries switched off for some 16-row groups, an empty query block and a range that starts inside an entry's
    second slab are all in there."""
    import flex_block_attn_amd as fba
    from flex_block_attn_amd import interface

    g = torch.Generator(device="cpu").manual_seed(31)
    m = torch.rand((1, 2, 12, 6), generator=g) < 0.5
    m[..., 3, :] = False
    for split in (None, "0"):
        monkeypatch.setattr(interface, "SPLIT_WORKSPACE_MIB", split)
        _run_case(oracle, gpu, 1, 2, 2, 768, 384, 64, 64, m, seed=32)
    # 24 halves against lists of up to 64 chunks
    m = torch.rand((1, 2, 12, 64), generator=g) < 0.5
    m[..., 3, :] = False
    q, k, v, _ = oracle.seeded_qkv(1, 2, 2, 768, 4096, seed=33)
    q, k, v = (t.to(torch.bfloat16) for t in (q, k, v))
    o_ref, lse_ref = oracle.c_attention_forward(q, k, v, m, 64, 64)
    lists = fba.lists_for(m.to(gpu), 64, 64)
    outs, res = [], {}
    for split in (None, "0"):
        monkeypatch.setattr(interface, "SPLIT_WORKSPACE_MIB", split)
        o, lse = fba.forward_with_lists(q.to(gpu), k.to(gpu), v.to(gpu), 64, 64, lists)
        _check(oracle, o, o_ref, f"o split {split}", res)
        assert torch.equal(torch.isinf(lse).flatten().cpu(), torch.isinf(lse_ref).flatten())
        outs.append(o)
    rows = (torch.arange(768) // 64 != 3).to(gpu)
    assert not torch.equal(outs[0][:, :, rows], outs[1][:, :, rows])  # the parts did sum in another order
    B, H, S, bs = 1, 9, 16384, 64  # 2304 halves of 128-row tiles on 512 slots
    nb = S // bs
    q, k, v = (torch.randn((B, H, S, 128), generator=g).to(torch.bfloat16).to(gpu) for _ in range(3))
    mask = (torch.rand((B, H, nb, nb), generator=g) < 0.15).to(gpu)
    lists = fba.lists_for(mask, bs, bs)
    assert lists.tiled
    outs = []
    for split in (None, "0"):
        monkeypatch.setattr(interface, "SPLIT_WORKSPACE_MIB", split)
        outs.append(fba.forward_with_lists(q, k, v, bs, bs, lists))
    (o_a, lse_a), (o_b, lse_b) = outs
    assert not torch.equal(o_a[:, -1], o_b[:, -1])  # the last tiles did sum in another order
    assert torch.equal(o_a[:, 0], o_b[:, 0]) and torch.equal(lse_a[:, 0], lse_b[:, 0])
    assert (o_a.float() - o_b.float()).abs().max().item() <= 2e-2
    both = torch.isfinite(lse_a) & torch.isfinite(lse_b)
    assert torch.equal(torch.isfinite(lse_a), torch.isfinite(lse_b)) and (lse_a[both] - lse_b[both]).abs().max().item() <= 1e-3


@pytest.mark.parametrize("bs", [128, 64])
def test_handover_with_a_workspace_too_small_for_the_lists_fails_loudly(gpu, bs):
    """A hand-over call whose lists number more pairs than the workspace is said to hold (lists rebuilt, a stale pair
    count): the host cannot see it, the kernels can.  Nothing is stored into the workspace and dQ, dK, dV come back as
    NaN; the same call with the true size gives what backward_with_lists gives.  Block lists and tile lists."""
    import ctypes

    import flex_block_attn_amd as fba
    from flex_block_attn_amd import _lib, interface
    from flex_block_attn_amd.interface import _ptr, _stream

    B, H, S = 1, 3, 1024
    g = torch.Generator(device="cpu").manual_seed(41 + bs)
    q, k, v, do = (torch.randn((B, H, S, 128), generator=g).to(torch.bfloat16).to(gpu) for _ in range(4))
    mask = (torch.rand((B, H, S // bs, S // bs), generator=g) < 0.5).to(gpu)
    lists = fba.lists_for(mask, bs, bs)
    assert lists.tiled == (bs == 64)
    o, lse = fba.forward_with_lists(q, k, v, bs, bs, lists)
    want = fba.backward_with_lists(q, k, v, o, lse, do, bs, bs, lists, hand_over=True)
    pairs, ws_bytes = interface.ds_workspace_bytes(lists, B, H, bs, bs)
    pair_bytes = ws_bytes // pairs
    ws = torch.full((ws_bytes,), 0x5A, dtype=torch.uint8, device=gpu)  # full size, so that nothing could leave the allocation
    stats = torch.empty((2, B, H, S), dtype=torch.float32, device=gpu)
    _split, sp_ptr, sp_bytes = interface._split_workspace(q.device)  # as backward_with_lists: same tiles split, same sums

    def call(n_pairs):
        dq, dk, dv = (torch.zeros_like(t) for t in (q, k, v))
        head = (_ptr(q), _ptr(k), _ptr(v), _ptr(o), _ptr(do), _ptr(lse), _ptr(stats), _ptr(ws), n_pairs * pair_bytes,
                _ptr(dq), _ptr(dk), _ptr(dv), _ptr(lists.q_cnt), _ptr(lists.q_idx), _ptr(lists.k_cnt), _ptr(lists.k_idx))
        shape = (n_pairs, lists.mask_bh, B, H, H, S, S, 128, bs, bs)
        if lists.tiled:
            _lib.call("fba_bwd_tiled_handover", *head, _ptr(lists.pair_base), _ptr(lists.k_slot), _ptr(lists.q_slot), *shape, sp_ptr, sp_bytes, _stream())
        else:
            _lib.call("fba_bwd_handover", *head, _ptr(lists.pair_base), _ptr(lists.q_slot), *shape, sp_ptr, sp_bytes, _stream())
        torch.cuda.synchronize()
        return dq, dk, dv

    for short in (pairs - 1, pairs // 2):
        got = call(short)
        for t in got:
            assert torch.isnan(t).all()
        assert (ws == 0x5A).all()
    for a, b in zip(call(pairs), want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("bs,keys", [(128, "64"), (128, "32"), (64, "32")])
def test_claimed_grid_indices_change_no_bit(gpu, monkeypatch, bs, keys):
    """Launches of four rounds and more let the dK/dV work-groups claim their grid indices (some work-groups more than
    indices, an XCD that is through early takes over from the others): which work-group computes a tile must not show in
    the result.  1152 key tiles; block lists with either dK/dV kernel, and tile lists."""
    import flex_block_attn_amd as fba

    B, H, S = 1, 9, 16384
    g = torch.Generator(device="cpu").manual_seed(51 + bs)
    q, k, v, do = (torch.randn((B, H, S, 128), generator=g).to(torch.bfloat16).to(gpu) for _ in range(4))
    mask = (torch.rand((B, H, S // bs, S // bs), generator=g) < 0.1).to(gpu)
    lists = fba.lists_for(mask, bs, bs)
    o, lse = fba.forward_with_lists(q, k, v, bs, bs, lists)
    monkeypatch.setenv("FBA_DKDV_KEYS_PER_WAVE", keys)
    outs = []
    for claim in ("0", None):
        if claim is None:
            monkeypatch.delenv("FBA_CLAIM_WORK", raising=False)
        else:
            monkeypatch.setenv("FBA_CLAIM_WORK", claim)
        outs.append(fba.backward_with_lists(q, k, v, o, lse, do, bs, bs, lists))
    for a, b in zip(*outs):
        assert torch.isfinite(a).all() and torch.equal(a, b)


def test_backward_memory_follows_the_sequence_length(gpu):
    """One head, S=30720, all 80 x 80 blocks of 384: the dS of that head (1.9 GB) is more than the default backward may
    allocate (six times the call's own tensors), so it recomputes instead and its peak allocation stays within twice the
    144.8 MB the reference's backward needs for the same problem (benchmark/full/results/full_memory_results_384.csv:4,
    column ptm_bwd_memory); forward + backward of the operator through autograd."""
    import flex_block_attn_amd as fba
    from flex_block_attn_amd import masks

    S, bs = 30720, 384
    g = torch.Generator(device="cpu").manual_seed(23)
    q, k, v = (torch.randn((1, 1, S, 128), generator=g).to(torch.bfloat16).to(gpu).requires_grad_(True) for _ in range(3))
    m = masks.full_block_mask(S // bs, S // bs).to(gpu)
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    o = fba.flex_block_attn_func(q, k, v, bs, bs, m)
    o.sum().backward()
    torch.cuda.synchronize()
    peak = torch.cuda.max_memory_allocated() - before + 3 * q.numel() * 2  # the reference's figure counts q, k, v too
    assert peak <= 2 * 144.8e6, f"peak {peak * 1e-6:.1f} MB"
    assert torch.isfinite(q.grad).all() and torch.isfinite(k.grad).all() and torch.isfinite(v.grad).all()
