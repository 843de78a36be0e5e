"""Backward through a dS workspace with a place for every pair (fba_bwd_dense) against the numbered hand-over, bit for bit, and
fba_lists with and without its key-major half against the entry points it stands for."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Skv,qbs,kbs,dims", [
    (1, 1, 1, 128, 128, 128, 128, 4),     # one pair
    (2, 4, 2, 1024, 768, 128, 256, 4),    # grouped heads, cross lengths, a mask per head
    (1, 3, 3, 1536, 1536, 384, 384, 2),   # one mask for all heads
    (1, 2, 1, 512, 384, 16, 64, 4),       # tile lists, grouped heads
    (2, 2, 2, 640, 640, 64, 64, 2),
])
def test_dense_numbering_changes_no_bit(gpu, B, Hq, Hkv, Sq, Skv, qbs, kbs, dims):
    import flex_block_attn_amd as fba
    from flex_block_attn_amd import _lib, interface
    from flex_block_attn_amd.interface import _ptr, _stream

    g = torch.Generator().manual_seed(Sq + qbs)
    nQ, nK = Sq // qbs, Skv // kbs
    m = (torch.rand((nQ, nK) if dims == 2 else (B, Hq, nQ, nK), generator=g) < 0.5)
    m[..., 0, :] = nQ == 1  # an empty query block, and with it shorter lists
    m = m.to(gpu)
    q, do = (torch.randn((B, Hq, Sq, 128), generator=g).to(torch.bfloat16).to(gpu) for _ in range(2))
    k, v = (torch.randn((B, Hkv, Skv, 128), generator=g).to(torch.bfloat16).to(gpu) for _ in range(2))
    print(f"dense B{B} Hq{Hq} Hkv{Hkv} Sq{Sq} Skv{Skv} q{qbs} k{kbs}", flush=True)
    lists = fba.lists_for(m, qbs, kbs)
    o, lse = fba.forward_with_lists(q, k, v, qbs, kbs, lists)
    assert interface.dense_ds_fits(q, k) and lists.pair_base is None
    dense = fba.backward_with_lists(q, k, v, o, lse, do, qbs, kbs, lists)
    assert lists.pair_base is None
    numbered = fba.backward_with_lists(q, k, v, o, lse, do, qbs, kbs, lists, hand_over=True)
    for name, a, b in zip(("dq", "dk", "dv"), dense, numbered):
        assert torch.equal(a, b), name
    # the same lists through fba_lists, whole and query-major alone
    for both in (True, False):
        got = [torch.full_like(t, -7) for t in (lists.q_cnt, lists.q_idx, lists.k_cnt, lists.k_idx)]
        _lib.call("fba_lists", _ptr(m), lists.mask_bh, nQ, nK, qbs, kbs, _ptr(got[0]), _ptr(got[1]), _ptr(got[2]) if both else None,
                  _ptr(got[3]) if both else None, _stream())
        torch.cuda.synchronize()
        assert torch.equal(got[0], lists.q_cnt) and torch.equal(got[1], lists.q_idx)
        if both:
            assert torch.equal(got[2], lists.k_cnt) and torch.equal(got[3], lists.k_idx)
        else:
            assert (got[2] == -7).all() and (got[3] == -7).all()


@pytest.mark.parametrize("H,S,keep,dense", [
    (24, 6912, 5, False),  # 54 key blocks: places for all pairs would be 2.3 GB, the selected ones are 0.2 GB
    (24, 2048, 2, True),   # 0.2 GB, all pairs
])
def test_backward_memory_of_a_sparse_call(gpu, H, S, keep, dense):
    """Outside small problems the dS workspace follows the selected pairs."""
    import flex_block_attn_amd as fba
    from flex_block_attn_amd import interface, masks

    n = S // 128
    q, k, v = (torch.randn((1, H, S, 128), device=gpu, dtype=torch.bfloat16).requires_grad_(True) for _ in range(3))
    mask = masks.random_block_mask(1, H, n, n, keep, 0).to(gpu)
    assert interface.dense_ds_fits(q, k) is dense
    print(f"memory of backward H{H} S{S} keep {keep}", flush=True)
    o = fba.flex_block_attn_func(q, k, v, 128, 128, mask)
    do = torch.randn_like(o)
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    torch.autograd.grad(o, (q, k, v), do)
    torch.cuda.synchronize()
    ds = interface.dense_ds_bytes(q, k) if dense else int(mask.sum()) * 128 * 128 * 2
    # the three gradients, statistics (two floats a row), the tail-splitting workspace, rounding by the allocator
    rest = 3 * q.numel() * 2 + 2 * H * S * 4 + interface._split_bytes() + 2 ** 22
    assert torch.cuda.max_memory_allocated() - before <= ds + rest


@pytest.mark.parametrize("cfg", [(2, 4, 2, 1024, 768, 128, 256, 4), (1, 3, 3, 1536, 1536, 384, 384, 2)])
def test_dense_numbering_with_32_keys_per_wave(gpu, monkeypatch, cfg):
    """The same in the dK/dV kernel kept for measurement."""
    monkeypatch.setenv("FBA_DKDV_KEYS_PER_WAVE", "32")
    test_dense_numbering_changes_no_bit(gpu, *cfg)
