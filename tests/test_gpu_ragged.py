"""Sequences that are no whole number of 128-row tiles go through padded copies made by the library.  Outputs and gradients
against the same call on inputs padded by torch: bit for bit, with shapes and strides of their own.  Query rows alone, keys
alone, both, shorter than a tile, many sequences, grouped heads, both mask ranks, with and without gradients, and in-place
changes of the output, which autograd has to notice."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Skv,qbs,kbs,dims", [
    (1, 1, 1, 16, 64, 16, 64, 2),         # less than a tile
    (2, 4, 2, 3136, 3136, 16, 64, 4),
    (1, 2, 2, 640, 576, 32, 64, 4),       # keys alone
    (1, 3, 1, 336, 768, 48, 192, 4),      # queries alone, appended in blocks of 384 rows
    (3, 2, 1, 320, 448, 64, 64, 2),
    (1, 17, 17, 144, 192, 16, 64, 4),     # a number of rows that is no multiple of a copy's block
])
def test_ragged_lengths(gpu, B, Hq, Hkv, Sq, Skv, qbs, kbs, dims):
    import math

    import flex_block_attn_amd as fba
    from flex_block_attn_amd.interface import FlexBlockAttnFunc

    g = torch.Generator().manual_seed(Sq + Skv)
    m = torch.rand(((B, Hq) if dims == 4 else ()) + (Sq // qbs, Skv // kbs), generator=g) < 0.5
    m[..., 0] = True
    m = m.to(gpu)
    q, do = (torch.randn((B, Hq, Sq, 128), generator=g).to(torch.bfloat16).to(gpu) for _ in range(2))
    k, v = (torch.randn((B, Hkv, Skv, 128), generator=g).to(torch.bfloat16).to(gpu) for _ in range(2))
    print(f"ragged B{B} Hq{Hq} Hkv{Hkv} Sq{Sq} Skv{Skv} q{qbs} k{kbs}", flush=True)

    def pads(n, block):
        return 0 if n % 128 == 0 else -n % math.lcm(block, 128)

    pq, pk = pads(Sq, qbs), pads(Skv, kbs)
    F = torch.nn.functional
    ref = [t.clone().requires_grad_(True) for t in (q, k, v)]
    mp = F.pad(m, (0, pk // kbs, 0, pq // qbs), value=False)
    o_ref = FlexBlockAttnFunc.apply(*(F.pad(t, (0, 0, 0, n)) for t, n in zip(ref, (pq, pk, pk))), qbs, kbs, mp, True)[:, :, :Sq]
    want = torch.autograd.grad(o_ref, ref, do)
    ins = [t.clone().requires_grad_(True) for t in (q, k, v)]
    o = fba.flex_block_attn_func(*ins, qbs, kbs, m)
    got = torch.autograd.grad(o, ins, do)
    with torch.no_grad():
        o_plain = fba.flex_block_attn_func(q, k, v, qbs, kbs, m)
    assert o.shape == q.shape and o.stride() == o_ref.stride()
    assert torch.equal(o, o_ref) and torch.equal(o_plain, o_ref)
    for name, t, a, b in zip(("dq", "dk", "dv"), ins, got, want):
        assert a.shape == t.shape and a.is_contiguous() and torch.equal(a, b), name

    o = fba.flex_block_attn_func(*ins, qbs, kbs, m)
    o.mul_(2)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        torch.autograd.grad(o, ins, do)
