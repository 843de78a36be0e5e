"""Gradients of outputs whose rows were cut: whatever layout the incoming gradient has (strided, expanded, off the 16-byte grid, fp32 through
a cast), the same bits as for a plain contiguous one; none at all for an output that enters nothing."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Skv,qbs,kbs", [(1, 2, 1, 336, 448, 16, 64), (2, 1, 1, 192, 256, 64, 64)])
def test_layouts_of_the_gradient(gpu, B, Hq, Hkv, Sq, Skv, qbs, kbs):
    import flex_block_attn_amd as fba

    g = torch.Generator().manual_seed(Sq)
    m = torch.ones((Sq // qbs, Skv // kbs), dtype=torch.bool, device=gpu)
    q = torch.randn((B, Hq, Sq, 128), generator=g).to(torch.bfloat16).to(gpu).requires_grad_(True)
    k, v = (torch.randn((B, Hkv, Skv, 128), generator=g).to(torch.bfloat16).to(gpu).requires_grad_(True) for _ in range(2))
    do = torch.randn((B, Hq, Sq, 128), generator=g).to(torch.bfloat16).to(gpu)
    print(f"ragged gradient B{B} Hq{Hq} Sq{Sq} q{qbs}", flush=True)

    def grads(do):
        return torch.autograd.grad(fba.flex_block_attn_func(q, k, v, qbs, kbs, m), (q, k, v), do)

    want = grads(do)
    off = torch.empty(do.numel() + 1, dtype=do.dtype, device=gpu)[1:].view(do.shape).copy_(do)
    assert off.data_ptr() % 16 != 0
    for other in (off, do.transpose(2, 3).contiguous().transpose(2, 3)):
        assert all(torch.equal(a, b) for a, b in zip(grads(other), want))
    ones = grads(torch.ones_like(do))
    assert all(torch.equal(a, b) for a, b in zip(grads(torch.ones((), dtype=do.dtype, device=gpu).expand_as(do)), ones))
    o = fba.flex_block_attn_func(q, k, v, qbs, kbs, m)
    assert all(torch.equal(a, b) for a, b in zip(torch.autograd.grad(o.float(), (q, k, v), do.float()), want))
    other = torch.ones((), device=gpu, requires_grad=True)
    o = fba.flex_block_attn_func(q, k, v, qbs, kbs, m)
    assert torch.autograd.grad(other * 2, (q,), allow_unused=True)[0] is None and o.shape == q.shape


@pytest.mark.parametrize("H,Sq,Skv", [
    (2, 1984, 1984),   # backward from the mask
    (1, 176, 320),
    (8, 3136, 3136),   # lists
])
def test_inputs_written_to_before_backward(gpu, H, Sq, Skv):
    """Lengths that are no whole tiles: backward reads copies of q, k, v, so they may be written to after the call."""
    import flex_block_attn_amd as fba

    g = torch.Generator().manual_seed(Sq + Skv)
    q, do = (torch.randn((1, H, Sq, 128), generator=g).to(torch.bfloat16).to(gpu) for _ in range(2))
    k, v = (torch.randn((1, H, Skv, 128), generator=g).to(torch.bfloat16).to(gpu) for _ in range(2))
    m = (torch.rand((Sq // 16, Skv // 64), generator=g) < 0.4).to(gpu)
    grads = []
    for write in (False, True):
        x = [t.clone().requires_grad_(True) for t in (q, k, v)]
        o = fba.flex_block_attn_func(*x, 16, 64, m)
        if write:
            with torch.no_grad():
                for t in x:
                    t.fill_(3.0)
        grads.append(torch.autograd.grad(o, x, do))
    for a, b in zip(*grads):
        assert torch.equal(a, b)
