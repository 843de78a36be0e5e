"""Calls of the operator under torch's function transforms: what the autograd function refuses stays refused on the native path,
and a traced call is recorded, not baked in."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _inputs(gpu, seed):
    g = torch.Generator().manual_seed(seed)
    return [torch.randn((1, 1, 256, 128), generator=g).to(torch.bfloat16).to(gpu) for _ in range(3)]


def test_forward_mode_is_refused(gpu):
    import flex_block_attn_amd as fba
    from torch.autograd import forward_ad

    q, k, v = _inputs(gpu, 0)
    mask = torch.ones((2, 2), dtype=torch.bool, device=gpu)
    with forward_ad.dual_level():
        with pytest.raises(RuntimeError):
            fba.flex_block_attn_func(forward_ad.make_dual(q, torch.ones_like(q)), k, v, 128, 128, mask)


def test_vmap_is_refused(gpu):
    import flex_block_attn_amd as fba

    q, k, v = (t[None] for t in _inputs(gpu, 1))
    mask = torch.ones((2, 2), dtype=torch.bool, device=gpu)
    with pytest.raises(RuntimeError):
        torch.vmap(lambda a, b, c: fba.flex_block_attn_func(a, b, c, 128, 128, mask))(q, k, v)


def test_traced_call_follows_its_inputs(gpu):
    import flex_block_attn_amd as fba

    mask = torch.ones((2, 2), dtype=torch.bool, device=gpu)

    def f(q, k, v):
        return fba.flex_block_attn_func(q, k, v, 128, 128, mask)

    traced = torch.jit.trace(f, _inputs(gpu, 2), check_trace=False)
    other = _inputs(gpu, 3)
    assert torch.equal(traced(*other), f(*other))


def test_saved_tensor_hooks_see_the_inputs(gpu):
    import flex_block_attn_amd as fba

    q, k, v = (t.requires_grad_(True) for t in _inputs(gpu, 4))
    mask = torch.ones((2, 2), dtype=torch.bool, device=gpu)
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t.shape) or t.cpu(), lambda t: t.to(gpu)):
        o = fba.flex_block_attn_func(q, k, v, 128, 128, mask)
    got = torch.autograd.grad(o, (q, k, v), torch.ones_like(o))
    assert len(packed) == 5  # q, k, v, o, lse
    want = torch.autograd.grad(fba.flex_block_attn_func(q, k, v, 128, 128, mask), (q, k, v), torch.ones_like(o))
    assert all(torch.equal(a, b) for a, b in zip(got, want))
