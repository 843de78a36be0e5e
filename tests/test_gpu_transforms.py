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


# what a saved-tensor hook may not turn a tensor into, by its place among (q, k, v, o, lse): the kernels read by raw pointer
BAD = {
    "fewer rows": (0, lambda t: t[:, :, :128].contiguous(), ValueError),
    "no batch": (1, lambda t: t[0], ValueError),
    "another type": (2, lambda t: t.float(), TypeError),
    "another type of o": (3, lambda t: t.half(), TypeError),
    "left on the host": (1, lambda t: t.cpu(), ValueError),
    "strided": (0, lambda t: t.transpose(2, 3).contiguous().transpose(2, 3), ValueError),
    "lse in half precision": (4, lambda t: t.half(), TypeError),
    "lse cut short": (4, lambda t: t[:, :, :-1], ValueError),
}


@pytest.mark.parametrize("what", BAD)
def test_unpacked_tensors_are_checked(gpu, what):
    import flex_block_attn_amd as fba

    place, change, error = BAD[what]
    q, k, v = (t.requires_grad_(True) for t in _inputs(gpu, 5))
    mask = torch.ones((2, 2), dtype=torch.bool, device=gpu)
    order = []

    def unpack(packed):
        number, t = packed
        return change(t) if number == place else t

    with torch.autograd.graph.saved_tensors_hooks(lambda t: order.append(0) or (len(order) - 1, t), unpack):
        o = fba.flex_block_attn_func(q, k, v, 128, 128, mask)
    with pytest.raises(error, match="saved"):
        torch.autograd.grad(o, (q, k, v), torch.ones_like(o))


def test_unpacked_output_may_be_strided(gpu):
    import flex_block_attn_amd as fba

    q, k, v = (t.requires_grad_(True) for t in _inputs(gpu, 6))
    mask = torch.ones((2, 2), dtype=torch.bool, device=gpu)
    order = []

    def unpack(packed):
        number, t = packed
        return t.transpose(2, 3).contiguous().transpose(2, 3) if number >= 3 else t

    with torch.autograd.graph.saved_tensors_hooks(lambda t: order.append(0) or (len(order) - 1, t), unpack):
        o = fba.flex_block_attn_func(q, k, v, 128, 128, mask)
    got = torch.autograd.grad(o, (q, k, v), torch.ones_like(o))
    want = torch.autograd.grad(fba.flex_block_attn_func(q, k, v, 128, 128, mask), (q, k, v), torch.ones_like(o))
    assert all(torch.equal(a, b) for a, b in zip(got, want))


class Marked(torch.Tensor):
    """A tensor subclass without semantics of its own."""


@pytest.mark.parametrize("S,bs", [(256, 128), (256, 64), (192, 64)])
def test_tensor_subclasses_keep_their_type(gpu, S, bs):
    """Results have the type that torch's own functions would give them: o that of q, gradients those of their tensors."""
    import flex_block_attn_amd as fba

    g = torch.Generator().manual_seed(S)
    plain = [torch.randn((1, 1, S, 128), generator=g).to(torch.bfloat16).to(gpu) for _ in range(4)]
    mask = torch.ones((S // bs, S // bs), dtype=torch.bool, device=gpu)
    leaves = [t.clone().requires_grad_() for t in plain[:3]]
    want_o = fba.flex_block_attn_func(*leaves, bs, bs, mask)
    want = torch.autograd.grad(want_o, leaves, plain[3])
    assert type(want_o) is torch.Tensor
    for which in ((0, 1, 2), (0,)):
        leaves = [t.clone().as_subclass(Marked).requires_grad_() if i in which else t.clone().requires_grad_() for i, t in enumerate(plain[:3])]
        o = fba.flex_block_attn_func(*leaves, bs, bs, mask)
        got = torch.autograd.grad(o, leaves, plain[3])
        assert type(o) is Marked and torch.equal(o.as_subclass(torch.Tensor), want_o)
        assert all(torch.equal(a.as_subclass(torch.Tensor), b) for a, b in zip(got, want))
        with torch.no_grad():
            assert type(fba.flex_block_attn_func(*leaves, bs, bs, mask)) is Marked
    assert type(fba.flex_block_attn_func(torch.nn.Parameter(plain[0].clone()), plain[1], plain[2], bs, bs, mask)) is torch.Tensor


@pytest.mark.parametrize("transform", ["grad", "vjp", "vmap"])
def test_function_transforms_are_refused_with_the_reason(gpu, transform):
    import flex_block_attn_amd as fba

    q, k, v = _inputs(gpu, 7)
    mask = torch.ones((2, 2), dtype=torch.bool, device=gpu)
    call = lambda x: fba.flex_block_attn_func(x, k, v, 128, 128, mask)
    with pytest.raises(RuntimeError, match="functorch transforms"):
        if transform == "grad":
            torch.func.grad(lambda x: call(x).float().sum())(q)
        elif transform == "vjp":
            torch.func.vjp(call, q)
        else:
            torch.vmap(call)(q[None])
