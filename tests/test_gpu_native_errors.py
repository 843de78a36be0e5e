"""What the native host path raises: the library's error codes as FbaError, from forward and from backward (where the exception
crosses the autograd engine) alike."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _misaligned(t):
    """The values of `t` in memory that starts two bytes behind a 16-byte boundary, contiguous."""
    buffer = torch.empty((t.numel() + 8,), dtype=t.dtype, device=t.device)
    return buffer[1: 1 + t.numel()].view(t.shape).copy_(t)


def _case(gpu, S, qbs, kbs):
    g = torch.Generator().manual_seed(S)
    q, k, v = (torch.randn((1, 2, S, 128), generator=g).to(torch.bfloat16).to(gpu).requires_grad_(True) for _ in range(3))
    return q, k, v, torch.ones((S // qbs, S // kbs), dtype=torch.bool, device=gpu)


@pytest.mark.parametrize("S,qbs,kbs,dense", [(256, 128, 128, True), (256, 64, 64, True), (256, 128, 128, False), (256, 64, 64, False)])
def test_backward_raises_the_library_error(gpu, monkeypatch, S, qbs, kbs, dense):
    import flex_block_attn_amd as fba
    from flex_block_attn_amd import _lib, interface

    if not dense:
        monkeypatch.setattr(interface, "DS_WORKSPACE_LIMIT_GIB", 0.0)
    q, k, v, mask = _case(gpu, S, qbs, kbs)
    o = fba.flex_block_attn_func(q, k, v, qbs, kbs, mask)
    with pytest.raises(_lib.FbaError, match="not 16-byte aligned") as raised:
        torch.autograd.grad(o, (q, k, v), _misaligned(torch.ones_like(o)))
    assert raised.value.code == _lib.FBA_ERR_INVALID and "d_o" in raised.value.message


def test_forward_raises_the_library_error(gpu):
    import flex_block_attn_amd as fba
    from flex_block_attn_amd import _lib

    q, k, v, mask = _case(gpu, 256, 128, 128)
    lists = fba.lists_for(mask, 128, 128)
    for call in (lambda: fba.flex_block_attn_func(_misaligned(q.detach()), k, v, 128, 128, mask),
                 lambda: fba.forward_with_lists(_misaligned(q.detach()), k, v, 128, 128, lists)):
        with pytest.raises(_lib.FbaError, match="q is not 16-byte aligned") as raised:
            call()
        assert raised.value.code == _lib.FBA_ERR_INVALID
