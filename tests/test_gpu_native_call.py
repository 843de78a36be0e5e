"""The native call path where a program uses more than one backward pass, stream or thread, and where memory is short."""
import threading

import pytest
import torch

pytestmark = pytest.mark.gpu


def _step(gpu, S, qbs, kbs, seed, H=2):
    """(q, k, v, do, function that runs forward) of a step on a mask of its own."""
    import flex_block_attn_amd as fba

    g = torch.Generator().manual_seed(seed)
    q, k, v, do = (torch.randn((1, H, S, 128), generator=g).to(torch.bfloat16).to(gpu) for _ in range(4))
    for t in (q, k, v):
        t.requires_grad_(True)
    mask = (torch.rand((1, H, S // qbs, S // kbs), generator=g) < 0.5).to(gpu)
    return q, k, v, do, lambda: fba.flex_block_attn_func(q, k, v, qbs, kbs, mask)


SIZES = [(768, 128, 128), (832, 64, 64)]  # block lists; tile lists with a padded length


@pytest.mark.parametrize("S,qbs,kbs", SIZES)
@pytest.mark.parametrize("dense", [True, False])
def test_backward_twice(gpu, monkeypatch, S, qbs, kbs, dense):
    from flex_block_attn_amd import interface

    if not dense:  # no room for all pairs, enough for the selected ones
        monkeypatch.setattr(interface, "DS_WORKSPACE_LIMIT_GIB", 0.9 * 2 * 2 * 768 ** 2 / 2 ** 30)
    q, k, v, do, forward = _step(gpu, S, qbs, kbs, 1)
    o = forward()
    first = torch.autograd.grad(o, (q, k, v), do, retain_graph=True)
    second = torch.autograd.grad(o, (q, k, v), do)
    assert all(torch.equal(a, b) for a, b in zip(first, second))
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(o, (q, k, v), do)


@pytest.mark.parametrize("S,qbs,kbs", SIZES)
def test_step_on_a_side_stream(gpu, S, qbs, kbs):
    q, k, v, do, forward = _step(gpu, S, qbs, kbs, 2)
    o = forward()
    want = (o, *torch.autograd.grad(o, (q, k, v), do))
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        o = forward()
        got = (o, *torch.autograd.grad(o, (q, k, v), do))
    torch.cuda.current_stream().wait_stream(side)
    assert all(torch.equal(a, b) for a, b in zip(got, want))


def test_steps_in_two_threads(gpu):
    steps = [_step(gpu, *SIZES[i], 3 + i) for i in range(2)]
    want, got = [None, None], [[], []]

    def once(i):
        q, k, v, do, forward = steps[i]
        o = forward()
        return (o.detach(), *torch.autograd.grad(o, (q, k, v), do))

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(8):
                got[i].append(once(i))
        torch.cuda.current_stream().synchronize()

    for i in range(2):
        want[i] = once(i)
    torch.cuda.synchronize()
    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    for i in range(2):
        assert len(got[i]) == 8 and all(torch.equal(a, b) for r in got[i] for a, b in zip(r, want[i]))


def test_backward_without_room_for_a_workspace(gpu):
    """The dS workspace (0.5 GB here) cannot be allocated: dQ recomputes S and dP."""
    from flex_block_attn_amd import interface

    S, H = 5632, 8
    q, k, v, do, forward = _step(gpu, S, 128, 128, 5, H)
    assert interface.dense_ds_fits(q, k)
    want = torch.autograd.grad(forward(), (q, k, v), do)
    o = forward()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    room = torch.cuda.memory_reserved() + 2 ** 28
    try:
        torch.cuda.set_per_process_memory_fraction(room / torch.cuda.get_device_properties(gpu).total_memory, gpu)
        torch.cuda.reset_peak_memory_stats()
        got = torch.autograd.grad(o, (q, k, v), do)
        torch.cuda.synchronize()
        assert torch.cuda.max_memory_reserved() <= room
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0, gpu)
    for a, b in zip(got, want):  # bf16 rounding of dS on one path only
        assert ((a.float() - b.float()).norm() / b.float().norm()).item() <= 1e-2
