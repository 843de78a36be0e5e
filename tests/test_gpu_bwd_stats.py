"""Backward statistics at the number of rows from which four rows go to 16 lanes, one row short of it and with remainders.  Against float64."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


@pytest.mark.parametrize("rows", [1, 63, 131071, 131072, 131088, 131137, 262143])
def test_backward_statistics(gpu, rows):
    from flex_block_attn_amd import _lib

    g = torch.Generator(device=gpu).manual_seed(rows)
    o, do = (torch.randn((rows, 128), generator=g, device=gpu, dtype=torch.bfloat16) for _ in range(2))
    lse = torch.randn((rows,), generator=g, device=gpu)
    stats = torch.full((2 * rows + 64,), 7.0, device=gpu)
    _lib.call("fba_bwd_stats", _ptr(o), _ptr(do), _ptr(lse), _ptr(stats), rows, 128, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    delta = (o.double() * do.double()).sum(-1)
    # 128 products, exact in fp32, summed in fp32: 2^-24 of the sum of their sizes for each of the 11 additions on the longest way
    bound = 11 * 2.0**-24 * (o.double() * do.double()).abs().sum(-1)
    assert torch.equal(stats[:rows], lse * 1.4426950408889634)
    assert bool(((stats[rows : 2 * rows].double() + delta).abs() <= bound).all())
    assert bool((stats[2 * rows :] == 7.0).all())
