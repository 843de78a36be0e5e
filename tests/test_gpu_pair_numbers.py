"""Numbers of the listed pairs and their values at the head boundaries (fba_pair_slots_bounds, fba_tile_slots_bounds): in one launch where
few rows lie in front of a head, in two beyond that.  One entry, a work-group's worth and one more, the largest head and the most rows
of the one launch and one more of each, as many work-groups as it may have and more, one mask for all heads, empty heads; the boundaries in device and in pinned host memory.  Exact."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _lists(m):
    from flex_block_attn_amd import compact_block_mask

    return compact_block_mask(m)


def _call(name, *args):
    from flex_block_attn_amd import _lib
    from flex_block_attn_amd.interface import _ptr, _stream

    _lib.call(name, *(_ptr(a) if torch.is_tensor(a) else a for a in args), _stream())
    torch.cuda.synchronize()


@pytest.mark.parametrize("M,nQ,nK,density", [
    (1, 1, 1, 1.0), (1, 1, 1, 0.0), (3, 16, 16, 0.4), (3, 257, 1, 0.5), (1, 7, 2048, 0.3), (1, 7, 2049, 0.3), (8, 5, 2048, 0.2), (129, 3, 127, 0.6), (2, 300, 63, 0.9),
    (5, 540, 180, 0.1), (6, 540, 180, 0.1),
])
@pytest.mark.parametrize("pinned", [False, True])
def test_pair_numbers(gpu, M, nQ, nK, density, pinned):
    g = torch.Generator().manual_seed(M * nQ + nK)
    m = torch.rand((1, M, nQ, nK), generator=g) < density
    m[:, M // 2] = False
    l = _lists(m.to(gpu))
    base = torch.full((M * nK + 1,), -7, dtype=torch.int32, device=gpu)
    slot = torch.full((M, nQ, nK), -7, dtype=torch.int32, device=gpu)
    bounds = torch.full((M + 1,), -7, dtype=torch.int32).pin_memory() if pinned else torch.full((M + 1,), -7, dtype=torch.int32, device=gpu)
    _call("fba_pair_slots_bounds", l.q_cnt, l.q_idx, l.k_cnt, l.k_idx, M, nQ, nK, base, slot, bounds)
    counts = m[0].sum(1).flatten()
    want = torch.cat([torch.zeros(1, dtype=torch.int64), counts.cumsum(0)])
    assert torch.equal(base.cpu().long(), want) and torch.equal(bounds.cpu().long(), want[::nK])
    number = torch.full((M, nQ, nK), -1, dtype=torch.int64)  # of every pair, by position
    h, j, i = m[0].transpose(1, 2).nonzero(as_tuple=True)
    number[h, i, j] = torch.arange(h.numel())
    order = torch.where(m[0], torch.arange(nK).expand_as(m[0]), nK).sort(dim=-1).indices  # selected blocks first, ascending
    listed = torch.arange(nK) < m[0].sum(-1, keepdim=True)
    assert torch.equal(slot.cpu().long(), torch.where(listed, number.gather(-1, order), -1))


def test_boundaries_of_tile_pairs(gpu):
    from flex_block_attn_amd import tile_block_mask

    g = torch.Generator().manual_seed(1)
    m = (torch.rand((1, 3, 24, 12), generator=g) < 0.2).to(gpu)  # 64 x 64 blocks: 12 x 6 tiles
    l = tile_block_mask(m, 64, 64)
    n_qt, n_kt = l.q_cnt.shape[1], l.k_cnt.shape[1]
    i32 = dict(dtype=torch.int32, device=gpu)
    base, bounds = torch.empty((3 * n_kt + 1,), **i32), torch.full((4,), -7, dtype=torch.int32).pin_memory()
    slot, table = torch.empty((3, n_kt, 4 * n_qt), **i32), torch.empty((3, n_qt, n_kt), **i32)
    _call("fba_tile_slots_bounds", l.k_cnt, l.k_idx, 3, n_qt, n_kt, base, slot, table, bounds)
    assert torch.equal(bounds, base[::n_kt].cpu()) and int(bounds[0]) == 0 and int(bounds[3]) == int((table >= 0).sum())
