"""Raster to tile order for q, k, v in one launch with the tile means on the way, and the sliding window inside the mask kernel:
bit for bit what the single steps give.  Tiles of 64 rows to the largest that fit the kernel's table, smaller and larger ones (single
steps again), remainders of 16 and 48 rows, grouped heads, batches; windows wider than the grid, even ones, asymmetric grids."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Hq,Hkv,grid,tile", [
    (1, 2, 2, (6, 8, 16), (6, 8, 8)),
    (2, 4, 2, (4, 24, 16), (2, 8, 8)),       # 128 rows
    (1, 3, 1, (2, 8, 12), (1, 8, 4)),        # 32 rows: single steps
    (1, 1, 1, (4, 8, 12), (2, 8, 4)),        # 64 rows
    (1, 2, 1, (6, 20, 12), (2, 10, 4)),      # 80 rows: 64 and a remainder
    (1, 1, 1, (8, 16, 32), (8, 16, 16)),     # 2048 rows: the whole table
    (1, 1, 1, (8, 32, 16), (8, 32, 16)),     # 4096 rows, one tile: single steps
])
def test_gather_is_the_single_steps(gpu, B, Hq, Hkv, grid, tile):
    import flex_block_attn_amd as fba
    from flex_block_attn_amd import video

    S, block = grid[0] * grid[1] * grid[2], tile[0] * tile[1] * tile[2]
    g = torch.Generator().manual_seed(S + block)
    q = torch.randn((B, Hq, S, 128), generator=g).to(torch.bfloat16).to(gpu)
    k, v = (torch.randn((B, Hkv, S, 128), generator=g).to(torch.bfloat16).to(gpu) for _ in range(2))
    print(f"gather B{B} Hq{Hq} Hkv{Hkv} {grid} {tile}", flush=True)
    ins = [t.clone().requires_grad_(True) for t in (q, k, v)]
    *tiled, q_mean, k_mean = video._TilePermuteAll.apply(*ins, grid, tile)
    for t, x in zip(tiled, (q, k, v)):
        assert torch.equal(t, fba.tile_tokens(x, grid, tile))
    assert torch.equal(q_mean, fba.block_mean(tiled[0].detach(), block)) and torch.equal(k_mean, fba.block_mean(tiled[1].detach(), block))
    assert not q_mean.requires_grad and not k_mean.requires_grad
    grads = torch.autograd.grad(tiled, ins, [t.detach().flip(2) for t in tiled])
    for got, t in zip(grads, tiled):
        assert torch.equal(got, fba.untile_tokens(t.detach().flip(2).contiguous(), grid, tile))
    only, = torch.autograd.grad(video._TilePermuteAll.apply(q, ins[1], v, grid, tile)[1], ins[1], tiled[1].detach())
    assert torch.equal(only, k)


@pytest.mark.parametrize("tiles,window", [((3, 4, 5), (3, 3, 3)), ((2, 3, 7), (5, 1, 3)), ((1, 1, 70), (1, 3, 5)), ((4, 2, 3), (2, 4, 1)), ((5, 6, 10), (3, 3, 3))])
@pytest.mark.parametrize("topk,sink", [(0, 0), (3, 1)])
def test_window_in_the_mask_kernel(gpu, tiles, window, topk, sink):
    import flex_block_attn_amd as fba
    from flex_block_attn_amd import masks, video

    n = tiles[0] * tiles[1] * tiles[2]
    g = torch.Generator().manual_seed(n)
    q_mean, k_mean = torch.randn((2, 4, n, 128), generator=g).to(gpu), torch.randn((2, 2, n, 128), generator=g).to(gpu)
    base = masks.sta_3d_block_mask(tiles, window).to(gpu)
    want = video.ssta_mask_from_means(q_mean, k_mean, 1, 1, topk, -1, sink, base)
    got = video._ssta_3d_mask_from_means(q_mean, k_mean, tiles, (1, 1, 1), window, topk, sink)
    assert torch.equal(got, want)
    if topk == 0 and sink == 0:
        assert torch.equal(got, base.expand_as(got))
