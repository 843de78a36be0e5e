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


@pytest.mark.parametrize("window", [(3.0, 3.0, 3.0), (3.5, 1.2, 5.0), (2**33, 1, 2**33 + 4), (2**31, 3, 2**40), (2**31 - 1, 1, 1), (-1, 3, 3), (float("nan"), 3, 3),
                                    torch.tensor([3, 1, 5]), torch.tensor([3.0, 1.0, 5.0])])
def test_extents_that_are_no_small_whole_numbers(gpu, window):
    """What the mask made of tensors takes, the operator takes, with the same result."""
    import flex_block_attn_amd as fba
    from flex_block_attn_amd import masks, video

    tiles, tile = (2, 3, 4), (1, 4, 4)
    grid = tuple(n * t for n, t in zip(tiles, tile))
    S = grid[0] * grid[1] * grid[2]
    g = torch.Generator().manual_seed(7)
    q, k, v = (torch.randn((1, 2, S, 128), generator=g).to(torch.bfloat16).to(gpu) for _ in range(3))
    base = masks.sta_3d_block_mask(tiles, window).to(gpu)
    want = fba.create_ssta_mask(q, k, 16, 16, topk=0, band=-1, sink_blocks=1, base_mask=base)
    assert torch.equal(video.create_ssta_3d_mask(q, k, grid, tile, window, topk=0), want)
    # the same through the whole operator (key blocks of 64 tokens and more)
    tile = (1, 8, 8)
    grid = tuple(n * t for n, t in zip(tiles, tile))
    q, k, v = (torch.randn((1, 2, grid[0] * grid[1] * grid[2], 128), generator=g).to(torch.bfloat16).to(gpu) for _ in range(3))
    qt, kt, vt = (fba.tile_tokens(x, grid, tile) for x in (q, k, v))
    o = fba.flex_block_attn_func(qt, kt, vt, 64, 64, fba.create_ssta_mask(qt, kt, 64, 64, topk=1, band=-1, sink_blocks=0, base_mask=base))
    assert torch.equal(video.ssta_3d_attention(q, k, v, grid, tile, window, topk=1, sink_blocks=0), fba.untile_tokens(o, grid, tile))


@pytest.mark.parametrize("window", [(3, 3), (3, 3, 3, 3), None, ("3", "3", "3"), torch.tensor([3, 3, 3])])
def test_refused_extents(gpu, window):
    from flex_block_attn_amd import video

    q = torch.randn((1, 1, 2 * 16 * 16, 128), device=gpu).to(torch.bfloat16)
    if isinstance(window, torch.Tensor):
        window = window.to(gpu)
    with pytest.raises((ValueError, TypeError, RuntimeError)):
        video.create_ssta_3d_mask(q, q, (2, 16, 16), (1, 8, 8), window)


def test_outputs_that_enter_nothing(gpu):
    """Only what has a gradient is gathered back: nothing is filled for the means, and inputs whose output enters nothing get no gradient."""
    import flex_block_attn_amd as fba
    from flex_block_attn_amd import video

    grid, tile = (2, 16, 16), (1, 8, 8)
    g = torch.Generator().manual_seed(3)
    q, k, v = (torch.randn((1, 2, 512, 128), generator=g).to(torch.bfloat16).to(gpu).requires_grad_(True) for _ in range(3))
    got = []
    inner = video._gather

    def gather(xs, grid, tile, to_tiles, means=()):
        if not to_tiles:
            got.append(len(xs))
        return inner(xs, grid, tile, to_tiles, means)

    video._gather = gather
    try:
        for used, n in ((0,), 1), ((1, 2), 2), ((0, 1, 2), 3):
            outs = video._TilePermuteAll.apply(q, k, v, grid, tile)
            weights = torch.randn((1, 2, 512, 128), generator=g).to(torch.bfloat16).to(gpu)
            grads = torch.autograd.grad([outs[j] for j in used], (q, k, v), [weights] * len(used), allow_unused=True)
            for j in range(3):
                assert (grads[j] is None) if j not in used else torch.equal(grads[j], fba.untile_tokens(weights, grid, tile))
            assert got.pop() == n and not got
        with torch.profiler.profile() as prof:
            torch.autograd.grad(video._TilePermuteAll.apply(q, k, v, grid, tile)[:3], (q, k, v), [weights] * 3)
        assert not [e.key for e in prof.key_averages() if "zero" in e.key or "fill" in e.key]
    finally:
        video._gather = inner
