"""What fba_fwd_blocks takes, as the library says it: block sizes, key blocks, rows of lists, and where it works on 64 rows (for 256 compute units).  The operator goes by that,
so a step whose lists are there anyway reads them where it would work on 128 rows."""
import pytest
import torch

TAKEN, LISTS, HALVES = 1, 2, 4


@pytest.mark.parametrize("mask_bh,B,H,Sq,Skv,qbs,kbs,use", [
    (1, 1, 24, 3072, 128 * 256, 128, 128, TAKEN | LISTS),
    (1, 1, 24, 3072, 128 * 257, 128, 128, 0),
    (1, 1, 24, 3072, 64 * 48, 128, 64, 0),
    (1, 1, 24, 3072, 3072, 64, 128, 0),
    (8, 1, 8, 8192, 8192, 128, 128, TAKEN | LISTS),     # 8 x 128 rows
    (8, 1, 8, 8320, 8192, 128, 128, TAKEN),
    (70, 1, 70, 128, 3584, 128, 128, TAKEN | HALVES),   # 70 tiles, lists of 112 steps
    (70, 1, 70, 128, 4096, 128, 128, TAKEN),
    (96, 1, 96, 128, 4736, 128, 128, TAKEN | HALVES),
    (96, 1, 96, 128, 4864, 128, 128, TAKEN),
    (2, 1, 2, 8192, 2048, 128, 128, TAKEN | LISTS | HALVES),  # 128 tiles
    (2, 1, 2, 8320, 2048, 128, 128, TAKEN | LISTS),
])
def test_limits(mask_bh, B, H, Sq, Skv, qbs, kbs, use):
    from flex_block_attn_amd import _lib

    assert _lib.load().fba_fwd_blocks_use(mask_bh, B, H, Sq, Skv, qbs, kbs) == use


@pytest.mark.gpu
@pytest.mark.parametrize("H,Sq,Skv", [(70, 128, 4096), (95, 128, 4736)])
def test_steps_with_lists_read_them(gpu, H, Sq, Skv):
    import flex_block_attn_amd as fba

    g = torch.Generator(device=gpu).manual_seed(H)
    m = torch.rand((1, H, Sq // 128, Skv // 128), generator=g, device=gpu) < 0.6
    m[:, ::5] = False  # lists that differ
    q, k, v = (torch.randn((1, H, S, 128), generator=g, device=gpu).to(torch.bfloat16) for S in (Sq, Skv, Skv))
    want, _ = fba.forward_with_lists(q, k, v, 128, 128, fba.lists_for(m, 128, 128))
    got = fba.flex_block_attn_func(q.requires_grad_(True), k, v, 128, 128, m)
    assert got.requires_grad and torch.equal(got, want)
