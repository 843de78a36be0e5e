"""Which key blocks a score-driven mask picks: the top-k of every query block, ties to the lower block, never a score that is NaN or -inf.
Whole-number means, so that scores are exact and full of ties; key blocks around one, four and sixteen score registers per lane (64 blocks
each), more to pick than there are, nothing to pick, a last work-group with one query block.  Exact against a stable sort."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Hq,Hkv,nQ,nK,topk", [
    (1, 1, 1, 1, 1, 1), (1, 2, 1, 9, 63, 5), (1, 1, 1, 8, 64, 64), (2, 2, 2, 7, 65, 16), (1, 1, 1, 17, 256, 3), (1, 1, 1, 5, 257, 16),
    (1, 3, 1, 3, 1024, 100), (1, 1, 1, 3, 1025, 16), (1, 1, 1, 2, 4096, 70), (1, 1, 1, 4, 30, 40), (1, 1, 1, 4, 30, 0),
])
@pytest.mark.parametrize("kind", ["ties", "alike", "special"])
def test_top_blocks(gpu, B, Hq, Hkv, nQ, nK, topk, kind):
    from flex_block_attn_amd.video import ssta_mask_from_means

    g = torch.Generator().manual_seed(nK + topk)
    q, k = (torch.randint(-1, 2, (B, h, n, 128), generator=g).float() for h, n in ((Hq, nQ), (Hkv, nK)))
    if kind == "alike":
        k[:] = k[:, :, :1]
    if kind == "special":
        k[:, :, ::3] = 0.0  # scores of 0
        k[:, :, 1::5, 0] = float("nan")
        k[:, :, 2::7, 0], q[..., 0] = float("-inf"), 1.0
        k[:, :, 4::11, 0] = float("inf")
    score = (q[:, :, :, None] * k.repeat_interleave(Hq // Hkv, 1)[:, :, None]).sum(-1)
    rank = torch.where(score > float("-inf"), score + 0.0, float("-inf")).nan_to_num(nan=float("-inf"), posinf=float("inf"), neginf=float("-inf"))
    order = rank.sort(dim=-1, descending=True, stable=True).indices
    want = torch.zeros(score.shape, dtype=torch.bool).scatter_(-1, order[..., :topk], True) & (rank > float("-inf"))
    got = ssta_mask_from_means(q.to(gpu), k.to(gpu), 128, 128, topk=topk, band=-1, sink_blocks=0)
    assert torch.equal(got.cpu(), want)


@pytest.mark.parametrize("nK", [5, 300, 1100])
def test_a_score_of_minus_zero_ties_with_zero(gpu, nK):
    """A negative product that underflows, added last to sums that are +0, leaves -0: as large as the +0 further on, so the lower block is picked."""
    from flex_block_attn_amd.video import ssta_mask_from_means

    q, k = torch.zeros((1, 1, 1, 128)), torch.zeros((1, 1, nK, 128))
    q[..., 0], q[..., 127] = 1.0, 1e-30
    k[..., 0] = -1.0
    k[0, 0, 1, 0], k[0, 0, 1, 127], k[0, 0, nK - 1, 0] = 0.0, -1e-30, 0.0
    got = ssta_mask_from_means(q.to(gpu), k.to(gpu), 128, 128, topk=1, band=-1, sink_blocks=0)
    assert got.flatten().nonzero().flatten().tolist() == [1]


@pytest.mark.parametrize("nQ,nK", [(9, 63), (5, 300), (3, 1100)])
@pytest.mark.parametrize("offset", [1, 2, 3])
def test_means_at_any_float(gpu, nQ, nK, offset):
    """Means that begin at a float that is no multiple of 16 bytes, as views of a longer buffer do."""
    from flex_block_attn_amd.video import ssta_mask_from_means

    g = torch.Generator().manual_seed(nK)
    q, k = (torch.randn((1, 2, n, 128), generator=g).to(gpu) for n in (nQ, nK))
    moved = []
    for t in (q, k):
        moved.append(torch.empty(t.numel() + 4, device=gpu)[offset:offset + t.numel()].view(t.shape).copy_(t))
        assert moved[-1].data_ptr() % 16 == 4 * offset and moved[-1].is_contiguous()
    want = ssta_mask_from_means(q, k, 128, 128, topk=7)
    assert torch.equal(ssta_mask_from_means(*moved, 128, 128, topk=7), want)
    assert torch.equal(ssta_mask_from_means(moved[0], k, 128, 128, topk=7), want)
