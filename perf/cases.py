"""The work that users of this package have it do, as cases that can be timed and compared: attention forward and training
steps under block masks, from one short head to the longest video latents, through the public entry points.

A case is a dict of plain values:
  mask        how the block mask comes about: "random" (every query block keeps `keep` key blocks of its own choice),
              "full", "tiles" (static sliding window over a `grid` of tiles), "scores" (top-k by block means, built from
              q and k in every pass) or "latent" (`video.ssta_3d_attention` on tokens in raster order of `grid`)
  per_head    whether every (batch, head) has a mask of its own ("random" only)
  batch, heads, kv_heads, q_len, kv_len, q_block, kv_block
  step        True: forward and backward, False: forward alone
"""
import math

import torch

import flex_block_attn_amd as fba
from flex_block_attn_amd import masks, video

DIM = 128
TILE = (6, 8, 8)  # tokens of one tile of a video latent: 384


def _case(name, mask, heads, q_len, q_block, *, kv_heads=0, kv_len=0, kv_block=0, batch=1, keep=0, per_head=False, step=False, grid="", window="", topk=0):
    case = {"mask": mask, "per_head": per_head, "batch": batch, "heads": heads, "kv_heads": kv_heads or heads, "q_len": q_len, "kv_len": kv_len or q_len,
            "q_block": q_block, "kv_block": kv_block or q_block, "keep": keep, "grid": grid, "window": window, "topk": topk, "step": step}
    return dict(case, name=name) if name else case


def listed():
    return [
        # The smallest call of the operator: one head, six blocks, no gradient.  Launches and host work are all of it.
        _case("short_forward", "random", 1, 768, 128, keep=3),
        # A small layer's training step (two heads of 1536 tokens, 384-token blocks, one mask for all heads).
        _case("small_step", "random", 2, 1536, 384, keep=2, step=True),
        # Grouped kv heads and a batch at a text-like length with fine-grained blocks, and a length that is no whole
        # number of 128-row tiles (49 key blocks of 64).
        _case("ragged_fine_step", "random", 8, 3136, 16, kv_heads=2, kv_block=64, batch=2, keep=12, per_head=True, step=True),
        # Grouped-query layer with 128-token blocks, a quarter of them kept.
        _case("grouped_step", "random", 16, 8192, 128, kv_heads=4, batch=2, keep=16, per_head=True, step=True),
        # One row of the operator's published benchmark sweep: a single head, 60 % of the blocks kept.
        _case("one_head_step", "random", 1, 30720, 384, keep=48, step=True),
        # A chunk of new queries against a long cache of keys (cross lengths, grouped heads): few query tiles, long lists.
        _case("chunk_forward", "random", 24, 768, 128, kv_heads=6, kv_len=30720, kv_block=128, keep=96, per_head=True),
        # Dense attention of a middle-sized layer, inference.
        _case("full_forward", "full", 24, 11520, 384),
        # The benchmark's default workload: 24 heads, 40 % of the blocks kept, a mask per head, training.
        _case("random_step", "random", 24, 30720, 384, keep=32, per_head=True, step=True),
        # The same density in 64-token blocks, which are finer than the kernels' tiles.
        _case("fine_step", "random", 24, 30720, 64, keep=192, per_head=True, step=True),
        # Score-driven masks with a query block smaller than the key block, built from q and k in every step.
        _case("score_mask_step", "scores", 24, 69120, 128, kv_block=384, topk=16, step=True),
        # Inference on a video latent in raster order: permutation, mask, attention, permutation back.
        _case("latent_forward", "latent", 24, 69120, 384, grid="18x48x80", window="3x3x3", topk=16),
        # Training on the longest latent: sliding 3 x 3 x 3 window over 5 x 6 x 10 tiles.
        _case("sliding_tile_step", "tiles", 24, 115200, 384, grid="5x6x10", window="3x3x3", step=True),
    ]


def _dims(text):
    return tuple(int(n) for n in text.split("x"))


def _log_uniform(rng, low, high):
    return math.exp(rng.uniform(math.log(low), math.log(high)))


def _draw_any(rng):
    kind = rng.choice(["random", "random", "random", "fine", "fine", "cross", "full", "scores", "latent", "tiles"])
    step = rng.random() < 0.6
    group = rng.choice([1, 1, 1, 2, 4])
    kv_heads = max(1, round(_log_uniform(rng, 1, 24 / group)))
    heads = kv_heads * group
    batch = rng.choice([1, 1, 1, 2])
    per_head = rng.random() < 0.7
    if kind in ("random", "full"):
        q_block, kv_block = rng.choice([(128, 128), (128, 384), (256, 256), (256, 128), (384, 384), (384, 384), (512, 512)])
        unit = max(q_block, kv_block)
        length = unit * max(1, round(_log_uniform(rng, 768, 61440) / unit))
        keep = max(1, round(length // kv_block * rng.uniform(0.1, 0.9)))
        return _case("", kind, heads, length, q_block, kv_heads=kv_heads, kv_block=kv_block, batch=batch, step=step, keep=keep if kind == "random" else 0,
                     per_head=per_head and kind == "random")
    if kind == "fine":
        q_block, kv_block = rng.choice([(16, 64), (16, 128), (32, 64), (64, 64), (64, 64), (64, 128), (128, 64), (64, 192), (192, 192), (64, 384)])
        unit = max(q_block, kv_block)
        length = unit * max(1, round(_log_uniform(rng, 768, 30720) / unit))
        keep = max(1, round(length // kv_block * rng.uniform(0.1, 0.6)))
        return _case("", "random", heads, length, q_block, kv_heads=kv_heads, kv_block=kv_block, batch=batch, step=step, keep=keep, per_head=per_head)
    if kind == "cross":
        q_len, kv_len = 128 * max(1, round(_log_uniform(rng, 128, 3072) / 128)), 128 * round(_log_uniform(rng, 3840, 61440) / 128)
        return _case("", "random", heads, q_len, 128, kv_heads=kv_heads, kv_len=kv_len, batch=batch, step=step, keep=max(1, round(kv_len // 128 * rng.uniform(0.1, 0.9))),
                     per_head=per_head)
    if kind == "scores":
        length = 384 * round(_log_uniform(rng, 7680, 69120) / 384)
        return _case("", "scores", heads, length, 128, kv_heads=kv_heads, kv_block=384, topk=rng.randint(4, 16), step=step)
    tiles = (rng.randint(1, 5), rng.randint(2, 6), rng.randint(2, 10))
    length = 384 * math.prod(tiles)
    window = "x".join(str(rng.choice([1, 3, 3])) for _ in tiles)
    if kind == "tiles":
        return _case("", "tiles", heads, length, 384, kv_heads=kv_heads, grid="x".join(map(str, tiles)), window=window, step=step)
    grid = "x".join(str(n * t) for n, t in zip(tiles, TILE))
    return _case("", "latent", heads, length, 384, kv_heads=kv_heads, grid=grid, window=window, topk=rng.randint(1, min(16, math.prod(tiles))), step=step)


def draw(rng):
    most = max(work(c)["flops"] for c in listed())
    while True:
        case = _draw_any(rng)
        # query blocks of 16 or 32 rows with a choice of their own make a 128-row tile walk the union of theirs
        spread = 128 / min(128, case["q_block"])
        if work(case)["flops"] * min(spread, case["kv_len"] / (case["kv_block"] * max(1, case["keep"]))) <= most:
            return case


def _base_mask(case):
    tiles = _dims(case["grid"])
    if case["mask"] == "latent":
        tiles = tuple(n // t for n, t in zip(tiles, TILE))
    return masks.sta_3d_block_mask(tiles, _dims(case["window"]))


def _selected_pairs(case):
    """Selected block pairs over all heads; for masks by score what independent scores give on average."""
    nq, nk = case["q_len"] // case["q_block"], case["kv_len"] // case["kv_block"]
    heads = case["batch"] * case["heads"]
    if case["mask"] == "random":
        return heads * nq * case["keep"]
    if case["mask"] == "full":
        return heads * nq * nk
    if case["mask"] == "tiles":
        return heads * int(_base_mask(case).sum())
    if case["mask"] == "latent":
        always = _base_mask(case)
    else:
        own = torch.arange(nq)[:, None] * case["q_block"] // case["kv_block"]
        always = (own - torch.arange(nk)[None, :]).abs() <= 1
    always[:, 0] = True  # the sink block
    fixed = int(always.sum())
    return heads * (fixed + (nq * nk - fixed) * min(1.0, case["topk"] / nk))


def _random_mask(case, gen):
    """Every query block keeps `keep` key blocks, its own neighbourhood among them."""
    nq, nk = case["q_len"] // case["q_block"], case["kv_len"] // case["kv_block"]
    shape = (case["batch"], case["heads"], nq, nk) if case["per_head"] else (nq, nk)
    score = torch.rand(shape, generator=gen, device="cuda")
    rows = torch.arange(nq, device="cuda")
    score[..., rows, rows * nk // nq] = 2.0
    mask = torch.zeros(shape, dtype=torch.bool, device="cuda")
    return mask.scatter_(-1, score.topk(case["keep"], dim=-1).indices, True)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def normal(heads, length):
        return torch.randn((case["batch"], heads, length, DIM), generator=gen, device="cuda", dtype=torch.bfloat16)

    q = normal(case["heads"], case["q_len"])
    k, v = (normal(case["kv_heads"], case["kv_len"]) for _ in range(2))
    state = {"case": case, "q": q, "k": k, "v": v}
    if case["step"]:
        for t in (q, k, v):
            t.requires_grad_(True)
        state["do"] = normal(case["heads"], case["q_len"])
    if case["mask"] == "random":
        state["mask"] = _random_mask(case, gen)
    elif case["mask"] == "full":
        state["mask"] = masks.full_block_mask(case["q_len"] // case["q_block"], case["kv_len"] // case["kv_block"], device="cuda")
    elif case["mask"] == "tiles":
        state["mask"] = _base_mask(case).cuda()
    return state


def run(state):
    case, q, k, v = state["case"], state["q"], state["k"], state["v"]
    with torch.set_grad_enabled(case["step"]):
        if case["mask"] == "latent":
            o = video.ssta_3d_attention(q, k, v, _dims(case["grid"]), TILE, _dims(case["window"]), case["topk"])
        elif case["mask"] == "scores":
            mask = fba.create_ssta_mask(q.detach(), k.detach(), case["q_block"], case["kv_block"], topk=case["topk"])
            o = fba.flex_block_attn_func(q, k, v, case["q_block"], case["kv_block"], mask)
        else:
            o = fba.flex_block_attn_func(q, k, v, case["q_block"], case["kv_block"], state["mask"])
    if not case["step"]:
        return o
    dq, dk, dv = torch.autograd.grad(o, (q, k, v), state["do"])
    return {"o": o.detach(), "dq": dq, "dk": dk, "dv": dv}


def work(case):
    """Every tensor moved once (q, k, v and o; with the backward pass dO and the three gradients too) and the mask; two
    products per selected pair in the forward pass and five in the backward pass."""
    q = case["batch"] * case["heads"] * case["q_len"] * DIM * 2
    kv = case["batch"] * case["kv_heads"] * case["kv_len"] * DIM * 2
    mask = (case["q_len"] // case["q_block"]) * (case["kv_len"] // case["kv_block"]) * (case["batch"] * case["heads"] if case["per_head"] else 1)
    pair = case["q_block"] * case["kv_block"] * DIM
    step = case["step"]
    return {"bytes": float((4 if step else 2) * (q + kv) + mask), "flops": float((14 if step else 4) * pair * _selected_pairs(case))}


def tolerance(case):
    """bf16 results of fp32 sums, with P and dS rounded to bf16 for the second products.  Against the dense formula on float32
    inputs every output is off by 2.2e-3 to 2.4e-3 (2-norm) and a single value by at most 1.8e-2 of the larger of its own size
    and the root mean square; the bounds are four times that."""
    return {"rel": 1e-2, "max": 0.07}
