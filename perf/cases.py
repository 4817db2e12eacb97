"""What users of this framework have it do, as cases that can be timed and compared.

A case names one use of the public entry points with its sizes: `prepare` makes what the user's program has in hand
(q, k, v, masks, permutation plans on the GPU), `run` is one pass as such a program makes it, `work` the bytes and
operations that no implementation can do without, `tolerance` what the data types allow.

Kinds of use:
  forward   flash_attention_custom_mask with a block mask the program keeps (one mask for every layer and step)
  dynamic   the same with a block mask that is new in every call (chosen from block scores, per head)
  dense_in  the block mask comes as a dense N x N bool tensor and is reduced in the call
  lse       flash_attention_custom_mask_lse with results in fp32 (partial results that the caller merges)
  train     forward and gradients through autograd, block mask
  token     forward and gradients through autograd, elementwise N x N mask (causal or sliding window)
  reorder   the token reorder around attention on video tokens: q, k, v before it, the result after it
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.abspath("customize-block-sparse-attention-with-triton_amd"))
import fa2_custom_mask as fm  # noqa: E402

TILE = 64
DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16}
COST_MAX = 1.0e12        # operations of the largest drawn case
MASK_BYTES_MAX = 320e6   # of a dense N x N mask


def _attn(name, kind, B, H, N, D, dtype, mask, keep, per_head=False):
    c = {"kind": kind, "B": B, "H": H, "N": N, "D": D, "dtype": dtype, "mask": mask, "keep": keep, "per_head": per_head}
    return dict(c, name=name) if name else c


def _reorder(name, H, frames, height, width, text, D, dtype):
    c = {"kind": "reorder", "H": H, "frames": frames, "height": height, "width": width, "text": text, "D": D, "dtype": dtype}
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest benchmark configuration: one short head, latency of a call
        _attn("forward_1k", "forward", 1, 1, 1024, 64, "f16", "uniform", 0.5),
        # a dense tile-constant mask on the way in, its reduction and the lists part of the call
        _attn("dense_in_6400", "dense_in", 1, 1, 6400, 64, "f16", "uniform", 0.1),
        # one long sparse head, mask kept: what sparsity has to pay back
        _attn("forward_17536_sparse", "forward", 1, 1, 17536, 64, "f16", "uniform", 0.1),
        # the reference script's eight heads, every tile kept
        _attn("forward_17536_full_8_heads", "forward", 1, 8, 17536, 64, "f16", "uniform", 1.0),
        # the reference script as it is: a mask per head, preprocessing in every call
        _attn("dynamic_17536_8_heads", "dynamic", 1, 8, 17536, 64, "f16", "uniform", 0.1, True),
        # the longest benchmark sequence, block-causal
        _attn("forward_32000_causal", "forward", 1, 1, 32000, 64, "f16", "causal", 1.0),
        # a video layer: 226 text + 13 x 30 x 45 image tokens (not whole tiles), 48 heads with a mask each
        _attn("forward_video_48_heads", "forward", 1, 48, 17776, 64, "bf16", "uniform", 0.2, True),
        # the largest head dimension, results in fp32 with their logsumexp
        _attn("lse_4096_d256", "lse", 1, 16, 4096, 256, "bf16", "causal", 0.5),
        # a training step of a long-context layer
        _attn("train_8192_d128", "train", 2, 16, 8192, 128, "bf16", "causal", 0.25),
        # a short training step with a ragged length: launches and host work count
        _attn("train_777", "train", 2, 4, 777, 64, "f16", "uniform", 0.6),
        # a sliding window of tokens, which cuts through tiles, ragged length
        _attn("token_window_4000_d128", "token", 1, 8, 4000, 128, "bf16", "window", 0.25),
        # the reorder before and after the video layer's attention
        _reorder("reorder_video_48_heads", 48, 13, 30, 45, 226, 64, "bf16"),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _length(rng, lo, hi):
    n = int(_log(rng, lo, hi))
    return n if rng.random() < 0.5 else max(TILE, n // TILE * TILE)


def draw(rng):
    kind = rng.choice(["forward", "forward", "forward", "dynamic", "dense_in", "lse", "train", "train", "token", "reorder"])
    dtype = rng.choice(["f16", "bf16"])
    if kind == "reorder":
        return _reorder(None, rng.randint(4, 48), rng.randint(3, 13), rng.randint(10, 30), rng.randint(16, 45),
                        rng.choice([0, 77, 226]), rng.choice([64, 64, 128]), dtype)
    D = rng.choice([64, 64, 64, 128, 128, 256])
    B = rng.choice([1, 1, 1, 2])
    H = max(1, round(_log(rng, 1, 48 if kind in ("forward", "dynamic") else 16)))
    mask = rng.choice(["uniform", "uniform", "causal"])
    keep = rng.choice([1.0, round(_log(rng, 0.05, 1.0), 3), round(_log(rng, 0.05, 1.0), 3)])
    if kind in ("forward", "dynamic", "lse"):
        N = _length(rng, 256, 32000)
    elif kind == "dense_in":
        N = max(512, int(_log(rng, 512, 17536)) // TILE * TILE)
    else:
        N = _length(rng, 256, 8192)
    if kind == "token":
        mask, keep = rng.choice([("window", round(rng.uniform(0.1, 0.6), 3)), ("causal", 1.0)])
    case = _attn(None, kind, B, H, N, D, dtype, mask, keep, kind == "dynamic" or (kind == "forward" and rng.random() < 0.3))
    while work(case)["flops"] > COST_MAX or (kind in ("dense_in", "token") and case["N"] ** 2 > MASK_BYTES_MAX):
        if case["H"] > 1:
            case["H"] = case["H"] // 2
        elif case["B"] > 1:
            case["B"] = 1
        else:
            case["N"] = max(TILE, case["N"] * 3 // 4)
            if kind == "dense_in":
                case["N"] = max(512, case["N"] // TILE * TILE)
    return case


def _randn(g, dtype, *shape):
    return torch.randn(*shape, generator=g, device="cuda").to(dtype)


def _block_scores(case, g):
    """Scores in [0, 1) per block; a block is kept where its score is below `keep`.  Blocks on the diagonal score 0,
    blocks above it (causal) 2."""
    nb = -(-case["N"] // TILE)
    b, h = (case["B"], case["H"]) if case["per_head"] else (1, 1)
    s = torch.rand(b, h, nb, nb, generator=g, device="cuda")
    if case["mask"] == "causal":
        s = s.masked_fill(torch.ones(nb, nb, dtype=torch.bool, device="cuda").triu(1), 2.0)
    s.diagonal(dim1=2, dim2=3).zero_()
    return s


def _window(case):
    """Keys a token sees: itself and the ones before it, at most this many."""
    return case["N"] if case["mask"] == "causal" else max(1, int(case["N"] * case["keep"]))


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    dtype = DTYPES[case["dtype"]]
    if case["kind"] == "reorder":
        T = case["text"] + case["frames"] * case["height"] * case["width"]
        q, k, v, o = (_randn(g, dtype, 1, case["H"], T, case["D"]) for _ in range(4))
        plan = {"permute": [torch.randint(0, 6, (case["H"],), generator=g, device="cuda")]}
        return {"case": case, "q": q, "k": k, "v": v, "o": o, "plan": plan}
    shape = (case["B"], case["H"], case["N"], case["D"])
    q, k, v, do = (_randn(g, dtype, *shape) for _ in range(4))
    state = {"case": case, "q": q, "k": k, "v": v, "sm_scale": case["D"] ** -0.5}
    if case["kind"] == "token":
        i = torch.arange(case["N"], device="cuda")
        d = i[:, None] - i[None, :]
        state["mask"] = ((d >= 0) & (d < _window(case)))[None, None]
    else:
        scores = _block_scores(case, g)
        if case["kind"] == "dynamic":
            state["scores"] = scores
        else:
            state["mask"] = scores < case["keep"]
        if case["kind"] == "dense_in":
            state["mask"] = state["mask"].repeat_interleave(TILE, 2).repeat_interleave(TILE, 3)
    if case["kind"] in ("train", "token"):
        state["do"] = do
        for x in (q, k, v):
            x.requires_grad_(True)
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "reorder":
        size = {"F": case["frames"], "H": case["height"], "W": case["width"], "n_text_tokens": case["text"]}
        q, k, v = fm.permute_qkv_triton(state["q"], state["k"], state["v"], state["plan"], 0, **size)
        return q, k, v, fm.inv_permute_attn_triton(state["o"], state["plan"], 0, **size)
    q, k, v, sm_scale = state["q"], state["k"], state["v"], state["sm_scale"]
    if kind == "forward":
        return fm.flash_attention_custom_mask(q, k, v, state["mask"], sm_scale)
    if kind == "dynamic":
        return fm.flash_attention_custom_mask(q, k, v, state["scores"] < case["keep"], sm_scale)
    if kind == "dense_in":
        return fm.flash_attention_custom_mask(q, k, v, fm.reduce_dense_mask(state["mask"]), sm_scale)
    if kind == "lse":
        return fm.flash_attention_custom_mask_lse(q, k, v, state["mask"], sm_scale, out_fp32=True)
    o = fm.flash_attention_custom_mask(q, k, v, state["mask"], sm_scale)
    return (o.detach(),) + torch.autograd.grad(o, (q, k, v), state["do"])


def _kept_tiles(case):
    """Expected number of kept 64 x 64 tiles of one head, the last row and column of tiles counted by what they hold."""
    n = case["N"] / TILE
    if case["kind"] == "token":
        w = _window(case) / TILE
        return n * w - w * w / 2 + n / 2
    off = n * n - n
    return n + case["keep"] * (off / 2 if case["mask"] == "causal" else off)


def work(case):
    if case["kind"] == "reorder":
        image = case["H"] * case["frames"] * case["height"] * case["width"] * case["D"] * 2
        return {"bytes": 4 * 2 * image, "flops": 0}
    heads = case["B"] * case["H"]
    tensor = heads * case["N"] * case["D"]
    train = case["kind"] in ("train", "token")
    flops = heads * _kept_tiles(case) * TILE * TILE * case["D"] * (14 if train else 4)
    nb = -(-case["N"] // TILE)
    if case["kind"] in ("dense_in", "token"):
        mask = case["N"] ** 2
    else:
        mask = nb * nb * (heads if case["per_head"] else 1) * (4 if case["kind"] == "dynamic" else 1)
    if train:                                 # q, k, v, dO in; O, dQ, dK, dV out
        moved = 8 * 2 * tensor
    elif case["kind"] == "lse":               # fp32 O and logsumexp out
        moved = (3 * 2 + 4) * tensor + 4 * heads * case["N"]
    else:
        moved = 4 * 2 * tensor
    return {"bytes": moved + mask, "flops": flops}


def tolerance(case):
    if case["kind"] == "reorder":
        return "exact"
    # P and the results are rounded to the inputs' type (2^-11 and 2^-8 relative at most); with fp32 results P and the
    # products' operands still have 16 bits
    if case["kind"] == "lse" or case["dtype"] == "f16":
        return {"rel": 2e-3}
    return {"rel": 1e-2}
