"""What a user of MaskedLinear and MaskedFFN has them do, as a list of cases that can be timed.

A transformer block over text and image tokens routes every token row to the weights of its modality:
the attention projections go through MaskedLinear, the feed-forward layer through MaskedFFN.  The cases
take both through the sizes of a model's life: single-token and batched decode, short and long prompts
(prefill), and training steps (forward and backward), over square and odd-sized layers.

    listed()          the fixed cases
    draw(rng)         one more case from the ranges that the fixed ones stand for
    prepare(case, s)  inputs and weights on the GPU, made from the seed s
    run(state)        one pass through the public entry points
    work(case)        bytes and operations that one pass cannot do without
    tolerance(case)   how far another correct implementation in the same precision may differ
"""
from __future__ import annotations

import random

import torch

from ffn_kernel_amd import MaskedFFN, MaskedLinear

# op: "linear" (y = x W), "ffn" (SwiGLU feed-forward); train: forward and backward instead of the forward alone.
# k, n: input and output features of the linear layer, or model width and intermediate size of the feed-forward layer.
# mask: "spans" (runs of image tokens between runs of text), "mixed" (each row on its own, as in a decode batch of
# unrelated sequences), "visual" / "text" (one modality only).
_LISTED = (
    # One token through a projection: nothing but latency.
    dict(name="linear_decode_1", op="linear", train=False, m=1, k=1024, n=1024, mask="text"),
    # A prompt of one sequence through a projection.
    dict(name="linear_fwd_2048", op="linear", train=False, m=2048, k=1024, n=1024, mask="spans"),
    # A projection whose extents are no multiples of a tile (nor of 64), odd row count.
    dict(name="linear_fwd_ragged", op="linear", train=False, m=3001, k=2056, n=1544, mask="spans"),
    # Training step of a projection, rows of both modalities fully interleaved.
    dict(name="linear_train_8192", op="linear", train=True, m=8192, k=1024, n=1024, mask="mixed"),
    # Single-stream decode of a large layer: one modality's weights are read from memory once.
    dict(name="ffn_decode_1", op="ffn", train=False, m=1, k=4096, n=14336, mask="text"),
    # A decode batch of sequences in both modalities, odd size.
    dict(name="ffn_decode_27", op="ffn", train=False, m=27, k=4096, n=14336, mask="mixed"),
    # The largest decode batch, one modality (a text-generation service).
    dict(name="ffn_decode_64", op="ffn", train=False, m=64, k=4096, n=14336, mask="text"),
    # A short prompt: too many rows to be memory-bound by far, too few to fill the chip with large tiles.
    dict(name="ffn_prefill_300", op="ffn", train=False, m=300, k=4096, n=14336, mask="spans"),
    # An ordinary prompt with an image in it, odd size.
    dict(name="ffn_prefill_1411", op="ffn", train=False, m=1411, k=4096, n=14336, mask="spans"),
    # Four sequences through the feed-forward layer of a small model.
    dict(name="ffn_small_8192", op="ffn", train=False, m=8192, k=1024, n=2048, mask="spans"),
    # A batch of long prompts through a large layer.
    dict(name="ffn_prefill_32768", op="ffn", train=False, m=32768, k=4096, n=14336, mask="spans"),
    # Training step of a large layer.
    dict(name="ffn_train_4096", op="ffn", train=True, m=4096, k=4096, n=14336, mask="spans"),
)

_MAX_FLOPS = 2 * 32768 * 4096 * 14336 * 3
_IMAGE_TOKENS = 576


def listed():
    return [dict(c) for c in _LISTED]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, round(lo * (hi / lo) ** rng.random())))


def _extent(rng, lo, hi):
    """A layer's extent: mostly a multiple of 64, as models have them, else a multiple of 8."""
    unit = 64 if rng.random() < 0.75 else 8
    return max(lo, _log_int(rng, lo, hi) // unit * unit)


def draw(rng: random.Random):
    kind = rng.choice(("linear_fwd", "linear_train", "ffn_decode", "ffn_prefill", "ffn_train"))
    while True:
        if kind.startswith("linear"):
            m = _log_int(rng, 65, 16384) if kind == "linear_train" else _log_int(rng, 1, 32768)
            k, n = _extent(rng, 512, 8192), _extent(rng, 512, 8192)
        else:
            k = _extent(rng, 1024, 8192)
            n = int(k * rng.uniform(2.0, 3.5)) // 64 * 64 if k % 64 == 0 else int(k * rng.uniform(2.0, 3.5)) // 8 * 8
            m = _log_int(rng, *{"ffn_decode": (1, 64), "ffn_prefill": (65, 32768), "ffn_train": (65, 8192)}[kind])
        mask = rng.choice(("mixed", "mixed", "visual", "text") if m <= 64 else ("spans", "spans", "mixed", "visual", "text"))
        case = dict(op=kind.split("_")[0], train=kind.endswith("train"), m=m, k=k, n=n,
                    mask=mask if m > 1 else rng.choice(("visual", "text")))
        if work(case)["flops"] <= _MAX_FLOPS:
            return case


def _mask(case, seed):
    m, kind = case["m"], case["mask"]
    rng = random.Random(seed)
    if kind in ("visual", "text"):
        return torch.full((m,), kind == "visual")
    if kind == "mixed":
        return torch.rand(m, generator=torch.Generator().manual_seed(seed)) < 0.5
    span = min(_IMAGE_TOKENS, max(1, m // 4))  # a short prompt holds a smaller image
    mask = torch.zeros(m, dtype=torch.bool)
    at = rng.randrange(span)
    while at < m:
        mask[at:at + span] = True
        at += span + rng.randrange(span // 2, span + span // 2 + 1)
    return mask


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def normal(rows, cols, std):
        return torch.randn((rows, cols), generator=gen, device="cuda", dtype=torch.float32).mul_(std).bfloat16()

    m, k, n, train = case["m"], case["k"], case["n"], case["train"]
    # Weights as nn.Linear holds them: [out features, in features].
    if case["op"] == "linear":
        shapes = [(n, k)] * 2                                               # visual, text
    else:
        shapes = [(n, k), (k, n), (n, k)] * 2                               # w1, w2, w3, u1, u2, u3
    state = dict(train=train, op=MaskedLinear if case["op"] == "linear" else MaskedFFN,
                 x=normal(m, k, 1.0).requires_grad_(train),                 # behind a normalisation layer
                 weights=[normal(*s, 0.02).requires_grad_(train) for s in shapes],
                 mask=_mask(case, seed).cuda())
    if train:
        state["grad"] = normal(m, shapes[1][0], 1.0)
    return state


def run(state):
    views = [w.T for w in state["weights"]]
    if not state["train"]:
        with torch.no_grad():
            return state["op"].apply(state["x"], *views, state["mask"])
    y = state["op"].apply(state["x"], *views, state["mask"])
    grads = torch.autograd.grad(y, [state["x"], *state["weights"]], state["grad"])
    return (y.detach(), *grads)


def work(case):
    m, k, n = case["m"], case["k"], case["n"]
    linear = case["op"] == "linear"
    present = 1 if case["mask"] in ("visual", "text") else 2
    per_set = k * n if linear else 3 * k * n
    out = n if linear else k
    flops = 2 * m * per_set
    nbytes = 2 * (present * per_set + m * k + m * out) + m
    if case["train"]:
        flops *= 3                                                          # dx, and the weights' gradients
        nbytes += 2 * (2 * per_set + m * out + m * k)                       # gradients of both sets, upstream in, dx out
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """About four times what the path differs from the same computation in float32 and above: the outputs' rounding to
    bf16 (linear: 1.7e-3 of the norm, 0.004 of a value), the intermediate's as well (feed-forward: 2.4e-3, 0.010), and
    the gradients' behind it (3.5e-3, 0.021)."""
    if case["op"] == "linear":
        return {"rel": 7e-3, "max": 0.016}
    if not case["train"]:
        return {"rel": 1e-2, "max": 0.04}
    return {"rel": 1.4e-2, "max": 0.08}
