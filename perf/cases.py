"""The work whose speed this repository is measured by: window attention as a model's layer has it done.

A layer holds queries, keys and values (the outputs of its projections) and calls either
`window_attention` or the chain `window_matmul` -> `band_softmax` -> `unwindow_matmul`; a training
step then sends the gradient of the layer's output back to the three projections.  Sizes are those of the
benchmark (`bench.py`), of the tests, and of the range between them.

A case is a dict:
  op      "attention": `window_attention`;  "chain": the three separate ops
  dtype   storage type of every tensor ("float32" is what a model has by default)
  batch, heads, M, N, w   sequences, heads, positions, head width, window (2w + 1 neighbours)
  layout  "heads": q, k, v are (batch, M, heads * N) projections seen as (batch, heads, M, N), and the gradient
          of the output comes back the same way;  "flat": contiguous (batch * heads, M, N) tensors;
          "columns": like "flat", with the keys of the chain stored as (batch * heads, N, M)
  train   forward and backward (True), or forward alone without a graph (inference)
  mask    whether neighbours outside the sequence are left out of the softmax (`mask_out_of_range`)
"""
import math
import os
import sys

import torch

_PACKAGE = os.path.join(os.getcwd(), "pytorch-window-matmul_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

from window_matmul import band_softmax, unwindow_matmul, window_attention, window_matmul  # noqa: E402

_BYTES = {"float32": 4, "bfloat16": 2, "float16": 2}


def _case(name, op, dtype, batch, heads, M, N, w, layout, train, mask):
    return {"name": name, "op": op, "dtype": dtype, "batch": batch, "heads": heads, "M": M, "N": N, "w": w,
            "layout": layout, "train": train, "mask": mask}


def listed():
    return [
        # a layer at toy size (unit tests, debugging, a first look): every microsecond is a launch or host work
        _case("toy step", "chain", "float32", 2, 1, 128, 64, 4, "columns", True, False),
        # one document with one head: a training step that cannot fill the chip
        _case("one short sequence step", "attention", "bfloat16", 1, 1, 4096, 128, 256, "heads", True, False),
        # ragged everything: odd batch, sequence no multiple of any tile, odd window
        _case("ragged step", "attention", "bfloat16", 7, 1, 3001, 80, 33, "flat", True, True),
        # a head width that the matrix instructions do not divide
        _case("odd head width step", "attention", "float16", 1, 8, 4096, 60, 64, "heads", True, False),
        # inference over one long document
        _case("one long sequence", "attention", "bfloat16", 1, 1, 16384, 128, 1024, "heads", False, True),
        # narrow local attention over long sequences, inference through the separate ops
        _case("narrow window", "chain", "bfloat16", 8, 12, 16384, 64, 8, "flat", False, False),
        # training of a local-attention encoder, in one call and through the separate ops
        _case("encoder step", "attention", "bfloat16", 8, 12, 4096, 64, 256, "heads", True, False),
        _case("encoder chain step", "chain", "bfloat16", 8, 12, 4096, 64, 256, "heads", True, False),
        # the same encoder in float32
        _case("float32 encoder step", "attention", "float32", 8, 12, 4096, 64, 256, "heads", True, False),
        # a window that covers most of a ragged sequence, float32, keys stored as columns
        _case("ragged wide float32 step", "chain", "float32", 7, 1, 3001, 80, 1500, "columns", True, False),
        # long-context training with wide heads, in one call and through the separate ops
        _case("long wide head step", "attention", "float16", 1, 16, 32768, 128, 512, "heads", True, True),
        _case("long wide head chain step", "chain", "float16", 1, 16, 32768, 128, 512, "flat", True, False),
    ]


def _spread(rng, low, high):
    """An integer of [low, high], spread over the logarithm."""
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def _cost(case):
    """Rough seconds of a pass, for the upper end of `draw` only."""
    w = work(case)
    return max(w["bytes"] / 4e12, w["flops"] / (80e12 if case["dtype"] == "float32" else 400e12))


def draw(rng):
    """A case anywhere between the smallest and the largest of the list."""
    most = max(_cost(c) for c in listed())
    while True:
        op = rng.choice(["attention", "attention", "chain"])
        layout = rng.choice(["heads", "heads", "flat", "columns" if op == "chain" else "flat"])
        M = _spread(rng, 128, 32768)
        if rng.random() < 0.5:  # as often as not a power-of-two-like length, otherwise whatever the document has
            M = (M + 63) // 64 * 64
        case = _case("", op, rng.choice(["bfloat16", "bfloat16", "float16", "float32"]), _spread(rng, 1, 8),
                     rng.choice([1, 2, 4, 8, 12, 16]), M, rng.choice([16, 32, 40, 48, 60, 64, 64, 64, 75, 80, 96, 128, 128]),
                     _spread(rng, 1, min(1500, M - 1)), layout, rng.random() < 0.65, rng.random() < 0.5)
        del case["name"]
        if _cost(case) <= most:
            return case


def _projection(case, generator):
    """One activation as its projection leaves it: N(0,1), in the layout of the case."""
    B, H, M, N = case["batch"], case["heads"], case["M"], case["N"]
    shape = (B, M, H * N) if case["layout"] == "heads" else (B * H, M, N)
    return torch.randn(shape, generator=generator, device="cuda", dtype=torch.float32).to(getattr(torch, case["dtype"]))


def _heads(case, x):
    if case["layout"] != "heads":
        return x
    return x.view(case["batch"], case["M"], case["heads"], case["N"]).transpose(1, 2)


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    q, k, v, grad = (_projection(case, g) for _ in range(4))
    if case["layout"] == "columns":
        k = k.transpose(1, 2).contiguous()
    if case["train"]:
        q, k, v = (t.requires_grad_(True) for t in (q, k, v))
    return {"case": case, "q": q, "k": k, "v": v, "grad": _heads(case, grad) if case["train"] else None}


def _forward(case, q, k, v):
    q, v = _heads(case, q), _heads(case, v)
    if case["op"] == "attention":
        return window_attention(q, _heads(case, k), v, case["w"], mask_out_of_range=case["mask"])
    columns = k if case["layout"] == "columns" else _heads(case, k).transpose(-1, -2)
    band = window_matmul(q, columns, case["w"])
    probs = band_softmax(band, 1.0 / math.sqrt(case["N"]), case["mask"])
    return unwindow_matmul(probs, v, case["w"])


def run(state):
    case, q, k, v = state["case"], state["q"], state["k"], state["v"]
    if not case["train"]:
        with torch.no_grad():
            return _forward(case, q, k, v)
    q.grad = k.grad = v.grad = None
    out = _forward(case, q, k, v)
    out.backward(state["grad"])
    return out.detach(), q.grad, k.grad, v.grad


def work(case):
    """Two products per pair of neighbours forward and four backward.  Every entry point reads its tensors once and
    writes its results once: four (B, M, N) tensors for an inference, eight for a training step; the separate
    ops hand a band from call to call, which is written or read 4 times forward and 6 times backward."""
    B, M, N, w, size = case["batch"] * case["heads"], case["M"], case["N"], case["w"], _BYTES[case["dtype"]]
    pairs = B * (M * (2 * w + 1) - w * (w + 1))
    rows, band = B * M * N * size, B * M * (2 * w + 1) * size
    if case["op"] == "attention":
        moved = (8 if case["train"] else 4) * rows
    else:  # forward q, k -> band -> probs, v -> out; backward grad, v, probs -> grad v, band; probs, band -> band; q, k, band -> grads
        moved = 4 * rows + 4 * band + ((7 * rows + 6 * band) if case["train"] else 0)
    return {"bytes": float(moved), "flops": (12.0 if case["train"] else 4.0) * pairs * N}


def tolerance(case):
    """Against the same chain in float64 on the same inputs, over the listed cases and thirty drawn ones, the outputs were off by at
    most (2-norm / single value): float32 8.7e-7 / 9.4e-6, float16 6.2e-4 / 7.8e-3 and bfloat16 4.9e-3 / 0.088 through the
    separate ops (which round the band twice), 5.6e-4 / 6.2e-3 and 2.7e-3 / 0.035 in one call.  About four times that, for
    bfloat16 twice."""
    return {"float32": {"rel": 3.5e-6, "max": 4e-5}, "float16": {"rel": 2.5e-3, "max": 0.03},
            "bfloat16": {"rel": 1e-2, "max": 0.2}}[case["dtype"]]
