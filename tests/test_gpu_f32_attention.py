"""Training of window attention in float32: the backward forms the gradient of the scores in one kernel, against float64 and
against the separate ops, whose accuracy it must keep."""
import math

import pytest
import torch

from conftest import seeded
from oracle import attention_oracle as ao

pytestmark = pytest.mark.gpu
# batch, heads, M, N, w: around a tile (128) and a chunk (32), one column group to eight, windows from the kernel's
# lower range to beyond the sequence; column shares (few tiles) and none
CASES = [(1, 1, 5, 8, 40), (2, 3, 129, 64, 32), (1, 2, 300, 80, 33), (2, 1, 127, 24, 64), (1, 2, 515, 128, 100), (1, 1, 700, 40, 800),
         (40, 16, 130, 16, 35)]


def _views(batch, heads, M, N, device, layout):
    flat = [seeded((batch, M, heads * N), 600 + s, torch.float32).to(device) for s in range(4)]
    views = [t.view(batch, M, heads, N).transpose(1, 2) for t in flat]
    return views if layout == "heads" else [t.reshape(batch * heads, M, N) for t in views]


def _error(got, want):
    return float((got.cpu().double().reshape(want.shape) - want).norm() / want.norm())


@pytest.mark.parametrize("layout", ["heads", "flat"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "B%dx%d_M%d_N%d_w%d" % c)
def test_step_keeps_the_accuracy_of_the_separate_ops(device, case, layout):
    import window_matmul_kernel as native
    from window_matmul import band_softmax, unwindow_matmul, window_matmul

    batch, heads, M, N, w = case
    views = _views(batch, heads, M, N, device, layout)
    host = [t.cpu().reshape(batch * heads, M, N) for t in views]
    scale = 1.0 / math.sqrt(N)
    for mask in (False, True):
        want = [torch.from_numpy(x) for x in ao.window_attention_backward(*host[:3], w, host[3], scale, mask)]
        errors = []
        for fused in (True, False):
            q, k, v = (t.detach().requires_grad_(True) for t in views[:3])
            if fused:
                out = native.window_attention_f32(q, k, v, w, scale, mask)
                assert type(out.grad_fn).__name__ == "WindowAttentionF32FuncBackward"
            else:
                out = unwindow_matmul(band_softmax(window_matmul(q, k.transpose(-1, -2), w), scale, mask), v, w)
            out.backward(views[3])
            errors.append([_error(t.grad, x) for t, x in zip((q, k, v), want)])
            assert q.grad.stride() == views[0].stride()
        # D is one sum of N products of float32 values, the separate ops' one of 2 w + 1: a few roundings either way
        for mine, theirs in zip(*errors):
            assert mine < 1.5 * theirs + 1e-7 and mine < 3e-6


def test_part_of_the_gradients_and_below_the_rule(device):
    from window_matmul import window_attention

    base = _views(1, 2, 200, 64, device, "heads")

    def grads(need):
        leaves = [t.detach().requires_grad_(n) for t, n in zip(base[:3], need)]
        window_attention(*leaves, 130).backward(base[3])
        return [t.grad for t in leaves]

    full = grads((True, True, True))
    for need in ((True, False, False), (False, True, False), (False, False, True), (False, True, True)):
        for n, x, y in zip(need, grads(need), full):
            assert (x is None) == (not n)
            assert x is None or torch.equal(x, y)
    out = window_attention(base[0].detach().requires_grad_(True), base[1], base[2], 127)
    assert type(out.grad_fn).__name__ == "UnwindowMatmulFuncBackward"
    out = window_attention(base[0].detach().requires_grad_(True), base[1], base[2], 128)
    assert type(out.grad_fn).__name__ == "WindowAttentionF32FuncBackward"
