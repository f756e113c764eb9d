"""Training of window attention in float32: the backward forms the gradient of the scores in one kernel, against float64 and
against the separate ops, whose accuracy it must keep."""
import ctypes
import math

import pytest
import torch

import wm_ctypes as abi
from conftest import seeded
from oracle import attention_oracle as ao

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


@pytest.mark.gpu
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


@pytest.mark.gpu
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


@pytest.mark.gpu
@pytest.mark.parametrize("batch,heads,M,N,w", [(1, 2, 131, 64, 16), (2, 1, 97, 80, 17), (1, 3, 260, 8, 16), (2, 2, 33, 128, 31),
                                               (40, 16, 131, 24, 17)])
def test_score_gradient_of_the_c_abi(device, batch, heads, M, N, w):
    """The entry point over its whole range of windows, below the one that training takes it from too, against float64 and
    the two separate ops that it stands for."""
    go, v, o = (t.reshape(batch * heads, M, N).contiguous() for t in _views(batch, heads, M, N, device, "heads")[:3])
    probs = torch.softmax(seeded((batch * heads, M, 2 * w + 1), 640, torch.float32).to(device), -1)
    o = abi.unwindow_forward(probs, v, w)
    want = torch.zeros(probs.shape, dtype=torch.float64, device=device)
    for j in range(2 * w + 1):  # column j of row i: position i + j - w
        i0, i1 = max(0, w - j), min(M, M + w - j)
        if i0 < i1:
            want[:, i0:i1, j] = (go[:, i0:i1].double() * v[:, i0 + j - w:i1 + j - w].double()).sum(-1)
    p = probs.double()
    want = 0.3 * p * (want - (p * want).sum(-1, keepdim=True))
    ga, _ = abi.unwindow_backward(probs, v, w, go, want_v=False)
    theirs = _error(abi.band_softmax_backward(probs, ga, 0.3), want.cpu())
    got = abi.score_gradient(go, v, o, probs, w, 0.3)
    assert _error(got, want.cpu()) < 1.5 * theirs + 1e-7  # as in the step above
    def view(t):
        return t.view(batch, heads, M, N).transpose(1, 2).contiguous().transpose(1, 2)
    assert torch.equal(abi.score_gradient(view(go), view(v), view(o), probs, w, 0.3), got)


def test_score_gradient_refuses_on_the_host():
    L, P = abi.lib(), ctypes.byref

    def status(B=1, M=64, N=64, w=20, scale=1.0, dtype=0, flags=0, heads=(0, 0, 0), data=(4096,) * 5, row=None, column=1):
        row = N if row is None else row
        rows = [abi.GroupedOperand(abi.Operand(d, M * row, row, column), h, 0) for d, h in zip(data, heads)]
        bands = [abi.Operand(d, M * (2 * w + 1), 2 * w + 1, 1) for d in data[3:]]
        return L.wm_grouped_score_gradient(P(rows[0]), P(rows[1]), P(rows[2]), P(bands[0]), P(bands[1]), B, M, N, w, scale,
                                           dtype, flags, None)

    assert status(B=0) == 0 and status(M=0) == 0                      # nothing to do
    assert all(status(data=tuple(None if i == j else 4096 for j in range(5))) == 1 for i in range(5))
    assert status(heads=(2, 3, 0)) == 2 and status(heads=(-1, 0, 0)) == 2 and status(scale=float("nan")) == 2
    assert status(w=-1) == 2 and status(dtype=9) == 3 and status(flags=0x80) == 4 and status(flags=abi.ANY_HEAD_WIDTH) == 4
    for declined in (dict(w=15), dict(N=20), dict(N=136), dict(dtype=1), dict(dtype=2), dict(dtype=3), dict(row=66), dict(column=2),
                     dict(data=(4100,) * 3 + (4096,) * 2), dict(flags=abi.FORCE_STRIDED), dict(flags=abi.NO_SPLIT_F32)):
        assert status(**declined) == abi.UNSUPPORTED, declined
