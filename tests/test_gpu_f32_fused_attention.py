"""The fused float32 attention (recomputing kernels at float32 accuracy) against float64 and against the separate ops, whose
accuracy it must keep."""
import ctypes
import math

import pytest
import torch

import wm_ctypes as abi
from conftest import seeded
from oracle import attention_oracle as ao

# batch, heads, M, N, w: every width class (16 columns) and widths that 8, 4 and 2 do not divide, sequences around a chunk (32) and a
# tile (128), windows from 1 through a chunk's and beyond the sequence
CASES = [(1, 1, 5, 8, 40), (1, 2, 33, 16, 1), (2, 3, 129, 24, 16), (1, 2, 127, 32, 31), (1, 1, 256, 40, 32), (2, 1, 131, 48, 33), (1, 2, 300, 64, 64),
         (1, 1, 515, 64, 600), (1, 2, 160, 75, 17), (2, 1, 97, 80, 97), (1, 1, 385, 96, 50), (1, 1, 200, 101, 63), (1, 1, 290, 112, 40), (1, 2, 260, 128, 100),
         (1, 1, 128, 9, 3), (1, 1, 161, 60, 20), (1, 1, 129, 127, 64)]


def _views(batch, heads, M, N, device, layout="heads"):
    flat = [seeded((batch, M, heads * N), 800 + s, torch.float32).to(device) for s in range(4)]
    views = [t.view(batch, M, heads, N).transpose(1, 2) for t in flat]
    return views if layout == "heads" else [t.reshape(batch * heads, M, N) for t in views]


def _error(got, want):
    return float((got.cpu().double().reshape(want.shape) - want).norm() / want.norm())


def _want(views, w, scale, mask):
    B, M, N = math.prod(views[0].shape[:-2]), *views[0].shape[-2:]
    host = [t.cpu().reshape(B, M, N) for t in views]
    out, _ = ao.window_attention_forward(*host[:3], w, scale, mask)
    return [torch.from_numpy(x) for x in (out, *ao.window_attention_backward(*host[:3], w, host[3], scale, mask))]


def _chain(views, w, scale, mask):
    from window_matmul import band_softmax, unwindow_matmul, window_matmul

    q, k, v = (t.detach().requires_grad_(True) for t in views[:3])
    out = unwindow_matmul(band_softmax(window_matmul(q, k.transpose(-1, -2), w), scale, mask), v, w)
    out.backward(views[3])
    return out.detach(), q.grad, k.grad, v.grad


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["heads", "flat"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "B%dx%d_M%d_N%d_w%d" % c)
def test_accuracy_of_the_separate_ops(device, case, layout):
    batch, heads, M, N, w = case
    views = _views(batch, heads, M, N, device, layout)
    scale = 1.0 / math.sqrt(N)
    for mask in (False, True):
        out, stats = abi.attention_f32_forward(*views[:3], w, scale, mask)
        got = (out, *abi.attention_f32_backward(*views[:3], out, stats, views[3], w, scale))
        for mine, theirs, want in zip(got, _chain(views, w, scale, mask), _want(views, w, scale, mask)):
            # a few roundings either way in the row statistics, as for the score gradient kernel
            assert _error(mine, want) < 1.5 * _error(theirs, want) + 1e-7 and _error(mine, want) < 3e-6
        again, _ = abi.attention_f32_forward(*views[:3], w, scale, mask, want_stats=False)
        assert torch.equal(again, out)


@pytest.mark.gpu
@pytest.mark.parametrize("N,w", [(64, 40), (128, 70)])
@pytest.mark.parametrize("factor", [1e-18, 30.0, 1e3])
def test_magnitudes(device, N, w, factor):
    """Scores that vanish, that put a row's weight on a few keys, and that leave one key with all of it; gradients of any size."""
    views = _views(1, 2, 300, N, device, "flat")
    views[0], views[3] = views[0] * factor, views[3] * 1e-12
    scale = 1.0 / math.sqrt(N)
    out, stats = abi.attention_f32_forward(*views[:3], w, scale)
    got = (out, *abi.attention_f32_backward(*views[:3], out, stats, views[3], w, scale))
    # a score s carries an error of s 2^-24 times a few, and so does the exponent of its probability: with them grows what
    # both ways are off by
    for mine, theirs, want in zip(got, _chain(views, w, scale, False), _want(views, w, scale, False)):
        assert bool(torch.isfinite(mine).all())
        assert _error(mine, want) < 1.5 * _error(theirs, want) + 1e-7


@pytest.mark.gpu
@pytest.mark.parametrize("N", [9, 41, 64, 75, 126, 128])
def test_rows_of_any_alignment(device, N):
    """Rows a word off every alignment, between words that must stay as they are."""
    B, M, w = 2, 150, 20
    def misaligned(t):
        big = torch.full((B, M + 2, N + 3), float("nan"), device=device)
        inner = big[:, 1:M + 1, 1:N + 1]
        inner.copy_(t)
        return big, inner
    plain = _views(B, 1, M, N, device, "flat")
    scale = 1.0 / math.sqrt(N)
    out, stats = abi.attention_f32_forward(*plain[:3], w, scale)
    grads = abi.attention_f32_backward(*plain[:3], out, stats, plain[3], w, scale)
    q, k, v, go = (misaligned(t)[1] for t in plain)
    big, o = misaligned(torch.zeros_like(out))
    _, stats2 = abi.attention_f32_forward(q, k, v, w, scale, out=o)
    assert torch.equal(o, out) and torch.equal(stats2, stats)
    assert bool(torch.isnan(big[:, 0]).all()) and bool(torch.isnan(big[:, -1]).all())
    assert bool(torch.isnan(big[:, :, 0]).all()) and bool(torch.isnan(big[:, :, N + 1:]).all())
    for got, want in zip(abi.attention_f32_backward(q, k, v, o, stats2, go, w, scale), grads):
        assert torch.equal(got, want)


@pytest.mark.gpu
@pytest.mark.parametrize("N", [32, 64, 80])
def test_part_of_the_gradients(device, N):
    views = _views(1, 2, 200, N, device)
    out, stats = abi.attention_f32_forward(*views[:3], 35, 0.2)
    full = abi.attention_f32_backward(*views[:3], out, stats, views[3], 35, 0.2)
    for want in ((True, False, False), (False, True, False), (False, False, True), (False, True, True)):
        part = abi.attention_f32_backward(*views[:3], out, stats, views[3], 35, 0.2, want=want)
        assert all((x is None) == (not n) and (x is None or torch.equal(x, y)) for n, x, y in zip(want, part, full))


@pytest.mark.gpu
@pytest.mark.parametrize("w", [16, 64, 256])
@pytest.mark.parametrize("N", [64, 96])
def test_poisoned_rows_stay_local(device, N, w):
    """As for the other matrix kernels: a NaN or an infinity reaches every row that the exact result gives it to, and no
    row farther than w + 320."""
    M, row = 2048, 1000
    q, k, v, go = _views(1, 1, M, N, device, "flat")
    scale = 1.0 / math.sqrt(N)
    out, stats = abi.attention_f32_forward(q, k, v, w, scale)
    clean = (out, *abi.attention_f32_backward(q, k, v, out, stats, go, w, scale))
    far = (torch.arange(M, device=device) - row).abs() > w + 320
    near = (torch.arange(M, device=device) - row).abs() <= w
    for which in range(4):
        for value in (float("nan"), float("inf")):
            xs = [t.clone() for t in (q, k, v, go)]
            xs[which][0, row, 5] = value
            o, st = abi.attention_f32_forward(*xs[:3], w, scale)
            dirty = (o, *abi.attention_f32_backward(*xs[:3], o, st, xs[3], w, scale))
            for c, d in zip(clean, dirty):
                assert torch.equal(c[:, far], d[:, far])
            if which == 2:
                assert not bool(torch.isfinite(o[0, near, 5]).any())
            if which == 0:
                assert not bool(torch.isfinite(o[0, row]).any())
            if which == 3:
                assert not bool(torch.isfinite(dirty[3][0, near, 5]).any()) and not bool(torch.isfinite(dirty[1][0, row]).any())


@pytest.mark.gpu
def test_in_a_captured_graph(device):
    views = _views(2, 4, 300, 64, device)
    out, stats = abi.attention_f32_forward(*views[:3], 40, 0.1)
    leaves = [t.clone().contiguous() for t in views]
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        o, st = abi.attention_f32_forward(*leaves[:3], 40, 0.1)
        abi.attention_f32_backward(*leaves[:3], o, st, leaves[3], 40, 0.1)
        side.synchronize()
        with torch.cuda.graph(graph, stream=side):
            o, st = abi.attention_f32_forward(*leaves[:3], 40, 0.1)
            grads = abi.attention_f32_backward(*leaves[:3], o, st, leaves[3], 40, 0.1)
    for turn in range(3):
        for t, x in zip(leaves, views):
            t.copy_(x * (1.0 - 0.25 * turn))
        graph.replay()
        torch.cuda.synchronize()
        want, stats = abi.attention_f32_forward(*leaves[:3], 40, 0.1)
        assert torch.equal(o, want)
        for x, y in zip(grads, abi.attention_f32_backward(*leaves[:3], want, stats, leaves[3], 40, 0.1)):
            assert torch.equal(x, y)


@pytest.mark.gpu
@pytest.mark.parametrize("heads,M,N,w,fused", [(8, 128, 64, 32, True), (7, 128, 64, 32, False), (8, 128, 64, 31, False), (2, 4096, 64, 257, False),
                                               (8, 128, 80, 128, False), (256, 128, 80, 127, False), (256, 128, 80, 128, True),
                                               (8, 128, 75, 32, True), (8, 128, 33, 64, True), (8, 128, 33, 63, False), (8, 128, 32, 64, False),
                                               (8, 128, 32, 63, False), (64, 128, 24, 100, False), (159, 128, 96, 128, False), (160, 128, 96, 128, True), (255, 128, 104, 128, False)])
def test_route_of_training_and_of_a_result_changed_in_place(device, heads, M, N, w, fused):
    from window_matmul import window_attention

    views = _views(1, heads, M, N, device)
    scale = 1.0 / math.sqrt(N)
    leaves = [t.detach().requires_grad_(True) for t in views[:3]]
    out = window_attention(*leaves, w)
    plain, stats = abi.attention_f32_forward(*views[:3], w, scale)
    assert torch.equal(out, plain) == fused
    if not fused:
        return
    assert type(out.grad_fn).__name__ == "WindowAttentionF32FuncBackward"
    out.add_(1.0)  # the separate ops kept nothing of their result: still allowed
    out.backward(views[3])
    for t, want in zip(leaves, abi.attention_f32_backward(*views[:3], plain, stats, views[3], w, scale)):
        assert torch.equal(t.grad, want) and t.grad.stride() == t.stride()
    with torch.no_grad():
        assert torch.equal(window_attention(*views[:3], w), plain)
        assert torch.equal(window_attention(*views[:3], 16), abi.attention_f32_forward(*views[:3], 16, scale)[0])
        assert not torch.equal(window_attention(*views[:3], 15), abi.attention_f32_forward(*views[:3], 15, scale)[0])


def test_refusals_on_the_host():
    L, P = abi.lib(), ctypes.byref

    def operands(n, M, N, heads, data, column):
        return [abi.GroupedOperand(abi.Operand(d, M * N, N, column), h, 0) for d, h in zip(data, heads)][:n]

    def forward(B=1, M=64, N=64, w=20, scale=1.0, dtype=0, flags=0, heads=(0,) * 8, data=(4096,) * 8, column=1):
        x = operands(4, M, N, heads, data, column)
        return L.wm_grouped_window_attention_f32_forward(*map(P, x), None, B, M, N, w, scale, 0, dtype, flags, None)

    def backward(B=1, M=64, N=64, w=20, scale=1.0, dtype=0, flags=0, heads=(0,) * 8, data=(4096,) * 8, column=1, stats=4096, delta=4096):
        x = operands(8, M, N, heads, data, column)
        return L.wm_grouped_window_attention_f32_backward(*map(P, x[:4]), stats, *map(P, x[4:]), delta, B, M, N, w, scale, dtype, flags, None)

    for status, n in ((forward, 4), (backward, 8)):
        assert status(B=0) == 0 and status(M=0) == 0
        assert all(status(data=tuple(None if i == j else 4096 for j in range(8))) == 1 for i in range(n))
        assert status(heads=(2, 3) + (0,) * 6) == 2 and status(heads=(-1,) + (0,) * 7) == 2 and status(scale=float("nan")) == 2
        assert status(w=-1) == 2 and status(dtype=9) == 3 and status(flags=0x80) == 4 and status(flags=abi.ANY_HEAD_WIDTH) == 4
        for declined in (dict(w=0), dict(N=7), dict(N=129), dict(dtype=1), dict(dtype=2), dict(dtype=3), dict(column=2), dict(scale=0.0), dict(scale=-1.0),
                         dict(data=(4098,) * 8), dict(flags=abi.FORCE_STRIDED), dict(flags=abi.NO_SPLIT_F32)):
            assert status(**declined) == abi.UNSUPPORTED, declined
    assert backward(stats=None) == 1 and backward(delta=None) == 1
