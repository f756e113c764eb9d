"""The native autograd nodes behind the public functions: the same gradients as the Python Function classes (which
torch.jit.trace and, for the two products, autocast take instead), saved tensors that are released, checked for in-place changes and kept under
retain_graph, and gradients only of the inputs that ask for one."""
import pytest
import torch

from conftest import seeded

pytestmark = pytest.mark.gpu

B, M, N, W = 2, 70, 32, 6


def inputs(device, n, columns=N):
    return [seeded((B, M, columns), s, torch.float32).to(device).to(torch.bfloat16).requires_grad_(True) for s in range(1, n + 1)]


def functions():
    from window_matmul import band_softmax, unwindow_matmul, window_attention, window_matmul
    from window_matmul.band_softmax import BandSoftmaxFunc
    from window_matmul.window_attention import WindowAttentionFunc
    from window_matmul.window_matmul import UnwindowMatmulFunc, WindowMatmulFunc

    def flip(f):
        return lambda q, k: f(q, k.transpose(-1, -2), W)

    return {
        "WindowMatmulFuncBackward": (flip(window_matmul), flip(WindowMatmulFunc.apply), (N, N)),
        "UnwindowMatmulFuncBackward": (lambda a, v: unwindow_matmul(a, v, W), lambda a, v: UnwindowMatmulFunc.apply(a, v, W),
                                       (2 * W + 1, N)),
        "BandSoftmaxFuncBackward": (lambda a: band_softmax(a, 0.5, True), lambda a: BandSoftmaxFunc.apply(a, 0.5, True),
                                    (2 * W + 1,)),
        "WindowAttentionFuncBackward": (lambda q, k, v: window_attention(q, k, v, W, 0.3),
                                        lambda q, k, v: WindowAttentionFunc.apply(q, k, v, W, 0.3, False), (N, N, N)),
    }


@pytest.mark.parametrize("name", ["WindowMatmulFuncBackward", "UnwindowMatmulFuncBackward", "BandSoftmaxFuncBackward",
                                  "WindowAttentionFuncBackward"])
def test_nodes(device, name):
    fn, python_fn, columns = functions()[name]
    xs = [inputs(device, i + 1, c)[i] for i, c in enumerate(columns)]
    out = fn(*xs)
    want = python_fn(*xs)
    assert type(out.grad_fn).__name__ == name and torch.equal(out, want)
    grad = seeded(tuple(out.shape), 9, torch.bfloat16).to(device)
    expect = torch.autograd.grad(want, xs, grad)
    for _ in range(2):  # retain_graph keeps what the node saved
        got = torch.autograd.grad(out, xs, grad, retain_graph=True)
        assert all(torch.equal(a, b) for a, b in zip(got, expect))
    for i, x in enumerate(xs):  # one input at a time, out of this graph and out of a graph of its own
        (one,) = torch.autograd.grad(out, [x], grad, retain_graph=True)
        alone = [t.detach().requires_grad_(j == i) for j, t in enumerate(xs)]
        fn(*alone).backward(grad)
        assert torch.equal(one, expect[i]) and torch.equal(alone[i].grad, expect[i])
        assert all(t.grad is None for j, t in enumerate(alone) if j != i)
    out.backward(grad)
    with pytest.raises(RuntimeError, match="second time"):
        out.backward(grad)
    with torch.no_grad():
        assert fn(*xs).grad_fn is None
    if name != "BandSoftmaxFuncBackward":  # a saved input that changes in between is noticed
        ys = [x.detach().requires_grad_(True) for x in xs]
        out = fn(*ys)
        with torch.no_grad():
            ys[-1].mul_(2)
        with pytest.raises(RuntimeError, match="modified by an inplace operation"):
            out.backward(grad)
