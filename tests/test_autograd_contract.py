"""What torch.autograd.Function does for its callers holds for the native nodes behind the public functions too."""
import pytest
import torch
import torch.autograd.forward_ad as forward_ad

from conftest import seeded

B, M, N, W = 2, 40, 32, 6
# name, columns of the inputs, dtype
OPS = [("window_matmul", (N, N), torch.bfloat16), ("unwindow_matmul", (2 * W + 1, N), torch.bfloat16),
       ("band_softmax", (2 * W + 1,), torch.bfloat16), ("window_attention", (N, N, N), torch.bfloat16),
       ("window_attention", (44, 44, 44), torch.float16), ("window_attention", (N, N, N), torch.float32),
       ("window_attention", (64, 64, 64), torch.float32)]
IDS = ["window_matmul", "unwindow_matmul", "band_softmax", "window_attention", "window_attention_N44", "window_attention_float32",
       "window_attention_float32_fused"]


def call(name, dtype):
    import window_matmul as wm

    if name == "window_matmul":
        return lambda q, k: wm.window_matmul(q, k.transpose(-1, -2), W)
    if name == "unwindow_matmul":
        return lambda a, v: wm.unwindow_matmul(a, v, W)
    if name == "band_softmax":
        return lambda a: wm.band_softmax(a, 0.5, True)
    return lambda q, k, v: wm.window_attention(q, k, v, 130 if dtype == torch.float32 else W)


def operands(columns, dtype, device="cpu"):
    batch = 8 if columns[0] == 64 else B  # eight tiles of rows: where the fused float32 kernels begin
    return [seeded((batch, M, c), 700 + i, dtype).to(device) for i, c in enumerate(columns)]


@pytest.mark.gpu
def test_the_float32_cases_take_the_route_with_the_band_and_the_one_without(device):
    import wm_ctypes as abi

    for (name, columns, dtype), fused in ((OPS[5], False), (OPS[6], True)):
        xs = operands(columns, dtype, device)
        plain, _ = abi.attention_f32_forward(*xs, 130, columns[0] ** -0.5)
        out = call(name, dtype)(*(x.requires_grad_(True) for x in xs))
        assert torch.equal(out, plain) == fused and type(out.grad_fn).__name__ == "WindowAttentionF32FuncBackward"


def refuses_tangents(name, columns, dtype, device):
    fn = call(name, dtype)
    for i in range(len(columns)):
        for other_needs_grad in (False, True):
            xs = [x.requires_grad_(other_needs_grad and j != i) for j, x in enumerate(operands(columns, dtype, device))]
            with forward_ad.dual_level():
                xs[i] = forward_ad.make_dual(xs[i], torch.ones_like(xs[i]))
                with pytest.raises(NotImplementedError):
                    fn(*xs)


@pytest.mark.gpu
@pytest.mark.parametrize("name,columns,dtype", OPS, ids=IDS)
def test_forward_mode_is_refused(device, name, columns, dtype):
    refuses_tangents(name, columns, dtype, device)


@pytest.mark.parametrize("name,columns", [("window_matmul", (N, N)), ("unwindow_matmul", (2 * W + 1, N)), ("band_softmax", (2 * W + 1,))])
def test_forward_mode_is_refused_before_anything_else(name, columns):
    refuses_tangents(name, columns, torch.float32, "cpu")


@pytest.mark.gpu
@pytest.mark.parametrize("name,columns,dtype", OPS, ids=IDS)
def test_traced_calls_replay(device, name, columns, dtype):
    """A trace holds the operation and not only the allocation of its result: other inputs give other results, with
    and without a graph, and gradients flow through the replay."""
    fn = call(name, dtype)
    for needs_grad in (False, True):
        first = [x.requires_grad_(needs_grad) for x in operands(columns, dtype, device)]
        traced = torch.jit.trace(lambda *xs: fn(*xs) + 0, tuple(first), check_trace=False)
        for factor in (1.0, 0.5):
            xs = [(x.detach() * factor).requires_grad_(needs_grad) for x in first]
            torch.empty(1 << 20, device=device).fill_(float("nan"))  # what a fresh allocation may find
            got, want = traced(*xs), fn(*xs)
            # a trace holds the separate ops: bit for bit what the route that keeps the band computes forward
            # (without it both are within some 8 * 2^-24 of the largest value, about 4)
            assert torch.equal(got, want) if columns[0] != 64 else torch.allclose(got, want, rtol=1e-5, atol=2e-6)
            if needs_grad:
                grad = torch.ones_like(want)
                for a, b in zip(torch.autograd.grad(got, xs, grad), torch.autograd.grad(want, xs, grad)):
                    # float32 attention is traced as the chain of the separate ops: the same sums in another order
                    assert torch.equal(a, b) if dtype != torch.float32 else torch.allclose(a, b, rtol=1e-4, atol=1e-5)


class StopsGradients(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x):
        return x.clone()

    @staticmethod
    def backward(ctx, grad):
        return None


@pytest.mark.gpu
@pytest.mark.parametrize("name,columns,dtype", OPS, ids=IDS)
def test_an_undefined_gradient_counts_as_zeros(device, name, columns, dtype):
    xs = [x.requires_grad_(True) for x in operands(columns, dtype, device)]
    StopsGradients.apply(call(name, dtype)(*xs)).sum().backward()
    for x in xs:
        assert x.grad is not None and x.grad.shape == x.shape and not x.grad.any()


@pytest.mark.gpu
@pytest.mark.parametrize("name,columns,dtype", OPS, ids=IDS)
def test_compiled_autograd(device, name, columns, dtype):
    fn = call(name, dtype)
    eager, compiled = ([x.requires_grad_(True) for x in operands(columns, dtype, device)] for _ in range(2))
    fn(*eager).sum().backward()
    out = fn(*compiled).sum()
    torch._dynamo.reset()
    with torch._dynamo.compiled_autograd._enable(torch.compile(backend="eager")):
        out.backward()
    for x, y in zip(eager, compiled):
        assert torch.equal(x.grad, y.grad)


@pytest.mark.gpu
@pytest.mark.parametrize("name,columns,dtype", OPS, ids=IDS)
def test_saved_tensor_hooks_and_checkpoints(device, name, columns, dtype):
    """Everything the backward reads goes through the hooks, their errors arrive as they are, and a checkpoint, which
    stops its second forward from inside a hook, gives the gradients of the plain call."""
    from torch.utils.checkpoint import checkpoint

    fn = call(name, dtype)
    xs, ys = ([x.requires_grad_(True) for x in operands(columns, dtype, device)] for _ in range(2))
    fn(*xs).sum().backward()
    with torch.autograd.graph.save_on_cpu():
        out = fn(*ys)
    out.sum().backward()
    assert all(torch.equal(x.grad, y.grad) for x, y in zip(xs, ys))
    for y in ys:
        y.grad = None
    checkpoint(fn, *ys, use_reentrant=False).sum().backward()
    assert all(torch.equal(x.grad, y.grad) for x, y in zip(xs, ys))

    def refuse(t):
        raise KeyError("from the hook")

    with torch.autograd.graph.saved_tensors_hooks(refuse, lambda t: t), pytest.raises(KeyError, match="from the hook"):
        fn(*ys)


@pytest.mark.gpu
@pytest.mark.parametrize("name,columns,dtype", OPS, ids=IDS)
def test_backward_on_a_side_stream(device, name, columns, dtype):
    """The backward runs on the stream of its forward whatever stream calls for it, and its inputs stay alive for it."""
    fn = call(name, dtype)
    xs, ys = ([x.requires_grad_(True) for x in operands(columns, dtype, device)] for _ in range(2))
    fn(*xs).sum().backward()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        out = fn(*ys).sum()
    out.backward()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    assert all(torch.equal(x.grad, y.grad) for x, y in zip(xs, ys))


@pytest.mark.gpu
@pytest.mark.parametrize("compiled", [False, True], ids=["eager", "compiled"])
@pytest.mark.parametrize("name,columns,dtype", [OPS[1], *OPS[4:]], ids=[IDS[1], *IDS[4:]])
def test_result_changed_in_place(device, name, columns, dtype, compiled):
    """The last result of the separate ops is not needed by their backward; the routes that took their place keep to that.
    The same gradients bit for bit as without the change."""
    fn = call(name, dtype)

    def gradients(change):
        xs = [x.requires_grad_(True) for x in operands(columns, dtype, device)]
        out = fn(*xs)
        loss = (change(out) * 1.0).sum()
        torch._dynamo.reset()
        if compiled:
            with torch._dynamo.compiled_autograd._enable(torch.compile(backend="eager")):
                loss.backward()
        else:
            loss.backward()
        return [x.grad for x in xs]

    plain = gradients(lambda out: out * 2)
    for x, y in zip(plain, gradients(lambda out: out.mul_(2))):
        assert torch.equal(x, y)
    for x, y in zip(plain, gradients(lambda out: out.mul_(2).add_(float("inf")))):
        assert torch.equal(x, y)


@pytest.mark.gpu
def test_result_that_stays_as_it_was_given(device):
    """float16 / bfloat16 training at multiples of 16: the backward reads the result and notices a change."""
    name, columns, dtype = OPS[3]
    out = call(name, dtype)(*(x.requires_grad_(True) for x in operands(columns, dtype, device)))
    out.mul_(2)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        out.sum().backward()


@pytest.mark.gpu
@pytest.mark.parametrize("columns,dtype", [(44, torch.float16), (N, torch.float32), (64, torch.float32), (N, torch.bfloat16)])
def test_inference_mode(device, columns, dtype):
    xs = operands((columns,) * 3, dtype, device)
    want = call("window_attention", dtype)(*xs)
    with torch.inference_mode():
        got = call("window_attention", dtype)(*xs)
    assert got.is_inference() and torch.equal(got, want)


@pytest.mark.gpu
@pytest.mark.parametrize("name,columns,dtype", OPS, ids=IDS)
def test_compiled_callers(device, name, columns, dtype):
    """torch.compile around a call breaks its graph there and gives the eager results and gradients."""
    fn = call(name, dtype)
    xs, ys = ([x.requires_grad_(True) for x in operands(columns, dtype, device)] for _ in range(2))
    want = fn(*xs) * 2
    torch._dynamo.reset()
    got = torch.compile(lambda *t: fn(*t) * 2, backend="eager")(*ys)
    assert torch.equal(got, want)
    want.sum().backward()
    got.sum().backward()
    assert all(torch.equal(x.grad, y.grad) for x, y in zip(xs, ys))
