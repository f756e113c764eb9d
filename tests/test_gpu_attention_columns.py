"""Attention on operands stored as columns, (..., N, M): the library's own transpose makes rows of them, as it does for the separate ops."""
import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from conftest import seeded


class Copies(TorchDispatchMode):
    """The general strided copies that run inside."""

    def __init__(self):
        super().__init__()
        self.seen = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        if func.overloadpacket in (torch.ops.aten.clone, torch.ops.aten.copy_, torch.ops.aten.contiguous):
            self.seen.append(str(func))
        return func(*args, **(kwargs or {}))


# dtype, shape of the keys' columns, window; the last ones have no aligned rows for the library's transpose and are copied
@pytest.mark.gpu
@pytest.mark.parametrize("dtype,lead,N,M,w,copies", [(torch.float32, (8,), 64, 160, 40, 0), (torch.float32, (2, 4), 64, 160, 40, 0), (torch.float32, (8,), 60, 129, 33, 0),
                                                     (torch.float16, (8,), 120, 160, 20, 0), (torch.float32, (8,), 75, 160, 40, 1), (torch.float32, (2, 4), 41, 131, 40, 1)])
@pytest.mark.parametrize("which", [0, 1, 2])
def test_columns(device, dtype, lead, N, M, w, copies, which):
    from window_matmul import window_attention

    shape = (*lead, M, N)
    rows = [seeded(shape, 500 + i, dtype).to(device) for i in range(4)]
    def run(columns):
        xs = [t.detach() for t in rows[:3]]
        if columns:
            xs[which] = xs[which].transpose(-1, -2).contiguous()
        xs = [t.requires_grad_(True) for t in xs]
        args = [t.transpose(-1, -2) if columns and i == which else t for i, t in enumerate(xs)]
        with Copies() as c:
            out = window_attention(*args, w)
        out.backward(rows[3])
        return out.detach(), [t.grad for t in xs], len(c.seen)
    out, grads, _ = run(False)
    got, got_grads, seen = run(True)
    assert torch.equal(got, out) and seen == copies
    got_grads[which] = got_grads[which].transpose(-1, -2)
    assert all(torch.equal(x, y) for x, y in zip(grads, got_grads))
