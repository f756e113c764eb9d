"""The fused float32 attention where not every gradient is wanted: the same bits, and none of the work that only the others need."""
import pytest
import torch

import wm_ctypes as abi
from test_gpu_f32_fused_attention import _views


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,w", [(200, 9, 20), (200, 24, 16), (290, 48, 33), (131, 60, 40), (300, 64, 100), (515, 75, 64), (200, 96, 50), (161, 101, 63), (260, 112, 600),
                                   (385, 128, 40)])
def test_part_of_the_gradients(device, M, N, w):
    views = _views(1, 2, M, N, device)
    out, stats = abi.attention_f32_forward(*views[:3], w, 0.2)
    full = abi.attention_f32_backward(*views[:3], out, stats, views[3], w, 0.2)
    for want in ((False, True, False), (False, False, True), (False, True, True), (True, True, False), (True, False, True)):
        part = abi.attention_f32_backward(*views[:3], out, stats, views[3], w, 0.2, want=want)
        assert all((x is None) == (not n) and (x is None or torch.equal(x, y)) for n, x, y in zip(want, part, full)), want


@pytest.mark.gpu
@pytest.mark.parametrize("N", [16, 64, 128])
def test_the_gradient_of_the_values_needs_no_row_sums(device, N):
    """grad_v is a product of the probabilities and the gradient of the result: the workspace for D stays as it was."""
    views = [t.contiguous() for t in _views(1, 2, 200, N, device)]
    out, stats = abi.attention_f32_forward(*views[:3], 35, 0.2)
    for wanted, touched in ((2, False), (1, True)):
        delta, grad = torch.full((2, 200), 7.0, device=device), torch.empty_like(views[2])
        operands = [abi.grouped_op(grad) if i == wanted else None for i in range(3)]
        status = abi.lib().wm_grouped_window_attention_f32_backward(
            *map(abi.grouped_op, views[:3]), abi.grouped_op(out), abi._pointer(stats), abi.grouped_op(views[3]), *operands,
            abi._pointer(delta), 2, 200, N, 35, 0.2, abi.DTYPES[torch.float32], 0, abi._stream())
        assert status == 0 and bool((delta != 7.0).any()) == touched
