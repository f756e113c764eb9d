"""Python API and autograd glue of the banded matmuls.

Mirrors reference window_matmul/window_matmul.py:7-76: the public functions
``window_matmul(inp, other, window_size)`` and ``unwindow_matmul(inp, other,
window_size)`` plus the two ``torch.autograd.Function`` classes they apply.
All arithmetic happens in the native module ``window_matmul_kernel`` (HIP
kernels for gfx950); if that module has not been built the import below fails,
on purpose -- there is no Python or CPU fallback behind this package.

Band convention: with ``W = 2 * window_size + 1``, column ``j`` of band row
``i`` refers to sequence position ``i + j - window_size``; positions outside
``[0, M)`` read as nothing and are written as exact zeros.
"""
from typing import Optional, Tuple

import torch

import window_matmul_kernel as _native

# Inside a CUDA/HIP autocast region the operands are cast to float16 and the
# body runs with autocast disabled (reference window_matmul.py:9,18,45,54).  The public functions take
# the two classes below there and under torch.jit.trace, which records a Function as one operation but of a native call
# only the allocation of its result, and the native module's own autograd nodes everywhere else.
_amp_forward = torch.amp.custom_fwd(device_type="cuda", cast_inputs=torch.float16)
_amp_backward = torch.amp.custom_bwd(device_type="cuda")
_tracing = torch._C._is_tracing  # what torch.jit.is_tracing asks, in a quarter of its time (0.4 us a call)


class WindowMatmulFunc(torch.autograd.Function):
    """``A[b, i, j] = sum_h inp[b, i, h] * other[b, h, i + j - w]``.

    ``inp`` is ``(..., M, N)``, ``other`` is ``(..., N, M)`` (the keys, transposed), the result is
    ``(..., M, 2w+1)`` with the leading dimensions of ``inp``.  Leading dimensions with at most two levels
    of strides (a projection seen as ``(batch, heads, M, N)``) are read in place, and gradients are laid out
    like the operand they belong to.  reference window_matmul.py:7-27.
    """

    @staticmethod
    @_amp_forward
    def forward(ctx, inp: torch.Tensor, other: torch.Tensor, window_size: int) -> torch.Tensor:
        ctx.save_for_backward(inp, other)
        return _native.window_matmul_forward(inp, other, window_size)

    @staticmethod
    @_amp_backward
    def backward(ctx, grad_output: torch.Tensor) -> Tuple[torch.Tensor, torch.Tensor, None]:
        inp, other = ctx.saved_tensors
        # the band width fixes the window: W = 2w + 1  (reference window_matmul.py:22)
        half_width = grad_output.shape[-1] // 2
        # a gradient nobody asked for is not computed (the reference always computes both)
        grad_inp, grad_other = _native.window_matmul_backward(
            inp, other, half_width, grad_output, ctx.needs_input_grad[0], ctx.needs_input_grad[1]
        )
        return grad_inp, grad_other, None


class UnwindowMatmulFunc(torch.autograd.Function):
    """``O[b, i, h] = sum_j inp[b, i, j] * other[b, i + j - w, h]``.

    ``inp`` is the band ``(..., M, 2w+1)``, ``other`` is ``(..., M, N)``, the result has the shape of
    ``other``; leading dimensions as in :class:`WindowMatmulFunc`.  reference window_matmul.py:43-63.
    """

    @staticmethod
    @_amp_forward
    def forward(ctx, inp: torch.Tensor, other: torch.Tensor, window_size: int) -> torch.Tensor:
        ctx.save_for_backward(inp, other)
        return _native.unwindow_matmul_forward(inp, other, window_size)

    @staticmethod
    @_amp_backward
    def backward(ctx, grad_output: torch.Tensor) -> Tuple[torch.Tensor, torch.Tensor, None]:
        inp, other = ctx.saved_tensors
        half_width = inp.shape[-1] // 2  # reference window_matmul.py:59
        grad_inp, grad_other = _native.unwindow_matmul_backward(
            inp, other, half_width, grad_output, ctx.needs_input_grad[0], ctx.needs_input_grad[1]
        )
        return grad_inp, grad_other, None


def window_matmul(inp: torch.Tensor, other: torch.Tensor, window_size: Optional[int]) -> torch.Tensor:
    """Band of ``inp @ other``: ``(..., M, N) x (..., N, M) -> (..., M, 2w+1)``.

    A falsy ``window_size`` keeps only the diagonal and is computed with plain
    torch ops, giving ``(..., M, 1)`` (reference window_matmul.py:33-34).  Any
    number of leading dimensions counts as one batch dimension
    (reference window_matmul.py:35-40 flattens them; here the kernels read them where they are).
    """
    if not window_size:
        return (inp * other.transpose(-1, -2)).sum(dim=-1, keepdim=True)
    seq_len, hidden_dim = inp.shape[-2:]
    if other.shape[-2:] != (hidden_dim, seq_len):  # reshaped to the keys' shape like the reference does
        other = other.reshape(-1, hidden_dim, seq_len)
    if torch.is_autocast_enabled("cuda") or _tracing():
        return WindowMatmulFunc.apply(inp, other, window_size)
    return _native.window_matmul(inp, other, window_size)


def unwindow_matmul(inp: torch.Tensor, other: torch.Tensor, window_size: Optional[int]) -> torch.Tensor:
    """Band times values: ``(..., M, 2w+1) x (..., M, N) -> (..., M, N)``.

    A falsy ``window_size`` is the elementwise product ``inp * other``
    (reference window_matmul.py:69-70); leading dimensions as in
    :func:`window_matmul` (reference window_matmul.py:71-76).
    """
    if not window_size:
        return inp * other
    band_shape = (other.shape[-2], 2 * window_size + 1)
    if inp.shape[-2:] != band_shape:
        inp = inp.reshape(-1, *band_shape)
    if torch.is_autocast_enabled("cuda") or _tracing():
        return UnwindowMatmulFunc.apply(inp, other, window_size)
    return _native.unwindow_matmul(inp, other, window_size)
