"""Window attention in one call: ``unwindow_matmul(softmax(scale * window_matmul(q, k^T, w)), v, w)``.

The reference package stops at the two banded matmuls; its callers write the chain above
themselves (reference tests/test_attention.py:57-63).  This function is that chain with the
same semantics, as an addition next to the unchanged two-function API.  For float16 /
bfloat16 inputs whose last dimension is 8 to 128 it runs fused kernels that
never write the ``(…, M, 2w+1)`` band to memory (forward keeps only the log-sum-exp of every
row, backward recomputes the probabilities), and for float32 inputs of such widths kernels that do the same at
float32 accuracy where they are faster; everything else runs the chain of the separate ops of this package, on the GPU as well.
"""
import math
from typing import Optional

import torch

import window_matmul_kernel as _native

from .band_softmax import band_softmax
from .window_matmul import _tracing, unwindow_matmul, window_matmul


# tensors below this many elements take the fused kernels: most of them are bound by the host's launches, of which those need fewer
_HOST_BOUND_ELEMENTS = 32 << 20


def _chain_is_faster(window_size: int, width: int, elements: int) -> bool:
    """Whether a training step is faster through the separate ops than through the fused kernels.
    Up to N = 64 the fused backward is one kernel at narrow windows and the fused step wins or nearly ties at
    every window (chain / fused on 100 M elements, us: N = 16 650 / 691 at w = 1 and 687 / 693 at w = 2, N = 32
    465 / 478 and 479 / 482).  Above N = 64 the recomputing two-kernel backward costs the same
    at every narrow window, and the chain wins up to w = 32 at N = 128 (B16 M32768: 356 / 535 at
    w = 4, 506 / 548 at w = 32, 597 / 583 at w = 40; B96 M4096: 372 / 396 at w = 32, 430 / 424 at w = 36, as
    (8, 12) projection views 388 / 422 at w = 32) and up to about w = 24 at N = 96 (B96 M4096: 303 / 305 at w = 24, 328 / 304 at
    w = 32; N = 80 232 / 252 at w = 16, 288 / 272 at w = 24).  Small problems are bound by the host, which issues seven
    launches for the chain and three for the fused step: at B7 M3001 83-90 / 47 at N = 80 and 128, w = 4 and 24, so below
    about 32 M elements per tensor the fused kernels are always taken.  (At 20 M elements neither side is bound by
    the host any more: N = 80 124 / 171 at w = 4, 207 / 183 at w = 24; N = 128 196 / 242 and 243 / 251; at 8 M 121 / 76.)
    Widths that 16 does not divide always are: the separate ops pad every operand there (B4x12 M16384: 1271 / 806 at N = 75,
    w = 4; 1979 / 949 at N = 120, w = 4; 1015 / 368 at N = 60, w = 1)."""
    if width <= 64 or width % 16 or elements < _HOST_BOUND_ELEMENTS:
        return False
    return window_size <= (24 if width <= 96 else 32)


class WindowAttentionFunc(torch.autograd.Function):
    """Fused kernels on ``(..., M, N)`` operands; ``k`` holds key rows (not transposed).  What
    :func:`window_attention` takes under ``torch.jit.trace``; elsewhere the native module's own node does the same."""

    @staticmethod
    def forward(ctx, q, k, v, window_size: int, scale: float, mask_out_of_range: bool):
        out, lse = _native.window_attention_forward(q, k, v, window_size, scale, mask_out_of_range)
        ctx.save_for_backward(q, k, v, out, lse)
        ctx.window_size = window_size
        ctx.scale = scale
        return out

    @staticmethod
    def backward(ctx, grad_output):
        q, k, v, out, lse = ctx.saved_tensors
        gq, gk, gv = _native.window_attention_backward(q, k, v, out, lse, grad_output, ctx.window_size, ctx.scale,
                                                       *ctx.needs_input_grad[:3])
        return gq, gk, gv, None, None, None


def window_attention(query: torch.Tensor, key: torch.Tensor, value: torch.Tensor, window_size: int,
                     scale: Optional[float] = None, mask_out_of_range: bool = False) -> torch.Tensor:
    """Local attention of every position over its ``2 * window_size + 1`` neighbours.

    ``query``, ``key``, ``value`` are ``(..., M, N)`` (``key`` NOT transposed, unlike the second
    argument of ``window_matmul``); the result is ``(..., M, N)``.  ``scale`` defaults to
    ``1 / sqrt(N)``.  With ``mask_out_of_range=False`` (default) the result equals the reference
    callers' chain exactly as they write it: neighbours that fall outside the sequence take part
    in the softmax with score 0 and add nothing to the output.  With ``True`` they are left out
    of the softmax, which is the usual definition of sliding-window attention.

    The result may be changed in place before the backward (``out += residual``), except for float16 /
    bfloat16 training whose last dimension is a multiple of 16: its backward may read the result, and then raises.
    """
    if query.shape != key.shape or query.shape != value.shape or query.dim() < 2:
        raise RuntimeError("Input mismatch")
    scale = 1.0 / math.sqrt(query.shape[-1]) if scale is None else float(scale)
    if not window_size:
        # a single neighbour: the softmax is 1 and the output is the value itself, as in the
        # chain (reference tests/test_attention.py:75-87); kept differentiable through torch ops
        score = (query * key).sum(-1, keepdim=True) * scale
        return torch.softmax(score, -1) * value
    # With a very narrow band the recomputing backward of the fused kernels costs more than the
    # band it avoids writing, so training there goes through the separate ops.
    training = torch.is_grad_enabled() and (query.requires_grad or key.requires_grad or value.requires_grad)
    autocast, tracing = torch.is_autocast_enabled("cuda"), _tracing()
    # Head widths that 16 does not divide: the chain computes in float16 inside an autocast region, so it stays there.
    if _native.window_attention_supported(query, window_size, scale, not autocast) and not (
            training and _chain_is_faster(window_size, query.shape[-1], query.numel())):
        fused = WindowAttentionFunc.apply if tracing else _native.window_attention
        return fused(query, key, value, window_size, scale, bool(mask_out_of_range))
    if not autocast and not tracing and _native.window_attention_f32_supported(query, window_size, scale, training):
        return _native.window_attention_f32(query, key, value, window_size, scale, bool(mask_out_of_range))
    att = window_matmul(query, key.transpose(-1, -2), window_size)
    return unwindow_matmul(band_softmax(att, scale, mask_out_of_range), value, window_size)
