"""The fused float32 attention at the limits of what it takes: empty problems, scores and scales of any size."""
import math

import pytest
import torch

import wm_ctypes as abi
from conftest import seeded
from test_gpu_f32_fused_attention import _error, _views, _want


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(2, 0, 64), (0, 128, 64), (8, 2, 0, 64)])
def test_empty_problems(device, shape):
    import window_matmul_kernel as native

    for needs_grad in (False, True):
        xs = [torch.empty(shape, device=device, requires_grad=needs_grad) for _ in range(3)]
        out = native.window_attention_f32(*xs, 40, 0.1, False)
        assert out.shape == shape
        if needs_grad:
            out.sum().backward()
            assert all(x.grad.shape == shape for x in xs)


@pytest.mark.gpu
@pytest.mark.parametrize("N,w", [(64, 40), (128, 70), (32, 300), (75, 33)])
@pytest.mark.parametrize("mask", [False, True])
@pytest.mark.parametrize("q_by,k_by,scale", [(1.0, 1.0, 1e29), (1e10, 1e8, 0.125), (1e18, 1e18, 1e-3), (1.0, 1e-12, 1e24), (1.0, 1.0, 1.3e-38), (1e25, 1.0, 1e-25)])
def test_scores_of_any_size(device, N, w, mask, q_by, k_by, scale):
    """Finite scores and scales give finite results, those of float64: with one key that has all of a row's weight, with equal
    weights, and anything between."""
    views = _views(1, 2, 300, N, device, "flat")
    views[0], views[1] = views[0] * q_by, views[1] * k_by
    out, stats = abi.attention_f32_forward(*views[:3], w, scale, mask)
    grads = abi.attention_f32_backward(*views[:3], out, stats, views[3], w, scale)
    assert all(bool(torch.isfinite(t).all()) for t in (out, *grads))
    # Where one key has all the weight the result is its value row, unless the two largest scores of a row lie within the error of the
    # scores, a few 2^-24 of their size: there, one row in some ten thousand of these, the weights differ.
    off = (out.cpu().double() - _want(views, w, scale, mask)[0]).abs().amax(-1)
    assert float((off > 1e-5).double().mean()) < 0.01


@pytest.mark.gpu
@pytest.mark.parametrize("mask", [False, True])
def test_rows_of_large_negative_scores(device, mask):
    """No neighbour of a row scores above -1e30, c s far below it: the weights go by the differences all the same."""
    views = [t.contiguous() for t in _views(1, 2, 300, 64, device, "flat")]
    views[0], views[1] = views[0].abs(), -views[1].abs()
    for scale in (1e28, 1e29):
        out, _ = abi.attention_f32_forward(*views[:3], 40, scale, mask)
        off = (out.cpu().double() - _want(views, 40, scale, mask)[0]).abs().amax(-1)
        assert bool(torch.isfinite(out).all()) and float((off > 1e-5).double().mean()) < 0.01


@pytest.mark.gpu
@pytest.mark.parametrize("scale", [1e-40, 1e-46, 1e31])
def test_scales_that_the_fused_kernels_leave_to_the_separate_ops(device, scale):
    import window_matmul_kernel as native
    from window_matmul import window_attention

    xs = _views(2, 8, 256, 64, device)[:3]
    assert not native.window_attention_f32_supported(xs[0], 32, scale, False)
    out = window_attention(*xs, 32, scale, True)
    assert bool(torch.isfinite(out).all())
    if scale < 1.0:  # equal weights
        want = _want(xs + [xs[0]], 32, scale, True)[0]
        assert _error(out, want) < 1e-6
