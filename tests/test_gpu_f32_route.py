"""Which float32 calls of window_attention the fused kernels take, on both sides of every line of the rule."""
import math

import pytest
import torch

import wm_ctypes as abi
from test_gpu_f32_fused_attention import _views


def _takes_the_fused_kernels(views, w, training):
    from window_matmul import window_attention

    xs = [t.detach().requires_grad_(training) for t in views[:3]]
    fused, _ = abi.attention_f32_forward(*views[:3], w, 1.0 / math.sqrt(views[0].shape[-1]))
    return torch.equal(window_attention(*xs, w).detach(), fused)


# few tiles of 128 rows: wide heads at wide windows, where a sequence is long enough for them
@pytest.mark.gpu
@pytest.mark.parametrize("heads,M,N,w,fused", [(8, 128, 8, 16, True), (8, 128, 64, 16, True), (8, 128, 64, 15, False), (7, 128, 64, 40, False), (8, 128, 75, 16, True), (8, 128, 24, 16, True),
                                               (2, 4096, 64, 257, True), (2, 4096, 80, 256, True), (2, 4096, 80, 257, False), (4, 4096, 80, 257, True), (1, 1024, 96, 256, True),
                                               (1, 1024, 104, 160, True), (1, 1024, 104, 161, False), (1, 1024, 128, 256, False), (1, 1024, 127, 256, True), (32, 128, 128, 256, True),
                                               (31, 128, 128, 256, True), (1, 4096, 128, 256, True)])
def test_inference(device, heads, M, N, w, fused):
    with torch.no_grad():
        assert _takes_the_fused_kernels(_views(1, heads, M, N, device), w, False) == fused


# widths beyond 112 that 8 does not divide (the other lines: test_route_of_training_and_of_a_result_changed_in_place)
@pytest.mark.gpu
@pytest.mark.parametrize("heads,M,N,w,fused", [(8, 128, 127, 32, True), (1023, 128, 127, 32, True), (1024, 128, 127, 39, False), (1024, 128, 127, 40, True), (1024, 128, 111, 32, True)])
def test_training(device, heads, M, N, w, fused):
    assert _takes_the_fused_kernels(_views(1, heads, M, N, device), w, True) == fused
