"""The fused float32 attention at the limits of what it takes."""
import pytest
import torch


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
