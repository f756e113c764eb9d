"""float32 attention as training takes it: whichever route a head width goes, no gradient is farther from float64 than the separate ops'."""
import math

import pytest
import torch

from window_matmul import band_softmax, unwindow_matmul, window_attention, window_matmul

def _float64(q, k, v, go, w, scale, mask):
    """One sequence after the other: (out, grad_q, grad_k, grad_v) of dense masked attention."""
    M = q.shape[1]
    i = torch.arange(M, device=q.device)
    outside = (i[None] - i[:, None]).abs() > w
    zeros = (w - i).clamp(min=0) + (i + w - (M - 1)).clamp(min=0) if not mask else torch.zeros_like(i)  # neighbours outside: score 0
    results = []
    for q, k, v, go in zip(*(t.double() for t in (q, k, v, go))):
        s = (q @ k.T * scale).masked_fill(outside, -math.inf)
        top = s.amax(-1, keepdim=True).clamp(min=0.0)
        p = torch.exp(s - top)
        p = p / (p.sum(-1, keepdim=True) + zeros[:, None] * torch.exp(-top))
        out = p @ v
        ds = scale * p * (go @ v.T - (go * out).sum(-1, keepdim=True))
        results.append((out, ds @ k, ds.T @ q, p.T @ go))
    return [torch.stack(t) for t in zip(*results)]


def _quotients(device, B, M, N, w, factor):
    """Root mean square of the relative distance over four inputs, with and without mask, window_attention over the separate ops:
    out, grad_q, grad_k, grad_v, and out without a graph."""
    mine, theirs = [0.0] * 5, [0.0] * 5
    for seed in range(4):
        g = torch.Generator(device=device).manual_seed(9000 + seed)
        q, k, v, go = (torch.randn((B, M, N), generator=g, device=device) for _ in range(4))
        q, scale, mask = q * factor, 1.0 / math.sqrt(N), bool(seed % 2)
        want = _float64(q, k, v, go, w, scale, mask)
        for total, separate in ((mine, False), (theirs, True)):
            xs = [t.detach().requires_grad_(True) for t in (q, k, v)]
            if separate:
                out = unwindow_matmul(band_softmax(window_matmul(xs[0], xs[1].transpose(-1, -2), w), scale, mask), xs[2], w)
            else:
                out = window_attention(*xs, w, scale, mask)
            grads = torch.autograd.grad(out, xs, go)
            with torch.no_grad():
                plain = out if separate else window_attention(q, k, v, w, scale, mask)
            for i, (x, y) in enumerate(zip((out.detach(), *grads, plain.detach()), (*want, want[0]))):
                total[i] += float(((x.double() - y).norm() / y.norm()) ** 2)
    return [(x / y) ** 0.5 for x, y in zip(mine, theirs)]


@pytest.mark.gpu
@pytest.mark.parametrize("factor", [1.0, 3.0])
@pytest.mark.parametrize("w", [64, 100])
@pytest.mark.parametrize("N", [8, 24, 32, 33, 40, 41, 48, 60, 64, 75, 101, 127])
def test_no_less_accurate_than_the_separate_ops(device, N, w, factor):
    """They are at 0.44 to 0.947 where the fused kernels run; training at N = 32 would be at 1.06 and goes through the separate ops."""
    quotients = _quotients(device, 32, 1024, N, w, factor)
    assert max(quotients) <= (1.0 if N <= 32 else 0.97) and quotients[4] <= 0.97, quotients


@pytest.mark.gpu
@pytest.mark.parametrize("N", [60, 64])
def test_a_row_with_one_neighbour_has_no_gradient_of_its_score(device, N):
    q, k, v = (torch.randn((16, 1, N), device=device, requires_grad=True) for _ in range(3))
    grads = torch.autograd.grad(window_attention(q, k, v, 40, None, True).sum(), (q, k, v))
    assert not grads[0].any() and not grads[1].any() and torch.equal(grads[2], torch.ones_like(v))


@pytest.mark.gpu
@pytest.mark.parametrize("N,w", [(33, 256), (33, 257), (36, 600), (39, 1500), (47, 256), (47, 600), (54, 600), (54, 601), (63, 1140), (70, 1500)])
def test_wide_windows_of_widths_that_8_does_not_divide(device, N, w):
    """The separate ops pad these beyond w = 256; the fused kernels would be at 1.04 to 1.13 up to N = 47, at 1.02 at N = 63, w = 1500."""
    quotients = _quotients(device, 8, 2048, N, w, 4.0)
    assert max(quotients) <= 1.0, quotients
