"""Band softmax of long rows, which sit in registers up to 3072 elements: the edges of the shape classes, against float64."""
import pytest
import torch

import wm_ctypes as abi
from conftest import seeded

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mask", [False, True], ids=["zero_filled", "masked"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=["float32", "bfloat16", "float16"])
@pytest.mark.parametrize("w", [639, 640, 767, 768, 1023, 1024, 1279, 1280, 1500, 1535, 1536])
def test_long_rows(device, w, dtype, mask):
    B, M, scale = 2, 9, 0.3
    W = 2 * w + 1
    a, go = (seeded((B, M, W), 700 + s, dtype, 3.0) for s in range(2))
    i, j = torch.arange(M)[:, None], torch.arange(W)[None, :] - w
    outside = (i + j < 0) | (i + j >= M) if mask else torch.zeros(M, W, dtype=torch.bool)
    x = a.double().masked_fill(outside, float("-inf"))
    want = torch.softmax(scale * x, -1)
    got = abi.band_softmax_forward(a.to(device), scale, mask)
    # one rounding of the result; before it, in float32, an exponent of up to 16 rounded once (2^-21 of a probability) and
    # a sum of up to 3073 terms over 64 lanes
    eps = {torch.float32: 2 ** -24, torch.bfloat16: 2 ** -8, torch.float16: 2 ** -11}[dtype]
    torch.testing.assert_close(got.cpu().double(), want, rtol=eps + 2 ** -20, atol=2 ** -25)
    assert bool((got.cpu()[:, outside] == 0).all())
    probs = want.to(dtype)
    got_ga = abi.band_softmax_backward(probs.to(device), go.to(device), scale, mask)
    p = probs.double()
    exact = scale * p * (go.double() - (p * go.double()).sum(-1, keepdim=True))
    torch.testing.assert_close(got_ga.cpu().double(), exact, rtol=eps + 2 ** -20, atol=2 ** -21)
