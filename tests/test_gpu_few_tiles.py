"""Fused window attention with few tiles: the streamed side of a tile is shared out among wavefronts, whose sums meet in
LDS.  The same problems in a batch large enough for the kernels that do not share must agree."""
import math

import pytest
import torch

import wm_ctypes as abi
from conftest import seeded
from oracle import attention_oracle as ao
from test_gpu_attention import close

pytestmark = pytest.mark.gpu

# B, M, N, w: one to four blocks of 32 result columns; sequences around a workgroup (64, 32 rows), a block (32) and a chunk
# (128); windows at the rule's lower end, inside a chunk, over several chunks, beyond the sequence; shares without any key
CASES = [(1, 5, 64, 40), (2, 33, 128, 32), (1, 64, 16, 33), (2, 65, 48, 64), (1, 127, 64, 100), (3, 129, 128, 300),
         (1, 500, 32, 80), (2, 1000, 64, 256), (1, 1030, 80, 200), (2, 777, 112, 95), (1, 2000, 128, 512)]


def _run(q, k, v, go, w, scale, mask, want=(True, True, True)):
    o, lse = abi.attention_forward(q, k, v, w, scale, mask)
    return (o, lse, *abi.attention_backward(q, k, v, o, lse, go, w, scale, want=want))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bfloat16", "float16"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "B%d_M%d_N%d_w%d" % c)
def test_shares_agree_with_oracle_and_with_large_batches(device, case, dtype):
    B, M, N, w = case
    scale = 1.0 / math.sqrt(N)
    host = [seeded((B, M, N), 500 + s, dtype) for s in range(4)]
    few = [t.to(device) for t in host]
    times = 257  # more tiles than any rule for sharing admits
    many = [t.repeat(times, 1, 1) for t in few]
    for mask in (False, True):
        got = _run(*few, w, scale, mask)
        want_o, want_lse = ao.window_attention_forward(*host[:3], w, scale, mask)
        want = ao.window_attention_backward(*host[:3], w, host[3], scale, mask)
        close(got[0], want_o)
        torch.testing.assert_close(got[1].cpu().double(), torch.from_numpy(want_lse), rtol=5e-3, atol=5e-3)
        for x, y in zip(got[2:], want):
            close(x, y)
        for x, y in zip(got, _run(*few, w, scale, mask)):
            assert torch.equal(x, y)  # the shares are added in a fixed order
        for x, y in zip(got, _run(*many, w, scale, mask)):
            # float32 sums in another order, then one rounding: one unit of the storage type, or where a result
            # cancels, of the few terms it is made of
            y = y.view(times, *x.shape)
            assert torch.equal(y[0], y[-1])
            torch.testing.assert_close(x.float(), y[0].float(), rtol=2e-2, atol=2e-2)


@pytest.mark.parametrize("M,N,w", [(100, 128, 40), (100, 64, 70)])
def test_rows_far_apart_are_not_shared_out(device, M, N, w):
    """Row strides at which 32-bit offsets reach the chunk past the last of the kernels that do not share, 192 rows beyond
    the sequence, but not that of the ones that do, 256: the bits of the former."""
    stride = (2 ** 30 // (M + 224)) // 64 * 64
    assert (M + 192) * stride * 2 < 2 ** 31 - 1 <= (M + 256) * stride * 2
    room = torch.empty(M * stride, dtype=torch.bfloat16, device=device)
    host = [seeded((1, M, N), 540 + s, torch.bfloat16) for s in range(4)]
    far = [room.as_strided((1, M, N), (M * stride, stride, 1), N * s).copy_(t) for s, t in enumerate(host)]
    near = [t.to(device) for t in host]
    times = 257
    many = [x[0] for x in _run(*(t.repeat(times, 1, 1) for t in near), w, 0.1, False) if x.dim() == 3]
    got = [x[0] for x in _run(*far, w, 0.1, False) if x.dim() == 3]
    shared = [x[0] for x in _run(*near, w, 0.1, False) if x.dim() == 3]
    assert all(torch.equal(x, y) for x, y in zip(got, many))
    assert not all(torch.equal(x, y) for x, y in zip(shared, many))  # otherwise the above says nothing


@pytest.mark.parametrize("N,w", [(60, 40), (76, 130), (126, 64), (127, 64)])
def test_shares_at_widths_16_does_not_divide(device, N, w):
    """Even widths; an odd one is no case for these kernels, whatever the window, and has to come out right all the same."""
    from window_matmul import window_attention

    host = [seeded((2, 300, N), 510 + s, torch.bfloat16) for s in range(4)]
    q, k, v = (t.to(device).requires_grad_(True) for t in host[:3])
    out = window_attention(q, k, v, w)
    out.backward(host[3].to(device))
    scale = 1.0 / math.sqrt(N)
    close(out, ao.window_attention_forward(*host[:3], w, scale, False)[0])
    for x, y in zip((q.grad, k.grad, v.grad), ao.window_attention_backward(*host[:3], w, host[3], scale, False)):
        close(x, y)


@pytest.mark.parametrize("part", [(True, False, False), (False, True, True), (False, True, False), (False, False, True)])
def test_part_of_the_gradients(device, part):
    q, k, v, go = (seeded((1, 300, 128), 520 + s, torch.bfloat16).to(device) for s in range(4))
    full = _run(q, k, v, go, 70, 0.1, False)[2:]
    for wanted, x, y in zip(part, _run(q, k, v, go, 70, 0.1, False, want=part)[2:], full):
        assert (x is None) == (not wanted)
        assert x is None or torch.equal(x, y)


def test_large_scores(device):
    """Every share raises its own maximum; scores far from zero in both directions, one share without a key in reach."""
    q, k, v = (seeded((1, 400, 64), 530 + s, torch.bfloat16, 4.0) for s in range(3))
    for mask in (False, True):
        want_o, want_lse = ao.window_attention_forward(q, k, v, 50, 1.0, mask)
        o, lse = abi.attention_forward(q.to(device), k.to(device), v.to(device), 50, 1.0, mask)
        torch.testing.assert_close(lse.cpu().double(), torch.from_numpy(want_lse), rtol=5e-3, atol=5e-3)
        torch.testing.assert_close(o.cpu().double(), torch.from_numpy(want_o), rtol=2e-2, atol=8e-2)  # values of size 4
