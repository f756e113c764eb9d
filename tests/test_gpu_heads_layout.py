"""Operands whose batch has two levels of strides: (batch, M, heads * N) projections seen as (batch, heads, M, N), the
way the reference's own tests build them (reference tests/utils.py:38-64), read in place.  The kernels, their
order of summation and their results are those of the same call on contiguous copies: equal bit for bit."""
import ctypes

import pytest
import torch

import wm_ctypes as abi
from conftest import seeded

F32, F16, BF16, F64 = torch.float32, torch.float16, torch.bfloat16, torch.float64

# (batch, heads, M, N, w, dtype): one shape per kernel family at a ragged M; batch and heads of one; head counts
# that are and are not multiples of the eight elements dealt to the chip's eight dies
SHAPES = [
    (3, 5, 133, 64, 2, BF16), (2, 8, 200, 64, 8, BF16), (3, 3, 259, 64, 33, F16), (2, 5, 700, 64, 256, BF16),
    (2, 3, 515, 128, 96, F16), (2, 9, 131, 16, 40, BF16), (1, 7, 300, 80, 20, BF16), (5, 1, 300, 80, 20, F16),
    (3, 5, 133, 64, 4, F32), (2, 3, 300, 64, 20, F32), (2, 3, 300, 80, 100, F32), (2, 3, 260, 40, 15, F32),
    (2, 3, 97, 20, 5, BF16), (2, 3, 97, 75, 9, F32), (2, 3, 65, 3, 4, F64), (2, 2, 90, 144, 9, BF16),
]


def head_view(batch, heads, M, N, seed, dtype, device):
    return seeded((batch, M, heads * N), seed, dtype).to(device).view(batch, M, heads, N).transpose(1, 2)


def flat(t):
    return t.reshape(-1, *t.shape[-2:]).contiguous()


def steps(fn, inputs, grad):
    inputs = [t.detach().requires_grad_(True) for t in inputs]
    out = fn(*inputs)
    return [out.detach()] + list(torch.autograd.grad(out, inputs, grad))


@pytest.mark.gpu
@pytest.mark.parametrize("batch,heads,M,N,w,dtype", SHAPES)
def test_projection_views_equal_contiguous_operands(device, batch, heads, M, N, w, dtype):
    from window_matmul import unwindow_matmul, window_attention, window_matmul

    q, k, v, go = (head_view(batch, heads, M, N, s, dtype, device) for s in (1, 2, 3, 4))
    band = seeded((batch, heads, M, 2 * w + 1), 5, dtype).to(device)
    pairs = [
        (lambda a, b: window_matmul(a, b.transpose(-1, -2), w), (q, k), band),
        (lambda a, b: unwindow_matmul(a, b, w), (band, v), go),
        (lambda a, b, c: window_attention(a, b, c, w), (q, k, v), go),
    ]
    for fn, inputs, grad in pairs:
        got = steps(fn, inputs, grad)
        want = steps(fn, [flat(t) for t in inputs], flat(grad))
        for x, y in zip(got, want):
            assert torch.equal(flat(x), y)
        for g, t in zip(got[1:], inputs):  # a gradient is laid out like the operand it belongs to
            assert N * dtype.itemsize % 16 or N > 128 or g.stride() == t.stride()


@pytest.mark.gpu
def test_more_levels_and_different_groupings(device):
    """Three levels of batch strides are copied; operands grouped differently, or expanded, meet in one call."""
    from window_matmul import window_attention

    M, N, w = 150, 64, 20
    base = seeded((2, 3, M, 4, N), 1, BF16).to(device).transpose(2, 3)                 # (2, 3, 4, M, N)
    k = seeded((2, 3, 4, M, N), 2, BF16).to(device)
    v = seeded((6, M, 2, 2 * N), 3, BF16).to(device)[..., :N].transpose(1, 2)          # (6, 2, M, N), padded rows
    v = torch.cat([v, v], 1).view(2, 3, 4, M, N)
    views = (base, k[:, :, :1].expand_as(k), v)
    three = base[:, ::2].expand(2, 2, 4, M, N)  # leading strides that do not merge
    for q in (base, three):
        kk, vv = (t[:, :q.shape[1]] for t in views[1:])
        got = window_attention(q, kk, vv, w)
        assert torch.equal(got.flatten(0, 2), window_attention(flat(q), flat(kk), flat(vv), w))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [F32, F16, BF16, F64])
@pytest.mark.parametrize("batch,heads,N,M,w", [(3, 5, 64, 133, 20), (2, 2, 128, 64, 9), (1, 3, 16, 1000, 40), (2, 3, 80, 97, 5)])
def test_keys_as_columns_of_a_channels_first_projection(device, dtype, batch, heads, N, M, w):
    """(batch, heads, N, M) keys cut out of a (batch, 3 * heads * N, M) projection: two batch levels and unit stride along M,
    made into key rows by the library's own transpose."""
    from window_matmul import window_matmul

    for pad in (0, 7):  # rows that start on a 16-byte boundary, and rows that do not
        qkv = seeded((batch, 3 * heads, N, M + pad), 11, dtype).to(device)
        k = qkv[:, heads:2 * heads, :, pad:]
        want = flat(k.transpose(-1, -2))
        assert torch.equal(abi.key_rows(k), want)
        q = seeded((batch, heads, M, N), 12, dtype).to(device)
        grad = seeded((batch, heads, M, 2 * w + 1), 13, dtype).to(device)
        got = steps(lambda a, b: window_matmul(a, b, w), (q, k), grad)
        same = steps(lambda a, b: window_matmul(a, b.transpose(-1, -2), w), (flat(q), want), flat(grad))
        assert torch.equal(flat(got[0]), same[0]) and torch.equal(flat(got[1]), same[1])
        assert torch.equal(flat(got[2].transpose(-1, -2)), same[2])


def test_grouped_operands_of_a_call_share_their_heads():
    L, P = abi.lib(), ctypes.byref
    plain = abi.Operand(ctypes.c_void_p(16), 0, 0, 0)
    two, three = (abi.GroupedOperand(plain, h, 0) for h in (2, 3))
    negative = abi.GroupedOperand(plain, -1, 0)
    assert L.wm_grouped_key_rows(P(negative), ctypes.c_void_p(16), 1, 8, 8, 2, None) == 2
    assert L.wm_grouped_key_rows(P(two), ctypes.c_void_p(16), 1, 8, 8, 2, None) == 7  # no unit column stride
    tail = (1, 4, 4, 1, 0, 0, None)
    assert L.wm_grouped_window_matmul_forward(P(two), P(three), P(plain), *tail) == 2
    assert L.wm_grouped_unwindow_matmul_forward(P(plain), P(negative), P(two), *tail) == 2
    assert L.wm_grouped_window_attention_forward(P(two), P(two), P(two), P(three), None, 1, 4, 16, 1, 1.0, 0, 1, 0, None) == 2


def test_heads_out_of_range_are_refused():
    """64-bit counts that 32 bits would turn into another grouping (2^32 + 2: into pairs) or into none at all (2^32)."""
    L, P = abi.lib(), ctypes.byref
    plain = abi.Operand(ctypes.c_void_p(16), 0, 0, 0)
    for heads in (2 ** 32 + 2, 2 ** 32, 2 ** 31, -1, -2 ** 32):
        odd = abi.GroupedOperand(plain, heads, 0)
        assert L.wm_grouped_window_matmul_forward(P(odd), P(odd), P(plain), 1, 4, 4, 1, 0, 0, None) == 2
        assert L.wm_grouped_unwindow_matmul_forward(P(plain), P(odd), P(odd), 1, 4, 4, 1, 0, 0, None) == 2
        assert L.wm_grouped_window_attention_forward(P(odd), P(odd), P(odd), P(odd), None, 1, 4, 16, 1, 1.0, 0, 1, 0, None) == 2
