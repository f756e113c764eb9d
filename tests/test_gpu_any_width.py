"""Fused window attention at head widths that 16 does not divide: rows are read and written where they lie, the last
16-byte piece of a row moved back so that it ends with the row."""
import math

import pytest
import torch

from conftest import seeded
from oracle import attention_oracle as ao
from test_gpu_attention import close

pytestmark = pytest.mark.gpu
BF16, F16 = torch.bfloat16, torch.float16

# batch, heads, M, N, w: one piece, odd piece counts, odd widths (rows of 2-byte alignment), every kernel of both directions
# (one-pass and chunked forward; one-kernel and two-kernel backward), sequences below and across a tile
CASES = [(2, 2, 70, 8, 3), (1, 3, 131, 12, 40), (2, 1, 300, 20, 16), (2, 3, 260, 40, 20), (1, 2, 515, 60, 64),
         (1, 5, 200, 60, 100), (3, 2, 129, 57, 33), (2, 2, 300, 75, 8), (1, 3, 333, 75, 70), (2, 1, 257, 72, 24),
         (1, 2, 400, 100, 130), (1, 2, 300, 127, 50), (1, 1, 5, 60, 2)]


def _views(batch, heads, M, N, dtype, device, fill=None):
    """(batch, heads, M, N) views of (batch, M, heads * N) projections: q, k, v, grad."""
    flat = [seeded((batch, M, heads * N), 300 + s, dtype).to(device) for s in range(4)]
    if fill is not None:
        for t in flat:
            t[..., N:] = fill
    return [t.view(batch, M, heads, N).transpose(1, 2) for t in flat]


def _step(views, w, mask):
    from window_matmul import window_attention

    q, k, v = (t.detach().requires_grad_(True) for t in views[:3])
    out = window_attention(q, k, v, w, mask_out_of_range=mask)
    assert type(out.grad_fn).__name__ == "WindowAttentionFuncBackward"
    out.backward(views[3])
    return out.detach(), q.grad, k.grad, v.grad


@pytest.mark.parametrize("dtype", [BF16, F16], ids=["bfloat16", "float16"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "B%dx%d_M%d_N%d_w%d" % c)
def test_step_against_oracle(device, case, dtype):
    batch, heads, M, N, w = case
    views = _views(batch, heads, M, N, dtype, device)
    flat = [t.reshape(batch * heads, M, N).contiguous() for t in views]
    host = [t.cpu() for t in flat]
    scale = 1.0 / math.sqrt(N)
    for mask in (False, True):
        want_o, _ = ao.window_attention_forward(*host[:3], w, scale, mask)
        want = [want_o, *ao.window_attention_backward(*host[:3], w, host[3], scale, mask)]
        got = _step(views, w, mask)
        for x, y in zip(got, want):
            close(x.reshape(batch * heads, M, N), y)
        for x, y in zip(got, _step(flat, w, mask)):  # another layout, the same bits
            assert torch.equal(x.reshape(batch * heads, M, N), y)
        assert got[1].stride() == views[0].stride()  # gradients are laid out like their operands


# N, w of launches with more workgroups than any rule for few tiles admits: even widths, which take the kernels that load
# straight into LDS in their streaming form, certain from w = 79 on to have chunks of 64 rows wholly inside the band of a
# wavefront's 32; one to four blocks of 32 result columns
@pytest.mark.parametrize("mask", [False, True], ids=["zero_filled", "masked"])
@pytest.mark.parametrize("N,w", [(60, 64), (60, 100), (14, 70), (22, 70), (42, 130), (90, 90), (76, 130), (100, 90), (100, 130), (126, 40), (36, 33)])
def test_streaming_kernels_against_oracle(device, N, w, mask):
    host = [seeded((1, 300, N), 330 + s, BF16) for s in range(4)]
    times = 257
    got = _step([t.to(device).repeat(times, 1, 1) for t in host], w, mask)
    scale = 1.0 / math.sqrt(N)
    want_o, _ = ao.window_attention_forward(*host[:3], w, scale, mask)
    for x, y in zip(got, [want_o, *ao.window_attention_backward(*host[:3], w, host[3], scale, mask)]):
        assert torch.equal(x[0], x[-1]) and torch.equal(x[0], x[100])
        close(x[:1], y)


# B, M, N, w: narrow and wide windows, up to and above N = 64, few tiles and more than any rule for few tiles admits
@pytest.mark.parametrize("B,M,N,w", [(2, 150, 41, 10), (2, 300, 41, 70), (2, 150, 75, 20), (2, 300, 75, 100), (1, 300, 127, 50),
                                     (270, 40, 41, 70), (270, 40, 75, 33)])
@pytest.mark.parametrize("rows", ["padded", "every second"])
def test_odd_widths_in_rows_on_dword_addresses(device, B, M, N, w, rows):
    """Rows that start on a multiple of 4 bytes although N is odd: their last piece does not, so they are no case for
    the loads straight into LDS and give the bits of contiguous rows."""
    def view(seed):
        if rows == "padded":
            return seeded((B, M, N + 5), seed, BF16).to(device)[..., :N]
        return seeded((B, 2 * M, N), seed, BF16).to(device)[:, ::2]

    views = [view(320 + s) for s in range(4)]
    assert all(t.stride(1) % 2 == 0 and t.data_ptr() % 4 == 0 for t in views)
    flat = [t.contiguous() for t in views]
    got, same = _step(views, w, False), _step(flat, w, False)
    host = [t[:2].cpu() for t in flat]
    scale = 1.0 / math.sqrt(N)
    want_o, _ = ao.window_attention_forward(*host[:3], w, scale, False)
    want = [want_o, *ao.window_attention_backward(*host[:3], w, host[3], scale, False)]
    for x, y, z in zip(got, same, want):
        assert torch.equal(x, y)
        close(x[:2], z)


@pytest.mark.parametrize("N,w", [(60, 20), (60, 100), (75, 20), (75, 100), (41, 60)])
def test_neighbours_in_memory_do_not_matter(device, N, w):
    """Row pieces never reach into the next head: with NaN in all other heads the first one keeps its bits."""
    clean = _step(_views(1, 3, 300, N, BF16, device), w, False)
    dirty = _step(_views(1, 3, 300, N, BF16, device, fill=float("nan")), w, False)
    for x, y in zip(clean, dirty):
        assert torch.equal(x[:, 0], y[:, 0])


def test_register_staged_kernels_agree(device):
    """Rows on dword addresses take the kernels that load straight into LDS, the same rows two bytes further the
    register-staged ones: the same sums, in float32, before one rounding."""
    from window_matmul import window_attention

    N, w = 60, 100
    q, k, v = (seeded((2, 300, N), s, F16).to(device) for s in range(3))

    def shifted(t):
        room = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:].view(t.shape)
        return room.copy_(t)

    a, b = window_attention(q, k, v, w), window_attention(*(shifted(t) for t in (q, k, v)), w)
    torch.testing.assert_close(a, b, rtol=2 ** -9, atol=2 ** -11)


def test_refused_without_the_flag_and_chain_under_autocast(device):
    from window_matmul import window_attention

    q = seeded((2, 64, 60), 1, BF16).to(device)
    with torch.autocast("cuda"):
        assert window_attention(q, q, q, 5).dtype == F16  # the separate ops compute in float16 there
    assert window_attention(q, q, q, 5).dtype == BF16
