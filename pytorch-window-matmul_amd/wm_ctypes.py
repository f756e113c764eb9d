"""ctypes binding of libwindow_matmul_hip.so (mirrors include/window_matmul_hip.h).

For callers that want the C ABI without the PyTorch extension in between: the tests,
the benchmark's per-kernel timing, and as a template for bindings from other hosts.
Tensors are only used as (pointer, strides) carriers; work is enqueued on torch's
current stream."""
import ctypes
import math
import os
import re

import torch

HERE = os.path.dirname(os.path.abspath(__file__))
REPO = os.path.dirname(HERE)
LIB_PATH = os.environ.get("WM_LIBRARY_PATH", os.path.join(HERE, "libwindow_matmul_hip.so"))
HEADER = os.path.join(REPO, "include", "window_matmul_hip.h")

DTYPES = {torch.float32: 0, torch.float16: 1, torch.bfloat16: 2, torch.float64: 3}
FORCE_STRIDED = 0x1
NO_ALIGNED_BAND = 0x2
NO_NARROW_BAND = 0x4
NO_LDS_DIRECT = 0x8
NO_SPLIT_F32 = 0x10
ANY_HEAD_WIDTH = 0x20


class Operand(ctypes.Structure):
    _fields_ = [
        ("data", ctypes.c_void_p),
        ("stride_b", ctypes.c_int64),
        ("stride_r", ctypes.c_int64),
        ("stride_c", ctypes.c_int64),
    ]


class GroupedOperand(ctypes.Structure):
    """Operand whose batch may have two levels: groups of `heads` elements, stride_g apart (heads = 0: plain)."""

    _fields_ = [("op", Operand), ("heads", ctypes.c_int64), ("stride_g", ctypes.c_int64)]


def declared_symbols():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(wm_[a-z_0-9]+)\s*\(", text)))


_LIB = None


def lib():
    global _LIB
    if _LIB is None:
        if not os.path.exists(LIB_PATH):
            raise FileNotFoundError(f"{LIB_PATH} is not built; run python pytorch-window-matmul_amd/build.py")
        L = ctypes.CDLL(LIB_PATH)
        P, i64, u32, vp = ctypes.POINTER(Operand), ctypes.c_int64, ctypes.c_uint, ctypes.c_void_p
        tail = [i64, i64, i64, i64, ctypes.c_int, u32, vp]
        L.wm_window_matmul_forward.argtypes = [P, P, P] + tail
        L.wm_unwindow_matmul_forward.argtypes = [P, P, P] + tail
        L.wm_window_matmul_backward.argtypes = [P, P, P, P, P] + tail
        L.wm_unwindow_matmul_backward.argtypes = [P, P, P, P, P] + tail
        L.wm_status_string.restype = ctypes.c_char_p
        L.wm_status_string.argtypes = [ctypes.c_int]
        L.wm_kernel_choice.restype = ctypes.c_char_p
        L.wm_kernel_choice.argtypes = [ctypes.c_int, i64, i64, i64, i64, ctypes.c_int, ctypes.c_int, u32]
        sm_tail = [i64, i64, i64, ctypes.c_double, ctypes.c_int, ctypes.c_int, u32, vp]
        L.wm_band_softmax_forward.argtypes = [P, P] + sm_tail
        L.wm_band_softmax_backward.argtypes = [P, P, P] + sm_tail
        L.wm_band_softmax_kernel_choice.restype = ctypes.c_char_p
        L.wm_band_softmax_kernel_choice.argtypes = [i64, ctypes.c_int, ctypes.c_int, ctypes.c_int, u32]
        L.wm_window_attention_forward.argtypes = [P, P, P, P, vp, i64, i64, i64, i64, ctypes.c_double, ctypes.c_int,
                                                  ctypes.c_int, u32, vp]
        L.wm_window_attention_backward.argtypes = [P, P, P, P, vp, P, P, P, P, vp, i64, i64, i64, i64, ctypes.c_double,
                                                   ctypes.c_int, u32, vp]
        G = ctypes.POINTER(GroupedOperand)
        L.wm_grouped_window_matmul_forward.argtypes = [G, G, P] + tail
        L.wm_grouped_window_matmul_backward.argtypes = [G, G, P, G, G] + tail
        L.wm_grouped_unwindow_matmul_forward.argtypes = [P, G, G] + tail
        L.wm_grouped_unwindow_matmul_backward.argtypes = [P, G, G, P, G] + tail
        L.wm_grouped_window_attention_forward.argtypes = [G, G, G, G, vp, i64, i64, i64, i64, ctypes.c_double, ctypes.c_int,
                                                          ctypes.c_int, u32, vp]
        L.wm_grouped_window_attention_backward.argtypes = [G, G, G, G, vp, G, G, G, G, vp, i64, i64, i64, i64,
                                                           ctypes.c_double, ctypes.c_int, u32, vp]
        L.wm_grouped_score_gradient.argtypes = [G, G, G, P, P, i64, i64, i64, i64, ctypes.c_double, ctypes.c_int, u32, vp]
        L.wm_grouped_window_attention_f32_forward.argtypes = [G, G, G, G, vp, i64, i64, i64, i64, ctypes.c_double, ctypes.c_int,
                                                              ctypes.c_int, u32, vp]
        L.wm_grouped_window_attention_f32_backward.argtypes = [G, G, G, G, vp, G, G, G, G, vp, i64, i64, i64, i64,
                                                               ctypes.c_double, ctypes.c_int, u32, vp]
        L.wm_window_attention_backward_static.argtypes = [P, P, P, P, vp, P, P, P, P, i64, i64, i64, i64,
                                                          ctypes.c_double, ctypes.c_int, u32, vp]
        L.wm_window_attention_supported.argtypes = [i64, i64, i64, ctypes.c_int, ctypes.c_double]
        L.wm_key_rows.argtypes = [P, vp, i64, i64, i64, ctypes.c_int, vp]
        L.wm_grouped_key_rows.argtypes = [G, vp, i64, i64, i64, ctypes.c_int, vp]
        _LIB = L
    return _LIB


def op(t):
    """Operand for a rank-3 tensor (None -> NULL pointer)."""
    if t is None:
        return None
    assert t.dim() == 3
    return ctypes.byref(Operand(t.data_ptr(), t.stride(0), t.stride(1), t.stride(2)))


def grouped_op(t):
    """Grouped operand for a rank-3 tensor, or a rank-4 one (batch, heads, rows, columns)."""
    step, heads, group = (t.stride(0), 0, 0) if t.dim() == 3 else (t.stride(1), t.shape[1], t.stride(0))
    return ctypes.byref(GroupedOperand(Operand(t.data_ptr(), step, t.stride(-2), t.stride(-1)), heads, group))


def _stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def _check(status, what):
    if status != 0:
        raise RuntimeError(f"{what}: {lib().wm_status_string(status).decode()} ({status})")


def window_forward(q, k, w, flags=0, out=None):
    """q (B,M,N), k (B,N,M) (any strides) -> a (B,M,2w+1)."""
    B, M, N = q.shape
    a = torch.empty(B, M, 2 * w + 1, dtype=q.dtype, device=q.device) if out is None else out
    _check(lib().wm_window_matmul_forward(op(q), op(k), op(a), B, M, N, w, DTYPES[q.dtype], flags, _stream()),
           "wm_window_matmul_forward")
    return a


def key_rows(k):
    """wm_key_rows: k (B,N,M), or for wm_grouped_key_rows (batch,heads,N,M), with unit stride along M -> contiguous key rows
    (B,M,N)."""
    *lead, N, M = k.shape
    B = math.prod(lead)
    rows = torch.empty(B, M, N, dtype=k.dtype, device=k.device)
    fn, operand = (lib().wm_key_rows, op(k)) if k.dim() == 3 else (lib().wm_grouped_key_rows, grouped_op(k))
    _check(fn(operand, ctypes.c_void_p(rows.data_ptr()), B, N, M, DTYPES[k.dtype], _stream()), "wm_key_rows")
    return rows


def window_backward(q, k, w, ga, flags=0, want_q=True, want_k=True):
    B, M, N = q.shape
    gq = torch.empty(B, M, N, dtype=q.dtype, device=q.device) if want_q else None
    gk = torch.empty(B, M, N, dtype=q.dtype, device=q.device).transpose(1, 2) if want_k else None
    _check(lib().wm_window_matmul_backward(op(q), op(k), op(ga), op(gq), op(gk), B, M, N, w, DTYPES[q.dtype], flags,
                                          _stream()), "wm_window_matmul_backward")
    return gq, gk


def unwindow_forward(a, v, w, flags=0):
    B, M, N = v.shape
    o = torch.empty(B, M, N, dtype=v.dtype, device=v.device)
    _check(lib().wm_unwindow_matmul_forward(op(a), op(v), op(o), B, M, N, w, DTYPES[v.dtype], flags, _stream()),
           "wm_unwindow_matmul_forward")
    return o


def unwindow_backward(a, v, w, go, flags=0, want_a=True, want_v=True):
    B, M, N = v.shape
    ga = torch.empty(B, M, 2 * w + 1, dtype=v.dtype, device=v.device) if want_a else None
    gv = torch.empty(B, M, N, dtype=v.dtype, device=v.device) if want_v else None
    _check(lib().wm_unwindow_matmul_backward(op(a), op(v), op(go), op(ga), op(gv), B, M, N, w, DTYPES[v.dtype], flags,
                                            _stream()), "wm_unwindow_matmul_backward")
    return ga, gv


def band_softmax_forward(a, scale=1.0, mask=False, flags=0, out=None):
    """a (B,M,2w+1) -> softmax(scale * a) along the band; out may be a itself."""
    B, M, W = a.shape
    p = torch.empty_like(a) if out is None else out
    _check(lib().wm_band_softmax_forward(op(a), op(p), B, M, W // 2, float(scale), int(mask), DTYPES[a.dtype], flags,
                                        _stream()), "wm_band_softmax_forward")
    return p


def band_softmax_backward(p, gp, scale=1.0, mask=False, flags=0, out=None):
    B, M, W = p.shape
    ga = torch.empty_like(p) if out is None else out
    _check(lib().wm_band_softmax_backward(op(p), op(gp), op(ga), B, M, W // 2, float(scale), int(mask),
                                         DTYPES[p.dtype], flags, _stream()), "wm_band_softmax_backward")
    return ga


def score_gradient(go, v, o, probs, w, scale=1.0, flags=0):
    """Gradient of the scores of o = unwindow(softmax(scale * scores), v) from the float32 probabilities (B,M,2w+1); go, v and
    o are (B,M,N) or (batch,heads,M,N)."""
    B, M, _ = probs.shape
    gs = torch.empty_like(probs)
    _check(lib().wm_grouped_score_gradient(grouped_op(go), grouped_op(v), grouped_op(o), op(probs), op(gs), B, M, v.shape[-1],
                                           w, float(scale), DTYPES[probs.dtype], flags, _stream()), "wm_grouped_score_gradient")
    return gs


UNSUPPORTED = 7


def attention_forward(q, k, v, w, scale=1.0, mask=False, flags=0, want_lse=True):
    """q, k, v (B,M,N) row-major (k holds key rows) -> (o (B,M,N), lse (B,M) float32 or None)."""
    B, M, N = q.shape
    o = torch.empty(B, M, N, dtype=q.dtype, device=q.device)
    lse = torch.empty(B, M, dtype=torch.float32, device=q.device) if want_lse else None
    _check(lib().wm_window_attention_forward(op(q), op(k), op(v), op(o),
                                            ctypes.c_void_p(lse.data_ptr()) if want_lse else None, B, M, N, w,
                                            float(scale), int(mask), DTYPES[q.dtype], flags, _stream()),
           "wm_window_attention_forward")
    return o, lse


STATIC_SCRATCH_ROWS = 1 << 21
SCRATCH_TOO_SMALL = 8


def attention_backward_static(q, k, v, o, lse, go, gq, gk, gv, w, scale=1.0, flags=0):
    """wm_window_attention_backward_static: outputs are the caller's (None skips one), the workspace the
    library's static array; the call itself allocates nothing.  Returns the status code."""
    B, M, N = q.shape
    return lib().wm_window_attention_backward_static(op(q), op(k), op(v), op(o), ctypes.c_void_p(lse.data_ptr()),
                                                     op(go), op(gq), op(gk), op(gv), B, M, N, w, float(scale),
                                                     DTYPES[q.dtype], flags, _stream())


def attention_backward(q, k, v, o, lse, go, w, scale=1.0, flags=0, want=(True, True, True)):
    """Gradients (gq, gk, gv), all (B,M,N) row-major, from the forward's o and lse; None where not wanted."""
    B, M, N = q.shape
    gq, gk, gv = (torch.empty(B, M, N, dtype=q.dtype, device=q.device) if x else None for x in want)
    delta = torch.empty(2, B, M, dtype=torch.float32, device=q.device)
    _check(lib().wm_window_attention_backward(op(q), op(k), op(v), op(o), ctypes.c_void_p(lse.data_ptr()), op(go),
                                             op(gq), op(gk), op(gv), ctypes.c_void_p(delta.data_ptr()), B, M, N, w,
                                             float(scale), DTYPES[q.dtype], flags, _stream()),
           "wm_window_attention_backward")
    return gq, gk, gv


def _pointer(t):
    return ctypes.c_void_p(t.data_ptr()) if t is not None else None


def attention_f32_forward(q, k, v, w, scale=1.0, mask=False, flags=0, want_stats=True, out=None):
    """q, k, v (B,M,N) or (batch,heads,M,N) float32 -> (o, stats (2,B,M) or None)."""
    B, M, N = math.prod(q.shape[:-2]), q.shape[-2], q.shape[-1]
    o = torch.empty_like(q) if out is None else out
    stats = torch.empty(2, B, M, dtype=torch.float32, device=q.device) if want_stats else None
    _check(lib().wm_grouped_window_attention_f32_forward(grouped_op(q), grouped_op(k), grouped_op(v), grouped_op(o), _pointer(stats),
                                                         B, M, N, w, float(scale), int(mask), DTYPES[q.dtype], flags, _stream()),
           "wm_grouped_window_attention_f32_forward")
    return o, stats


def attention_f32_backward(q, k, v, o, stats, go, w, scale=1.0, flags=0, want=(True, True, True)):
    """Gradients (gq, gk, gv) laid out like their operands, None where not wanted."""
    B, M, N = math.prod(q.shape[:-2]), q.shape[-2], q.shape[-1]
    grads = [torch.empty_like(t) if x else None for t, x in zip((q, k, v), want)]
    delta = torch.empty(B, M, dtype=torch.float32, device=q.device)
    operands = [grouped_op(t) if t is not None else None for t in grads]
    _check(lib().wm_grouped_window_attention_f32_backward(grouped_op(q), grouped_op(k), grouped_op(v), grouped_op(o), _pointer(stats),
                                                          grouped_op(go), *operands, _pointer(delta), B, M, N, w, float(scale),
                                                          DTYPES[q.dtype], flags, _stream()),
           "wm_grouped_window_attention_f32_backward")
    return tuple(grads)
