// Python module `window_matmul_kernel` for PyTorch-ROCm: the same four functions the
// reference's native module exports (reference csrc/window_matmul/window_matmul.cpp:100-106),
// implemented as a thin layer over the C ABI in include/window_matmul_hip.h.
//
// What this layer does: argument checks with the reference's error
// texts (reference cuda/utils.cuh:3-4, cuda/window_matmul_cuda.cu:226-232, 323-329),
// layout normalisation, output allocation with the input's dtype and device, device
// guard, current-stream lookup, and the call into libwindow_matmul_hip.so; and, in its second half, the
// differentiable forms of these functions, which the Python package calls.
//
// There is deliberately no CPU implementation behind this module: tensors that do not
// live on the GPU raise, as the reference does for GPU tensors in a CPU-only build
// (reference window_matmul.cpp:15).
#include <torch/extension.h>

#include <algorithm>
#include <stdexcept>
#include <string>
#include <vector>

#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>

#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_cpp_function.h>

#include <tuple>

#include "../../include/window_matmul_hip.h"

namespace {

void check_gpu(const torch::Tensor &t, const char *name) {
  TORCH_CHECK(t.device().is_cuda(), name,
              " must be CUDA tensor (window_matmul_kernel is built for MI355X only and has no CPU path)");
}

int abi_dtype(const torch::Tensor &t, const char *op) {
  switch (t.scalar_type()) {
    case at::kFloat: return WM_DTYPE_F32;
    case at::kHalf: return WM_DTYPE_F16;
    case at::kBFloat16: return WM_DTYPE_BF16;
    case at::kDouble: return WM_DTYPE_F64;
    default: TORCH_CHECK(false, "\"", op, "\" not implemented for '", c10::toString(t.scalar_type()), "'");
  }
  return -1;
}

bool aligned16(const torch::Tensor &t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; }

// A tensor (..., R, C) is a batch of (R, C) matrices.  Its leading dimensions are read in place when they amount to
// at most two levels of strides: contiguous leading dimensions are one, a (batch, M, heads * N) projection
// seen as (batch, heads, M, N) is two.  False when there are more.
bool batch_steps(const torch::Tensor &t, int64_t *step, int64_t *heads, int64_t *group) {
  int64_t size[2] = {1, 1}, stride[2] = {0, 0};
  int levels = 0;
  for (int64_t d = t.dim() - 3; d >= 0; --d) {  // innermost level first
    if (t.size(d) == 1) continue;
    if (levels > 0 && t.stride(d) == stride[levels - 1] * size[levels - 1]) {
      size[levels - 1] *= t.size(d);
    } else {
      if (levels == 2) return false;
      size[levels] = t.size(d), stride[levels] = t.stride(d), ++levels;
    }
  }
  *step = stride[0], *heads = levels == 2 ? size[0] : 0, *group = levels == 2 ? stride[1] : 0;
  return true;
}

int64_t batch_of(const torch::Tensor &t) {
  int64_t B = 1;
  for (int64_t d = 0; d < t.dim() - 2; ++d) B *= t.size(d);
  return B;
}
// Sizes of `like` with the last dimension replaced.
std::vector<int64_t> with_columns(const torch::Tensor &like, int64_t columns) {
  auto sizes = like.sizes().vec();
  sizes.back() = columns;
  return sizes;
}

// Unit column stride, 16-byte aligned rows and batch elements, at most two batch levels: what the kernels read in place.
bool readable_in_place(const torch::Tensor &t) {
  const int64_t es = t.element_size();
  int64_t step, heads, group;
  return t.stride(-1) == 1 && (t.stride(-2) * es) % 16 == 0 && aligned16(t) && batch_steps(t, &step, &heads, &group) &&
         (step * es) % 16 == 0 && (group * es) % 16 == 0;
}

// The operands of a call share one grouping of the batch (include/window_matmul_hip.h); the first tensor with two levels
// of batch strides decides it.
struct Heads {
  int64_t heads = 0;
  bool admit(const torch::Tensor &t) {
    int64_t step, h, group;
    if (!batch_steps(t, &step, &h, &group)) return false;
    if (h != 0 && heads == 0) heads = h;
    return h == 0 || h == heads;
  }
};

// `t` where the kernels can read it in place, else a contiguous copy.
torch::Tensor vector_friendly(const torch::Tensor &t) {
  if (t.numel() == 0 || readable_in_place(t)) return t;
  const bool alignable = (t.size(-1) * t.element_size()) % 16 == 0;
  if (t.is_contiguous()) {
    // rows that cannot be aligned (N * element size not a multiple of 16): the tile kernels take
    // the tensor as it is; alignable rows behind a misaligned pointer (a view at a storage offset)
    // move into a fresh allocation so that the tuned kernels apply
    return alignable ? t.clone(at::MemoryFormat::Contiguous) : t;
  }
  auto c = t.contiguous();
  return aligned16(c) || !alignable ? c : c.clone(at::MemoryFormat::Contiguous);
}

torch::Tensor vector_friendly(const torch::Tensor &t, Heads &heads) {
  auto r = vector_friendly(t);
  return heads.admit(r) ? r : r.contiguous();
}

// Storage for a result of the shape of `t`, in the memory layout of `t` where the kernels can write that (the
// gradient of a projection view is then laid out like the projection and needs no copy on its way back).
torch::Tensor empty_like_rows(const torch::Tensor &t, int64_t columns, Heads &heads) {
  if (t.size(-1) == columns) {
    auto g = torch::empty_like(t);
    if (readable_in_place(g) && heads.admit(g)) return g;
  }
  return torch::empty(with_columns(t, columns), t.options());
}

// Band tensors (rows of odd length 2w+1) need to be contiguous and start on a 16-byte boundary.
torch::Tensor band_friendly(const torch::Tensor &t) {
  auto c = t.contiguous();
  return aligned16(c) || c.numel() == 0 ? c : c.clone(at::MemoryFormat::Contiguous);
}

// Head widths that the tuned kernels do not take -- N not a multiple of 16 for 16-bit storage, of 8
// for float32 -- are padded with zero columns to the next such width (up to 128): zero columns add
// nothing to a dot product and produce result columns that are cut off again, and two or three
// passes over the (B,M,N) tensors cost less than the element-by-element tile kernels, which take such
// shapes otherwise.  float64 needs none of this: its kernels take every head width.  Nor does float32
// up to w = 256, where the tile kernels were measured level with or ahead of padding and slicing
// (B96 M4096 N60: 109 against 151 us at w = 8, 184 against 245 us at w = 64; B16 M4096 N256 w256:
// 298 against 287 us; at w = 1500 the tuned kernels are 1.5 times faster again).
constexpr int64_t kTileUpToWindowF32 = 256;
bool tiles_preferred(const torch::Tensor &t, int64_t w) { return t.scalar_type() == at::kFloat && w <= kTileUpToWindowF32; }

int64_t padded_width(const torch::Tensor &t, int64_t w) {
  const int64_t N = t.size(-1);
  if (tiles_preferred(t, w)) return N;
  int64_t unit;
  switch (t.scalar_type()) {
    case at::kHalf:
    case at::kBFloat16: unit = 16; break;
    case at::kFloat: unit = 8; break;
    default: return N;
  }
  const int64_t Np = (N + unit - 1) / unit * unit;
  return N > 0 && Np <= 128 ? Np : N;
}
torch::Tensor pad_columns(const torch::Tensor &t, int64_t Np) {
  const int64_t N = t.size(-1);
  if (N == Np) return t;
  auto padded = torch::zeros(with_columns(t, Np), t.options());
  padded.narrow(-1, 0, N).copy_(t);
  return padded;
}
torch::Tensor cut_columns(const torch::Tensor &t, int64_t N) {
  return t.size(-1) == N ? t : t.narrow(-1, 0, N).contiguous();
}

// Head widths beyond 128 (the widest the tuned kernels take) are worked on in slices of 128 columns:
// results with N columns are independent per slice, bands are the sum over the slices.  The slices
// of a band are computed and summed in float32 whatever the storage type (a 16-bit partial band
// would be rounded at the magnitude of the partial sums, which shows where the slices cancel) and
// the sum is rounded once.  float64 is not sliced: its kernels take every head width.
constexpr int64_t kMaxWidth = 128;
bool sliced_width(const torch::Tensor &t, int64_t w) {
  return t.size(-1) > kMaxWidth && !tiles_preferred(t, w) && (t.scalar_type() == at::kHalf || t.scalar_type() == at::kBFloat16 || t.scalar_type() == at::kFloat);
}

// A contiguous band (..., M, W) as an operand.
wm_operand band_operand(const torch::Tensor &t) {
  return wm_operand{t.data_ptr(), t.size(-2) * t.size(-1), t.size(-1), 1};
}
wm_grouped_operand grouped(const torch::Tensor &t) {
  wm_grouped_operand g{{t.data_ptr(), 0, t.stride(-2), t.stride(-1)}, 0, 0};
  TORCH_CHECK(batch_steps(t, &g.op.stride_b, &g.heads, &g.stride_g), "more than two levels of batch strides");
  return g;
}

void raise_on_error(int status, const char *op) {
  TORCH_CHECK(status == WM_OK, op, ": ", wm_status_string(status), " (status ", status, ")");
}

void *current_stream(const torch::Tensor &t) {
  return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream();
}

// K comes as (...,N,M).  The kernels want key rows contiguous, which is what a
// transposed view of a row-major (...,M,N) tensor already is; anything else is
// copied into that layout once (the reference always copies: cuda:236).
// A tensor that is laid out as (B,N,M) with unit stride along M goes through the library's own
// transpose (one read and one write at memory speed; a general strided copy reaches a quarter of that), with one level of
// batch strides or two.
torch::Tensor key_rows(const torch::Tensor &k, Heads &heads) {
  auto view = k.transpose(-2, -1);
  if (view.stride(-1) == 1 || k.stride(-1) != 1 || k.numel() == 0 || !k.is_cuda()) return vector_friendly(view, heads);
  const int64_t es = k.element_size();
  int64_t step, h, group;
  if ((es != 2 && es != 4 && es != 8) || !batch_steps(k, &step, &h, &group)) return vector_friendly(view, heads);
  auto rows = torch::empty(view.sizes(), k.options());
  const wm_grouped_operand src = grouped(k);
  const int dtype = es == 2 ? WM_DTYPE_BF16 : es == 4 ? WM_DTYPE_F32 : WM_DTYPE_F64;  // only the element size matters
  const int status = wm_grouped_key_rows(&src, rows.data_ptr(), batch_of(k), k.size(-2), k.size(-1), dtype, current_stream(k));
  if (status == WM_ERR_UNSUPPORTED) return vector_friendly(view, heads);  // odd alignment: the general copy
  raise_on_error(status, "key rows");
  return rows;
}


// The operands may have any number of leading dimensions, which need not be the same as long as they amount to
// the same number of batch elements.
void check_window_inputs(const torch::Tensor &src, const torch::Tensor &other) {
  check_gpu(src, "A");
  check_gpu(other, "B");
  TORCH_CHECK(src.dim() >= 2 && other.dim() >= 2, "Input mismatch");
  TORCH_CHECK(batch_of(src) == batch_of(other), "Input mismatch");
  TORCH_CHECK(src.size(-1) == other.size(-2), "Input mismatch");
  TORCH_CHECK(src.size(-2) == other.size(-1), "Input mismatch");
  TORCH_CHECK(src.scalar_type() == other.scalar_type(), "Input mismatch");
  TORCH_CHECK(src.device() == other.device(), "Input mismatch");
}

void check_unwindow_inputs(const torch::Tensor &src, const torch::Tensor &other, int64_t w) {
  check_gpu(src, "A");
  check_gpu(other, "B");
  TORCH_CHECK(src.dim() >= 2 && other.dim() >= 2, "Input mismatch");
  TORCH_CHECK(batch_of(src) == batch_of(other), "Input mismatch");
  TORCH_CHECK(src.size(-1) == 2 * w + 1, "Input mismatch");
  TORCH_CHECK(src.size(-2) == other.size(-2), "Input mismatch");
  TORCH_CHECK(src.scalar_type() == other.scalar_type(), "Input mismatch");
  TORCH_CHECK(src.device() == other.device(), "Input mismatch");
}

// `g` has the leading dimensions and rows of `like`, and this many columns.
void check_grad(const torch::Tensor &g, const torch::Tensor &like, int64_t columns) {
  check_gpu(g, "grad_C");
  TORCH_CHECK(g.sizes().vec() == with_columns(like, columns), "Input mismatch");
  TORCH_CHECK(g.scalar_type() == like.scalar_type() && g.device() == like.device(), "Input mismatch");
}

// reference: window_matmul_forward -> window_matmul_fw_cuda (window_matmul.cpp:74-78, cuda:224-270)
torch::Tensor window_matmul_forward(torch::Tensor src, torch::Tensor other, int64_t window_size) {
  TORCH_CHECK(window_size >= 0, "Input mismatch");
  check_window_inputs(src, other);
  const int dtype = abi_dtype(src, "window_matmul_fw_cuda");
  at::hip::HIPGuardMasqueradingAsCUDA guard(src.device());
  if (sliced_width(src, window_size)) {
    torch::Tensor band;
    for (int64_t h = 0; h < src.size(-1); h += kMaxWidth) {
      const int64_t n = std::min(kMaxWidth, src.size(-1) - h);
      auto part = window_matmul_forward(src.narrow(-1, h, n).to(at::kFloat), other.narrow(-2, h, n).to(at::kFloat), window_size);
      if (h == 0) band = part; else band.add_(part);
    }
    return band.to(src.scalar_type());
  }
  const int64_t B = batch_of(src), M = src.size(-2), N = padded_width(src, window_size);
  Heads heads;
  auto q = vector_friendly(pad_columns(src, N), heads);
  auto kt = pad_columns(key_rows(other, heads), N).transpose(-2, -1);  // (...,N,M) view of key rows
  auto out = torch::empty(with_columns(src, 2 * window_size + 1), src.options());
  const wm_grouped_operand oq = grouped(q), ok = grouped(kt);
  const wm_operand oa = band_operand(out);
  raise_on_error(wm_grouped_window_matmul_forward(&oq, &ok, &oa, B, M, N, window_size, dtype, 0, current_stream(src)),
                 "window_matmul_forward");
  return out;
}

// reference: window_matmul_backward -> window_matmul_bw_cuda (window_matmul.cpp:80-85, cuda:272-319)
// need_src / need_other (extensions of the reference signature, both true by default) let the
// autograd Function skip the kernel of a gradient nobody asked for; a skipped one comes back as None.
std::tuple<c10::optional<torch::Tensor>, c10::optional<torch::Tensor>> window_matmul_backward(
    torch::Tensor src, torch::Tensor other, int64_t window_size, torch::Tensor grad_output, bool need_src,
    bool need_other) {
  TORCH_CHECK(window_size >= 0, "Input mismatch");
  check_window_inputs(src, other);
  const int64_t B = batch_of(src), M = src.size(-2), N = src.size(-1);
  check_grad(grad_output, src, 2 * window_size + 1);
  const int dtype = abi_dtype(src, "window_matmul_bw_cuda");
  at::hip::HIPGuardMasqueradingAsCUDA guard(src.device());
  if (sliced_width(src, window_size)) {
    std::vector<torch::Tensor> gq, gk;
    for (int64_t h = 0; h < N; h += kMaxWidth) {
      const int64_t n = std::min(kMaxWidth, N - h);
      auto part = window_matmul_backward(src.narrow(-1, h, n), other.narrow(-2, h, n), window_size, grad_output, need_src, need_other);
      if (need_src) gq.push_back(*std::get<0>(part));
      if (need_other) gk.push_back(*std::get<1>(part));
    }
    c10::optional<torch::Tensor> grad_q, grad_k;
    if (need_src) grad_q = torch::cat(gq, -1);
    if (need_other) grad_k = torch::cat(gk, -2);
    return std::make_tuple(grad_q, grad_k);
  }
  const int64_t Np = padded_width(src, window_size);
  Heads heads;
  auto q = vector_friendly(pad_columns(src, Np), heads);
  auto kt = pad_columns(key_rows(other, heads), Np).transpose(-2, -1);
  auto ga = band_friendly(grad_output);
  c10::optional<torch::Tensor> grad_q, grad_k;
  if (need_src) grad_q = empty_like_rows(src, Np, heads);
  // grad_k is produced row-major per key row and handed back in the (...,N,M)
  // orientation of `other` as a transposed view, like the reference (cuda:318).
  if (need_other) grad_k = empty_like_rows(other.transpose(-2, -1), Np, heads).transpose(-2, -1);
  const wm_grouped_operand oq = grouped(q), ok = grouped(kt);
  const wm_operand oga = band_operand(ga);
  wm_grouped_operand ogq{}, ogk{};
  if (need_src) ogq = grouped(*grad_q);
  if (need_other) ogk = grouped(*grad_k);
  raise_on_error(wm_grouped_window_matmul_backward(&oq, &ok, &oga, need_src ? &ogq : nullptr, need_other ? &ogk : nullptr,
                                                   B, M, Np, window_size, dtype, 0, current_stream(src)),
                 "window_matmul_backward");
  if (need_src) grad_q = cut_columns(*grad_q, N);
  if (need_other && Np != N) grad_k = grad_k->narrow(-2, 0, N);
  return std::make_tuple(grad_q, grad_k);
}

// reference: unwindow_matmul_forward -> unwindow_matmul_fw_cuda (window_matmul.cpp:87-91, cuda:321-358)
torch::Tensor unwindow_matmul_forward(torch::Tensor src, torch::Tensor other, int64_t window_size) {
  TORCH_CHECK(window_size >= 0, "Input mismatch");
  check_unwindow_inputs(src, other, window_size);
  const int dtype = abi_dtype(src, "unwindow_matmul_fw_cuda");
  at::hip::HIPGuardMasqueradingAsCUDA guard(src.device());
  const int64_t B = batch_of(other), M = other.size(-2), N = other.size(-1);
  if (sliced_width(other, window_size)) {
    std::vector<torch::Tensor> parts;
    for (int64_t h = 0; h < N; h += kMaxWidth)
      parts.push_back(unwindow_matmul_forward(src, other.narrow(-1, h, std::min(kMaxWidth, N - h)), window_size));
    return torch::cat(parts, -1);
  }
  const int64_t Np = padded_width(other, window_size);
  auto a = band_friendly(src);
  Heads heads;
  auto v = vector_friendly(pad_columns(other, Np), heads);
  auto out = torch::empty(with_columns(other, Np), src.options());
  const wm_operand oa = band_operand(a);
  const wm_grouped_operand ov = grouped(v), oo = grouped(out);
  raise_on_error(wm_grouped_unwindow_matmul_forward(&oa, &ov, &oo, B, M, Np, window_size, dtype, 0, current_stream(src)),
                 "unwindow_matmul_forward");
  return cut_columns(out, N);
}

// reference: unwindow_matmul_backward -> unwindow_matmul_bw_cuda (window_matmul.cpp:93-98, cuda:360-416)
std::tuple<c10::optional<torch::Tensor>, c10::optional<torch::Tensor>> unwindow_matmul_backward(
    torch::Tensor src, torch::Tensor other, int64_t window_size, torch::Tensor grad_output, bool need_src,
    bool need_other) {
  TORCH_CHECK(window_size >= 0, "Input mismatch");
  check_unwindow_inputs(src, other, window_size);
  const int64_t B = batch_of(other), M = other.size(-2), N = other.size(-1);
  check_grad(grad_output, other, N);
  const int dtype = abi_dtype(src, "unwindow_matmul_bw_cuda");
  at::hip::HIPGuardMasqueradingAsCUDA guard(src.device());
  if (sliced_width(other, window_size)) {
    c10::optional<torch::Tensor> grad_a, grad_v;
    std::vector<torch::Tensor> gv;
    for (int64_t h = 0; h < N; h += kMaxWidth) {
      const int64_t n = std::min(kMaxWidth, N - h);
      if (need_other)
        gv.push_back(*std::get<1>(unwindow_matmul_backward(src, other.narrow(-1, h, n), window_size, grad_output.narrow(-1, h, n), false, true)));
      if (need_src) {  // grad_a = band of grad_output against other: in float32, as in window_matmul_forward
        auto part = window_matmul_forward(grad_output.narrow(-1, h, n).to(at::kFloat), other.narrow(-1, h, n).transpose(-2, -1).to(at::kFloat), window_size);
        if (h == 0) grad_a = part; else grad_a->add_(part);
      }
    }
    if (need_src) grad_a = grad_a->to(src.scalar_type()).view(src.sizes());
    if (need_other) grad_v = torch::cat(gv, -1);
    return std::make_tuple(grad_a, grad_v);
  }
  const int64_t Np = padded_width(other, window_size);
  auto a = band_friendly(src);
  Heads heads;
  auto v = vector_friendly(pad_columns(other, Np), heads);
  auto go = vector_friendly(pad_columns(grad_output, Np), heads);
  c10::optional<torch::Tensor> grad_a, grad_v;
  if (need_src) grad_a = torch::empty(src.sizes(), src.options());
  if (need_other) grad_v = empty_like_rows(other, Np, heads);
  const wm_operand oa = band_operand(a);
  const wm_grouped_operand ov = grouped(v), ogo = grouped(go);
  wm_operand oga{};
  wm_grouped_operand ogv{};
  if (need_src) oga = band_operand(*grad_a);
  if (need_other) ogv = grouped(*grad_v);
  raise_on_error(wm_grouped_unwindow_matmul_backward(&oa, &ov, &ogo, need_src ? &oga : nullptr, need_other ? &ogv : nullptr,
                                                     B, M, Np, window_size, dtype, 0, current_stream(src)),
                 "unwindow_matmul_backward");
  if (need_other) grad_v = cut_columns(*grad_v, N);
  return std::make_tuple(grad_a, grad_v);
}

// Softmax over the band dimension, the step callers put between the two ops
// (reference tests/test_attention.py:60-61); not part of the reference's native module.
torch::Tensor band_softmax_forward(torch::Tensor src, double scale, bool mask_out_of_range) {
  check_gpu(src, "A");
  TORCH_CHECK(src.dim() >= 2 && src.size(-1) % 2 == 1, "Input mismatch");
  const int dtype = abi_dtype(src, "band_softmax_forward");
  at::hip::HIPGuardMasqueradingAsCUDA guard(src.device());
  auto a = band_friendly(src);
  auto out = torch::empty_like(a);
  const wm_operand oa = band_operand(a), oo = band_operand(out);
  raise_on_error(wm_band_softmax_forward(&oa, &oo, batch_of(a), a.size(-2), a.size(-1) / 2, scale, mask_out_of_range,
                                         dtype, 0, current_stream(src)),
                 "band_softmax_forward");
  return out;
}

torch::Tensor band_softmax_backward(torch::Tensor probs, torch::Tensor grad_output, double scale,
                                    bool mask_out_of_range) {
  check_gpu(probs, "P");
  check_gpu(grad_output, "grad_P");
  TORCH_CHECK(probs.dim() >= 2 && probs.size(-1) % 2 == 1, "Input mismatch");
  TORCH_CHECK(grad_output.sizes() == probs.sizes() && grad_output.scalar_type() == probs.scalar_type() &&
                  grad_output.device() == probs.device(),
              "Input mismatch");
  const int dtype = abi_dtype(probs, "band_softmax_backward");
  at::hip::HIPGuardMasqueradingAsCUDA guard(probs.device());
  auto p = band_friendly(probs);
  auto g = band_friendly(grad_output);
  auto out = torch::empty_like(p);
  const wm_operand op = band_operand(p), og = band_operand(g), oo = band_operand(out);
  raise_on_error(wm_band_softmax_backward(&op, &og, &oo, batch_of(p), p.size(-2), p.size(-1) / 2, scale,
                                          mask_out_of_range, dtype, 0, current_stream(probs)),
                 "band_softmax_backward");
  return out;
}

// Fused window attention (no counterpart in the reference's native module): forward returns
// (o, lse); q, k, v are (..., M, N) with k holding key rows.  Raises when the fused kernels do not
// cover the problem; window_attention_supported() lets the caller choose the separate ops first.
// any_width: also head widths from 8 on that are no multiple of 16.
bool window_attention_supported(torch::Tensor q, int64_t window_size, double scale, bool any_width) {
  if (q.dim() < 2 || !q.device().is_cuda()) return false;
  int dtype;
  switch (q.scalar_type()) {
    case at::kHalf: dtype = WM_DTYPE_F16; break;
    case at::kBFloat16: dtype = WM_DTYPE_BF16; break;
    default: return false;
  }
  const int64_t N = q.size(-1), unit = any_width && N >= 8 ? (N + 15) / 16 * 16 : N;
  return wm_window_attention_supported(q.size(-2), unit, window_size, dtype, scale) != 0;
}

// Operands of the fused attention.  Its kernels for widths that 16 does not divide take rows of any alignment.
bool ragged_width(const torch::Tensor &t) { return t.size(-1) % 16 != 0; }
unsigned attention_flags(const torch::Tensor &t) { return ragged_width(t) ? WM_FLAG_ANY_HEAD_WIDTH : 0; }
bool ragged_rows_in_place(const torch::Tensor &t) {
  int64_t step, heads, group;
  return t.stride(-1) == 1 && batch_steps(t, &step, &heads, &group);
}
torch::Tensor attention_rows(const torch::Tensor &t, Heads &heads) {  // rows of any alignment
  if (t.stride(-1) != 1 && t.stride(-2) == 1) return key_rows(t.transpose(-2, -1), heads);  // keys of a channels-first projection
  return ragged_rows_in_place(t) && heads.admit(t) ? t : t.contiguous();
}
torch::Tensor attention_rows_like(const torch::Tensor &t, Heads &heads) {
  auto g = torch::empty_like(t);
  return ragged_rows_in_place(g) && heads.admit(g) ? g : torch::empty(t.sizes(), t.options());
}
torch::Tensor attention_operand(const torch::Tensor &t, Heads &heads) {
  return ragged_width(t) ? attention_rows(t, heads) : vector_friendly(t, heads);
}
torch::Tensor attention_gradient(const torch::Tensor &t, Heads &heads) {
  return ragged_width(t) ? attention_rows_like(t, heads) : empty_like_rows(t, t.size(-1), heads);
}

void check_attention_inputs(const torch::Tensor &q, const torch::Tensor &k, const torch::Tensor &v) {
  check_gpu(q, "Q");
  check_gpu(k, "K");
  check_gpu(v, "V");
  TORCH_CHECK(q.dim() >= 2 && k.sizes() == q.sizes() && v.sizes() == q.sizes(), "Input mismatch");
  TORCH_CHECK(k.scalar_type() == q.scalar_type() && v.scalar_type() == q.scalar_type(), "Input mismatch");
  TORCH_CHECK(k.device() == q.device() && v.device() == q.device(), "Input mismatch");
}

std::tuple<torch::Tensor, torch::Tensor> window_attention_forward(torch::Tensor q, torch::Tensor k, torch::Tensor v,
                                                                  int64_t window_size, double scale,
                                                                  bool mask_out_of_range) {
  check_attention_inputs(q, k, v);
  const int dtype = abi_dtype(q, "window_attention_forward");
  at::hip::HIPGuardMasqueradingAsCUDA guard(q.device());
  const int64_t B = batch_of(q), M = q.size(-2), N = q.size(-1);
  Heads heads;
  auto qq = attention_operand(q, heads), kk = attention_operand(k, heads), vv = attention_operand(v, heads);
  auto o = torch::empty(q.sizes(), q.options());
  auto lse = torch::empty({B, M}, q.options().dtype(at::kFloat));
  const wm_grouped_operand oq = grouped(qq), ok = grouped(kk), ov = grouped(vv), oo = grouped(o);
  raise_on_error(wm_grouped_window_attention_forward(&oq, &ok, &ov, &oo, lse.data_ptr<float>(), B, M, N, window_size, scale,
                                                     mask_out_of_range, dtype, attention_flags(q), current_stream(q)),
                 "window_attention_forward");
  return std::make_tuple(o, lse);
}

std::tuple<c10::optional<torch::Tensor>, c10::optional<torch::Tensor>, c10::optional<torch::Tensor>>
window_attention_backward(torch::Tensor q, torch::Tensor k, torch::Tensor v, torch::Tensor o, torch::Tensor lse,
                          torch::Tensor grad_output, int64_t window_size, double scale, bool need_q, bool need_k,
                          bool need_v) {
  check_attention_inputs(q, k, v);
  const int64_t B = batch_of(q), M = q.size(-2), N = q.size(-1);
  check_grad(grad_output, q, N);
  check_grad(o, q, N);
  TORCH_CHECK(lse.device() == q.device() && lse.scalar_type() == at::kFloat && lse.dim() == 2 &&
                  lse.size(0) == B && lse.size(1) == M && lse.is_contiguous(),
              "Input mismatch");
  const int dtype = abi_dtype(q, "window_attention_backward");
  at::hip::HIPGuardMasqueradingAsCUDA guard(q.device());
  Heads heads;
  auto qq = attention_operand(q, heads), kk = attention_operand(k, heads), vv = attention_operand(v, heads),
       oo = attention_operand(o, heads), go = attention_operand(grad_output, heads);
  c10::optional<torch::Tensor> gq, gk, gv;
  wm_grouped_operand f{}, g{}, h{};
  if (need_q) gq = attention_gradient(q, heads), f = grouped(*gq);
  if (need_k) gk = attention_gradient(k, heads), g = grouped(*gk);
  if (need_v) gv = attention_gradient(v, heads), h = grouped(*gv);
  auto delta = torch::empty({2, B, M}, lse.options());  // row sums and log2-scaled log-sum-exp
  const wm_grouped_operand a = grouped(qq), b = grouped(kk), c = grouped(vv), d = grouped(oo), e = grouped(go);
  raise_on_error(wm_grouped_window_attention_backward(&a, &b, &c, &d, lse.data_ptr<float>(), &e, need_q ? &f : nullptr,
                                                      need_k ? &g : nullptr, need_v ? &h : nullptr,
                                                      delta.data_ptr<float>(), B, M, N, window_size, scale, dtype,
                                                      attention_flags(q), current_stream(q)),
                 "window_attention_backward");
  return std::make_tuple(gq, gk, gv);
}

// Differentiable forms of the functions above.  The public functions of the package call these: an autograd.Function in
// Python costs 20-30 us of host time per call and direction, which a small problem cannot hide (a training
// step of the fused attention at B 7, M 3001 keeps the GPU busy for 33 us).  They are torch's own C++ Functions, so that
// saved-tensor hooks, compiled autograd, functorch's refusal and undefined gradients are dealt with as in Python; what a node
// written by hand saves over that is about 1 us a call.
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// There are no forward-mode derivatives: inputs that carry a tangent are refused with the error type of a Python Function
// without a jvp.
void refuse_tangents(std::initializer_list<const torch::Tensor *> inputs) {
  for (const auto *t : inputs)
    TORCH_CHECK_NOT_IMPLEMENTED(!t->_fw_grad(0).defined(), "no forward-mode derivative is implemented for the banded products, "
                                "the band softmax and the window attention");
}

torch::Tensor or_none(const c10::optional<torch::Tensor> &t) { return t ? *t : torch::Tensor(); }

// A result that the backward reads although the caller may change it in place: what is kept has a version counter of its own,
// and a tensor of no elements that shares the result's counter, 0 for a fresh tensor, tells the backward whether the
// values are still those.
torch::Tensor keep_changeable(AutogradContext *ctx, const torch::Tensor &out) {
  if (!out.is_inference()) {
    TORCH_INTERNAL_ASSERT(out._version() == 0);
    auto counter = torch::empty({0});
    torch::autograd::impl::set_version_counter(counter, torch::autograd::impl::version_counter(out));
    ctx->saved_data["counter"] = std::move(counter);
  }
  return out.variable_data();
}
bool changed_since(AutogradContext *ctx) {
  const auto counter = ctx->saved_data.find("counter");
  return counter != ctx->saved_data.end() && counter->second.toTensor()._version() != 0;
}

struct WindowMatmulFunc : torch::autograd::Function<WindowMatmulFunc> {
  static torch::Tensor forward(AutogradContext *ctx, const torch::Tensor &src, const torch::Tensor &other, int64_t window_size) {
    ctx->save_for_backward({src, other});
    at::AutoDispatchBelowADInplaceOrView below;
    return window_matmul_forward(src, other, window_size);
  }
  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    at::NoGradGuard no_grad;  // no second derivative
    const auto t = ctx->get_saved_variables();
    const int64_t window_size = grads[0].size(-1) / 2;  // the band width fixes the window: W = 2w + 1
    auto g = window_matmul_backward(t[0], t[1], window_size, grads[0], ctx->needs_input_grad(0), ctx->needs_input_grad(1));
    return {or_none(std::get<0>(g)), or_none(std::get<1>(g)), torch::Tensor()};
  }
};

torch::Tensor window_matmul(const torch::Tensor &src, const torch::Tensor &other, int64_t window_size) {
  refuse_tangents({&src, &other});
  return WindowMatmulFunc::apply(src, other, window_size);
}

struct UnwindowMatmulFunc : torch::autograd::Function<UnwindowMatmulFunc> {
  static torch::Tensor forward(AutogradContext *ctx, const torch::Tensor &src, const torch::Tensor &other, int64_t window_size) {
    ctx->save_for_backward({src, other});
    at::AutoDispatchBelowADInplaceOrView below;
    return unwindow_matmul_forward(src, other, window_size);
  }
  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    at::NoGradGuard no_grad;
    const auto t = ctx->get_saved_variables();
    auto g = unwindow_matmul_backward(t[0], t[1], t[0].size(-1) / 2, grads[0], ctx->needs_input_grad(0), ctx->needs_input_grad(1));
    return {or_none(std::get<0>(g)), or_none(std::get<1>(g)), torch::Tensor()};
  }
};

torch::Tensor unwindow_matmul(const torch::Tensor &src, const torch::Tensor &other, int64_t window_size) {
  refuse_tangents({&src, &other});
  return UnwindowMatmulFunc::apply(src, other, window_size);
}

struct BandSoftmaxFunc : torch::autograd::Function<BandSoftmaxFunc> {
  static torch::Tensor forward(AutogradContext *ctx, const torch::Tensor &src, double scale, bool mask_out_of_range) {
    ctx->saved_data["scale"] = scale;
    ctx->saved_data["mask_out_of_range"] = mask_out_of_range;
    at::AutoDispatchBelowADInplaceOrView below;
    auto probs = band_softmax_forward(src, scale, mask_out_of_range);
    ctx->save_for_backward({probs});
    return probs;
  }
  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    at::NoGradGuard no_grad;
    const auto t = ctx->get_saved_variables();
    return {band_softmax_backward(t[0], grads[0], ctx->saved_data["scale"].toDouble(), ctx->saved_data["mask_out_of_range"].toBool()),
            torch::Tensor(), torch::Tensor()};
  }
};

torch::Tensor band_softmax(const torch::Tensor &src, double scale, bool mask_out_of_range) {
  refuse_tangents({&src});
  return BandSoftmaxFunc::apply(src, scale, mask_out_of_range);
}

struct WindowAttentionFunc : torch::autograd::Function<WindowAttentionFunc> {
  static torch::Tensor forward(AutogradContext *ctx, const torch::Tensor &q, const torch::Tensor &k, const torch::Tensor &v,
                               int64_t window_size, double scale, bool mask_out_of_range) {
    ctx->saved_data["window_size"] = window_size;
    ctx->saved_data["scale"] = scale;
    ctx->saved_data["mask_out_of_range"] = mask_out_of_range;
    at::AutoDispatchBelowADInplaceOrView below;
    auto [out, lse] = window_attention_forward(q, k, v, window_size, scale, mask_out_of_range);
    // The separate ops keep nothing of their last result, so it may be changed in place before the backward.  At the widths
    // that ran through them until these kernels took rows of any width, that holds on.
    ctx->save_for_backward({q, k, v, ragged_width(q) ? keep_changeable(ctx, out) : out, lse});
    return out;
  }
  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    at::NoGradGuard no_grad;
    auto t = ctx->get_saved_variables();
    const int64_t window_size = ctx->saved_data["window_size"].toInt();
    const double scale = ctx->saved_data["scale"].toDouble();
    if (changed_since(ctx))  // made again, bit for bit
      std::tie(t[3], t[4]) = window_attention_forward(t[0], t[1], t[2], window_size, scale, ctx->saved_data["mask_out_of_range"].toBool());
    auto g = window_attention_backward(t[0], t[1], t[2], t[3], t[4], grads[0], window_size, scale, ctx->needs_input_grad(0),
                                       ctx->needs_input_grad(1), ctx->needs_input_grad(2));
    return {or_none(std::get<0>(g)), or_none(std::get<1>(g)), or_none(std::get<2>(g)), torch::Tensor(), torch::Tensor(), torch::Tensor()};
  }
};

torch::Tensor window_attention(const torch::Tensor &q, const torch::Tensor &k, const torch::Tensor &v, int64_t window_size,
                               double scale, bool mask_out_of_range) {
  refuse_tangents({&q, &k, &v});
  return WindowAttentionFunc::apply(q, k, v, window_size, scale, mask_out_of_range);
}

// Window attention in float32.  Two routes beside the separate ops: the fused kernels (wm_attention_f32.hip), which recompute
// everything from q, k and v with six bf16 products for every float32 one, and for training the separate ops forward
// with a backward that forms the gradient of the scores in one kernel, which has the band in memory.
//
// Fused, us of the separate ops / of the fused kernels; T is tiles of 128 rows, and the route compared with in training
// is the better of the other two:
//   inference  T = 3072: N = 64 117 / 122 at w = 8, 149 / 113 at w = 16, 886 / 420 at w = 256; N = 128 323 / 317 at w = 16, 1249 / 710 at
//              256.  Few tiles leave CUs idle where the separate ops share a tile out: N = 128 T = 32 39 / 29 at w = 64, 53 / 55 at w = 256,
//              T = 64 138 / 167 at w = 1024, T = 128 196 / 170; N = 64 T = 32 105 / 92 at w = 1024.  T = 8 of one sequence: N = 128 49 / 46 at w =
//              160, 50 / 51 at 180, 53 / 59 at 256, N = 96 52 / 50 at 256, N = 127 104 / 59 at 256; T = 32 N = 128 59 / 60 at 256.
//   training   Narrow heads would gain as well (N = 32 329 / 287 at w = 24, 707 / 360 at w = 64, N = 16 276 / 227), but up to N = 32 the separate ops,
//              whose row sums of P dP have 2 w + 1 terms, are the more accurate: distance to float64 in 1e-7, theirs / fused, grad_k N = 16
//              2.30 / 2.57 at w = 40, N = 24 2.07 / 2.11, N = 32 2.77 / 2.81 at w = 64; with scores three times as large N = 32 w = 64 grad_q
//              3.97 / 4.20, grad_k 3.90 / 4.07.  From N = 33 on none is worse (N = 33 ... 128, w = 32 ... 300, scores of one, three and six times
//              the size, four inputs each), up to w = 256.  Beyond, the separate ops pad widths that 8 does not divide and take the split products
//              as well, and the row sums tell again: quotients of the distances, fused / theirs, N = 36 1.01 at w = 300, 1.07 at 600, N = 47 0.99 and
//              1.04, N = 54 0.94 at w = 600, 1.01 at 1000, N = 63 0.97 at w = 1000, 1.02 at 1500, N = 70 0.98 at w = 1500, 1.02 at 3000, N = 85 0.99 at
//              6000.  Widths that 8 divides had D = sum dO O from w = 128 on before: 0.92 ... 0.99 at w = 1500 ... 6000.
//              N = 64: T = 3072 567 / 576 at w = 24, 678 / 561 at w = 32, 2096 / 1456 at w = 256; T = 32 96 / 66 at
//              w = 64, 142 / 132 at w = 256, 177 / 200 at w = 400, T = 64 346 / 420 at w = 1024, T = 128 438 / 402.
//              N > 64: a wavefront of the key kernel needs the registers of a whole SIMD: T = 3072 N = 80 1096 / 1112 at w = 64, N = 96
//              1551 / 1640 at w = 100, 2709 / 2390 at w = 256, N = 128 2090 / 2074 at w = 128, 3553 / 3130 at w = 256; T = 168 N = 80 226 / 212 at
//              w = 300, 766 / 687 at w = 1500, T = 128 N = 80 477 / 514 at w = 1000; T = 256 N = 128 251 / 251 and 791 / 792 at w = 200 and 1000.
//              Widths that 8 does not divide, which the separate ops take to the tile kernels: T = 3072 N = 60 616 / 602
//              at w = 16, 748 / 580 at w = 32, N = 75 5062 / 2346 at w = 256; T = 32 N = 75 216 / 216 at w = 300.
//              N = 127 T = 1536 694 / 720 at w = 32, 879 / 885 at 48, 971 / 882 at 64, T = 256 156 / 131 at w = 32, 182 / 148 at 48; N = 110 T = 1536
//              658 / 655 at w = 32.  With few tiles the separate ops wait for the host, 105 to 145 us by the machine: T = 8 N = 127
//              143 / 101 at w = 32, 139 / 133 at 64, 142 / 150 at 80, 158 / 169 at 100, 188 / 189 at 140.
// Below 8 tiles, whose routes differ in launches alone, a problem gives what it gave before these kernels, traced or not, bit for bit.  That
// costs time: T = 8 takes 144 / 86 us for a step and 38 / 17 for inference (8 x M128 N64 w40); one sequence with T = 8, N = 64 at w = 257
// 56 / 40 for inference and at w = 1000 66 / 51, T = 16 103 / 90.
// An infinite operand gives NaN where the exact result is infinite, as in the separate ops on split products (wm_f32_split.hip); where those
// run on the float32 instruction, which gives the infinity, that is a difference between the routes: widths that 8 does not divide
// up to w = 256, values of N <= 32, and up to w = 28 (queries and keys: 31) widths of 16, 32, 48 and 64.
bool f32_fused(const torch::Tensor &q, int64_t window_size, double scale, bool training) {
  const int64_t N = q.size(-1), M = q.size(-2);
  if (q.numel() == 0) return false;
  if (N < 8 || N > kMaxWidth || M > (1 << 30) || window_size < 16 || window_size > (1 << 28) || !(scale > 1.2e-38 && scale < 1.0e30)) return false;
  const int64_t tiles = batch_of(q) * ((M + 127) / 128);
  if (tiles < 8 || tiles > 0x7fffff00 || (tiles < 128 && window_size > 256 && (training || N > 64))) return false;
  if (!training) return tiles >= 32 || N <= 96 || N % 8 != 0 || std::min(window_size, M / 4) <= 160;
  if (M < 16) return false;  // few neighbours: gradients of scores that cancel, with a single neighbour to exact zeros in the separate ops
  if (N % 8 != 0 && std::min(window_size, M) > std::max<int64_t>(256, 60 * (N - 44))) return false;
  if (N > 64 && N % 8 == 0) return window_size >= 128 && tiles >= (N <= 96 ? 160 : 256);
  if (N > 112 && tiles >= 1024) return window_size >= 40;
  return N >= 40 ? window_size >= 32 : N > 32 && window_size >= 64;
}

bool window_attention_f32_supported(const torch::Tensor &q, int64_t window_size, double scale, bool training) {
  if (q.dim() < 2 || !q.device().is_cuda() || q.scalar_type() != at::kFloat || q.numel() == 0) return false;
  if (f32_fused(q, window_size, scale, training)) return true;
  // The gradient of the scores in one kernel, from w = 128 on.  A training step through the separate ops / with it, us, B96 M4096: N = 64
  // 931 / 953 at w = 64, 1251 / 1257 at w = 100, 2313 / 2093 at w = 256; N = 128 1521 / 1572, 2044 / 2027, 3609 / 3438; B8 M3001
  // N = 16 191 / 174 at w = 256.  In a narrow band the pieces at its two edges, read element by element, cost more than
  // the passes that are saved (N = 80, w = 32: 802 / 880).
  return training && q.size(-1) >= 8 && q.size(-1) <= kMaxWidth && q.size(-1) % 8 == 0 && window_size >= 128 && window_size <= (1 << 28) &&
         scale == scale;
}

std::tuple<torch::Tensor, torch::Tensor> f32_fused_forward(const torch::Tensor &q, const torch::Tensor &k, const torch::Tensor &v,
                                                           int64_t window_size, double scale, bool mask_out_of_range, bool training) {
  at::hip::HIPGuardMasqueradingAsCUDA guard(q.device());
  const int64_t B = batch_of(q), M = q.size(-2), N = q.size(-1);
  Heads heads;
  auto qq = attention_rows(q, heads), kk = attention_rows(k, heads), vv = attention_rows(v, heads);
  auto o = torch::empty(q.sizes(), q.options());
  auto stats = training ? torch::empty({2, B, M}, q.options()) : torch::Tensor();
  const wm_grouped_operand oq = grouped(qq), ok = grouped(kk), ov = grouped(vv), oo = grouped(o);
  raise_on_error(wm_grouped_window_attention_f32_forward(&oq, &ok, &ov, &oo, training ? stats.data_ptr<float>() : nullptr, B, M, N,
                                                         window_size, scale, mask_out_of_range, WM_DTYPE_F32, 0, current_stream(q)),
                 "window_attention_f32");
  return std::make_tuple(o, stats);
}

variable_list f32_fused_backward(const torch::Tensor &q, const torch::Tensor &k, const torch::Tensor &v, const torch::Tensor &o,
                                 const torch::Tensor &stats, const torch::Tensor &grad, int64_t window_size, double scale, bool need_q,
                                 bool need_k, bool need_v) {
  variable_list g(7);
  if (!need_q && !need_k && !need_v) return g;
  at::hip::HIPGuardMasqueradingAsCUDA guard(q.device());
  const int64_t B = batch_of(q), M = q.size(-2), N = q.size(-1);
  Heads heads;
  auto qq = attention_rows(q, heads), kk = attention_rows(k, heads), vv = attention_rows(v, heads), oo = attention_rows(o, heads),
       go = attention_rows(grad, heads);
  wm_grouped_operand x{}, y{}, z{};
  if (need_q) g[0] = attention_rows_like(q, heads), x = grouped(g[0]);
  if (need_k) g[1] = attention_rows_like(k, heads), y = grouped(g[1]);
  if (need_v) g[2] = attention_rows_like(v, heads), z = grouped(g[2]);
  auto delta = torch::empty({B, M}, q.options());
  const wm_grouped_operand a = grouped(qq), b = grouped(kk), c = grouped(vv), d = grouped(oo), e = grouped(go);
  raise_on_error(wm_grouped_window_attention_f32_backward(&a, &b, &c, &d, stats.data_ptr<float>(), &e, need_q ? &x : nullptr,
                                                          need_k ? &y : nullptr, need_v ? &z : nullptr, delta.data_ptr<float>(), B, M, N,
                                                          window_size, scale, WM_DTYPE_F32, 0, current_stream(q)),
                 "window_attention_f32 backward");
  return g;
}

// An undefined result: the kernel does not take the problem (more workgroups than a launch can have; layouts are made to fit).
torch::Tensor score_gradient(const torch::Tensor &probs, const torch::Tensor &v, const torch::Tensor &o, const torch::Tensor &grad_output,
                             int64_t window_size, double scale) {
  at::hip::HIPGuardMasqueradingAsCUDA guard(v.device());
  Heads heads;
  auto vv = vector_friendly(v, heads), oo = vector_friendly(o, heads), go = vector_friendly(grad_output, heads);
  auto p = band_friendly(probs), gs = torch::empty_like(p);
  const wm_grouped_operand a = grouped(go), b = grouped(vv), c = grouped(oo);
  const wm_operand d = band_operand(p), e = band_operand(gs);
  const int status = wm_grouped_score_gradient(&a, &b, &c, &d, &e, batch_of(v), v.size(-2), v.size(-1), window_size, scale,
                                               WM_DTYPE_F32, 0, current_stream(v));
  if (status == WM_ERR_UNSUPPORTED) return torch::Tensor();
  raise_on_error(status, "score_gradient");
  return gs;
}

struct WindowAttentionF32Func : torch::autograd::Function<WindowAttentionF32Func> {
  static torch::Tensor forward(AutogradContext *ctx, const torch::Tensor &q, const torch::Tensor &k, const torch::Tensor &v,
                               int64_t window_size, double scale, bool mask_out_of_range, bool training) {
    check_attention_inputs(q, k, v);
    const bool fused = f32_fused(q, window_size, scale, training);
    ctx->saved_data["fused"] = fused;
    ctx->saved_data["window_size"] = window_size;
    ctx->saved_data["scale"] = scale;
    ctx->saved_data["mask_out_of_range"] = mask_out_of_range;
    at::AutoDispatchBelowADInplaceOrView below;
    if (fused) {
      auto [out, stats] = f32_fused_forward(q, k, v, window_size, scale, mask_out_of_range, training);
      if (training) ctx->save_for_backward({q, k, v, stats, keep_changeable(ctx, out)});
      return out;
    }
    auto probs = band_softmax_forward(window_matmul_forward(q, k.transpose(-1, -2), window_size), scale, mask_out_of_range);
    auto out = unwindow_matmul_forward(probs, v, window_size);
    ctx->save_for_backward({q, k, v, probs, keep_changeable(ctx, out)});
    return out;
  }
  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    at::NoGradGuard no_grad;
    const auto t = ctx->get_saved_variables();
    const auto &q = t[0], &k = t[1], &v = t[2], &grad = grads[0];
    const int64_t window_size = ctx->saved_data["window_size"].toInt();
    const double scale = ctx->saved_data["scale"].toDouble();
    const bool mask_out_of_range = ctx->saved_data["mask_out_of_range"].toBool();
    const bool need_q = ctx->needs_input_grad(0), need_k = ctx->needs_input_grad(1), need_v = ctx->needs_input_grad(2);
    check_grad(grad, v, v.size(-1));
    if (ctx->saved_data["fused"].toBool()) {
      auto stats = t[3], out = t[4];
      if (changed_since(ctx)) std::tie(out, stats) = f32_fused_forward(q, k, v, window_size, scale, mask_out_of_range, true);  // again, bit for bit
      return f32_fused_backward(q, k, v, out, stats, grad, window_size, scale, need_q, need_k, need_v);
    }
    const auto &probs = t[3];
    variable_list g(7);
    if (need_v) g[2] = or_none(std::get<1>(unwindow_matmul_backward(probs, v, window_size, grad, false, true)));
    if (!need_q && !need_k) return g;
    const auto out = changed_since(ctx) ? unwindow_matmul_forward(probs, v, window_size) : t[4];  // again, bit for bit
    auto gs = score_gradient(probs, v, out, grad, window_size, scale);
    if (!gs.defined())
      gs = band_softmax_backward(probs, *std::get<0>(unwindow_matmul_backward(probs, v, window_size, grad, true, false)), scale,
                                 mask_out_of_range);
    auto qk = window_matmul_backward(q, k.transpose(-1, -2), window_size, gs, need_q, need_k);
    if (need_q) g[0] = *std::get<0>(qk);
    if (need_k) g[1] = std::get<1>(qk)->transpose(-1, -2);
    return g;
  }
};

torch::Tensor window_attention_f32(const torch::Tensor &q, const torch::Tensor &k, const torch::Tensor &v, int64_t window_size,
                                   double scale, bool mask_out_of_range) {
  refuse_tangents({&q, &k, &v});
  const bool training = at::GradMode::is_enabled() && (q.requires_grad() || k.requires_grad() || v.requires_grad());
  return WindowAttentionF32Func::apply(q, k, v, window_size, scale, mask_out_of_range, training);
}

// What Python shows as the grad_fn of a result: an object of a class of this name.
template <typename Func>
void name_node(const char *name) {
  using namespace torch::autograd;
  static PyTypeObject type;
  TORCH_CHECK(_initFunctionPyTypeObject(type, name, nullptr, nullptr) != nullptr, "no Python type for ", name);
  registerCppFunction(typeid(CppNode<Func>), &type);
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.doc() = "MI355X banded matmul kernels behind the window_matmul package";
  // The argument lists and workspace sizes of the C ABI change with WM_ABI_VERSION (version 4 doubled
  // the float workspace of wm_window_attention_backward to 2 B M values): a library of another
  // version next to this module would be called with the wrong contract, so refuse to load.
  if (wm_abi_version() != WM_ABI_VERSION)
    throw std::runtime_error("window_matmul_kernel was built against ABI " + std::to_string(WM_ABI_VERSION) +
                             " of libwindow_matmul_hip.so, the library that was loaded reports " +
                             std::to_string(wm_abi_version()));
  m.def("window_matmul_forward", &window_matmul_forward, "WindowMatmul forward");
  m.def("window_matmul_backward", &window_matmul_backward, "WindowMatmul backward", py::arg("src"), py::arg("other"),
        py::arg("window_size"), py::arg("grad_output"), py::arg("need_src") = true, py::arg("need_other") = true);
  m.def("unwindow_matmul_forward", &unwindow_matmul_forward, "UnwindowMatmul forward");
  m.def("unwindow_matmul_backward", &unwindow_matmul_backward, "UnwindowMatmul backward", py::arg("src"),
        py::arg("other"), py::arg("window_size"), py::arg("grad_output"), py::arg("need_src") = true,
        py::arg("need_other") = true);
  m.def("band_softmax_forward", &band_softmax_forward, "softmax over the band dimension", py::arg("src"),
        py::arg("scale") = 1.0, py::arg("mask_out_of_range") = false);
  m.def("band_softmax_backward", &band_softmax_backward, "backward of band_softmax_forward", py::arg("probs"),
        py::arg("grad_output"), py::arg("scale") = 1.0, py::arg("mask_out_of_range") = false);
  m.def("window_attention_supported", &window_attention_supported, "whether the fused attention kernels cover q",
        py::arg("q"), py::arg("window_size"), py::arg("scale"), py::arg("any_width") = false);
  m.def("window_attention_forward", &window_attention_forward, "fused window attention forward -> (o, lse)",
        py::arg("q"), py::arg("k"), py::arg("v"), py::arg("window_size"), py::arg("scale"),
        py::arg("mask_out_of_range") = false);
  m.def("window_attention_backward", &window_attention_backward, "fused window attention backward -> (gq, gk, gv)",
        py::arg("q"), py::arg("k"), py::arg("v"), py::arg("o"), py::arg("lse"), py::arg("grad_output"),
        py::arg("window_size"), py::arg("scale"), py::arg("need_q") = true, py::arg("need_k") = true,
        py::arg("need_v") = true);
  name_node<WindowMatmulFunc>("WindowMatmulFuncBackward");
  name_node<UnwindowMatmulFunc>("UnwindowMatmulFuncBackward");
  name_node<BandSoftmaxFunc>("BandSoftmaxFuncBackward");
  name_node<WindowAttentionFunc>("WindowAttentionFuncBackward");
  name_node<WindowAttentionF32Func>("WindowAttentionF32FuncBackward");
  m.def("window_attention_f32_supported", &window_attention_f32_supported, "whether window_attention_f32 covers q", py::arg("q"),
        py::arg("window_size"), py::arg("scale"), py::arg("training") = true);
  m.def("window_attention_f32", torch::wrap_pybind_function(window_attention_f32), "window attention in float32, differentiable", py::arg("q"), py::arg("k"),
        py::arg("v"), py::arg("window_size"), py::arg("scale"), py::arg("mask_out_of_range"));
  m.def("window_matmul", torch::wrap_pybind_function(window_matmul), "WindowMatmul, differentiable", py::arg("src"), py::arg("other"), py::arg("window_size"));
  m.def("unwindow_matmul", torch::wrap_pybind_function(unwindow_matmul), "UnwindowMatmul, differentiable", py::arg("src"), py::arg("other"),
        py::arg("window_size"));
  m.def("band_softmax", torch::wrap_pybind_function(band_softmax), "softmax over the band dimension, differentiable", py::arg("src"), py::arg("scale"),
        py::arg("mask_out_of_range"));
  m.def("window_attention", torch::wrap_pybind_function(window_attention), "fused window attention, differentiable", py::arg("q"), py::arg("k"),
        py::arg("v"), py::arg("window_size"), py::arg("scale"), py::arg("mask_out_of_range"));
  m.def("abi_version", []() { return wm_abi_version(); }, "ABI version of libwindow_matmul_hip.so");
}
