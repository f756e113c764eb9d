// Shared declarations of the gfx950 banded-matmul kernels.
//
// The six products of the path (window forward, grad_q, grad_k, unwindow
// forward, grad_a, grad_v) are three primitives over row-major views:
//   P1 band-out            C[b,i,j] = sum_h X[b,i,h] * Y[b,i+j-w,h]      (+0 out of range)
//   P2 band-in             C[b,i,h] = sum_j A[b,i,j] * Y[b,i+j-w,h]
//   P3 transposed band-in  C[b,c,h] = sum_r A[b,r,c-r+w] * Y[b,r,h]
// with X, Y, C(P2,P3) of logical shape (B,M,N) and the band of shape (B,M,2w+1).
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>
#include <stdint.h>

#include "../../include/window_matmul_hip.h"

namespace wm {

// Position of a batch element: element r of group g.  The batch of an operand is one level of strides (heads = 0:
// g = 0, r = b) or groups of `heads` elements: a (batch, M, heads * N) projection seen as batch * heads
// elements of (M, N) has step N from element to element and M * heads * N from group to group.  All operands of
// a launch share `heads`, so that a workgroup divides once and keeps two scalars: with a division per operand
// the one-kernel attention backward (eight operands) spilled scalar registers and lost 1.5 %.
struct BatchPos {
  unsigned g, r;
};
__device__ __forceinline__ BatchPos batch_pos(int64_t b, int heads) {
  if (heads <= 0) return BatchPos{0u, (unsigned)b};
  const unsigned g = (unsigned)b / (unsigned)heads;
  return BatchPos{g, (unsigned)b - g * (unsigned)heads};
}
struct BatchStep {
  int64_t step, group;
  int heads;
  __device__ __forceinline__ int64_t at(BatchPos p) const { return (int64_t)p.g * group + (int64_t)p.r * step; }
};

// Rank-3 view handed to kernels: element strides, 64-bit.
struct View {
  void *data;
  BatchStep sb;
  int64_t sr, sc;
};

inline View make_view(const wm_operand *op) {
  return View{op->data, BatchStep{op->stride_b, 0, 0}, op->stride_r, op->stride_c};
}
// heads outside 0 ... 2^31 - 1 become -1, which no call accepts (common_heads).
inline View make_view(const wm_grouped_operand *g) {
  const int heads = g->heads < 0 || g->heads > 0x7fffffff ? -1 : (int)g->heads;
  return View{g->op.data, BatchStep{g->op.stride_b, g->stride_g, heads}, g->op.stride_r, g->op.stride_c};
}
// Same storage seen with rows and columns swapped: (B,N,M) <-> (B,M,N).
inline View transposed(const View &v) { return View{v.data, v.sb, v.sc, v.sr}; }

struct Problem {
  int64_t B, M, N, w;
  int dtype;
  unsigned flags;
  hipStream_t stream;
};

// Workgroups of a tiled launch over B batch elements of nblk blocks each (the decode_block of the
// kernels maps them back): whole elements for every full group of 8, the rest of the tiles in eight
// equal ranges.  No surplus workgroups: the dispatcher places workgroups in order, and ones that
// return at once still shift the others onto fewer CUs.
inline int64_t tiled_grid(int64_t B, int64_t nblk) { return 8 * ((B >> 3) * nblk + ((B & 7) * nblk + 7) / 8); }

// Workgroup -> (batch, block).  Workgroups are dealt round-robin to the 8 XCDs, each with its
// own L2: XCD x runs ids x, x + 8, ...  Every full group of 8 batch elements gives one element to
// each XCD, so that neighbouring blocks of an element find the rows they share (the +-w halo) in
// that L2; the B % 8 elements left over are cut into 8 contiguous ranges of tiles, one per XCD
// (a whole element per XCD would leave one XCD idle at B = 7).  The launch uses tiled_grid():
// at most 7 workgroups at the end of the grid have no tile and return at once.
__device__ __forceinline__ bool decode_block(int nblk, int B, int *b, int *blk) {
  const int id = blockIdx.x, xcd = id & 7, slot = id >> 3;
  const int full = (B >> 3) * nblk;  // slots of the full groups
  if (slot < full) {
    *b = (slot / nblk) * 8 + xcd;
    *blk = slot % nblk;
    return true;
  }
  const int64_t tiles = (int64_t)(B & 7) * nblk, per = (tiles + 7) / 8, t = xcd * per + (slot - full);
  if (slot - full >= per || t >= tiles) return false;
  *b = (B & ~7) + (int)(t / nblk);
  *blk = (int)(t % nblk);
  return true;
}

// Launchers return hipSuccess or the launch error.  The strided family accepts
// any dtype and layout; the MFMA family reports whether it took the problem.
hipError_t launch_strided_p1(const Problem &p, const View &x, const View &y, const View &c);
hipError_t launch_strided_p2(const Problem &p, const View &a, const View &y, const View &c);
hipError_t launch_strided_p3(const Problem &p, const View &a, const View &y, const View &c);

// Returns true and sets *err when the MFMA family handles the problem.
bool try_launch_mfma_p1(const Problem &p, const View &x, const View &y, const View &c, hipError_t *err);
bool try_launch_mfma_p2(const Problem &p, const View &a, const View &y, const View &c, hipError_t *err);
bool try_launch_mfma_p3(const Problem &p, const View &a, const View &y, const View &c, hipError_t *err);
// Whether the band-in kernels of that family that load their tiles straight into LDS accept the
// layout of band `a` and operand `y` (the shape aside): what the narrow-band family asks before it
// leaves a window to them.
bool lds_direct_layout_ok(const Problem &p, const View &a, const View &y);
// Narrow-band family (w <= 32; P2 and P3 while their LDS images fit 64 KB; float32 at N <= 64).
bool try_launch_small_p1(const Problem &p, const View &x, const View &y, const View &c, hipError_t *err);
bool try_launch_small_p2(const Problem &p, const View &a, const View &y, const View &c, hipError_t *err);
bool try_launch_small_p3(const Problem &p, const View &a, const View &y, const View &c, hipError_t *err);
bool small_supports(int op, int64_t M, int64_t N, int64_t w, int dtype, unsigned flags);
bool small_f32_in_supports(int64_t M, int64_t N, int64_t w);  // float32 band-in kernels of the narrow-band family
bool small_f32_p1_supports(int64_t M, int64_t N, int64_t w);  // float32 band-out kernel of the narrow-band family
// Vector-ALU kernels for the narrowest windows: 16-bit up to w = 3 (band-in) and w = 2 (band-out),
// float32 up to w = 14 (the band-out product only where the narrow-band float32 kernel does not apply).
bool try_launch_vector_p1(const Problem &p, const View &x, const View &y, const View &c, hipError_t *err);
bool try_launch_vector_p2(const Problem &p, const View &a, const View &y, const View &c, hipError_t *err);
bool try_launch_vector_p3(const Problem &p, const View &a, const View &y, const View &c, hipError_t *err);
bool vector_supports(int op, int64_t M, int64_t N, int64_t w, int dtype);
// Both gradients of an op in one launch of the vector-ALU kernels, for small problems (false: not taken,
// nothing launched; the caller then launches the two products separately).
bool try_launch_vector_window_backward(const Problem &p, const View &ga, const View &k, const View &q, const View &gq,
                                       const View &gk, hipError_t *err);
bool try_launch_vector_unwindow_backward(const Problem &p, const View &a, const View &v, const View &go, const View &ga,
                                         const View &gv, hipError_t *err);
// float32 MFMA family (N multiple of 8 up to 128, w >= 4).
bool try_launch_f32_p1(const Problem &p, const View &x, const View &y, const View &c, hipError_t *err);
bool try_launch_f32_p2(const Problem &p, const View &a, const View &y, const View &c, hipError_t *err);
bool try_launch_f32_p3(const Problem &p, const View &a, const View &y, const View &c, hipError_t *err);
bool f32_supports(int op, int64_t M, int64_t N, int64_t w, int dtype);
// The same products on the bf16 matrix instruction through an exact three-way split of every float32
// value (wm_f32_split.hip); taken ahead of the kernels above from a window size on.
bool try_launch_f32_split_p1(const Problem &p, const View &x, const View &y, const View &c, hipError_t *err);
bool try_launch_f32_split_p2(const Problem &p, const View &a, const View &y, const View &c, hipError_t *err);
bool try_launch_f32_split_p3(const Problem &p, const View &a, const View &y, const View &c, hipError_t *err);
// dS = scale * P * (dO V^T - rowsum(dO * O)) in band form, by the band-out kernel of that family.
bool try_launch_f32_split_score_gradient(const Problem &p, const View &go, const View &v, const View &o, const View &probs,
                                         const View &gs, double scale, hipError_t *err);
bool f32_split_supports(int op, int64_t M, int64_t N, int64_t w, int dtype, unsigned flags);
// Tile family: float64, and whatever the families above decline in 16-bit and float32 storage;
// 64 x 64 tiles on the 16x16x4 matrix instructions, any strides, any N and w.
bool try_launch_tile_p1(const Problem &p, const View &x, const View &y, const View &c, hipError_t *err);
bool try_launch_tile_p2(const Problem &p, const View &a, const View &y, const View &c, hipError_t *err);
bool try_launch_tile_p3(const Problem &p, const View &a, const View &y, const View &c, hipError_t *err);
bool tile_supports(int op, int64_t M, int64_t N, int64_t w, int dtype);
// Pure predicate behind the wide-band 16-bit functions above (shape/dtype only).
bool mfma_supports(int op, int64_t B, int64_t M, int64_t N, int64_t w, int dtype);

// Softmax along the band dimension (wm_softmax.hip).  `mask` non-zero treats entries outside
// the sequence as -infinity.  In-place use (out aliasing an input) is allowed.
hipError_t launch_band_softmax_forward(const Problem &p, const View &a, const View &out, double scale, int mask);
hipError_t launch_band_softmax_backward(const Problem &p, const View &probs, const View &grad_probs,
                                        const View &grad_a, double scale, int mask);
// Whether rows of length W get the LDS-staged kernel (given contiguous, 16-byte aligned tensors).
bool band_softmax_staged(int64_t W, int dtype, bool backward);

// Fused window attention forward (wm_attention.hip): q, k, v, o row-major (B,M,N) views, lse an
// optional float32 (B,M) buffer.  Returns false when the kernel does not take the problem.
bool attention_supports(int64_t M, int64_t N, int64_t w, int dtype, double scale);
bool try_launch_attention_forward(const Problem &p, const View &q, const View &k, const View &v, const View &o,
                                  float *lse, double scale, int mask, hipError_t *err);

// The same pair for head widths that 16 does not divide (N >= 8, WM_FLAG_ANY_HEAD_WIDTH set): rows of any alignment.
bool try_launch_attention_forward_ragged(const Problem &p, const View &q, const View &k, const View &v, const View &o,
                                         float *lse, double scale, int mask, hipError_t *err);
bool try_launch_attention_backward_ragged(const Problem &p, const View &q, const View &k, const View &v, const View &o,
                                          const View &go, const float *lse, float *delta, const View &gq,
                                          const View &gk, const View &gv, double scale, hipError_t *err);

// Backward of the fused attention (wm_attention_bwd.hip): two kernels on p.stream; `delta` is a
// float32 (2,B,M) workspace the first one fills and the second one reads (-D and the log-sum-exp in log2 units).
bool try_launch_attention_backward(const Problem &p, const View &q, const View &k, const View &v, const View &o,
                                   const View &go, const float *lse, float *delta, const View &gq, const View &gk,
                                   const View &gv, double scale, hipError_t *err);

// Fused window attention in float32 (wm_attention_f32.hip): stats is a float32 (2,B,M) buffer that the forward fills (it may be
// null) and the backward reads, delta a float32 (B,M) workspace of the backward.
bool attention_f32_supports(const Problem &p, double scale);
bool try_launch_attention_f32_forward(const Problem &p, const View &q, const View &k, const View &v, const View &o, float *stats,
                                      double scale, int mask, hipError_t *err);
bool try_launch_attention_f32_backward(const Problem &p, const View &q, const View &k, const View &v, const View &o, const View &go,
                                       const float *stats, float *delta, const View &gq, const View &gk, const View &gv,
                                       double scale, hipError_t *err);
hipError_t launch_attention_f32_key_wide(const Problem &p, const View &q, const View &k, const View &v, const View &go, const float *stats,
                                         const float *delta, const View &gk, const View &gv, double scale);  // N > 96

// Batched transpose of the last two dimensions (wm_transpose.hip): src (B,R,C) with unit column stride and
// batch / row strides ssb / ssr (elements), dst contiguous (B,C,R).  Returns false, nothing launched,
// unless dst is 16-byte aligned, R is a multiple of 16 bytes and elem_size is 2, 4 or 8.
bool try_launch_transpose(const void *src, void *dst, int64_t B, int64_t R, int64_t C, BatchStep ssb, int64_t ssr,
                          int elem_size, hipStream_t stream, hipError_t *err);

inline size_t dtype_size(int dtype) {
  switch (dtype) {
    case WM_DTYPE_F32: return 4;
    case WM_DTYPE_F16: return 2;
    case WM_DTYPE_BF16: return 2;
    case WM_DTYPE_F64: return 8;
    default: return 0;
  }
}

// Unit column stride, every row start 16-byte aligned: what the vector paths need.
inline bool fast_layout(const View &v, int dtype) {
  const int64_t es = (int64_t)dtype_size(dtype);
  if (v.sc != 1) return false;
  if (((uintptr_t)v.data) % 16 != 0) return false;
  return (v.sr * es) % 16 == 0 && (v.sb.step * es) % 16 == 0 && (v.sb.heads <= 0 || (v.sb.group * es) % 16 == 0);
}

// The fused attention kernels that share the streamed side of a tile out among wavefronts (workgroups of `rows` rows)
// are taken while all their workgroups start at once, one on a CU: up to there they are faster at the windows from
// 32 on, or as fast (the key kernel at exactly 256 workgroups), beyond it the second round makes them slower.  us without / with, tiles of 128 rows in the launch:
//   forward (64 rows)       N = 128 w = 1024: 64 tiles 45 / 25, 128 46 / 27, 192 46 / 47;  w = 256: 128 tiles 18 / 13, 192 18.7 / 23.7
//                           N = 64 w = 256: 128 tiles 12.5 / 9.4, 192 12.6 / 13.2;  w = 64: 128 tiles 8.0 / 7.2
//   query kernel (64 rows)  N = 128 w = 256: 128 tiles 23.8 / 18.2, 192 26 / 33;  w = 64: 14.2 / 13.5;  N = 96 w = 20: 9.1 / 9.8
//   key kernel (32 rows)    N = 128 w = 256: 64 tiles 29.5 / 18.2, 128 29.1 / 29.1, 192 30 / 42;  w = 64: 64 tiles 17.7 / 14.0
inline bool shares_pay(int64_t B, int64_t M, int64_t w, int rows) { return w >= 32 && B * ((M + rows - 1) / rows) <= 256; }

// Whether 32-bit byte offsets reach `past` rows beyond the M rows of a 16-bit batch element: the kernels that load straight
// into LDS address it so and request whole chunks up to some past the last one, each launch as many rows as its kernel says.
inline bool rows_in_reach(const View &v, int64_t M, int64_t past) { return v.sr > 0 && (M + past) * v.sr * 2 < 0x7fffffff; }

// 16-bit rows of N elements whose pieces all start on a multiple of 4 bytes, which is what loads straight into LDS need: the
// rows themselves, and the last piece, which starts at column N - 8 (HeadWidth), so an odd N never qualifies.
inline bool dword_pieces(const View &v, int64_t N) {
  return N % 2 == 0 && (uintptr_t)v.data % 4 == 0 && v.sr % 2 == 0 && v.sb.step % 2 == 0 &&
         (v.sb.heads <= 0 || v.sb.group % 2 == 0);
}

// Band operands are only required to be contiguous per batch (rows of odd
// length 2w+1 are never 16-byte aligned); the kernels realign in LDS.
inline bool band_layout(const View &v, int64_t W) { return v.sc == 1 && v.sr == W; }

}  // namespace wm
