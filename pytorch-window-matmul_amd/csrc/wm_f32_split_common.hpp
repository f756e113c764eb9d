// float32 values as three bf16 planes, for products at float32 accuracy on the bf16 matrix instruction (wm_f32_split.hip says why
// and with what error).
#pragma once

#include "wm_mfma_common.hpp"

namespace wm {
namespace {

constexpr int kStage = 32 + 4;     // staged result row: 32 floats, rows 16 bytes apart mod 128

struct __attribute__((packed, aligned(4))) Chunk4 {
  f32x4 v;
};
__device__ __forceinline__ f32x4 load4(const float *p) { return reinterpret_cast<const Chunk4 *>(p)->v; }
__device__ __forceinline__ void store4(float *p, f32x4 v) { reinterpret_cast<Chunk4 *>(p)->v = v; }

// The three bf16 planes of four consecutive floats, each plane as 8 bytes (element e in bits 16 e .. 16 e + 15).
struct Planes4 {
  u32x2 p[3];
};
__device__ __forceinline__ uint32_t high_halves(uint32_t hi, uint32_t lo) {
  return __builtin_amdgcn_perm(hi, lo, 0x07060302u);  // (hi & 0xffff0000) | (lo >> 16)
}
__device__ __forceinline__ Planes4 split4(f32x4 v) {
  uint32_t a[4], b[4], c[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    a[e] = __float_as_uint(v[e]);
    const float r1 = v[e] - __uint_as_float(a[e] & 0xffff0000u);  // exact: the low 16 bits of the significand
    b[e] = __float_as_uint(r1);
    c[e] = __float_as_uint(r1 - __uint_as_float(b[e] & 0xffff0000u));  // at most 8 significant bits left
  }
  Planes4 r;
  r.p[0] = u32x2{high_halves(a[1], a[0]), high_halves(a[3], a[2])};
  r.p[1] = u32x2{high_halves(b[1], b[0]), high_halves(b[3], b[2])};
  r.p[2] = u32x2{high_halves(c[1], c[0]), high_halves(c[3], c[2])};
  return r;
}

__device__ __forceinline__ f32x16 mma16(u32x4 a, u32x4 b, f32x16 c) { return Mma<bf16_t>::run(a, b, c); }
// acc += x y for the split operands xa (A side) and xb (B side), smallest terms first
__device__ __forceinline__ f32x16 mma_split(const u32x4 (&xa)[3], const u32x4 (&xb)[3], f32x16 acc) {
  acc = mma16(xa[2], xb[0], acc);
  acc = mma16(xa[0], xb[2], acc);
  acc = mma16(xa[1], xb[1], acc);
  acc = mma16(xa[1], xb[0], acc);
  acc = mma16(xa[0], xb[1], acc);
  acc = mma16(xa[0], xb[0], acc);
  return acc;
}

}  // namespace
}  // namespace wm
