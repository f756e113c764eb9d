// Vector work dealt out among matrix instructions, for kernels of one wavefront per SIMD.
#pragma once

#include <type_traits>
#include <utility>

#include "wm_mfma_common.hpp"

namespace wm {
namespace {

// A matrix instruction of 32 cycles leaves its wavefront free to issue five or six vector instructions beside it (measured: 35 cycles
// alone, 42 with six), but the compiler puts the ones first and the others after them.  Where a SIMD holds one wavefront nothing
// else fills the time.  So the vector work comes as a list of small steps, and deal() runs slot i of SLOTS with its share
// of them, fenced against reordering.  What it brings stands at forward_stages() in wm_attention_f32.hip; with two wavefronts per SIMD nothing.
template <int... I, typename F>
__device__ __forceinline__ void each_of(std::integer_sequence<int, I...>, F &&f) {
  (f(std::integral_constant<int, I>()), ...);
}
template <int N, typename F>
__device__ __forceinline__ void each(F &&f) {
  each_of(std::make_integer_sequence<int, N>(), f);
}
template <int SLOTS, int STEPS, typename Slot, typename Step>
__device__ __forceinline__ void deal(Slot &&slot, Step &&step) {
  each<SLOTS>([&](auto i) {
    constexpr int from = i * STEPS / SLOTS, to = (i + 1) * STEPS / SLOTS;
    slot(i);
    each<to - from>([&](auto j) { step(std::integral_constant<int, from + decltype(j)::value>()); });
    __builtin_amdgcn_sched_barrier(0);
  });
}

}  // namespace
}  // namespace wm
