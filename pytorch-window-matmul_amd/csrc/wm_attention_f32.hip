// Fused window attention in float32, forward and backward: what wm_attention.hip and wm_attention_bwd.hip do for 16-bit storage,
// with every product at float32 accuracy on the bf16 matrix instruction (three planes per operand, six products per pair,
// wm_f32_split.hip).  The band never reaches memory: through the separate ops a training step writes or reads it eleven
// times, 807 MB each at B96 M4096 N64 w256.
//
//   forward       a workgroup owns 128 queries, 32 per wavefront, and walks over the keys its band can reach in chunks of 32:
//                 S^T = K Q^T, an online softmax with a running maximum that is raised lazily, O^T += V^T P^T.  For the backward
//                 it leaves two float32 values per row, the score m the exponentials were taken against (the maximum, or a
//                 little below it) and 1 / l, l the sum of them.  A log-sum-exp in one float would be off by half a unit in its last place, for a
//                 value around 10 that is 5e-7, a relative error of every probability of the row; m and 1 / l are exact and
//                 correctly rounded.
//   query kernel  128 queries: S^T, dP^T = V dO^T, dS^T, dQ^T += K^T dS^T.  Also writes D / l, D = sum_h dO O, for
//   key kernel    128 keys, walks over the queries: S, dP, dV^T += dO^T P, dK^T += Q^T dS, or what one of the two needs.
// The backward works on exp2(c (S - m)), not yet divided by l: dO is multiplied by 1 / l on its way in instead.
//
// Layouts are those of the 16-bit kernels: in a 32 x 32 score tile a lane owns one stationary row and sixteen streamed ones, the
// stationary operands stay in registers as planes, P and dS come out arranged as B operands.  A streamed chunk goes through
// registers, is split once per workgroup and stored as swizzled bf16 planes (LdsTile), read by rows and transposed.
//
// Head widths (training through window_attention begins at N = 33, f32_fused() in binding.cpp; the backward of narrower ones is for
// callers of the C ABI): any N = 8 ... 128, in pieces of eight columns, the last one moved back to end with the row (HeadWidth).  The
// columns it shares with the piece before are cleared in the stationary operands; as result columns they come out twice.
//
// With F32_KEY_WIDE set (wm_attention_f32_key_wide.hip) this translation unit holds the key kernel for N > 96 alone, which wants
// a compiler option of its own (FILE_FLAGS in build.py).
#include "wm_deal.hpp"
#include "wm_f32_split_common.hpp"

#ifndef F32_KEY_WIDE
#define F32_KEY_WIDE 0
#endif

namespace wm {
namespace {

constexpr int FA_TM = 128;  // stationary rows per workgroup
constexpr int FA_KC = 32;   // streamed rows per chunk
constexpr float kRaiseBy = 8.0f;

// Chunks in LDS.  With three, the first products of a chunk run one iteration ahead of the rest, their vector work dealt out among
// the matrix instructions (deal() below).  That is for one wavefront per SIMD: us at B96 M4096 w256, two stages / three, each kernel over and
// over (the clock falls under that load: the forward at N = 64 takes 326 with pauses and 304-312 in a training step): forward
// N = 32 191 / 203, N = 64 430 / 430 (B2 M4096 w1024, one wavefront per SIMD there too: 121 / 92), N = 128 735 / 712; query kernel
// N = 64 520 / 595 (two wavefronts only on two stages), N = 80 789 / 703, N = 128 1087 / 1005; key kernel and D N = 32 w = 64 166 / 237,
// N = 64 853 / 782, N = 80 1073 / 959, N = 96 1146 / 1053, N = 128 1450 / 1817 (there its registers do not suffice).
constexpr int forward_stages(int NK) { return NK <= 3 ? 2 : 3; }
constexpr int query_stages(int NK) { return NK <= 4 ? 2 : 3; }
constexpr int key_stages(int NK) { return NK >= 3 && NK <= 6 ? 3 : 2; }

// A chunk of two streamed tensors as it lies in LDS.
template <int NK>
struct PlaneTile {
  static constexpr int NB = (NK + 1) / 2, PPR = NK <= 4 ? 8 : 16, ROWB = 16 * PPR;
  static constexpr int SLOTS = FA_KC * PPR / kThreads;  // pieces of eight columns per thread and tensor
  static constexpr int PLANE = FA_KC * PPR * 8;         // elements of a plane
  static constexpr int STAGE_BYTES = 2 * 3 * PLANE * 2;
  typedef LdsTile<FA_KC, PPR> Tile;
};

// The pieces of a chunk that a thread moves: row of the chunk, column in memory, byte offset in a plane.
template <int NK>
struct ChunkPieces {
  int row[PlaneTile<NK>::SLOTS], column[PlaneTile<NK>::SLOTS], at[PlaneTile<NK>::SLOTS];
  __device__ __forceinline__ ChunkPieces(HeadWidth<true, NK> width, int tid) {
    typedef PlaneTile<NK> TL;
    const int pieces = width.pieces();
#pragma unroll
    for (int u = 0; u < TL::SLOTS; ++u) {
      const int q = min(tid + kThreads * u, FA_KC * pieces - 1);  // an idle thread repeats the last piece
      row[u] = q / pieces;
      const int piece = q - row[u] * pieces;
      column[u] = width.column(piece);
      at[u] = row[u] * TL::ROWB + ((piece ^ swz<TL::PPR>(row[u])) << 4);
    }
  }
};

struct Eight {
  f32x4 lo, hi;
};
__device__ __forceinline__ Eight load8(const float *p) { return Eight{load4(p), load4(p + 4)}; }
__device__ __forceinline__ void split8(const Eight &v, u32x4 (&planes)[3]) {
  const Planes4 lo = split4(v.lo), hi = split4(v.hi);
#pragma unroll
  for (int p = 0; p < 3; ++p) planes[p] = u32x4{lo.p[p][0], lo.p[p][1], hi.p[p][0], hi.p[p][1]};
}
__device__ __forceinline__ void split_to_lds(char *plane0, int plane_bytes, int at, const Eight &v) {
  u32x4 planes[3];
  split8(v, planes);
#pragma unroll
  for (int p = 0; p < 3; ++p) *reinterpret_cast<u32x4 *>(plane0 + p * plane_bytes + at) = planes[p];
}
// Piece of a row that stays in registers: the columns it shares with the piece before are zeros, rows outside too.
template <int NK>
__device__ __forceinline__ Eight mask_piece(HeadWidth<true, NK> width, Eight v, bool valid, int piece) {
  const bool there = valid && piece < width.pieces();
  const int first = width.first(piece);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    v.lo[e] = there && e >= first ? v.lo[e] : 0.0f;
    v.hi[e] = there && e + 4 >= first ? v.hi[e] : 0.0f;
  }
  return v;
}
// All pieces of the rows of two tensors, one row per lane: every load in flight before the first is waited for.
template <int NK>
__device__ __forceinline__ void fetch_pieces(HeadWidth<true, NK> width, const float *row, const float *safe, bool valid, int half,
                                             Eight (&v)[NK]) {
#pragma unroll
  for (int ks = 0; ks < NK; ++ks)
    v[ks] = load8(valid && 2 * ks + half < width.pieces() ? row + width.column(2 * ks + half) : safe);
}
template <int NK>
__device__ __forceinline__ Eight stationary_piece(HeadWidth<true, NK> width, const float *row, const float *safe, bool valid,
                                                  int piece) {
  return mask_piece(width, load8(valid && piece < width.pieces() ? row + width.column(piece) : safe), valid, piece);
}

__device__ __forceinline__ float both_halves_max(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float both_halves_sum(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// 2^(c (s - m)), c > 0 and a normal number.  The difference comes first: it is 0 at the maximum whatever the size of the scores,
// where c s rounded against c m exact leaves half a unit of c m, which from 2^31 on overflows the exponential of that entry or
// empties a row.  One instruction more per entry than a fused multiply-add, and no time: a training step at B96 M4096 N64 w256 takes
// 1475 us, 1472 with that.
__device__ __forceinline__ float exp2_above(float s, float m, float c) { return __builtin_amdgcn_exp2f((s - m) * c); }

// split4 in three steps: two elements, the other two, the planes.
struct Split4Steps {
  uint32_t a[4], b[4], c[4];
  template <int STEP>
  __device__ __forceinline__ void run(const f32x4 &v, u32x4 (&planes)[3], int part) {
    if (STEP < 2) {
#pragma unroll
      for (int e = 2 * STEP; e < 2 * STEP + 2 && STEP < 2; ++e) {
        a[e] = __float_as_uint(v[e]);
        const float r1 = v[e] - __uint_as_float(a[e] & 0xffff0000u);
        b[e] = __float_as_uint(r1);
        c[e] = __float_as_uint(r1 - __uint_as_float(b[e] & 0xffff0000u));
      }
    } else {
      planes[0][2 * part] = high_halves(a[1], a[0]), planes[0][2 * part + 1] = high_halves(a[3], a[2]);
      planes[1][2 * part] = high_halves(b[1], b[0]), planes[1][2 * part + 1] = high_halves(b[3], b[2]);
      planes[2][2 * part] = high_halves(c[1], c[0]), planes[2][2 * part + 1] = high_halves(c[3], c[2]);
    }
  }
};
// A piece of eight columns on its way into LDS in seven steps.
struct StashSteps {
  Split4Steps s;
  u32x4 planes[3];
  template <int STEP>
  __device__ __forceinline__ void run(const Eight &v, char *plane0, int plane_bytes, int at) {
    if constexpr (STEP < 3) {
      s.run<STEP>(v.lo, planes, 0);
    } else if constexpr (STEP < 6) {
      s.run<STEP - 3>(v.hi, planes, 1);
    } else {
#pragma unroll
      for (int p = 0; p < 3; ++p) *reinterpret_cast<u32x4 *>(plane0 + p * plane_bytes + at) = planes[p];
    }
  }
};
// Matrix instruction I of the six of a split product that sums the products of the leading planes and the rest apart, each
// rounding at its own magnitude (relative distance to float64 at N = 128, w = 100: 2.7e-7 against 3.8e-7 with one sum).
// SWAPPED takes the products in the order that they have with the operands exchanged.  The key kernel, whose A operand are the
// queries, forms the scores with it, bit for bit those of the forward: where scores are large a difference in their last
// bit is one of the probabilities against the row's sum.
template <int I, bool SWAPPED = false>
__device__ __forceinline__ void mma_step_two(const u32x4 (&xa)[3], const u32x4 (&xb)[3], f32x16 &lead, f32x16 &rest) {
  constexpr int X[6] = {2, 0, 0, 1, 1, 0}, Y[6] = {0, 0, 2, 1, 0, 1};
  constexpr int a = SWAPPED ? Y[I] : X[I], b = SWAPPED ? X[I] : Y[I];
  if (I == 1)
    lead = mma16(xa[a], xb[b], lead);
  else
    rest = mma16(xa[a], xb[b], rest);
}
template <bool SWAPPED = false>
__device__ __forceinline__ void mma_split_two(const u32x4 (&xa)[3], const u32x4 (&xb)[3], f32x16 &lead, f32x16 &rest) {
  each<6>([&](auto i) { mma_step_two<decltype(i)::value, SWAPPED>(xa, xb, lead, rest); });
}
template <int I>
__device__ __forceinline__ void mma_step(const u32x4 (&xa)[3], const u32x4 (&xb)[3], f32x16 &acc) {
  constexpr int A[6] = {2, 0, 1, 1, 0, 0}, B[6] = {0, 2, 1, 0, 1, 0};
  acc = mma16(xa[A[I]], xb[B[I]], acc);
}

// Accumulator v of a lane stands for streamed row r0 + 8 (v / 4) + 4 half + v % 4 and stationary row `mine`; entries outside the
// band or the sequence become -infinity.
__device__ __forceinline__ void mask_band_edge(f32x16 &s, int r0, int half, int mine, int w, int M) {
  const int d0 = r0 + 4 * half - mine;
  const int first = -w - d0, last = min(w - d0, M - 1 - r0 - 4 * half);
  const int origin = last < first ? 0x100000 : first;
  const unsigned span = last < first ? 0u : (unsigned)(last - first);
  const float ninf = -__builtin_huge_valf();
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const int ofs = 8 * (v / 4) + v % 4;
    s[v] = (unsigned)(ofs - origin) <= span ? s[v] : ninf;
  }
}

// The wavefront's 32 result rows (lane % 32) leave through a private LDS area, 32 columns at a time, in 16-byte pieces of
// which eight lanes write 128 consecutive bytes.
template <int NK>
__device__ __forceinline__ void store_f32_rows(float *stage, const f32x16 (&acc)[(NK + 1) / 2], float mul, float *C, int64_t csr,
                                               int row0, int M, HeadWidth<true, NK> width, int lane) {
  const int half = lane >> 5, r32 = lane & 31;
#pragma unroll
  for (int hb = 0; hb < (NK + 1) / 2; ++hb) {
    wave_sync_lds();
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<f32x4 *>(stage + r32 * kStage + 8 * g + 4 * half) =
          f32x4{acc[hb][4 * g] * mul, acc[hb][4 * g + 1] * mul, acc[hb][4 * g + 2] * mul, acc[hb][4 * g + 3] * mul};
    wave_sync_lds();
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int rr = (lane >> 3) + 8 * s, x = 4 * (lane & 7), piece = 4 * hb + (x >> 3);
      if (row0 + rr < M && piece < width.pieces())
        store4(C + (int64_t)(row0 + rr) * csr + width.column(piece) + (x & 4),
               *reinterpret_cast<const f32x4 *>(stage + rr * kStage + x));
    }
  }
}

// ---------------------------------------------------------------------------------------------
// forward
// ---------------------------------------------------------------------------------------------
template <int NK, bool MASK>  // 16 NK - 15 <= N <= 16 NK
__global__ __launch_bounds__(kThreads, NK <= 4 ? 2 : 1) void attention_f32_forward_kernel(
    const float *__restrict__ Q, const float *__restrict__ K, const float *__restrict__ V, float *__restrict__ O,
    float *__restrict__ stats, int B, int M, int w, int nblk, int n, float c, BatchStep qsb, int64_t qsr, BatchStep ksb,
    int64_t ksr, BatchStep vsb, int64_t vsr, BatchStep osb, int64_t osr) {
  typedef PlaneTile<NK> TL;
  typedef typename TL::Tile Tile;
  constexpr int NB = TL::NB, SLOTS = TL::SLOTS, PLANE = TL::PLANE, STAGES = forward_stages(NK);
  constexpr bool AHEAD = STAGES == 3;
  extern __shared__ __attribute__((aligned(1024))) uint16_t fa_lds[];  // [stage][K, V][plane]
  auto tile = [&](int buf, int tensor, int p) { return fa_lds + ((buf * 2 + tensor) * 3 + p) * PLANE; };

  const HeadWidth<true, NK> width{n};
  int b, blk;
  if (!decode_block(nblk, B, &b, &blk)) return;
  const BatchPos bp = batch_pos(b, ksb.heads);
  const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i0 = blk * FA_TM;
  const int qw0 = i0 + 32 * wave, qi = qw0 + (lane & 31);
  const float *Kb = K + ksb.at(bp), *Vb = V + vsb.at(bp);

  const int kc_lo = max(i0 - w, 0) / FA_KC;
  const int kc_hi = min(i0 + FA_TM - 1 + w, M - 1) / FA_KC;
  const ChunkPieces<NK> mine(width, tid);
  Eight kreg[SLOTS], vreg[SLOTS];
  // Rows past the end of the sequence, and the chunk after the last one, repeat the last row: their keys are masked out.
  auto fetch = [&](int kc) {
#pragma unroll
    for (int u = 0; u < SLOTS; ++u) {
      const int key = min(kc * FA_KC + mine.row[u], M - 1);
      kreg[u] = load8(Kb + (int64_t)key * ksr + mine.column[u]);
      vreg[u] = load8(Vb + (int64_t)key * vsr + mine.column[u]);
    }
  };
  auto stash = [&](int buf) {
#pragma unroll
    for (int u = 0; u < SLOTS; ++u) {
      split_to_lds(reinterpret_cast<char *>(tile(buf, 0, 0)), 2 * PLANE, mine.at[u], kreg[u]);
      split_to_lds(reinterpret_cast<char *>(tile(buf, 1, 0)), 2 * PLANE, mine.at[u], vreg[u]);
    }
  };
  fetch(kc_lo);
  // pieces of a row past the last one are never written and must read as zeros
  if (width.pieces() < TL::PPR) {
    for (int e = tid; e < STAGES * TL::STAGE_BYTES / 16; e += kThreads) reinterpret_cast<u32x4 *>(fa_lds)[e] = u32x4{0u, 0u, 0u, 0u};
    __syncthreads();
  }

  u32x4 qop[NK][3];  // B operand of the first product: this lane's query, split
  {
    const float *qr = Q + qsb.at(bp) + (int64_t)qi * qsr;
#pragma unroll
    for (int ks = 0; ks < NK; ++ks) split8(stationary_piece(width, qr, Q, qi < M, 2 * ks + half), qop[ks]);
  }
  const uint32_t row_at = Tile::row_at(lane), tr_at = Tile::tr_at(lane);
  f32x16 o[NB];
#pragma unroll
  for (int hb = 0; hb < NB; ++hb)
#pragma unroll
    for (int v = 0; v < 16; ++v) o[hb][v] = 0.0f;
  float m_used = -__FLT_MAX__, l_part = 0.0f;

  // Chunk kc's scores are formed one iteration ahead of their use: the products of chunk kc + 1 with the queries run while the
  // vector ALU takes the exponentials of chunk kc and splits them, the products of chunk kc with the values while it splits
  // the rows of chunk kc + 2.
  auto scores = [&](int buf, f32x16 &s, f32x16 &rest) {
#pragma unroll
    for (int v = 0; v < 16; ++v) s[v] = 0.0f, rest[v] = 0.0f;
#pragma unroll
    for (int ks = 0; ks < NK; ++ks) {
      u32x4 ka[3];
#pragma unroll
      for (int p = 0; p < 3; ++p) ka[p] = Tile::rows(tile(buf, 0, p), row_at, 0, ks);
      mma_split_two(ka, qop[ks], s, rest);
    }
  };
  auto row_max = [&](const f32x16 &s) {
    float a = fmaxf(s[0], s[1]), bb = fmaxf(s[2], s[3]);
#pragma unroll
    for (int v = 4; v < 16; v += 4) a = fmaxf(fmaxf(a, s[v]), s[v + 1]), bb = fmaxf(fmaxf(bb, s[v + 2]), s[v + 3]);
    return both_halves_max(fmaxf(a, bb));
  };
  auto raise_to = [&](float bm) {
    const bool raise = (bm - m_used) * c > kRaiseBy;
    if (__builtin_amdgcn_ballot_w64(raise) != 0) {
      const float m_new = raise ? bm : m_used;
      const float alpha = exp2_above(m_used, m_new, c);
      m_used = m_new;
      l_part *= alpha;
#pragma unroll
      for (int hb = 0; hb < NB; ++hb)
#pragma unroll
        for (int v = 0; v < 16; ++v) o[hb][v] *= alpha;
    }
  };
  auto probabilities = [&](const f32x16 &s, u32x4 (&pf)[2][3]) {
    float p[16], sum[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int v = 0; v < 16; ++v) p[v] = exp2_above(s[v], m_used, c), sum[v / 4] += p[v];
    l_part += (sum[0] + sum[1]) + (sum[2] + sum[3]);
#pragma unroll
    for (int t = 0; t < 2; ++t)
      split8(Eight{f32x4{p[8 * t], p[8 * t + 1], p[8 * t + 2], p[8 * t + 3]},
                   f32x4{p[8 * t + 4], p[8 * t + 5], p[8 * t + 6], p[8 * t + 7]}}, pf[t]);
  };
  auto values = [&](int buf, const u32x4 (&pf)[2][3]) {
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int hb = 0; hb < NB; ++hb) {
        u32x4 va[3];
#pragma unroll
        for (int p3 = 0; p3 < 3; ++p3) va[p3] = Tile::cols(tile(buf, 1, p3), tr_at, 16 * t, hb);
        o[hb] = mma_split(va, pf[t], o[hb]);
      }
  };
  auto in_band = [&](int kc) { return kc <= kc_hi && kc * FA_KC + 31 >= qw0 - w && kc * FA_KC <= qw0 + 31 + w; };
  auto whole = [&](int kc) { return kc * FA_KC >= qw0 + 31 - w && kc * FA_KC + 31 <= qw0 + w && kc * FA_KC + 31 < M; };
  auto after = [](int buf) { return buf + 1 == STAGES ? 0 : buf + 1; };

  stash(0);
  int kc = kc_lo, buf = 0;
  if constexpr (!AHEAD) {
    __syncthreads();
    for (; kc <= kc_hi; ++kc) {
      const int next = after(buf);
      fetch(kc + 1);
      __builtin_amdgcn_sched_barrier(0);
      if (in_band(kc)) {
        f32x16 s, rest;
        scores(buf, s, rest);
#pragma unroll
        for (int v = 0; v < 16; ++v) s[v] += rest[v];
        if (!whole(kc)) mask_band_edge(s, kc * FA_KC, half, qi, w, M);
        raise_to(row_max(s));
        u32x4 pf[2][3];
        probabilities(s, pf);
        values(buf, pf);
      }
      __builtin_amdgcn_sched_barrier(0);
      stash(next);
      __syncthreads();
      buf = next;
    }
  } else {
    f32x16 s;
#pragma unroll
    for (int v = 0; v < 16; ++v) s[v] = 0.0f;
    float bm = 0.0f;
    fetch(kc_lo + 1);
    __syncthreads();
    if (in_band(kc_lo)) {
      f32x16 rest;
      scores(0, s, rest);
#pragma unroll
      for (int v = 0; v < 16; ++v) s[v] += rest[v];
      if (!whole(kc_lo)) mask_band_edge(s, kc_lo * FA_KC, half, qi, w, M);
      bm = row_max(s);
    }
    stash(1);
    __syncthreads();
    // chunks [fast_lo, fast_hi]: they and the one after meet the wavefront's band
    const int fast_lo = max(kc_lo, (qw0 - w) >> 5);
    const int fast_hi = min(kc_hi, (qw0 + 31 + w) >> 5) - 1;
    auto general = [&]() {
      const int next = after(buf), free = after(next);
      fetch(kc + 2);
      f32x16 ns, rest;
      const bool more = in_band(kc + 1);
      if (more) {
        scores(next, ns, rest);
#pragma unroll
        for (int v = 0; v < 16; ++v) ns[v] += rest[v];
        if (!whole(kc + 1)) mask_band_edge(ns, (kc + 1) * FA_KC, half, qi, w, M);
      }
      if (in_band(kc)) {
        raise_to(bm);
        u32x4 pf[2][3];
        probabilities(s, pf);
        values(buf, pf);
      }
      if (more) s = ns, bm = row_max(ns);
      stash(free);
      __syncthreads();
      ++kc, buf = next;
    };
    const int lead_end = fast_lo <= fast_hi ? fast_lo : kc_hi + 1;
    while (kc < lead_end) general();
    while (kc <= fast_hi) {
      const int next = after(buf), free = after(next);
      raise_to(bm);
      fetch(kc + 2);
      __builtin_amdgcn_sched_barrier(0);
      f32x16 ns, rest;
#pragma unroll
      for (int v = 0; v < 16; ++v) ns[v] = 0.0f, rest[v] = 0.0f;
      u32x4 pf[2][3], ka[2][3], va[2][3];
      auto read_key = [&](auto ks) {
#pragma unroll
        for (int p = 0; p < 3; ++p) ka[ks % 2][p] = Tile::rows(tile(next, 0, p), row_at, 0, ks);
      };
      auto read_value = [&](auto x) {  // x = NB t + hb
#pragma unroll
        for (int p = 0; p < 3; ++p) va[x % 2][p] = Tile::cols(tile(buf, 1, p), tr_at, 16 * (x / NB), x % NB);
      };
      read_key(std::integral_constant<int, 0>());
      float pr[16], sum[4] = {0.0f, 0.0f, 0.0f, 0.0f};
      Split4Steps sp;
      deal<6 * NK, 24>(
          [&](auto i) {
            constexpr int ks = i / 6;
            if constexpr (i % 6 == 0 && ks + 1 < NK) read_key(std::integral_constant<int, ks + 1>());
            if constexpr (i == 6 * NK - 6) read_value(std::integral_constant<int, 0>());
            mma_step_two<i % 6>(ka[ks % 2], qop[ks], ns, rest);
          },
          [&](auto j) {
            constexpr int g = j / 6, r = j % 6;
            if constexpr (r < 2) {
#pragma unroll
              for (int v = 4 * g + 2 * r; v < 4 * g + 2 * r + 2; ++v)
                pr[v] = exp2_above(s[v], m_used, c), sum[g] += pr[v];
            } else if constexpr (r < 5) {
              sp.run<r - 2>(f32x4{pr[4 * g], pr[4 * g + 1], pr[4 * g + 2], pr[4 * g + 3]}, pf[g / 2], g % 2);
            } else if constexpr (g == 3) {
              l_part += (sum[0] + sum[1]) + (sum[2] + sum[3]);
            }
          });
      StashSteps st;
      float top[2];
      deal<12 * NB, 8 + 14 * SLOTS>(
          [&](auto i) {
            constexpr int x = i / 6;
            if constexpr (i % 6 == 0 && x + 1 < 2 * NB) read_value(std::integral_constant<int, x + 1>());
            mma_step<i % 6>(va[x % 2], pf[x / NB], o[x % NB]);
          },
          [&](auto j) {
            if constexpr (j < 8) {
              s[2 * j] = ns[2 * j] + rest[2 * j], s[2 * j + 1] = ns[2 * j + 1] + rest[2 * j + 1];
              if (j < 2)
                top[j] = fmaxf(s[2 * j], s[2 * j + 1]);
              else
                top[j % 2] = fmaxf(fmaxf(top[j % 2], s[2 * j]), s[2 * j + 1]);
            } else {
              constexpr int u = (j - 8) / 14, tensor = (j - 8) / 7 % 2;
              st.run<(j - 8) % 7>(tensor ? vreg[u] : kreg[u], reinterpret_cast<char *>(tile(free, tensor, 0)), 2 * PLANE, mine.at[u]);
            }
          });
      if (whole(kc + 1)) {
        bm = both_halves_max(fmaxf(top[0], top[1]));
      } else {
        mask_band_edge(s, (kc + 1) * FA_KC, half, qi, w, M);
        bm = row_max(s);
      }
      __syncthreads();
      ++kc, buf = next;
    }
    while (kc <= kc_hi) general();
  }

  float l = both_halves_sum(l_part);
  float alpha = 1.0f;
  if (!MASK) {  // band entries outside the sequence: score 0 each, no value row
    const int n_out = max(0, w - qi) + max(0, qi + w - (M - 1));
    const float m_new = n_out > 0 ? fmaxf(m_used, 0.0f) : m_used;
    alpha = exp2_above(m_used, m_new, c);
    l = l * alpha + (float)n_out * exp2_above(0.0f, fmaxf(m_new, 0.0f), c);  // no entries outside: 0 times a finite value
    m_used = m_new;
  }
  if (qi >= M) l = 1.0f;  // rows past the end: keep the arithmetic finite, nothing is stored
  if (stats != nullptr && half == 0 && qi < M) {
    stats[(int64_t)b * M + qi] = m_used;
    stats[((int64_t)B + b) * M + qi] = 1.0f / l;
  }
  // every wavefront is past the last barrier: the tiles stage the result rows
  store_f32_rows<NK>(reinterpret_cast<float *>(fa_lds) + wave * (32 * kStage), o, alpha / l, O + osb.at(bp), osr, qw0, M, width, lane);
}

// ---------------------------------------------------------------------------------------------
// backward: D / l of every row, when grad_k is wanted and grad_q is not (else the query kernel writes it)
// ---------------------------------------------------------------------------------------------
template <int NK>
__global__ __launch_bounds__(kThreads) void attention_f32_delta_kernel(const float *__restrict__ O, const float *__restrict__ dO,
                                                                     const float *__restrict__ stats, float *__restrict__ D,
                                                                     int B, int M, int nblk, int n, BatchStep osb, int64_t osr,
                                                                     BatchStep gsb, int64_t gsr) {
  const HeadWidth<true, NK> width{n};
  int b, blk;
  if (!decode_block(nblk, B, &b, &blk)) return;
  const BatchPos bp = batch_pos(b, gsb.heads);
  const int lane = threadIdx.x & 63, half = lane >> 5;
  const int qi = blk * FA_TM + 32 * (threadIdx.x >> 6) + (lane & 31);
  const float *gr = dO + gsb.at(bp) + (int64_t)qi * gsr, *orow = O + osb.at(bp) + (int64_t)qi * osr;
  const float inv_l = qi < M ? stats[((int64_t)B + b) * M + qi] : 0.0f;
  float delta = 0.0f;
#pragma unroll
  for (int ks = 0; ks < NK; ++ks) {
    const Eight g = stationary_piece(width, gr, dO, qi < M, 2 * ks + half), x = stationary_piece(width, orow, O, qi < M, 2 * ks + half);
#pragma unroll
    for (int e = 0; e < 4; ++e) delta += (g.lo[e] * inv_l) * x.lo[e] + (g.hi[e] * inv_l) * x.hi[e];
  }
  delta = both_halves_sum(delta);
  if (qi < M && half == 0) D[(int64_t)b * M + qi] = delta;
}

// ---------------------------------------------------------------------------------------------
// backward: query kernel
// ---------------------------------------------------------------------------------------------
// Above N = 64 the masks of the three rows that are loaded together take more scalar registers than there are: 20 to 91 of them go
// through vector lanes, once per tile before its loop.
template <int NK>
__global__ __launch_bounds__(kThreads, NK <= 4 ? 2 : 1) void attention_f32_query_kernel(
    const float *__restrict__ Q, const float *__restrict__ K, const float *__restrict__ V, const float *__restrict__ O,
    const float *__restrict__ dO, const float *__restrict__ stats, float *__restrict__ dQ, float *__restrict__ D, int B, int M,
    int w, int nblk, int n, float scale, float c, BatchStep qsb, int64_t qsr, BatchStep ksb, int64_t ksr, BatchStep vsb,
    int64_t vsr, BatchStep osb, int64_t osr, BatchStep gsb, int64_t gsr, BatchStep dqsb, int64_t dqsr) {
  typedef PlaneTile<NK> TL;
  typedef typename TL::Tile Tile;
  constexpr int NB = TL::NB, SLOTS = TL::SLOTS, PLANE = TL::PLANE, STAGES = query_stages(NK);
  constexpr bool AHEAD = STAGES == 3;
  extern __shared__ __attribute__((aligned(1024))) uint16_t fa_lds[];  // [stage][K, V][plane]
  auto tile = [&](int buf, int tensor, int p) { return fa_lds + ((buf * 2 + tensor) * 3 + p) * PLANE; };

  const HeadWidth<true, NK> width{n};
  int b, blk;
  if (!decode_block(nblk, B, &b, &blk)) return;
  const BatchPos bp = batch_pos(b, ksb.heads);
  const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i0 = blk * FA_TM;
  const int qw0 = i0 + 32 * wave, qi = qw0 + (lane & 31);
  const bool q_ok = qi < M;
  const float *Kb = K + ksb.at(bp), *Vb = V + vsb.at(bp);

  const int kc_lo = max(i0 - w, 0) / FA_KC;
  const int kc_hi = min(i0 + FA_TM - 1 + w, M - 1) / FA_KC;
  const ChunkPieces<NK> mine(width, tid);
  Eight kreg[SLOTS], vreg[SLOTS];
  auto fetch = [&](int kc) {  // as in the forward
#pragma unroll
    for (int u = 0; u < SLOTS; ++u) {
      const int key = min(kc * FA_KC + mine.row[u], M - 1);
      kreg[u] = load8(Kb + (int64_t)key * ksr + mine.column[u]);
      vreg[u] = load8(Vb + (int64_t)key * vsr + mine.column[u]);
    }
  };
  auto stash = [&](int buf) {
#pragma unroll
    for (int u = 0; u < SLOTS; ++u) {
      split_to_lds(reinterpret_cast<char *>(tile(buf, 0, 0)), 2 * PLANE, mine.at[u], kreg[u]);
      split_to_lds(reinterpret_cast<char *>(tile(buf, 1, 0)), 2 * PLANE, mine.at[u], vreg[u]);
    }
  };
  fetch(kc_lo);
  if (width.pieces() < TL::PPR) {
    for (int e = tid; e < STAGES * TL::STAGE_BYTES / 16; e += kThreads) reinterpret_cast<u32x4 *>(fa_lds)[e] = u32x4{0u, 0u, 0u, 0u};
    __syncthreads();
  }

  // stationary: the query, and its row of dO times 1 / l
  u32x4 qop[NK][3], gop[NK][3];
  const float m = q_ok ? stats[(int64_t)b * M + qi] : 0.0f;
  float delta = 0.0f;
  {
    const float inv_l = q_ok ? stats[((int64_t)B + b) * M + qi] : 0.0f;
    const float *qr = Q + qsb.at(bp) + (int64_t)qi * qsr, *gr = dO + gsb.at(bp) + (int64_t)qi * gsr,
                *orow = O + osb.at(bp) + (int64_t)qi * osr;
    Eight xs[NK], gs[NK], os[NK];
    fetch_pieces(width, gr, dO, q_ok, half, gs);
    fetch_pieces(width, orow, O, q_ok, half, os);
    fetch_pieces(width, qr, Q, q_ok, half, xs);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int ks = 0; ks < NK; ++ks) {
      split8(mask_piece(width, xs[ks], q_ok, 2 * ks + half), qop[ks]);
      Eight g = mask_piece(width, gs[ks], q_ok, 2 * ks + half);
      const Eight x = mask_piece(width, os[ks], q_ok, 2 * ks + half);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        g.lo[e] *= inv_l, g.hi[e] *= inv_l;
        delta += g.lo[e] * x.lo[e] + g.hi[e] * x.hi[e];
      }
      split8(g, gop[ks]);
    }
  }
  delta = both_halves_sum(delta);
  if (q_ok && half == 0) D[(int64_t)b * M + qi] = delta;

  const uint32_t row_at = Tile::row_at(lane), tr_at = Tile::tr_at(lane);
  f32x16 dq[NB];
#pragma unroll
  for (int hb = 0; hb < NB; ++hb)
#pragma unroll
    for (int v = 0; v < 16; ++v) dq[hb][v] = 0.0f;

  auto first_products = [&](int buf, f32x16 &s, f32x16 &dp) {
    f32x16 s1, dp1;
#pragma unroll
    for (int v = 0; v < 16; ++v) s[v] = 0.0f, dp[v] = 0.0f, s1[v] = 0.0f, dp1[v] = 0.0f;
#pragma unroll
    for (int ks = 0; ks < NK; ++ks) {
      u32x4 ka[3], va[3];
#pragma unroll
      for (int p = 0; p < 3; ++p) ka[p] = Tile::rows(tile(buf, 0, p), row_at, 0, ks), va[p] = Tile::rows(tile(buf, 1, p), row_at, 0, ks);
      mma_split_two(ka, qop[ks], s, s1);
      mma_split_two(va, gop[ks], dp, dp1);
    }
#pragma unroll
    for (int v = 0; v < 16; ++v) s[v] += s1[v], dp[v] += dp1[v];
  };
  auto second_products = [&](int buf, const f32x16 &s, const f32x16 &dp) {
    float ds[16];
#pragma unroll
    for (int v = 0; v < 16; ++v) ds[v] = exp2_above(s[v], m, c) * (dp[v] - delta);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      u32x4 df[3];
      split8(Eight{f32x4{ds[8 * t], ds[8 * t + 1], ds[8 * t + 2], ds[8 * t + 3]},
                   f32x4{ds[8 * t + 4], ds[8 * t + 5], ds[8 * t + 6], ds[8 * t + 7]}}, df);
#pragma unroll
      for (int hb = 0; hb < NB; ++hb) {
        u32x4 ka[3];
#pragma unroll
        for (int p = 0; p < 3; ++p) ka[p] = Tile::cols(tile(buf, 0, p), tr_at, 16 * t, hb);
        dq[hb] = mma_split(ka, df, dq[hb]);
      }
    }
  };
  auto in_band = [&](int kc) { return kc <= kc_hi && kc * FA_KC + 31 >= qw0 - w && kc * FA_KC <= qw0 + 31 + w; };
  auto whole = [&](int kc) { return kc * FA_KC >= qw0 + 31 - w && kc * FA_KC + 31 <= qw0 + w && kc * FA_KC + 31 < M; };
  auto after = [](int buf) { return buf + 1 == STAGES ? 0 : buf + 1; };

  f32x16 s, dp;
  stash(0);
  int kc = kc_lo, buf = 0;
  if constexpr (!AHEAD) {
    __syncthreads();
    for (; kc <= kc_hi; ++kc) {
      const int next = after(buf);
      fetch(kc + 1);
      __builtin_amdgcn_sched_barrier(0);
      if (in_band(kc)) {
        first_products(buf, s, dp);
        if (!whole(kc)) mask_band_edge(s, kc * FA_KC, half, qi, w, M);
        second_products(buf, s, dp);
      }
      __builtin_amdgcn_sched_barrier(0);
      stash(next);
      __syncthreads();
      buf = next;
    }
  } else {  // S and dP one chunk ahead of their use, as in the forward
    fetch(kc_lo + 1);
    __syncthreads();
    if (in_band(kc_lo)) {
      first_products(0, s, dp);
      if (!whole(kc_lo)) mask_band_edge(s, kc_lo * FA_KC, half, qi, w, M);
    }
    stash(1);
    __syncthreads();
    const int fast_lo = max(kc_lo, (qw0 - w) >> 5);
    const int fast_hi = min(kc_hi, (qw0 + 31 + w) >> 5) - 1;
    auto general = [&]() {
      const int next = after(buf), free = after(next);
      fetch(kc + 2);
      f32x16 ns, ndp;
      const bool more = in_band(kc + 1);
      if (more) {
        first_products(next, ns, ndp);
        if (!whole(kc + 1)) mask_band_edge(ns, (kc + 1) * FA_KC, half, qi, w, M);
      }
      if (in_band(kc)) second_products(buf, s, dp);
      if (more) s = ns, dp = ndp;
      stash(free);
      __syncthreads();
      ++kc, buf = next;
    };
    const int lead_end = fast_lo <= fast_hi ? fast_lo : kc_hi + 1;
    while (kc < lead_end) general();
    while (kc <= fast_hi) {
      const int next = after(buf), free = after(next);
      fetch(kc + 2);
      f32x16 ns, ns1, ndp, ndp1;
#pragma unroll
      for (int v = 0; v < 16; ++v) ns[v] = 0.0f, ns1[v] = 0.0f, ndp[v] = 0.0f, ndp1[v] = 0.0f;
      u32x4 ra[2][2][3], ca[2][3], df[2][3];
      auto read_rows = [&](auto ks) {
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
          for (int p = 0; p < 3; ++p) ra[ks % 2][x][p] = Tile::rows(tile(next, x, p), row_at, 0, ks);
      };
      auto read_cols = [&](auto y) {  // y = NB t + hb
#pragma unroll
        for (int p = 0; p < 3; ++p) ca[y % 2][p] = Tile::cols(tile(buf, 0, p), tr_at, 16 * (y / NB), y % NB);
      };
      read_rows(std::integral_constant<int, 0>());
      __builtin_amdgcn_sched_barrier(0);
      f32x4 s4;
      Split4Steps sd;
      deal<12 * NK, 20>(
          [&](auto i) {
            constexpr int ks = i / 12, r = i % 12;
            if constexpr (r == 0 && ks + 1 < NK) read_rows(std::integral_constant<int, ks + 1>());
            if constexpr (i == 12 * NK - 12) read_cols(std::integral_constant<int, 0>());
            if constexpr (r % 2 == 0)
              mma_step_two<r / 2>(ra[ks % 2][0], qop[ks], ns, ns1);
            else
              mma_step_two<r / 2>(ra[ks % 2][1], gop[ks], ndp, ndp1);
          },
          [&](auto j) {
            constexpr int g = j / 5, r = j % 5;
            if constexpr (r < 2) {
#pragma unroll
              for (int e = 2 * r; e < 2 * r + 2; ++e)
                s4[e] = exp2_above(s[4 * g + e], m, c) * (dp[4 * g + e] - delta);
            } else {
              sd.run<r - 2>(s4, df[g / 2], g % 2);
            }
          });
      StashSteps st;
      deal<12 * NB, 8 + 14 * SLOTS>(
          [&](auto i) {
            constexpr int y = i / 6;
            if constexpr (i % 6 == 0 && y + 1 < 2 * NB) read_cols(std::integral_constant<int, y + 1>());
            mma_step<i % 6>(ca[y % 2], df[y / NB], dq[y % NB]);
          },
          [&](auto j) {
            if constexpr (j < 8) {
              s[2 * j] = ns[2 * j] + ns1[2 * j], s[2 * j + 1] = ns[2 * j + 1] + ns1[2 * j + 1];
              dp[2 * j] = ndp[2 * j] + ndp1[2 * j], dp[2 * j + 1] = ndp[2 * j + 1] + ndp1[2 * j + 1];
            } else {
              constexpr int u = (j - 8) / 14, tensor = (j - 8) / 7 % 2;
              st.run<(j - 8) % 7>(tensor ? vreg[u] : kreg[u], reinterpret_cast<char *>(tile(free, tensor, 0)), 2 * PLANE, mine.at[u]);
            }
          });
      if (!whole(kc + 1)) mask_band_edge(s, (kc + 1) * FA_KC, half, qi, w, M);
      __syncthreads();
      ++kc, buf = next;
    }
    while (kc <= kc_hi) general();
  }
  store_f32_rows<NK>(reinterpret_cast<float *>(fa_lds) + wave * (32 * kStage), dq, scale, dQ + dqsb.at(bp), dqsr, qw0, M, width, lane);
}

// ---------------------------------------------------------------------------------------------
// backward: key kernel
// ---------------------------------------------------------------------------------------------
// DK, DV: the results that are wanted.  Without dK neither dP nor D is needed, nor the values; without dV P is not split.  A training
// step for grad_v alone / grad_q and grad_k, us at B96 M4096, separate ops, fused with all four products, fused with those needed:
// N = 64 w = 32 345, 446, 252 / 586, 561, 527; N = 80 w = 256 1290, 1505, 1095 / 2192, 2177, 2021; N = 128 w = 128 1114, 1470, 1008 / 1922,
// 2148, 1944, w = 256 1787, 2147, 1513 / 2986, 3150, 2852.
template <int NK, bool DK, bool DV>
__global__ __launch_bounds__(kThreads, NK <= 2 ? 2 : 1) void attention_f32_key_kernel(
    const float *__restrict__ Q, const float *__restrict__ K, const float *__restrict__ V, const float *__restrict__ dO,
    const float *__restrict__ stats, const float *__restrict__ D, float *__restrict__ dK, float *__restrict__ dV, int B, int M,
    int w, int nblk, int n, float scale, float c, BatchStep qsb, int64_t qsr, BatchStep ksb, int64_t ksr, BatchStep vsb,
    int64_t vsr, BatchStep gsb, int64_t gsr, BatchStep dksb, int64_t dksr, BatchStep dvsb, int64_t dvsr) {
  typedef PlaneTile<NK> TL;
  typedef typename TL::Tile Tile;
  constexpr int NB = TL::NB, SLOTS = TL::SLOTS, PLANE = TL::PLANE, STAGES = key_stages(NK);
  extern __shared__ __attribute__((aligned(1024))) uint16_t fa_lds[];  // [stage][Q, dO][plane], then [stage][m, D][row]
  auto tile = [&](int buf, int tensor, int p) { return fa_lds + ((buf * 2 + tensor) * 3 + p) * PLANE; };
  float *const row_lds = reinterpret_cast<float *>(fa_lds + STAGES * TL::STAGE_BYTES / 2);

  const HeadWidth<true, NK> width{n};
  int b, blk;
  if (!decode_block(nblk, B, &b, &blk)) return;
  const BatchPos bp = batch_pos(b, qsb.heads);
  const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c0 = blk * FA_TM;
  const int kw0 = c0 + 32 * wave, kj = kw0 + (lane & 31);
  const bool k_ok = kj < M;
  const float *Qb = Q + qsb.at(bp), *Gb = dO + gsb.at(bp);
  const float *m_rows = stats + (int64_t)b * M, *inv_rows = stats + ((int64_t)B + b) * M, *d_rows = D + (int64_t)b * M;

  const int qc_lo = max(c0 - w, 0) / FA_KC;
  const int qc_hi = min(c0 + FA_TM - 1 + w, M - 1) / FA_KC;
  const ChunkPieces<NK> mine(width, tid);
  Eight qreg[SLOTS], greg[SLOTS];
  float inv_reg[SLOTS], stat_reg;
  auto fetch = [&](int qc) {
#pragma unroll
    for (int u = 0; u < SLOTS; ++u) {
      const int row = min(qc * FA_KC + mine.row[u], M - 1);
      qreg[u] = load8(Qb + (int64_t)row * qsr + mine.column[u]);
      greg[u] = load8(Gb + (int64_t)row * gsr + mine.column[u]);
      inv_reg[u] = inv_rows[row];
    }
    stat_reg = (DK && (tid & 32) ? d_rows : m_rows)[min(qc * FA_KC + (tid & 31), M - 1)];
  };
  auto stash = [&](int buf) {
#pragma unroll
    for (int u = 0; u < SLOTS; ++u) {
      split_to_lds(reinterpret_cast<char *>(tile(buf, 0, 0)), 2 * PLANE, mine.at[u], qreg[u]);
      Eight g = greg[u];
#pragma unroll
      for (int e = 0; e < 4; ++e) g.lo[e] *= inv_reg[u], g.hi[e] *= inv_reg[u];
      split_to_lds(reinterpret_cast<char *>(tile(buf, 1, 0)), 2 * PLANE, mine.at[u], g);
    }
    if (tid < 64) row_lds[64 * buf + tid] = stat_reg;
  };
  fetch(qc_lo);
  if (width.pieces() < TL::PPR) {
    for (int e = tid; e < STAGES * TL::STAGE_BYTES / 16; e += kThreads) reinterpret_cast<u32x4 *>(fa_lds)[e] = u32x4{0u, 0u, 0u, 0u};
    __syncthreads();
  }

  u32x4 kop[NK][3], vop[DK ? NK : 1][3];
  {
    const float *kr = K + ksb.at(bp) + (int64_t)kj * ksr, *vr = V + vsb.at(bp) + (int64_t)kj * vsr;
    Eight x[NK], y[NK];
    fetch_pieces(width, kr, K, k_ok, half, x);
    if constexpr (DK) fetch_pieces(width, vr, V, k_ok, half, y);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int ks = 0; ks < NK; ++ks) {
      split8(mask_piece(width, x[ks], k_ok, 2 * ks + half), kop[ks]);
      if constexpr (DK) split8(mask_piece(width, y[ks], k_ok, 2 * ks + half), vop[ks]);
    }
  }
  const uint32_t row_at = Tile::row_at(lane), tr_at = Tile::tr_at(lane);
  f32x16 dk[NB], dv[NB];
#pragma unroll
  for (int hb = 0; hb < NB; ++hb)
#pragma unroll
    for (int v = 0; v < 16; ++v) dk[hb][v] = 0.0f, dv[hb][v] = 0.0f;

  // S and dP of the chunk at `buf`: lead and rest of each (mma_split_two)
  auto first_products = [&](int buf, f32x16 &s, f32x16 &dp) {
    f32x16 s1, dp1;
#pragma unroll
    for (int v = 0; v < 16; ++v) s[v] = 0.0f, dp[v] = 0.0f, s1[v] = 0.0f, dp1[v] = 0.0f;
#pragma unroll
    for (int ks = 0; ks < NK; ++ks) {
      u32x4 qa[3], ga[3];
#pragma unroll
      for (int p = 0; p < 3; ++p) {
        qa[p] = Tile::rows(tile(buf, 0, p), row_at, 0, ks);
        if constexpr (DK) ga[p] = Tile::rows(tile(buf, 1, p), row_at, 0, ks);
      }
      mma_split_two<true>(qa, kop[ks], s, s1);
      if constexpr (DK) mma_split_two(ga, vop[ks], dp, dp1);
    }
#pragma unroll
    for (int v = 0; v < 16; ++v) s[v] += s1[v], dp[v] += dp1[v];
  };
  // the maxima (which = 0) or D / l (1) of the lane's queries 8 g + 4 half .. + 3 of the chunk
  auto row_stats = [&](int buf, int which, int g) {
    return *reinterpret_cast<const f32x4 *>(row_lds + 64 * buf + 32 * which + 8 * g + 4 * half);
  };
  auto second_products = [&](int buf, const f32x16 &s, const f32x16 &dp) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      Eight pr, ds;
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        const f32x4 m4 = row_stats(buf, 0, 2 * t + g), d4 = DK ? row_stats(buf, 1, 2 * t + g) : m4;
        f32x4 p4, s4;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int v = 8 * t + 4 * g + e;
          p4[e] = exp2_above(s[v], m4[e], c);
          s4[e] = p4[e] * (dp[v] - d4[e]);
        }
        if (g == 0) pr.lo = p4, ds.lo = s4;
        else pr.hi = p4, ds.hi = s4;
      }
      u32x4 pf[3], df[3];
      if constexpr (DV) split8(pr, pf);
      if constexpr (DK) split8(ds, df);
#pragma unroll
      for (int hb = 0; hb < NB; ++hb) {
        u32x4 ga[3], qa[3];
#pragma unroll
        for (int p = 0; p < 3; ++p) {
          if constexpr (DV) ga[p] = Tile::cols(tile(buf, 1, p), tr_at, 16 * t, hb);
          if constexpr (DK) qa[p] = Tile::cols(tile(buf, 0, p), tr_at, 16 * t, hb);
        }
        if constexpr (DV) dv[hb] = mma_split(ga, pf, dv[hb]);
        if constexpr (DK) dk[hb] = mma_split(qa, df, dk[hb]);
      }
    }
  };
  auto in_band = [&](int qc) { return qc <= qc_hi && qc * FA_KC + 31 >= kw0 - w && qc * FA_KC <= kw0 + 31 + w; };
  auto whole = [&](int qc) { return qc * FA_KC >= kw0 + 31 - w && qc * FA_KC + 31 <= kw0 + w && qc * FA_KC + 31 < M; };
  auto after = [](int buf) { return buf + 1 == STAGES ? 0 : buf + 1; };

  f32x16 s, dp;
  stash(0);
  int qc = qc_lo, buf = 0;
  if constexpr (STAGES == 3) {  // as in the forward: S and dP one chunk ahead of their use
    fetch(qc_lo + 1);
    __syncthreads();
    if (in_band(qc_lo)) {
      first_products(0, s, dp);
      if (!whole(qc_lo)) mask_band_edge(s, qc_lo * FA_KC, half, kj, w, M);
    }
    stash(1);
    __syncthreads();
    const int fast_lo = max(qc_lo, (kw0 - w) >> 5);
    const int fast_hi = min(qc_hi, (kw0 + 31 + w) >> 5) - 1;
    auto general = [&]() {
      const int next = after(buf), free = after(next);
      fetch(qc + 2);
      f32x16 ns, ndp;
      const bool more = in_band(qc + 1);
      if (more) {
        first_products(next, ns, ndp);
        if (!whole(qc + 1)) mask_band_edge(ns, (qc + 1) * FA_KC, half, kj, w, M);
      }
      if (in_band(qc)) second_products(buf, s, dp);
      if (more) s = ns, dp = ndp;
      stash(free);
      __syncthreads();
      ++qc, buf = next;
    };
    const int lead_end = fast_lo <= fast_hi ? fast_lo : qc_hi + 1;
    while (qc < lead_end) general();
    while (qc <= fast_hi) {
      const int next = after(buf), free = after(next);
      fetch(qc + 2);
      f32x16 ns, ns1, ndp, ndp1;
#pragma unroll
      for (int v = 0; v < 16; ++v) ns[v] = 0.0f, ns1[v] = 0.0f, ndp[v] = 0.0f, ndp1[v] = 0.0f;
      u32x4 ra[2][2][3], ca[2][2][3], pf[2][3], df[2][3];
      auto read_rows = [&](auto ks) {
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
          for (int p = 0; p < 3; ++p)
            if (x == 0 || DK) ra[ks % 2][x][p] = Tile::rows(tile(next, x, p), row_at, 0, ks);
      };
      auto read_cols = [&](auto y) {  // y = NB t + hb
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
          for (int p = 0; p < 3; ++p)
            if (x == 0 ? DK : DV) ca[y % 2][x][p] = Tile::cols(tile(buf, x, p), tr_at, 16 * (y / NB), y % NB);
      };
      auto row_delta = [&](int g) { return DK ? row_stats(buf, 1, g) : f32x4{0.0f, 0.0f, 0.0f, 0.0f}; };
      f32x4 m4 = row_stats(buf, 0, 0), d4 = row_delta(0), p4, s4;
      read_rows(std::integral_constant<int, 0>());
      __builtin_amdgcn_sched_barrier(0);
      Split4Steps sp, sd;
      constexpr int FIRST = DK ? 2 : 1, SECOND = DK && DV ? 2 : 1;  // products of either kind
      deal<6 * FIRST * NK, 32>(
          [&](auto i) {
            constexpr int ks = i / (6 * FIRST), r = i % (6 * FIRST);
            if constexpr (r == 0 && ks + 1 < NK) read_rows(std::integral_constant<int, ks + 1>());
            if constexpr (r == 0 && ks + 1 == NK) read_cols(std::integral_constant<int, 0>());
            if constexpr (r % FIRST == 0)
              mma_step_two<r / FIRST, true>(ra[ks % 2][0], kop[ks], ns, ns1);
            else
              mma_step_two<r / FIRST>(ra[ks % 2][1], vop[ks], ndp, ndp1);
          },
          [&](auto j) {
            constexpr int g = j / 8, r = j % 8;
            if constexpr (r < 2) {
#pragma unroll
              for (int e = 2 * r; e < 2 * r + 2; ++e) {
                p4[e] = exp2_above(s[4 * g + e], m4[e], c);
                s4[e] = p4[e] * (dp[4 * g + e] - d4[e]);
              }
              if constexpr (r == 1 && g < 3) m4 = row_stats(buf, 0, g + 1), d4 = row_delta(g + 1);
            } else if constexpr (r < 5) {
              if constexpr (DV) sp.run<r - 2>(p4, pf[g / 2], g % 2);
            } else if constexpr (DK) {
              sd.run<r - 5>(s4, df[g / 2], g % 2);
            }
          });
      StashSteps st;
      deal<12 * SECOND * NB, 8 + 15 * SLOTS>(
          [&](auto i) {
            constexpr int y = i / (6 * SECOND), r = i % (6 * SECOND);
            if constexpr (r == 0 && y + 1 < 2 * NB) read_cols(std::integral_constant<int, y + 1>());
            if constexpr (DV && r % SECOND == 0)
              mma_step<r / SECOND>(ca[y % 2][1], pf[y / NB], dv[y % NB]);
            else
              mma_step<r / SECOND>(ca[y % 2][0], df[y / NB], dk[y % NB]);
          },
          [&](auto j) {
            if constexpr (j < 8) {
              s[2 * j] = ns[2 * j] + ns1[2 * j], s[2 * j + 1] = ns[2 * j + 1] + ns1[2 * j + 1];
              dp[2 * j] = ndp[2 * j] + ndp1[2 * j], dp[2 * j + 1] = ndp[2 * j + 1] + ndp1[2 * j + 1];
            } else {
              constexpr int u = (j - 8) / 15, r = (j - 8) % 15;
              if constexpr (r < 7) {
                st.run<r>(qreg[u], reinterpret_cast<char *>(tile(free, 0, 0)), 2 * PLANE, mine.at[u]);
              } else if constexpr (r == 7) {
#pragma unroll
                for (int e = 0; e < 4; ++e) greg[u].lo[e] *= inv_reg[u], greg[u].hi[e] *= inv_reg[u];
              } else {
                st.run<r - 8>(greg[u], reinterpret_cast<char *>(tile(free, 1, 0)), 2 * PLANE, mine.at[u]);
              }
            }
          });
      if (tid < 64) row_lds[64 * free + tid] = stat_reg;
      if (!whole(qc + 1)) mask_band_edge(s, (qc + 1) * FA_KC, half, kj, w, M);
      __syncthreads();
      ++qc, buf = next;
    }
    while (qc <= qc_hi) general();
  } else {
    __syncthreads();
    for (; qc <= qc_hi; ++qc) {
      const int next = after(buf);
      fetch(qc + 1);
      __builtin_amdgcn_sched_barrier(0);
      if (in_band(qc)) {
        first_products(buf, s, dp);
        if (!whole(qc)) mask_band_edge(s, qc * FA_KC, half, kj, w, M);
        second_products(buf, s, dp);
      }
      __builtin_amdgcn_sched_barrier(0);
      stash(next);
      __syncthreads();
      buf = next;
    }
  }
  float *stage = reinterpret_cast<float *>(fa_lds) + wave * (32 * kStage);
  if constexpr (DK) store_f32_rows<NK>(stage, dk, scale, dK + dksb.at(bp), dksr, kw0, M, width, lane);
  if constexpr (DV) store_f32_rows<NK>(stage, dv, 1.0f, dV + dvsb.at(bp), dvsr, kw0, M, width, lane);
}

// ---------------------------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------------------------
// More LDS than a kernel gets without asking: the call changes an attribute of the function, it allocates nothing.
hipError_t allow_lds(const void *kernel, int bytes) {
  return bytes <= 65536 ? hipSuccess : hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
}

constexpr double kLog2eD = 1.4426950408889634;

template <int NK>
hipError_t launch_key(const Problem &p, const View &q, const View &k, const View &v, const View &go, const float *stats, const float *delta,
                      const View &gk, const View &gv, double scale) {
  const int nblk = (int)((p.M + FA_TM - 1) / FA_TM);
  constexpr int BYTES = key_stages(NK) * (PlaneTile<NK>::STAGE_BYTES + 2 * FA_KC * 4);
  const auto kernel = gv.data == nullptr   ? attention_f32_key_kernel<NK, true, false>
                      : gk.data == nullptr ? attention_f32_key_kernel<NK, false, true>
                                           : attention_f32_key_kernel<NK, true, true>;
  if (const hipError_t err = allow_lds(reinterpret_cast<const void *>(kernel), BYTES); err != hipSuccess) return err;
  hipLaunchKernelGGL(kernel, dim3((unsigned)tiled_grid(p.B, nblk)), dim3(kThreads), BYTES, p.stream, (const float *)q.data,
                     (const float *)k.data, (const float *)v.data, (const float *)go.data, stats, delta, (float *)gk.data,
                     (float *)gv.data, (int)p.B, (int)p.M, (int)p.w, nblk, (int)p.N, (float)scale, (float)(scale * kLog2eD), q.sb, q.sr,
                     k.sb, k.sr, v.sb, v.sr, go.sb, go.sr, gk.sb, gk.sr, gv.sb, gv.sr);
  return hipGetLastError();
}

#if !F32_KEY_WIDE
template <int NK>
hipError_t launch_forward(const Problem &p, const View &q, const View &k, const View &v, const View &o, float *stats, double scale,
                          int mask) {
  const int nblk = (int)((p.M + FA_TM - 1) / FA_TM);
  constexpr int BYTES = forward_stages(NK) * PlaneTile<NK>::STAGE_BYTES;
  const auto kernel = mask ? attention_f32_forward_kernel<NK, true> : attention_f32_forward_kernel<NK, false>;
  if (const hipError_t err = allow_lds(reinterpret_cast<const void *>(kernel), BYTES); err != hipSuccess) return err;
  hipLaunchKernelGGL(kernel, dim3((unsigned)tiled_grid(p.B, nblk)), dim3(kThreads), BYTES, p.stream,
                     (const float *)q.data, (const float *)k.data, (const float *)v.data, (float *)o.data, stats, (int)p.B, (int)p.M,
                     (int)p.w, nblk, (int)p.N, (float)(scale * kLog2eD), q.sb, q.sr, k.sb, k.sr, v.sb, v.sr, o.sb, o.sr);
  return hipGetLastError();
}

template <int NK>
hipError_t launch_backward(const Problem &p, const View &q, const View &k, const View &v, const View &o, const View &go,
                           const float *stats, float *delta, const View &gq, const View &gk, const View &gv, double scale) {
  const int nblk = (int)((p.M + FA_TM - 1) / FA_TM);
  const dim3 grid((unsigned)tiled_grid(p.B, nblk)), block(kThreads);
  const float c = (float)(scale * kLog2eD);
  constexpr int BYTES = query_stages(NK) * PlaneTile<NK>::STAGE_BYTES;
  if (gq.data != nullptr) {
    const auto kernel = attention_f32_query_kernel<NK>;
    if (const hipError_t err = allow_lds(reinterpret_cast<const void *>(kernel), BYTES); err != hipSuccess) return err;
    hipLaunchKernelGGL(kernel, grid, block, BYTES, p.stream, (const float *)q.data, (const float *)k.data, (const float *)v.data,
                       (const float *)o.data, (const float *)go.data, stats, (float *)gq.data, delta, (int)p.B, (int)p.M, (int)p.w,
                       nblk, (int)p.N, (float)scale, c, q.sb, q.sr, k.sb, k.sr, v.sb, v.sr, o.sb, o.sr, go.sb, go.sr, gq.sb, gq.sr);
  } else if (gk.data != nullptr) {
    hipLaunchKernelGGL(attention_f32_delta_kernel<NK>, grid, block, 0, p.stream, (const float *)o.data, (const float *)go.data, stats,
                       delta, (int)p.B, (int)p.M, nblk, (int)p.N, o.sb, o.sr, go.sb, go.sr);
  }
  const hipError_t err = hipGetLastError();
  if (err != hipSuccess || (gk.data == nullptr && gv.data == nullptr)) return err;
  if constexpr (NK >= 7) return launch_attention_f32_key_wide(p, q, k, v, go, stats, delta, gk, gv, scale);
  else return launch_key<NK>(p, q, k, v, go, stats, delta, gk, gv, scale);
}

bool rows_ok(std::initializer_list<const View *> views) {
  for (const View *t : views)
    if (t->data != nullptr && (t->sc != 1 || (uintptr_t)t->data % 4 != 0)) return false;  // absent outputs have no layout
  return true;
}

#endif

}  // namespace

#if F32_KEY_WIDE
hipError_t launch_attention_f32_key_wide(const Problem &p, const View &q, const View &k, const View &v, const View &go, const float *stats,
                                         const float *delta, const View &gk, const View &gv, double scale) {
  return p.N > 112 ? launch_key<8>(p, q, k, v, go, stats, delta, gk, gv, scale) : launch_key<7>(p, q, k, v, go, stats, delta, gk, gv, scale);
}
#else
bool attention_f32_supports(const Problem &p, double scale) {
  if (p.dtype != WM_DTYPE_F32 || (p.flags & (WM_FLAG_FORCE_STRIDED | WM_FLAG_NO_SPLIT_F32))) return false;
  if (p.N < 8 || p.N > 128 || p.M < 1 || p.w < 1 || p.w > 0x3fffffff) return false;
  if (p.M > 0x7fffffff - p.w - 2 * FA_TM) return false;  // row and key indices are 32-bit in the kernels
  if (tiled_grid(p.B, (p.M + FA_TM - 1) / FA_TM) > 0x7fffffff) return false;
  return scale > 1.2e-38 && scale < 1.0e30;  // as a float32 a normal number, times log2(e) as well
}

bool try_launch_attention_f32_forward(const Problem &p, const View &q, const View &k, const View &v, const View &o, float *stats,
                                      double scale, int mask, hipError_t *err) {
  if (!attention_f32_supports(p, scale) || !rows_ok({&q, &k, &v, &o})) return false;
  switch ((p.N + 15) / 16) {
#define WM_CASE(NK) case NK: *err = launch_forward<NK>(p, q, k, v, o, stats, scale, mask); break;
    WM_CASE(1) WM_CASE(2) WM_CASE(3) WM_CASE(4) WM_CASE(5) WM_CASE(6) WM_CASE(7) WM_CASE(8)
#undef WM_CASE
  }
  return true;
}

bool try_launch_attention_f32_backward(const Problem &p, const View &q, const View &k, const View &v, const View &o, const View &go,
                                       const float *stats, float *delta, const View &gq, const View &gk, const View &gv, double scale,
                                       hipError_t *err) {
  if (!attention_f32_supports(p, scale) || !rows_ok({&q, &k, &v, &o, &go, &gq, &gk, &gv})) return false;
  switch ((p.N + 15) / 16) {
#define WM_CASE(NK) case NK: *err = launch_backward<NK>(p, q, k, v, o, go, stats, delta, gq, gk, gv, scale); break;
    WM_CASE(1) WM_CASE(2) WM_CASE(3) WM_CASE(4) WM_CASE(5) WM_CASE(6) WM_CASE(7) WM_CASE(8)
#undef WM_CASE
  }
  return true;
}

#endif

}  // namespace wm
