// Frame-window attention of the action branches' cached attention
// (multics/models/blocks.py:256-375: mouse temporal self-attention and
// keyboard cross-attention over a rolling cache).  Key j is visible to query i
// when k_frame[j] / n_block <= q_frame[i] / n_block and, with a window,
// q_frame[i] - k_frame[j] < local_attn.  Scores, softmax weights and sums are
// fp32 (the weights multiply V as three bf16 parts where the matrix cores do it).
//
// Three kernels, by the queries and keys of a sequence and by how many
// sequences and heads there are:
//
// seq_kernel    few queries (the temporal branch: one sequence per spatial
//               token, a block's 3 frames against a window of 24).  Bound by
//               reading K and V once.  One wave owns a (sequence, head) and up
//               to 8 of its queries: it loads the window's rows at once (D / 8
//               lanes per row, up to 8 groups of rows: 8 KB each of K and V),
//               scores them for every query from registers and adds the row
//               groups' sums at the end.  2,200 sequences x 24 heads of 128,
//               3 x 24 keys: 115 us, 6.1 TB/s (155 us, 4.5 TB/s, when each
//               query read the rows for itself, four keys at a time).
// slot_kernel   a short window (a rollout's first blocks, small windows).  8 or
//               4 queries per wave, each by D / 8 lanes, key after key.
//               1,970 x 12 heads of 64, 3 x 8 keys: 17.5 us (23.2 as
//               seq_kernel, whose fixed work is the larger part there).
// tile_kernel   more (the keyboard branch: 660 video tokens against 96 keyboard
//               tokens per player): 128 queries per workgroup on the matrix
//               cores, 64-key tiles of K and V in LDS, the next tile's rows
//               loaded during the current one.  Bound by the latency of its
//               few steps.  10 x 24 heads, 660 x 96 keys: 40 us (329 us with
//               one key at a time per query).
//
// seq_kernel and tile_kernel give every key a weight, 0 where the mask hides it, and 0 times an
// infinity or a NaN is a NaN.  A hidden row counts for nothing whatever it
// holds, so where results are not all finite, or a query's weights sum to 0,
// a wave computes its queries again from their visible keys alone, a key at a
// time (visible_only).  The check costs the keyboard branch 2 us of 40, waves
// of 7 or 8 queries 1-3 %, the temporal branch nothing.
#include "hier_common.h"
#include "hier_launch.h"
#include "hier_tile.h"
#include "hier_window.h"

namespace {

using namespace hier::tile;
using hier::Window;

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kNoMax = -1e30f;       // running max of a row without a visible key

__device__ __forceinline__ float lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }

template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true));
}
__device__ __forceinline__ float fold32(float a, float b) {   // lanes 0-31: a over both halves; 32-63: b
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float fold16(float a, float b) {   // rows 0, 2: a's pairs of rows; 1, 3: b's
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float max16(float v) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// Sum of packed results: infinite or NaN if one of them is.
__device__ __forceinline__ float probe(uint32_t w, float sum) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, w),
                                         __builtin_bit_cast(bf16x2, 0x3f803f80u), sum, false);
}
// A weight sum of 0, or it or a sum of results infinite or NaN.  (By their bits and out
// of the compiler's sight: this is built to assume that no NaN occurs.)
__device__ __forceinline__ bool is_odd(float l, float sum) {
  uint32_t w = __float_as_uint(l), x = __float_as_uint(sum);
  asm("" : "+v"(w), "+v"(x));
  return w - 1u >= 0x7f7fffffu || (x & 0x7f800000u) == 0x7f800000u;
}

// Queries [q0, q0 + nq) of a (sequence, head) by one wave, from the keys that
// each sees and no others: D / 8 lanes per query, a key at a time, the running
// maximum from -infinity.
template <int D>
__device__ __forceinline__ void visible_only(const HierFrameAttnArgs& a, int64_t b, int64_t h,
                                             int q0, int nq) {
  // (a score is rounded before the maximum is taken off: fused, what that
  // leaves of -1e31 is not 0)
#pragma clang fp contract(off)
  constexpr int LPR = D / 8, R = 64 / LPR;
  const int lane = threadIdx.x & 63, c = lane % LPR, r = lane / LPR;
  const uint16_t* const kb = a.k + b * a.k_sb + h * a.k_sh + 8 * c;
  const uint16_t* const vb = a.v + b * a.v_sb + h * a.v_sh + 8 * c;
  const float c2 = a.scale * kLog2e;
#pragma unroll 1
  for (int i = r; i - r < nq; i += R) {
    const bool mine = i < nq && q0 + i < a.Lq;
    const int qi = min(q0 + i, a.Lq - 1);
    const u32x4 q = *reinterpret_cast<const u32x4*>(a.q + b * a.q_sb + (int64_t)qi * a.q_ss +
                                                    h * a.q_sh + 8 * c);
    Window win;
    win.init(a.q_frame[qi], a.n_block, a.local_attn);
    float m = -INFINITY, l = 0.f, o[8] = {};
#pragma unroll 1
    for (int j = 0; j < a.Lk; ++j) {
      const u32x4 k = *reinterpret_cast<const u32x4*>(kb + (int64_t)j * a.k_ss);
      const u32x4 v = *reinterpret_cast<const u32x4*>(vb + (int64_t)j * a.v_ss);
      float s = 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t x = q[e], y = k[e];
        s = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, x),
                                            __builtin_bit_cast(bf16x2, y), s, false);
      }
#pragma unroll
      for (int d = 1; d < LPR; d <<= 1) s += __shfl_xor(s, d, 64);
      if (!win.sees(a.k_frame[j])) continue;
      const float t = s * c2, mn = fmaxf(m, t);
      const float alpha = __builtin_amdgcn_exp2f(m - mn);   // m = -inf: 0
      const float p = __builtin_amdgcn_exp2f(t - mn);
      l = fmaf(l, alpha, p);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        o[2 * e] = fmaf(p, lo(v[e]), o[2 * e] * alpha);
        o[2 * e + 1] = fmaf(p, hi(v[e]), o[2 * e + 1] * alpha);
      }
      m = mn;
    }
    const float inv = l > 0.f ? 1.f / l : 0.f;
    u32x4 w;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      w[e] = (uint32_t)f2bf(o[2 * e] * inv) | ((uint32_t)f2bf(o[2 * e + 1] * inv) << 16);
    if (mine)
      *reinterpret_cast<u32x4*>(a.o + b * a.o_sb + (int64_t)qi * a.o_ss + h * a.o_sh + 8 * c) = w;
  }
}

// ---- short windows -----------------------------------------------------------

// A wave serves 64 / (D / 8) (sequence, query) slots of one head: D / 8 lanes
// per query, each query over its own sequence's keys (slots of one sequence
// read the same rows), four of them loaded before any is used.  Bound by its
// instructions per query and key, and by one trip's latency per four keys; it
// holds no rows and sums nothing across them, which on a short window is most of a seq_kernel wave's work.
template <int D>
__global__ __launch_bounds__(64) void slot_kernel(HierFrameAttnArgs a) {
#pragma clang fp contract(off)   // (as in visible_only)
  constexpr int LPR = D / 8, R = 64 / LPR, G = 4;
  const int lane = threadIdx.x, c = lane % LPR, h = blockIdx.y;
  const uint32_t slot = blockIdx.x * R + lane / LPR;      // (fewer than 2^28)
  const bool mine = slot < (uint32_t)a.B * (uint32_t)a.Lq;
  const uint32_t seq = mine ? slot / (uint32_t)a.Lq : 0u;
  const int qi = mine ? (int)(slot - seq * (uint32_t)a.Lq) : 0;
  const int64_t b = seq;
  const u32x4 q = *reinterpret_cast<const u32x4*>(a.q + b * a.q_sb + (int64_t)qi * a.q_ss +
                                                  (int64_t)h * a.q_sh + 8 * c);
  Window win;
  win.init(a.q_frame[qi], a.n_block, a.local_attn);
  const uint16_t* const kb = a.k + b * a.k_sb + (int64_t)h * a.k_sh + 8 * c;
  const uint16_t* const vb = a.v + b * a.v_sb + (int64_t)h * a.v_sh + 8 * c;
  const float c2 = a.scale * kLog2e;
  float m = -INFINITY, l = 0.f, o[8] = {};
  for (int j0 = 0; j0 < a.Lk; j0 += G) {
    u32x4 k[G], v[G];
    int kf[G];
#pragma unroll
    for (int u = 0; u < G; ++u) {
      const int j = min(j0 + u, a.Lk - 1);
      k[u] = *reinterpret_cast<const u32x4*>(kb + (int64_t)j * a.k_ss);
      v[u] = *reinterpret_cast<const u32x4*>(vb + (int64_t)j * a.v_ss);
      kf[u] = a.k_frame[j];
    }
#pragma unroll
    for (int u = 0; u < G; ++u) {
      if (j0 + u >= a.Lk) break;
      float s = 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t x = q[e], y = k[u][e];
        s = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, x),
                                            __builtin_bit_cast(bf16x2, y), s, false);
      }
#pragma unroll
      for (int d = 1; d < LPR; d <<= 1) s += __shfl_xor(s, d, 64);
      if (!win.sees(kf[u])) continue;
      const float t = s * c2, mn = fmaxf(m, t);
      const float alpha = __builtin_amdgcn_exp2f(m - mn);   // m = -inf: 0
      const float p = __builtin_amdgcn_exp2f(t - mn);
      l = fmaf(l, alpha, p);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        o[2 * e] = fmaf(p, lo(v[u][e]), o[2 * e] * alpha);
        o[2 * e + 1] = fmaf(p, hi(v[u][e]), o[2 * e + 1] * alpha);
      }
      m = mn;
    }
  }
  if (!mine) return;
  const float inv = l > 0.f ? 1.f / l : 0.f;
  u32x4 w;
#pragma unroll
  for (int e = 0; e < 4; ++e)
    w[e] = (uint32_t)f2bf(o[2 * e] * inv) | ((uint32_t)f2bf(o[2 * e + 1] * inv) << 16);
  *reinterpret_cast<u32x4*>(a.o + b * a.o_sb + (int64_t)qi * a.o_ss + (int64_t)h * a.o_sh + 8 * c) = w;
}

// ---- up to 8 queries per sequence ------------------------------------------

// One wave: NQ queries of a (sequence, head), the keys in one chunk of G row
// groups or (LOOP) in several.  A sequence's ceil(Lq / NQ) waves sit side by side (in one
// workgroup as a rule).  ONCE: that is one wave, and a row is read by it alone.
template <int D, int NQ, int G, bool LOOP, bool ONCE>
__global__ __launch_bounds__(256, LOOP || NQ > 4 ? 2 : 3) void seq_kernel(HierFrameAttnArgs a,
                                                                     uint32_t nqg, uint32_t units) {
  constexpr int LPR = D / 8;          // lanes per row
  constexpr int R = 64 / LPR;         // rows per group
  const int lane = threadIdx.x & 63;
  const uint32_t unit = (blockIdx.y * gridDim.x + blockIdx.x) * 4 + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  if (unit >= units) return;
  const uint32_t bh = unit / nqg, b = bh / (uint32_t)a.H;
  const int h = (int)(bh - b * (uint32_t)a.H), q0 = (int)(unit - bh * nqg) * NQ;
  const int c = lane % LPR, r = lane / LPR;
  // rows stepped by a uniform stride; a lane past the last key repeats it, unseen
  const uint16_t* const kb = a.k + (int64_t)b * a.k_sb + (int64_t)h * a.k_sh + 8 * c;
  const uint16_t* const vb = a.v + (int64_t)b * a.v_sb + (int64_t)h * a.v_sh + 8 * c;
  const uint16_t* const kl = kb + (int64_t)(a.Lk - 1) * a.k_ss;
  const uint16_t* const vl = vb + (int64_t)(a.Lk - 1) * a.v_ss;
  const uint16_t* const kr = kb + (int64_t)r * a.k_ss;
  const uint16_t* const vr = vb + (int64_t)r * a.v_ss;
  u32x4 k[G], v[G];
  int kf[G];
  // a row read once: past the caches.  24 keys x 24 heads of 128, 3 queries,
  // plain / past them: 2,200 sequences 133 / 116 us, 400 27 / 25, 40 6.0 / 6.0.
  // Two waves read the same rows: 2,200 sequences, 16 queries 309 / 321 us, 12
  // queries 250 / 254, 40 sequences 9.5 / 10.4.  In a loop the rows' neighbours
  // follow (1,000 keys: 34 / 47).
  auto load = [&](const uint16_t* p) {
    const u32x4* w = reinterpret_cast<const u32x4*>(p);
    if constexpr (LOOP || !ONCE) return *w;
    else return __builtin_nontemporal_load(w);
  };
  auto fetch = [&](int j0) {          // a chunk's rows, all before any is used
#pragma unroll
    for (int g = 0; g < G; ++g)
      k[g] = load(j0 + g * R + r < a.Lk ? kr + (int64_t)(j0 + g * R) * a.k_ss : kl);
#pragma unroll
    for (int g = 0; g < G; ++g) kf[g] = a.k_frame[min(j0 + g * R + r, a.Lk - 1)];
#pragma unroll
    for (int g = 0; g < G; ++g)
      v[g] = load(j0 + g * R + r < a.Lk ? vr + (int64_t)(j0 + g * R) * a.v_ss : vl);
  };
  u32x4 q[NQ];
#pragma unroll
  for (int i = 0; i < NQ; ++i)
    q[i] = *reinterpret_cast<const u32x4*>(a.q + (int64_t)b * a.q_sb +
                                           (int64_t)min(q0 + i, a.Lq - 1) * a.q_ss +
                                           (int64_t)h * a.q_sh + 8 * c);
  const int qf = a.q_frame[min(q0 + min(lane, NQ - 1), a.Lq - 1)];   // lane i: query i
  // a window of one chunk: its rows in flight before the first wait (as a
  // loop's carried state they would cost as many registers again; the barrier
  // keeps the compiler from moving V's loads to where they are used)
  if (!LOOP && a.Lk > 0) fetch(0);
  __builtin_amdgcn_sched_barrier(0);
  Window win[NQ];
  {
    Window w;
    w.init(qf, a.n_block, a.local_attn);
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      win[i].first = __builtin_amdgcn_readlane(w.first, i);
      win[i].span = (uint32_t)__builtin_amdgcn_readlane((int)w.span, i);
    }
  }
  const float c2 = a.scale * kLog2e;
  float m[NQ], l[NQ], o[NQ][8];
#pragma unroll
  for (int i = 0; i < NQ; ++i) {
    m[i] = kNoMax;
    l[i] = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[i][e] = 0.f;
  }
  auto chunk = [&](int j0) {
#pragma unroll
    for (int g = 0; g < G; ++g) kf[g] = j0 + g * R + r < a.Lk ? kf[g] : INT_MAX;
    float s[G][NQ], mx[NQ];
#pragma unroll
    for (int i = 0; i < NQ; ++i) mx[i] = -INFINITY;
#pragma unroll
    for (int g = 0; g < G; ++g) {
#pragma unroll
      for (int i = 0; i < NQ; ++i) {
        float t = 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint32_t x = q[i][e], y = k[g][e];
          t = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, x),
                                              __builtin_bit_cast(bf16x2, y), t, false);
        }
        t += dpp<0xB1>(t);                      // the row's lanes: quad_perm [1,0,3,2]
        t += dpp<0x4E>(t);                      // quad_perm [2,3,0,1]
        if constexpr (LPR == 16) {
          t += dpp<0x124>(t);                   // row_ror:4
          t += dpp<0x128>(t);                   // row_ror:8
        } else {
          t += dpp<0x141>(t);                   // row_half_mirror
        }
        s[g][i] = win[i].sees(kf[g]) ? t * c2 : -INFINITY;
        mx[i] = fmaxf(mx[i], s[g][i]);
      }
    }
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      if constexpr (LPR == 8) mx[i] = fmaxf(mx[i], dpp<0x128>(mx[i]));
      const float mn = fmaxf(m[i], pair_max(max16(mx[i])));
      if constexpr (LOOP) {               // (one chunk: nothing summed yet)
        const float alpha = __builtin_amdgcn_exp2f(m[i] - mn);
        l[i] *= alpha;
#pragma unroll
        for (int e = 0; e < 8; ++e) o[i][e] *= alpha;
      }
      m[i] = mn;
    }
#pragma unroll
    for (int g = 0; g < G; ++g) {
      float x[8];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t w = v[g][e];
        x[2 * e] = lo(w);
        x[2 * e + 1] = hi(w);
      }
#pragma unroll
      for (int i = 0; i < NQ; ++i) {
        const float p = __builtin_amdgcn_exp2f(s[g][i] - m[i]);
        l[i] += p;
#pragma unroll
        for (int e = 0; e < 8; ++e) o[i][e] = fmaf(p, x[e], o[i][e]);
      }
    }
  };
  if constexpr (LOOP) {
    for (int j0 = 0; j0 < a.Lk; j0 += G * R) {
      fetch(j0);
      chunk(j0);
    }
  } else if (a.Lk > 0) {
    chunk(0);
  }
  // Sums over the row groups, four queries at a time: lane row 0 / 1 / 2 / 3
  // (16 lanes) ends up with query 0 / 2 / 1 / 3 of the four, and stores it.
  const int rw = lane >> 4, qr = (rw & 1) << 1 | rw >> 1;
  bool odd[(NQ + 3) / 4];
#pragma unroll
  for (int i0 = 0; i0 < NQ; i0 += 4) {
    auto fold = [&](auto get) {
      float x[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        x[i] = i0 + i < NQ ? get(min(i0 + i, NQ - 1)) : 0.f;
        if constexpr (LPR == 8) x[i] += dpp<0x128>(x[i]);
      }
      return fold16(fold32(x[0], x[1]), fold32(x[2], x[3]));
    };
    const float lt = fold([&](int i) { return l[i]; });
    const float inv = lt > 0.f ? 1.f / lt : 0.f;
    u32x4 w;
    float sum = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float x = fold([&](int i) { return o[i][2 * e]; }) * inv;
      const float y = fold([&](int i) { return o[i][2 * e + 1]; }) * inv;
      w[e] = (uint32_t)f2bf(x) | ((uint32_t)f2bf(y) << 16);
      sum = probe(w[e], sum);
    }
    const bool mine = i0 + qr < NQ && q0 + i0 + qr < a.Lq;
    odd[i0 / 4] = __ballot(mine && is_odd(lt, sum)) != 0;
    if (!odd[i0 / 4] && mine && (LPR == 16 || (lane & 8) == 0))
      *reinterpret_cast<u32x4*>(a.o + (int64_t)b * a.o_sb + (int64_t)(q0 + i0 + qr) * a.o_ss +
                                (int64_t)h * a.o_sh + 8 * c) = w;
  }
  if (odd[0]) visible_only<D>(a, b, h, q0, min(NQ, 4));
  if constexpr (NQ > 4)
    if (odd[1]) visible_only<D>(a, b, h, q0 + 4, NQ - 4);
}

// ---- more queries: matrix-core tiles ----------------------------------------
//
// Four waves of 32 queries.  S^T = K Q^T leaves each lane one query and 16 keys
// of a 32-key block (hier_tile.h); P goes from the accumulators into the
// operand of O^T += V^T P^T as the bf16 of P, the bf16 of what that rounding
// left and the bf16 of what is left then: all 24 bits of P (the products with
// bf16 V are exact, the sums fp32).  The rows reach LDS through registers: any
// row stride works.

template <int D>
__global__ __launch_bounds__(256, 2) void tile_kernel(HierFrameAttnArgs a, int q_tiles, int total) {
  constexpr int NC = Geo<D>::NC, NDB = Geo<D>::NDB, CPR = Geo<D>::CPR, ROWB = Geo<D>::ROWB;
  constexpr int NL = kSlab * CPR / 256;     // 16-byte chunks per thread and tile
  __shared__ __align__(16) char lds_k[Geo<D>::TILEB], lds_v[Geo<D>::TILEB];
  __shared__ __align__(16) int lds_f[kSlab];
  // the query tiles of one sequence and head on one XCD, which then reads
  // their keys from memory once
  const int logical = hier::xcd_logical((int)(blockIdx.y * gridDim.x + blockIdx.x),
                                        (int)(gridDim.x * gridDim.y));
  if (logical >= total) return;
  const int bh = logical / q_tiles, b = bh / a.H, h = bh - b * a.H;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int q0 = (logical - bh * q_tiles) * 128 + wave * 32;
  const bool active = q0 < a.Lq;
  const int qi = min(q0 + (lane & 31), a.Lq - 1);
  const uint16_t* const kb = a.k + (int64_t)b * a.k_sb + (int64_t)h * a.k_sh;
  const uint16_t* const vb = a.v + (int64_t)b * a.v_sb + (int64_t)h * a.v_sh;
  u32x4 kr[NL], vr[NL];
  int fr = INT_MAX;
  auto fetch = [&](int j0) {                // rows past the last repeat it, unseen
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int x = tid + 256 * i, row = min(j0 + x / CPR, a.Lk - 1), ch = x % CPR;
      kr[i] = *reinterpret_cast<const u32x4*>(kb + (int64_t)row * a.k_ss + 8 * ch);
      vr[i] = *reinterpret_cast<const u32x4*>(vb + (int64_t)row * a.v_ss + 8 * ch);
    }
    if (tid < kSlab) {
      const int f = a.k_frame[min(j0 + tid, a.Lk - 1)];
      fr = j0 + tid < a.Lk ? f : INT_MAX;
    }
  };
  if (a.Lk > 0) fetch(0);
  bf16x8 q[NC];
  Window win;
  {
    const uint16_t* p = a.q + (int64_t)b * a.q_sb + (int64_t)qi * a.q_ss + (int64_t)h * a.q_sh +
                        8 * (lane >> 5);
#pragma unroll
    for (int i = 0; i < NC; ++i) q[i] = *reinterpret_cast<const bf16x8*>(p + 16 * i);
    win.init(a.q_frame[qi], a.n_block, a.local_attn);
  }
  const float c2 = a.scale * kLog2e;
  int ka[NC], va[NDB];
#pragma unroll
  for (int i = 0; i < NC; ++i) ka[i] = row_read_off<D, kRowRead>(lane, i);
#pragma unroll
  for (int i = 0; i < NDB; ++i) va[i] = tr_read_off<D, kTrRead>(lane, i, 0);
  constexpr int HALF = (8 / Geo<D>::NI) * ROWB;   // rows of keys +8
  f32x16 o[NDB];
#pragma unroll
  for (int i = 0; i < NDB; ++i) o[i] = f32x16{};
  float m = kNoMax, l = 0.f;
  for (int j0 = 0; j0 < a.Lk; j0 += kSlab) {
    __syncthreads();                        // every wave is done with the tile in LDS
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int x = tid + 256 * i, row = x / CPR, ch = x % CPR;
      *reinterpret_cast<u32x4*>(lds_k + prow<D>(row) * ROWB + 16 * (ch ^ swz<D, kRowRead>(row))) = kr[i];
      *reinterpret_cast<u32x4*>(lds_v + prow<D>(row) * ROWB + 16 * (ch ^ swz<D, kTrRead>(row))) = vr[i];
    }
    if (tid < kSlab) lds_f[tid] = fr;
    __syncthreads();
    if (j0 + kSlab < a.Lk) fetch(j0 + kSlab);
    if (!active) continue;
    // one 32-key block at a time (the last tile may hold one)
#pragma unroll 1
    for (int kb32 = 0; kb32 < 2 && j0 + 32 * kb32 < a.Lk; ++kb32) {
      const char* kt = lds_k + kb32 * 32 * ROWB;
      const char* vt0 = lds_v + kb32 * 32 * ROWB;
      f32x16 s = {};
#pragma unroll
      for (int i = 0; i < NC; ++i) s = mfma(*reinterpret_cast<const bf16x8*>(kt + ka[i]), q[i], s);
      float mx = -INFINITY;
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4) {
        const u32x4 f = *reinterpret_cast<const u32x4*>(&lds_f[kb32 * 32 + 8 * g4 + 4 * (lane >> 5)]);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float x = win.sees((int)f[e]) ? s[4 * g4 + e] * c2 : -INFINITY;
          s[4 * g4 + e] = x;
          mx = fmaxf(mx, x);
        }
      }
      const float mn = fmaxf(m, pair_max(mx));
      if (__ballot(mn > m) != 0) {
        const float alpha = __builtin_amdgcn_exp2f(m - mn);
        l *= alpha;
#pragma unroll
        for (int i = 0; i < NDB; ++i)
#pragma unroll
          for (int e = 0; e < 16; ++e) o[i][e] *= alpha;
        m = mn;
      }
      bf16x8 ph[2], pm[2], pl[2];
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const float p = __builtin_amdgcn_exp2f(s[e] - m);
        l += p;
        const __bf16 t = (__bf16)p;
        ph[e >> 3][e & 7] = t;
        const float left = p - (float)t;         // exact, as the next
        const __bf16 u = (__bf16)left;
        pm[e >> 3][e & 7] = u;
        pl[e >> 3][e & 7] = (__bf16)(left - (float)u);
      }
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int i = 0; i < NDB; ++i) {
          const char* p0 = vt0 + j * 16 * ROWB + va[i];
          const bf16x8 vt = tr_read(p0, p0 + HALF);
          o[i] = mfma(vt, ph[j], o[i]);
          o[i] = mfma(vt, pm[j], o[i]);
          o[i] = mfma(vt, pl[j], o[i]);
        }
    }
  }
  if (!active) return;
  const float lt = pair_sum(l);
  const float inv = lt > 0.f ? 1.f / lt : 0.f;
  u32x2 res[NDB][4];
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < NDB; ++i)
#pragma unroll
    for (int g4 = 0; g4 < 4; ++g4)
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const uint32_t w = (uint32_t)f2bf(o[i][4 * g4 + 2 * e] * inv) |
                           ((uint32_t)f2bf(o[i][4 * g4 + 2 * e + 1] * inv) << 16);
        res[i][g4][e] = w;
        sum = probe(w, sum);
      }
  const bool stored = q0 + (lane & 31) < a.Lq;
  if (__ballot(stored && is_odd(lt, sum)) != 0) {
    visible_only<D>(a, b, h, q0, 32);
    return;
  }
  if (!stored) return;
  uint16_t* op = a.o + (int64_t)b * a.o_sb + (int64_t)qi * a.o_ss + (int64_t)h * a.o_sh;
#pragma unroll
  for (int i = 0; i < NDB; ++i)
#pragma unroll
    for (int g4 = 0; g4 < 4; ++g4)
      *reinterpret_cast<u32x2*>(op + i * 32 + 8 * g4 + 4 * (lane >> 5)) = res[i][g4];
}

// Queries that one wave of seq_kernel holds: 8 of a window of one chunk (32 or
// 64 keys), 4 where it loops over chunks (each waits for its rows).
bool one_chunk(const HierFrameAttnArgs& a) { return a.Lk <= 8 * (512 / a.D); }
int query_groups(const HierFrameAttnArgs& a) { return one_chunk(a) ? (a.Lq + 7) / 8 : (a.Lq + 3) / 4; }
// slot_kernel's time goes with queries x keys; a seq_kernel wave costs a chunk
// of 16 keys (D = 64) or 8 (128) at least, a tile_kernel workgroup 32 x 32, and
// with few sequences the chip waits for slot_kernel's trips of four keys.
// slot_kernel / seq_kernel, us: D = 64, 23,640 (sequence, head) pairs: 1 query x
// 1 key 4.9 / 13.8, 3 x 3 9.5 / 22.7, 3 x 8 17.5 / 23.2, 7 x 12 38 / 40, 3 x 15
// 28.5 / 25.1; 4,800 pairs: 3 x 3 4.8 / 7.2, 3 x 8 7.1 / 7.3, 3 x 12 8.8 / 7.5, 16 x 12
// 17.4 / 19.8; 1,600: 1 x 4 3.4 / 3.7, 3 x 8 5.8 / 4.7, 16 x 10 9.0 / 10.1; 800: 1 x 4
// 3.4 / 3.1.  D = 128, 23,640: 3 x 3 18.2 / 22.5, 4 x 4 24.9 / 26.1, 3 x 6 27.7 /
// 24.1; 3,600: 3 x 4 6.7 / 6.5, 8 x 4 8.7 / 10.4.
// slot_kernel / tile_kernel, D = 128: 240 pairs: 660 x 3 27.7 / 30.9, 660 x 6
// 38.3 / 31.2, 20 x 6 5.9 / 5.3; 1,600: 24 x 10 16.6 / 17.1, 48 x 5 18.5 / 22.4, 48 x
// 8 22.5 / 22.3; 24,000: 17 x 12 150 / 217, 32 x 8 202 / 240, 32 x 10 246 / 241.
bool use_slots(const HierFrameAttnArgs& a) {
  const int64_t pairs = (int64_t)a.B * a.H;
  if ((int64_t)a.B * a.Lq >= 1ll << 28) return false;   // its grid along x
  if (a.Lq > 16) return a.Lk <= 4 || ((int64_t)a.Lq * a.Lk <= 256 && pairs >= 512);
  if (a.Lk <= 2) return true;
  const int64_t queries = pairs * a.Lq;
  if (a.D == 128) return a.Lk <= 4 && queries >= 8192;
  return a.Lk <= 12 && queries >= (a.Lk <= 4 ? 2048 : a.Lk <= 8 ? 8192 : 20480);
}
// tile_kernel works on 32 queries whether they are there or not.  Windows of one
// chunk (2,200 x 24 heads, 24 keys, D = 128), seq_kernel / tile_kernel: 8
// queries 173 / 445 us, 16 309 / 475, 24 472 / 508, 32 612 / 533; 40 x 24 heads:
// 16 9.8 / 10.0, 24 13.4 / 10.4.  Longer (40 x 24 heads, 200 keys): 3 21 / 33 us,
// 5 29 / 33, 8 33 / 34; 8 heads, 1,000 keys: 5 59 / 43.
bool use_seq(const HierFrameAttnArgs& a) { return a.Lq <= (one_chunk(a) ? 16 : 4); }

template <int D, int NQ, bool ONCE>
void launch_seq(const HierFrameAttnArgs& a, hipStream_t st) {
  const int nqg = query_groups(a);
  const int64_t units = (int64_t)a.B * a.H * nqg;
  const hier::Grid gr = hier::launch_grid((units + 3) / 4, 256);
  const dim3 grid(gr.x, gr.y), block(256);
  const int groups = (a.Lk + 512 / D - 1) / (512 / D);   // of 512 / D rows
#define HIER_SEQ(G, LOOP) \
  hipLaunchKernelGGL((seq_kernel<D, NQ, G, LOOP, ONCE>), grid, block, 0, st, a, (uint32_t)nqg, (uint32_t)units)
  if (groups <= 2) HIER_SEQ(2, false);
  else if (groups <= 3) HIER_SEQ(3, false);
  else if (groups <= 4) HIER_SEQ(4, false);
  else if (groups <= 6) HIER_SEQ(6, false);
  else if (groups <= 8) HIER_SEQ(8, false);
  else if constexpr (ONCE && NQ <= 4) HIER_SEQ(8, true);
#undef HIER_SEQ
}

template <int D>
void launch_seq_d(const HierFrameAttnArgs& a, hipStream_t st) {
  const int nqg = query_groups(a);
  // (up to 8 queries, or 4 in a loop, are one wave's; 9 to 16 are two waves' of 5 to 8)
#define HIER_NQ(N) return nqg == 1 ? launch_seq<D, N, true>(a, st) : launch_seq<D, N, false>(a, st)
  switch ((a.Lq + nqg - 1) / nqg) {
    case 1: return launch_seq<D, 1, true>(a, st);
    case 2: return launch_seq<D, 2, true>(a, st);
    case 3: return launch_seq<D, 3, true>(a, st);
    case 4: return launch_seq<D, 4, true>(a, st);
    case 5: HIER_NQ(5);
    case 6: HIER_NQ(6);
    // (7 as 8, 1,970 x 12 heads, 14 keys, D = 64: 50.9 us, as 7 46.9)
    case 7: HIER_NQ(7);
    default: HIER_NQ(8);
  }
#undef HIER_NQ
}

}  // namespace

extern "C" int hier_frame_attn(const HierFrameAttnArgs* args, void* stream) {
  hier::clear_error();
  HIER_REQUIRE(args != nullptr, HIER_EINVAL, "args is NULL");
  const HierFrameAttnArgs& a = *args;
  HIER_REQUIRE(a.D == 128 || a.D == 64, HIER_EUNSUPPORTED, "head_dim must be 64 or 128, got %d", a.D);
  HIER_REQUIRE(a.B >= 0 && a.Lq >= 0 && a.Lk >= 0 && a.H >= 1 && a.n_block >= 1 &&
                   a.local_attn >= -1 && a.local_attn != 0,
               HIER_EINVAL, "invalid B=%d Lq=%d Lk=%d H=%d n_block=%d local_attn=%d", a.B, a.Lq,
               a.Lk, a.H, a.n_block, a.local_attn);
  if (a.B == 0 || a.Lq == 0) return HIER_OK;
  HIER_REQUIRE(a.q && a.k && a.v && a.o && a.q_frame && (a.k_frame || a.Lk == 0), HIER_EINVAL,
               "NULL pointer");
  auto al16 = [](const void* p) { return ((uintptr_t)p & 15u) == 0; };
  HIER_REQUIRE(al16(a.q) && al16(a.k) && al16(a.v) && al16(a.o), HIER_EINVAL,
               "q/k/v/o must be 16-byte aligned");
  HIER_REQUIRE(a.q_sb % 8 == 0 && a.q_ss % 8 == 0 && a.q_sh % 8 == 0 && a.k_sb % 8 == 0 &&
                   a.k_ss % 8 == 0 && a.k_sh % 8 == 0 && a.v_sb % 8 == 0 && a.v_ss % 8 == 0 &&
                   a.v_sh % 8 == 0 && a.o_sb % 8 == 0 && a.o_ss % 8 == 0 && a.o_sh % 8 == 0,
               HIER_EINVAL, "strides must keep 16-byte rows aligned");
  HIER_REQUIRE(a.H <= 65535, HIER_EUNSUPPORTED, "at most 65535 heads");
  const int64_t q_tiles = ((int64_t)a.Lq + 127) / 128;
  const int64_t wgs = (int64_t)a.B * a.H * (use_seq(a) ? query_groups(a) : q_tiles);
  const hier::Grid gr = hier::launch_grid(hier::xcd_grid(wgs), 256);
  HIER_REQUIRE(wgs <= hier::kMaxLaunchItems && gr.x != 0, HIER_EUNSUPPORTED, "too many queries");
  const hipStream_t st = (hipStream_t)stream;
  if (use_slots(a)) {
    const int64_t groups = ((int64_t)a.B * a.Lq + 512 / a.D - 1) / (512 / a.D);
    const dim3 sg((unsigned)groups, a.H);
    if (a.D == 128) hipLaunchKernelGGL(slot_kernel<128>, sg, dim3(64), 0, st, a);
    else hipLaunchKernelGGL(slot_kernel<64>, sg, dim3(64), 0, st, a);
    return hier::check_launch("slot_kernel");
  }
  if (use_seq(a)) {
    if (a.D == 128) launch_seq_d<128>(a, st);
    else launch_seq_d<64>(a, st);
    return hier::check_launch("seq_kernel");
  }
  const dim3 grid(gr.x, gr.y);
  if (a.D == 128)
    hipLaunchKernelGGL(tile_kernel<128>, grid, dim3(256), 0, st, a, (int)q_tiles, (int)wgs);
  else
    hipLaunchKernelGGL(tile_kernel<64>, grid, dim3(256), 0, st, a, (int)q_tiles, (int)wgs);
  return hier::check_launch("tile_kernel");
}
