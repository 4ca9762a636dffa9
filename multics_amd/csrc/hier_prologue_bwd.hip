// Backward of the Q/K projection tail (camera add, RMSNorm, gain, RoPE):
// the autograd of SelfAttention._project_self_attn_qkv after the three GEMMs
// (multics/models/attention.py:355-365, 307-320, 231-242; rope.py:248-254).
//
// Forward, per token and projection (x = q(x) or k(x), dim = H * D):
//   a = bf16(x + bf16(cam . Wc^T))      camera adapter (when present)
//   r = rsqrt(mean(a^2) + eps)
//   y = bf16(a * r),  z = bf16(y * w),  out = bf16(rotate(z, theta))
// Backward, given d_out:
//   dz = rotate(d_out, -theta)                    (the rotation's transpose)
//   dw += dz * y                                  (gain gradient, summed over tokens)
//   dy = dz * w
//   da = r * dy - r^3 * a * sum(dy * a) / dim     (RMSNorm)
//   dx = da                                       (the add passes it through)
// in fp32 from the saved inputs: a and r are recomputed from x, the camera
// row and the weights (the forward keeps nothing extra).  The gain gradient
// takes y before its rounding (r * a in fp32).
//
// HBM-bound: four bf16 rows per token and projection (x and d_out in, dx out).
// One workgroup owns `tpw` consecutive tokens of one projection (blockIdx.y:
// 0 = q, 1 = k) and a thread owns 8 channels of every one of them, so the sums
// over tokens (gain gradient, camera-weight gradient) stay in registers and
// only the two row sums (mean square, dy . a) cross threads.  Tokens go two at
// a time, the next two loaded meanwhile; their four row sums are folded
// together: one lane-swap tree per wave leaves a value per 16-lane row, one
// LDS slot per wave and value, one barrier, one DPP row sum.
//
// The camera-weight gradient is dWc = sum over tokens of dx (x) cam.  The
// camera row is the same for every token of a player's frame, so a thread sums
// its dx while the row stays and puts the sum into one of the workgroup's 12
// slots where it changes; grad_sum_kernel multiplies slots and rows.  A
// workgroup that meets more than 12 rows turns its slots into the 12 columns
// of its own dWc and adds the products there (slow, but no real camera changes
// that often).  All sums are added in a fixed order.
//
// 18,816 tokens x 3,072 of q and k, camera on: 694 MB in 146-150 us (4.6-4.8 TB/s; a
// copy reaches 5.05) plus 9 us for the sums.  One wave per 16 tokens with no
// loads ahead took 465 us, plus 26 us for the gain sums and 131 us for the
// camera-weight gradients as two GEMMs over dx.
#include "hier_common.h"

#include <algorithm>

namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }
__device__ __forceinline__ uint32_t pack(float a, float b) {
  const f32x2 v = {a, b};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}
__device__ __forceinline__ float dot2(uint32_t a, uint32_t b, float c) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, a), __builtin_bit_cast(bf16x2, b),
                                         c, false);
}

// Sum over the 16 lanes of a row, in each of them.
__device__ __forceinline__ float row_sum(float v) {
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xF, 0xF, false));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xF, 0xF, false));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x124, 0xF, 0xF, false));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128, 0xF, 0xF, false));
  return v;
}
// Lanes 0-31: a summed over its two halves; lanes 32-63: b.
__device__ __forceinline__ float fold32(float a, float b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// Rows 0 and 2: a's rows 0 + 1 and 2 + 3; rows 1 and 3: b's.
__device__ __forceinline__ float fold16(float a, float b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

constexpr int kCpt = 8;        // channels of a thread
constexpr int kTrip = 2;       // tokens of a trip
constexpr int kMaxWaves = 16;  // LDS slots per row sum (at most 8 waves run)
constexpr int kSlots = 12;     // camera sums of a workgroup: as many as dWc has columns
constexpr int kSegInts = 16;   // ints per workgroup: count (-1: dWc columns), then slot tokens

// What a trip reads: projection and gradient words, cos / sin, and (lane
// l < 12) dword l of the two camera rows and the same dword of the row before.
struct Trip {
  u32x4 x[kTrip], d[kTrip];
  float4 c[kTrip], s[kTrip];
  uint32_t cam, cam_prev;
};

template <int NCH, int C>
__global__ __launch_bounds__(64 * NCH, 2) void prologue_bwd_kernel(
    HierPrologueBwdArgs a, float* dwc_q, float* dwc_k, int32_t* seg, int tpw) {
  constexpr int dim = 512 * NCH, CW = C > 0 ? C / 2 : 1, NV = 2 * kTrip;
  __shared__ float red[2][NV][kMaxWaves];
  __shared__ int seg_tok[NCH][kSlots];       // each wave its own copy
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool is_k = blockIdx.y != 0;
  const int c0 = tid * kCpt;
  const int head = c0 / a.D, d0 = c0 - head * a.D, half = a.D / 2, m0 = d0 / 2;
  const int s_begin = (int)min((int64_t)a.S, (int64_t)blockIdx.x * tpw);
  const int s_end = (int)min((int64_t)a.S, (int64_t)s_begin + tpw);
  const float inv_dim = 1.f / (float)dim;
  const uint16_t* const xin = is_k ? a.kx : a.qx;
  const uint16_t* const din = (is_k ? a.dk : a.dq) + (int64_t)head * (is_k ? a.dk_sh : a.dq_sh) + d0;
  const int64_t d_ss = is_k ? a.dk_ss : a.dq_ss;
  uint16_t* const dx = is_k ? a.dkx : a.dqx;
  const bool cam_w = C > 0 && dwc_q != nullptr;
  int32_t* const my_seg = seg + ((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * kSegInts;

  for (int i = tid; i < 2 * NV * kMaxWaves; i += 64 * NCH) (&red[0][0][0])[i] = 0.f;
  float g[kCpt], dw[kCpt], sdx[kCpt];        // gains; gain gradient; dx summed over one camera row
  {
    const u32x4 w = *reinterpret_cast<const u32x4*>((is_k ? a.norm_k_w : a.norm_q_w) + c0);
#pragma unroll
    for (int e = 0; e < kCpt / 2; ++e) {
      g[2 * e] = lo(w[e]);
      g[2 * e + 1] = hi(w[e]);
    }
  }
#pragma unroll
  for (int e = 0; e < kCpt; ++e) dw[e] = sdx[e] = 0.f;
  int n_seg = 0, row_tok = s_begin;          // slots filled; a token with sdx's camera row
  uint32_t cp[kCpt / 2];                     // bf16 camera product of the current row
#pragma unroll
  for (int e = 0; e < kCpt / 2; ++e) cp[e] = 0;

  // camera rows from the one before s_begin (or s_begin, for the first token)
  const int cam0 = s_begin > 0 ? CW : 0;
  const uint32_t* const camw =
      reinterpret_cast<const uint32_t*>(a.cam) + (int64_t)s_begin * CW - cam0;
  // Past the range a trip repeats its last token, and stores its row again:
  // with a store that may or may not be outstanding the compiler waits for the
  // stores of one trip before the arithmetic of the next.  The uniform row offsets
  // are pinned to scalar registers: left to itself the compiler forms each
  // address with a quarter-rate vector multiply.
  auto fetch = [&](Trip& f, int s) {
#pragma unroll
    for (int t = 0; t < kTrip; ++t) {
      const int st = min(s + t, s_end - 1);
      int64_t xo = (int64_t)st * dim, ro = (int64_t)st * half;
      asm("" : "+s"(xo), "+s"(ro));
      f.x[t] = *reinterpret_cast<const u32x4*>(xin + xo + (uint32_t)c0);
      f.d[t] = *reinterpret_cast<const u32x4*>(din + (int64_t)st * d_ss);
      f.c[t] = *reinterpret_cast<const float4*>(a.rope_cos + ro + (uint32_t)m0);
      f.s[t] = *reinterpret_cast<const float4*>(a.rope_sin + ro + (uint32_t)m0);
    }
    if constexpr (C > 0) {
      // (lanes past the range read its last dword)
      const int i = cam0 + min((s - s_begin) * CW + lane, (s_end - s_begin) * CW - 1);
      f.cam = camw[(uint32_t)i];
      f.cam_prev = camw[(uint32_t)max(i - CW, 0)];
    }
  };
  // puts sdx, the sum over the tokens of row_tok's camera row, away
  auto flush = [&]() {
    if (!cam_w) return;
    // (the address is formed here, not held in registers between the flushes)
    int ch = c0;
    asm volatile("" : "+v"(ch));
    float* const slots = (is_k ? dwc_k : dwc_q) + (int64_t)blockIdx.x * kSlots * dim + ch;
    auto at = [&](int j, int q) { return reinterpret_cast<float4*>(slots + (int64_t)j * dim + 4 * q); };
    const uint16_t* cam = a.cam;
    auto cam_at = [&](int tok, int c) {
      return __uint_as_float((uint32_t)cam[(int64_t)tok * C + c] << 16);
    };
    if (n_seg < kSlots) {
#pragma unroll
      for (int q = 0; q < 2; ++q)
        *at(n_seg, q) = make_float4(sdx[4 * q], sdx[4 * q + 1], sdx[4 * q + 2], sdx[4 * q + 3]);
      if (lane == 0) seg_tok[wave][n_seg] = row_tok;
      ++n_seg;
    } else {
      if (n_seg == kSlots) {                 // the slots' products take the slots' place
#pragma unroll 1
        for (int e = 0; e < kCpt; ++e) {     // (one channel at a time: few registers)
          float v[kSlots];
#pragma unroll
          for (int j = 0; j < kSlots; ++j) v[j] = slots[(int64_t)j * dim + e];
#pragma unroll 1
          for (int c = 0; c < C; ++c) {
            float w = 0.f;
#pragma unroll
            for (int j = 0; j < kSlots; ++j) w = fmaf(v[j], cam_at(seg_tok[wave][j], c), w);
            slots[(int64_t)c * dim + e] = w;
          }
        }
        ++n_seg;
      }
#pragma unroll 1
      for (int c = 0; c < C; ++c) {
        const float m = cam_at(row_tok, c);
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          float4 w = *at(c, q);
          w.x = fmaf(sdx[4 * q], m, w.x); w.y = fmaf(sdx[4 * q + 1], m, w.y);
          w.z = fmaf(sdx[4 * q + 2], m, w.z); w.w = fmaf(sdx[4 * q + 3], m, w.w);
          *at(c, q) = w;
        }
      }
    }
#pragma unroll
    for (int e = 0; e < kCpt; ++e) sdx[e] = 0.f;
  };
  auto trip = [&](int s, int par, const Trip& use, Trip& nxt) {
    uint64_t diff = 0;                       // bit CW t + c: word c of token t's row is new
    if constexpr (C > 0) diff = __ballot(use.cam != use.cam_prev);
    auto is_new = [&](int t) {
      return C > 0 && s + t < s_end && ((diff >> (CW * t)) & ((1ull << CW) - 1)) != 0;
    };
    fetch(nxt, s + kTrip);
    uint32_t av[kTrip][kCpt / 2];            // a, packed
    float z[kTrip][kCpt], v[NV];
#pragma unroll
    for (int t = 0; t < kTrip; ++t) {
      if (C > 0 && (is_new(t) || (t == 0 && s == s_begin))) {   // uniform
        int ch = c0;                           // (formed here, as in flush)
        asm volatile("" : "+v"(ch));
        const uint32_t* wr = reinterpret_cast<const uint32_t*>(is_k ? a.w_cam_k : a.w_cam_q) + ch * CW;
#pragma unroll
        for (int e = 0; e < kCpt / 2; ++e) {
          // exact products, fp32 sums in c order (as the forward)
          const uint32_t* w32 = wr + 2 * e * CW;
          float p0 = 0.f, p1 = 0.f;
#pragma unroll
          for (int c = 0; c < CW; ++c) {
            const uint32_t cw = __builtin_amdgcn_readlane((int)use.cam, CW * t + c);
            p0 = dot2(w32[c], cw, p0);
            p1 = dot2(w32[CW + c], cw, p1);
          }
          cp[e] = pack(p0, p1);
          __builtin_amdgcn_sched_barrier(0);   // two channels' weights in registers at a time
        }
      }
      float ss = 0.f, dot = 0.f;
#pragma unroll
      for (int e = 0; e < kCpt / 2; ++e) {
        uint32_t u = use.x[t][e];
        if constexpr (C > 0) u = pack(lo(u) + lo(cp[e]), hi(u) + hi(cp[e]));
        ss = dot2(u, u, ss);                 // bf16 squares are exact in fp32
        const uint32_t dv = use.d[t][e];
        const float co = e == 0 ? use.c[t].x : e == 1 ? use.c[t].y : e == 2 ? use.c[t].z : use.c[t].w;
        const float si = e == 0 ? use.s[t].x : e == 1 ? use.s[t].y : e == 2 ? use.s[t].z : use.s[t].w;
        const float q0 = lo(dv), q1 = hi(dv);
        const float z0 = q0 * co + q1 * si, z1 = q1 * co - q0 * si;
        dot = fmaf(z0 * lo(u), g[2 * e], dot);
        dot = fmaf(z1 * hi(u), g[2 * e + 1], dot);
        av[t][e] = u;
        z[t][2 * e] = z0;
        z[t][2 * e + 1] = z1;
      }
      v[t] = ss;
      v[kTrip + t] = dot;
    }
    // four values, one per 16-lane row, in the order 0 2 1 3
    const float w = row_sum(fold16(fold32(v[0], v[1]), fold32(v[2], v[3])));
    const int rw = lane >> 4;
    if ((lane & 15) == 0) red[par][(rw & 1) << 1 | rw >> 1][wave] = w;
    hier::barrier_lds();                     // the next trip's loads stay in flight
    const float tot = row_sum(red[par][rw][lane & 15]);
    auto total = [&](int i) {
      return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(tot), 16 * i));
    };
#pragma unroll
    for (int t = 0; t < kTrip; ++t) {
      const float r = __builtin_amdgcn_rsqf(total(t) * inv_dim + a.eps);
      const float k2 = r * r * total(kTrip + t) * inv_dim;
      if (is_new(t)) {
        if (s + t > s_begin) flush();
        row_tok = s + t;
      }
      // past the end: the last token's row once more, and nothing to the sums
      const bool live = s + t < s_end;
      const float rl = live ? r : 0.f;
      u32x4 o;
#pragma unroll
      for (int e = 0; e < kCpt / 2; ++e) {
        float dv[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int ch = 2 * e + h;
          const float ac = h ? hi(av[t][e]) : lo(av[t][e]);
          dw[ch] = fmaf(z[t][ch] * ac, rl, dw[ch]);
          const float dyn = fmaf(-k2, ac, z[t][ch] * g[ch]);
          dv[h] = dyn * r;
          sdx[ch] = fmaf(dyn, rl, sdx[ch]);
        }
        o[e] = pack(dv[0], dv[1]);
      }
      int64_t xo = (int64_t)min(s + t, s_end - 1) * dim;
      asm("" : "+s"(xo));
      *reinterpret_cast<u32x4*>(dx + xo + (uint32_t)c0) = o;
    }
  };
  __syncthreads();   // red cleared
  float4* dst = reinterpret_cast<float4*>((is_k ? a.dw_k_partial : a.dw_q_partial) +
                                          (int64_t)blockIdx.x * dim + c0);
  if (s_begin < s_end) {
    Trip pa, pb;
    fetch(pa, s_begin);
    // two stores after the loads, as every later trip has (the wait counts of
    // the loop must hold on the way into it as well); overwritten below
    dst[0] = dst[1] = make_float4(0.f, 0.f, 0.f, 0.f);
    // (the second trip unconditionally: with a way round it the compiler
    // waits for the loads in flight before it issues the next ones)
    for (int s = s_begin; s < s_end; s += 2 * kTrip) {
      trip(s, 0, pa, pb);
      trip(s + kTrip, 1, pb, pa);
    }
    flush();
  }
  dst[0] = make_float4(dw[0], dw[1], dw[2], dw[3]);
  dst[1] = make_float4(dw[4], dw[5], dw[6], dw[7]);
  if (cam_w && wave == 0 && lane <= kSlots)
    my_seg[lane] = lane == 0 ? (n_seg > kSlots ? -1 : n_seg) : lane <= n_seg ? seg_tok[0][lane - 1] : 0;
}

// Sums of the workgroups' rows, rounded to bf16: the gain gradient and (CAM)
// the camera weights' ([dim][12]).  blockIdx.y = projection.  A workgroup sums
// 16 channels: 4 threads of 4 channels times 64 row groups.
template <bool CAM>
__global__ __launch_bounds__(256) void grad_sum_kernel(HierPrologueGradArgs g, const uint16_t* cam,
                                                       const float* dw_q, const float* dw_k,
                                                       int rows, int dim) {
  constexpr int NO = CAM ? 13 : 1;
  __shared__ float part[64][NO][17];         // (padded: the column sums read across the first index)
  const int tx = threadIdx.x & 3, ty = threadIdx.x >> 2;
  const int col = blockIdx.x * 16 + 4 * tx;
  const bool is_k = blockIdx.y != 0;
  float s[NO][4] = {};
  auto add = [&](float* d, const float4& v, float m) {
    d[0] = fmaf(v.x, m, d[0]); d[1] = fmaf(v.y, m, d[1]);
    d[2] = fmaf(v.z, m, d[2]); d[3] = fmaf(v.w, m, d[3]);
  };
  for (int r = ty; r < rows; r += 64) {
    add(s[0], *reinterpret_cast<const float4*>((is_k ? dw_k : dw_q) + (int64_t)r * dim + col), 1.f);
    if constexpr (CAM) {
      const float* slots = (is_k ? g.dwc_k_partial : g.dwc_q_partial) + (int64_t)r * kSlots * dim + col;
      const int32_t* sg = g.segments + ((int64_t)blockIdx.y * rows + r) * kSegInts;
      const int n = sg[0];
      for (int j = 0; j < n; ++j) {
        const float4 v = *reinterpret_cast<const float4*>(slots + (int64_t)j * dim);
        const uint32_t* cw = reinterpret_cast<const uint32_t*>(cam) + (int64_t)sg[1 + j] * 6;
#pragma unroll
        for (int c = 0; c < 6; ++c) {
          const uint32_t w = cw[c];
          add(s[1 + 2 * c], v, lo(w));
          add(s[2 + 2 * c], v, hi(w));
        }
      }
      if (n < 0)
#pragma unroll
        for (int c = 0; c < 12; ++c)
          add(s[1 + c], *reinterpret_cast<const float4*>(slots + (int64_t)c * dim), 1.f);
    }
  }
#pragma unroll
  for (int o = 0; o < NO; ++o)
#pragma unroll
    for (int e = 0; e < 4; ++e) part[ty][o][4 * tx + e] = s[o][e];
  __syncthreads();
  if (threadIdx.x >= 16 * NO) return;
  const int o = threadIdx.x >> 4, ch = threadIdx.x & 15;
  float t = 0.f;
  for (int i = 0; i < 64; ++i) t += part[i][o][ch];
  const uint16_t b = __builtin_bit_cast(uint16_t, (__bf16)t);
  const int64_t c = blockIdx.x * 16 + ch;
  if (o == 0) (is_k ? g.dnorm_k : g.dnorm_q)[c] = b;
  else (is_k ? g.dw_cam_k : g.dw_cam_q)[c * 12 + o - 1] = b;
}

int launch_bwd(const HierPrologueBwdArgs& a, float* dwc_q, float* dwc_k, int32_t* seg,
               hipStream_t st) {
  HIER_REQUIRE(a.S >= 0 && a.H >= 1 && a.H <= 4096 && (a.D == 64 || a.D == 128) &&
                   a.tokens_per_wave >= 1,
               HIER_EUNSUPPORTED, "prologue backward supports head_dim 64/128, got H=%d D=%d",
               a.H, a.D);
  const int dim = a.H * a.D;
  const int nch = dim / 512;
  HIER_REQUIRE(dim % 512 == 0 && nch >= 1 && nch <= 8, HIER_EUNSUPPORTED,
               "prologue backward supports model dims that are multiples of 512 up to 4096, got %d",
               dim);
  HIER_REQUIRE(a.qx && a.kx && a.dq && a.dk && a.dqx && a.dkx && a.norm_q_w && a.norm_k_w &&
                   a.rope_cos && a.rope_sin && a.dw_q_partial && a.dw_k_partial,
               HIER_EINVAL, "NULL pointer");
  const bool cam = a.cam != nullptr;
  HIER_REQUIRE(!cam || (a.C == 12 && a.w_cam_q && a.w_cam_k), HIER_EUNSUPPORTED,
               "camera adapter supports C=12 with both weights, got C=%d", a.C);
  auto al16 = [](const void* p) { return ((uintptr_t)p & 15u) == 0; };
  HIER_REQUIRE(al16(a.qx) && al16(a.kx) && al16(a.dq) && al16(a.dk) && al16(a.dqx) &&
                   al16(a.dkx) && al16(a.norm_q_w) && al16(a.norm_k_w) && al16(a.rope_cos) &&
                   al16(a.rope_sin) && al16(a.dw_q_partial) && al16(a.dw_k_partial) &&
                   (!cam || (((uintptr_t)a.cam & 3u) == 0 && ((uintptr_t)a.w_cam_q & 3u) == 0 &&
                             ((uintptr_t)a.w_cam_k & 3u) == 0)),
               HIER_EINVAL, "tensors must be 16-byte aligned (camera rows and weights 4-byte)");
  HIER_REQUIRE(a.dq_ss >= 0 && a.dq_sh >= 0 && a.dk_ss >= 0 && a.dk_sh >= 0 && a.dq_ss % 8 == 0 &&
                   a.dq_sh % 8 == 0 && a.dk_ss % 8 == 0 && a.dk_sh % 8 == 0,
               HIER_EINVAL, "gradient strides must be non-negative multiples of 8");
  HIER_REQUIRE((int64_t)a.S * dim <= ((int64_t)1 << 40), HIER_EUNSUPPORTED, "too many tokens");
  if (a.S == 0) return HIER_OK;
  const int rows = hier_qk_prologue_bwd_waves(&a);
  HIER_REQUIRE(rows > 0, HIER_EUNSUPPORTED, "too many waves");
  const dim3 grid(rows, 2);
#define HIER_PBWD(N)                                                                          \
  if (nch == N) {                                                                             \
    if (cam) hipLaunchKernelGGL((prologue_bwd_kernel<N, 12>), grid, dim3(64 * N), 0, st, a,    \
                                dwc_q, dwc_k, seg, a.tokens_per_wave);                        \
    else hipLaunchKernelGGL((prologue_bwd_kernel<N, 0>), grid, dim3(64 * N), 0, st, a, dwc_q,  \
                            dwc_k, seg, a.tokens_per_wave);                                   \
  }
  HIER_PBWD(1) HIER_PBWD(2) HIER_PBWD(3) HIER_PBWD(4) HIER_PBWD(5) HIER_PBWD(6) HIER_PBWD(7)
  HIER_PBWD(8)
#undef HIER_PBWD
  return hier::check_launch("prologue_bwd_kernel");
}

}  // namespace

extern "C" int hier_qk_prologue_bwd_waves(const HierPrologueBwdArgs* args) {
  if (!args || args->S < 0 || args->tokens_per_wave < 1) return -1;
  const int64_t waves = ((int64_t)args->S + args->tokens_per_wave - 1) / args->tokens_per_wave;
  return waves > (1ll << 28) ? -1 : (int)((waves + 3) / 4 * 4);
}

extern "C" int hier_qk_prologue_bwd(const HierPrologueBwdArgs* args, void* stream) {
  hier::clear_error();
  HIER_REQUIRE(args != nullptr, HIER_EINVAL, "args is NULL");
  return launch_bwd(*args, nullptr, nullptr, nullptr, (hipStream_t)stream);
}

extern "C" int hier_qk_prologue_grads(const HierPrologueBwdArgs* args,
                                      const HierPrologueGradArgs* grads, void* stream) {
  hier::clear_error();
  HIER_REQUIRE(args != nullptr && grads != nullptr, HIER_EINVAL, "args is NULL");
  const HierPrologueGradArgs& g = *grads;
  const bool cam_w = g.dw_cam_q != nullptr;
  HIER_REQUIRE(g.dnorm_q && g.dnorm_k && (cam_w == (g.dw_cam_k != nullptr)), HIER_EINVAL,
               "NULL gradient pointer");
  HIER_REQUIRE(!cam_w || (args->cam && g.dwc_q_partial && g.dwc_k_partial && g.segments &&
                          (((uintptr_t)g.dwc_q_partial | (uintptr_t)g.dwc_k_partial) & 15u) == 0),
               HIER_EINVAL, "camera-weight gradients need camera rows and 16-byte aligned partials");
  const int rc = launch_bwd(*args, cam_w ? g.dwc_q_partial : nullptr,
                            cam_w ? g.dwc_k_partial : nullptr, g.segments, (hipStream_t)stream);
  if (rc != HIER_OK || args->S == 0) return rc;
  const int dim = args->H * args->D, rows = hier_qk_prologue_bwd_waves(args);
  const dim3 grid(dim / 16, 2);
  if (cam_w)
    hipLaunchKernelGGL(grad_sum_kernel<true>, grid, dim3(256), 0, (hipStream_t)stream, g, args->cam,
                       args->dw_q_partial, args->dw_k_partial, rows, dim);
  else
    hipLaunchKernelGGL(grad_sum_kernel<false>, grid, dim3(256), 0, (hipStream_t)stream, g, args->cam,
                       args->dw_q_partial, args->dw_k_partial, rows, dim);
  return hier::check_launch("grad_sum_kernel");
}
