// kernels_decode.h -- small per-call kernels: the router and the test hook of
// the wave reduction.  The expert vecmats are in kernels_rows.h.
#pragma once

#include "device_common.h"

// ---------------------------------------------------------------------------
// Router, one wave per token (E <= 1024).  Scores, selection bias, top-k (ties
// -> lower id), weights from the unbiased scores, renorm with the 2^-14 floor,
// scale (glm_dsa/moe_block.h:48-91).  A NaN score is picked only when no number
// is left, lowest id first, so the ids of a token are always k different experts.
//
// Bound by latency: a token's scores stay in its wave's registers (lane l holds
// experts l, l + 64, ...), and a round of the top-k is one wave maximum over
// DPP and one ballot, with no LDS and no barrier.  Kernel trace, median of 200
// in a row: 256 experts, top-8, T = 512 13.9 -> 5.8 us, T = 1 12.3 -> 4.5; 32
// experts, top-4, T = 1 6.0 -> 2.3; 1024 experts, T = 512 25.3 -> 13.3 (against a
// 256-thread workgroup per token, scores in LDS, shuffles in every round).  The
// first launch of a process takes about 20 us.
#define MOE_ROUTE_MAX_E 1024

// Score of one logit for the element-wise score functions (mode 1: sigmoid,
// 2: sqrt(softplus)); softmax (mode 0) needs the whole row.
__device__ __forceinline__ float route_score(float v, int mode) {
  return mode == 1 ? __fdiv_rn(1.0f, 1.0f + expf(-v)) : sqrtf(v > 20.0f ? v : log1pf(expf(v)));
}

// NJ: experts per lane (E <= 64 * NJ).  grid T, 64 threads; k <= 64.
template <int NJ>
__global__ __launch_bounds__(64) void k_route(const float *__restrict__ logits, const float *__restrict__ bias, int E, int k,
                                              int mode, int norm, float scale, int32_t *__restrict__ ids,
                                              float *__restrict__ wts) {
  const int t = blockIdx.x, lane = threadIdx.x;
  const float *l = logits + (size_t)t * E;
  float p[NJ], sel[NJ];
#pragma unroll
  for (int j = 0; j < NJ; j++) p[j] = lane + 64 * j < E ? l[lane + 64 * j] : 0.0f;
#pragma unroll
  for (int j = 0; j < NJ; j++) sel[j] = bias && lane + 64 * j < E ? bias[lane + 64 * j] : 0.0f;
  if (mode == 0) {  // softmax: exp(l - max), sum in double, scale by (float)(1/sum)
    float mx = -INFINITY;
#pragma unroll
    for (int j = 0; j < NJ; j++)
      if (lane + 64 * j < E) mx = fmaxf(mx, p[j]);
    mx = wave_max(mx);
    double s[4] = {0.0, 0.0, 0.0, 0.0};  // experts l + 64 * (w + 4i): a sum per w, over i, then over the lanes
#pragma unroll
    for (int j = 0; j < NJ; j++) {
      p[j] = lane + 64 * j < E ? expf(p[j] - mx) : 0.0f;
      s[j & 3] += (double)p[j];
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1)
#pragma unroll
      for (int w = 0; w < (NJ < 4 ? NJ : 4); w++) s[w] += __shfl_xor(s[w], off);
    const float inv = (float)(1.0 / (((s[0] + s[1]) + s[2]) + s[3]));
#pragma unroll
    for (int j = 0; j < NJ; j++) p[j] = p[j] * inv;
  } else {
#pragma unroll
    for (int j = 0; j < NJ; j++) p[j] = route_score(p[j], mode);
  }
  uint32_t left = 0;  // bit j: expert lane + 64 j may still be picked
#pragma unroll
  for (int j = 0; j < NJ; j++) {
    sel[j] = bias ? p[j] + sel[j] : p[j];
    if (lane + 64 * j < E) left |= 1u << j;
  }
  int my_id = 0;  // lane s: the expert and the weight of slot s
  float my_w = 0.0f;
  for (int s = 0; s < k; s++) {
    // this lane's largest score left (the lowest id of equal ones); a NaN never wins
    float bv = -INFINITY, bp = 0.0f;
    int bj = -1;
#pragma unroll
    for (int j = 0; j < NJ; j++)
      if (((left >> j) & 1u) && (sel[j] > bv || (bj < 0 && sel[j] == bv))) {
        bv = sel[j];
        bp = p[j];
        bj = j;
      }
    const float mx = wave_max(bv);
    uint64_t m = __ballot(bj >= 0 && bv == mx);
    if (m == 0) {  // only NaN scores are left: the lowest id of any lane
#pragma unroll
      for (int j = NJ - 1; j >= 0; j--)
        if ((left >> j) & 1u) {
          bj = j;
          bp = p[j];
        }
      m = __ballot(bj >= 0);
    }
    int src = __ffsll((unsigned long long)m) - 1;
    int id = src + 64 * __builtin_amdgcn_readlane(bj, src);
    for (uint64_t r = m & (m - 1); r; r &= r - 1) {  // equal scores on several lanes: the lowest id
      const int o = __ffsll((unsigned long long)r) - 1, oid = o + 64 * __builtin_amdgcn_readlane(bj, o);
      if (oid < id) {
        id = oid;
        src = o;
      }
    }
    const float w = readlane_f(bp, src);
    if (lane == src) left &= ~(1u << bj);
    if (lane == s) {
      my_id = id;
      my_w = w;
    }
  }
  if (norm) {  // by max(sum, 2^-14), the sum in slot order
    double sum = 0.0;
    for (int s = 0; s < k; s++) sum += (double)readlane_f(my_w, s);
    float fs = (float)sum;
    fs = fs < 6.103515625e-5f ? 6.103515625e-5f : fs;
    my_w = __fdiv_rn(my_w, fs);
  }
  if (scale != 0.0f && scale != 1.0f) my_w = __fmul_rn(my_w, scale);
  if (lane < k) {
    ids[(size_t)t * k + lane] = my_id;
    wts[(size_t)t * k + lane] = my_w;
  }
}

// ---------------------------------------------------------------------------
// Router logits for the moe-server protocol: logits[t][e] = sum_h W[e][h] *
// x[t][h] in f32 (ggml_mul_mat of ffn_gate_inp [H, E] with x [H, T],
// nano-glm/lib/models/glm_dsa/moe_block.h:52).  One wave per expert and 4
// tokens: each lane accumulates a strided quarter-row slice with FMAs, then
// wave_sum.  grid (ceil(E/4), ceil(T/4)), 256 threads; H % 4 == 0, rows
// 16-byte aligned.
// x rounded to the router weight's type before the products (XR: 0 f32 = as
// is, 1 f16, 2 bf16, each round to nearest even): ggml-cpu's mul_mat converts
// src1 to src0's vec_dot_type (f16 -> f16, bf16 -> bf16) and accumulates the
// products in f32.  A product of two f16 (or two bf16) values is exact in
// f32, so only the order of the f32 sum differs from ggml's.
template <int XR>
__device__ __forceinline__ float router_x(float v) {
  if (XR == 1) return (float)(_Float16)v;
  if (XR == 2) {
    const uint32_t u = __builtin_bit_cast(uint32_t, v);
    if ((u & 0x7fffffffu) > 0x7f800000u) return v;  // NaN stays NaN
    return __builtin_bit_cast(float, (u + 0x7fffu + ((u >> 16) & 1u)) & 0xffff0000u);
  }
  return v;
}

template <int XR>
__global__ __launch_bounds__(256) void k_router_logits(const float *__restrict__ W, const float *__restrict__ x,
                                                       int T, int E, int H, float *__restrict__ logits) {
  const int lane = threadIdx.x & 63;
  const int e = blockIdx.x * 4 + (threadIdx.x >> 6), t0 = blockIdx.y * 4;
  if (e >= E) return;  // whole waves
  const float4 *w4 = reinterpret_cast<const float4 *>(W + (size_t)e * H);
  float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int i = lane; i < H / 4; i += 64) {
    const float4 w = w4[i];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      if (t0 + j >= T) break;
      const float4 v = reinterpret_cast<const float4 *>(x + (size_t)(t0 + j) * H)[i];
      acc[j] = fmaf(w.x, router_x<XR>(v.x),
                    fmaf(w.y, router_x<XR>(v.y), fmaf(w.z, router_x<XR>(v.z), fmaf(w.w, router_x<XR>(v.w), acc[j]))));
    }
  }
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const float v = wave_sum(acc[j]);
    if (lane == 0 && t0 + j < T) logits[(size_t)(t0 + j) * E + e] = v;
  }
}

// ---------------------------------------------------------------------------
// test hook: one wave_sum per 64 inputs
__global__ __launch_bounds__(64) void k_debug_wave_sum(const float *__restrict__ x,
                                                       float *__restrict__ out) {
  const float v = wave_sum(x[blockIdx.x * 64 + threadIdx.x]);
  out[blockIdx.x * 64 + threadIdx.x] = v;
}
