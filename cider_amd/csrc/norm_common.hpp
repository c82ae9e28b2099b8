// Elementwise and reduction helpers of the model's producer ops (RMSNorm,
// residual add, SwiGLU) shared by the producer kernels (fused.hip) and the
// M == 1 linears that run a producer inside their x staging (gemv.hip).  Both
// use these same definitions, with the same 8-element chunk per thread and
// the same reduction order, so a fused launch is bit-identical to the pair of
// launches it replaces.
#pragma once

#include "common.hpp"

namespace cider {

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v = v + __shfl_xor(v, off);
  return v;
}

__device__ __forceinline__ uint16_t lo16(int32_t w) { return (uint16_t)((uint32_t)w & 0xffffu); }
__device__ __forceinline__ uint16_t hi16(int32_t w) { return (uint16_t)((uint32_t)w >> 16); }
__device__ __forceinline__ int32_t pack2(uint16_t a, uint16_t b) {
  return (int32_t)((uint32_t)a | ((uint32_t)b << 16));
}

// h(a + b) elementwise on 8 fp16 values
__device__ __forceinline__ i32x4 add8(i32x4 a, i32x4 b) {
  i32x4 r;
#pragma unroll
  for (int j = 0; j < 4; ++j)
    r[j] = pack2(f2h(h2f(lo16(a[j])) + h2f(lo16(b[j]))), f2h(h2f(hi16(a[j])) + h2f(hi16(b[j]))));
  return r;
}

__device__ __forceinline__ float sumsq8(i32x4 v, float s) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float a = h2f(lo16(v[j])), b = h2f(hi16(v[j]));
    s = s + a * a;
    s = s + b * b;
  }
  return s;
}

// RMSNorm output of one element: h(f32(w) * f32(h(x * r)))
__device__ __forceinline__ uint16_t norm1(uint16_t x, uint16_t w, float r) {
  return f2h(h2f(w) * h2f(f2h(h2f(x) * r)));
}

__device__ __forceinline__ i32x4 norm8(i32x4 v, i32x4 w, float r) {
  i32x4 o;
#pragma unroll
  for (int j = 0; j < 4; ++j)
    o[j] = pack2(norm1(lo16(v[j]), lo16(w[j]), r), norm1(hi16(v[j]), hi16(w[j]), r));
  return o;
}

// SwiGLU of one element: h(f32(h(silu(g))) * f32(u)), silu(g) = g / (1 + e^-g)
// in fp32 from the hardware exp2 (v_exp_f32, 2^x) and reciprocal
// (v_rcp_f32), each within about one ulp of binary32: the fp32 silu lands
// within a few ulps of the exact quotient, so its fp16 rounding h(silu(g))
// is the exact one or a neighbour only for values within those few ulps of
// a rounding boundary.  (The correctly rounded expf and division took about
// 30 VALU operations per element and bound the SwiGLU kernels.)  Infinities
// map as in the exact expression: g = -inf gives NaN, +inf gives +inf, and
// e^-g overflowing to +inf gives a signed zero.
__device__ __forceinline__ uint16_t swiglu1(uint16_t g, uint16_t u) {
  const float gf = h2f(g);
  constexpr float kLog2e = 1.4426950408889634f;  // 1 / ln 2
  const float e = __builtin_amdgcn_exp2f(-gf * kLog2e);
  const uint16_t a = f2h(gf * __builtin_amdgcn_rcpf(1.0f + e));
  return f2h(h2f(a) * h2f(u));
}

__device__ __forceinline__ i32x4 swiglu8(i32x4 g, i32x4 u) {
  i32x4 o;
#pragma unroll
  for (int j = 0; j < 4; ++j)
    o[j] = pack2(swiglu1(lo16(g[j]), lo16(u[j])), swiglu1(hi16(g[j]), hi16(u[j])));
  return o;
}

// ---------------------------------------------------------------------------
// per-head q/k RMSNorm + RoPE + KV-cache write (head_dim 128)
// ---------------------------------------------------------------------------
// Eight lanes per (token, head) of the fused projection row [q heads | k
// heads | v heads], eight heads per wave: lane j of a head holds elements
// [8j, 8j + 8) and [64 + 8j, 64 + 8j + 8), which are the pairs the
// rotate-half RoPE mixes, so every access is 16 bytes.  The head's sum of
// squares: each lane's 16 squares in order, then pairs, quads and the 8-lane
// group by DPP moves.  Per element: n = h(w * h(x * r)), out = h(h(n * cos) +
// h(-n' * sin)) for the first half (n' its partner) and h(h(n * cos) +
// h(n' * sin)) for the second.  (One wave per head with 2-byte lanes ran the
// 2048-token prefill's 2048 x 48 heads in 29.5 us per call; this layout in
// 15.6 us.)
__device__ __forceinline__ float group8_sum(float v) {
  v = v + __builtin_bit_cast(float, dpp_mov<kDppXor1>(__builtin_bit_cast(int32_t, v)));
  v = v + __builtin_bit_cast(float, dpp_mov<kDppXor2>(__builtin_bit_cast(int32_t, v)));
  v = v + __builtin_bit_cast(float, dpp_mov<kDppMirror8>(__builtin_bit_cast(int32_t, v)));
  return v;
}

// Per-head RMSNorm (head dimension 128) and rotate-half RoPE, eight lanes per
// head: lane j holds elements 8j .. 8j+7 (x0) and 64 + 8j .. (x1), the pairs
// RoPE mixes; w, c and s the norm weight, cos and sin at the same elements.
// head_sumsq: the head's sum of squares, in every lane of its group.
__device__ __forceinline__ float head_sumsq(i32x4 x0, i32x4 x1) {
  float ss = 0.0f;
  ss = sumsq8(x0, ss);
  ss = sumsq8(x1, ss);
  return group8_sum(ss);
}
__device__ __forceinline__ void norm_rope8(i32x4 x0, i32x4 x1, i32x4 w0, i32x4 w1, i32x4 c0,
                                           i32x4 c1, i32x4 s0, i32x4 s1, float ss, float eps,
                                           i32x4& o0, i32x4& o1) {
  const float r = 1.0f / sqrtf(ss / 128.0f + eps);
  const i32x4 n0 = norm8(x0, w0, r), n1 = norm8(x1, w1, r);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    uint16_t lo[2], hi[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const float a = h2f(h ? hi16(n0[e]) : lo16(n0[e]));
      const float b = h2f(h ? hi16(n1[e]) : lo16(n1[e]));
      const float ca = h2f(h ? hi16(c0[e]) : lo16(c0[e]));
      const float sa = h2f(h ? hi16(s0[e]) : lo16(s0[e]));
      const float cb = h2f(h ? hi16(c1[e]) : lo16(c1[e]));
      const float sb = h2f(h ? hi16(s1[e]) : lo16(s1[e]));
      // out = x * cos + rotate_half(x) * sin, rotate_half(x) = [-x[64:], x[:64]]
      lo[h] = f2h(h2f(f2h(a * ca)) + h2f(f2h(-(b * sa))));
      hi[h] = f2h(h2f(f2h(b * cb)) + h2f(f2h(a * sb)));
    }
    o0[e] = pack2(lo[0], lo[1]);
    o1[e] = pack2(hi[0], hi[1]);
  }
}

__device__ __forceinline__ float block_sum4(float v, float* red) {
  const int wave = threadIdx.x >> 6;
  v = wave_sum(v);
  __syncthreads();  // red may still be read from the previous reduction
  if ((threadIdx.x & 63) == 0) red[wave] = v;
  __syncthreads();
  return ((red[0] + red[1]) + red[2]) + red[3];
}

}  // namespace cider
