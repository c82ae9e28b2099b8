// M == 1 decode MV: fp16 activation x int8 weight, no activation quantization.
//
// Reference semantics (cider/kernels/w8a8_int8_mv.metal:26-70 per-channel,
// cider/kernels/pergroup_int8_mv.metal:35-105 per-group): for each output row
// n, 32 lanes each own elements 256b + 8l + i (i < 8) of every 256-wide block
// b; lane l forms  d = sum_i f32(w) * f32(x)  left to right (the products are
// exact), accumulates  r_l += d  (per-channel) or  r_l += f32(sw[g,n] * d)
// with g = (256b + 8l) / gs  (per-group) over the blocks in order, the 32
// lanes are summed by an xor butterfly (16, 8, 4, 2, 1), and
//   per-channel: y = h(f32(sw[n] * R) + f32(bias[n]))
//   per-group:   y = h(f32(R + f32(bias[n])))
// This kernel reproduces exactly that order, for every shape.  It serves the
// shapes outside the table of the streaming MV (mv_stream.hip, which sums in
// its own order within the fp32 reassociation bound): K < 1024, K > 16384,
// K % 256 != 0, or unaligned operands.  launch_mv and launch_mv_producer pick
// between the two by the same rule, so a fused producer launch still equals
// the producer launch followed by launch_mv bit for bit.
//
// MI355X design
//   * 16 lanes per row, four rows per 64-lane wave.  Lane j carries the two
//     reference lanes 2j and 2j+1, so each block costs it one 16-byte weight
//     load (the 16 consecutive bytes 256b + 16j ..) instead of two 8-byte
//     ones.  The butterfly over reference lanes 16, 8, 4, 2 is a shuffle over
//     physical lanes 8, 4, 2, 1; offset 1 is the in-register sum of the pair.
//   * x is staged once per workgroup in LDS (zero-padded to whole blocks);
//     its reads are issued first, the first 2U weight blocks right after, so
//     the weight stream starts before the staging barrier.  Two register
//     buffers of U blocks (U * 16 bytes per lane each) keep it in flight
//     while blocks reduce.
//     Per-group scales of the workgroup's rows are staged in LDS as well.
//   * Rows per workgroup (4, 8 or 16) are chosen so the grid has enough
//     waves to cover HBM latency on short-N shapes.
#include "common.hpp"
#include "kernels.hpp"
#include "norm_common.hpp"

namespace cider {

namespace {

constexpr int kLanesPerRow = 16;

// d = sum_{i<8} f32(w_i) * f32(x_i), left to right, from 8 weight bytes
// (two dwords) and 8 fp16 values (four dwords).
__device__ __forceinline__ float dot8(uint32_t w0, uint32_t w1, uint32_t x0, uint32_t x1,
                                      uint32_t x2, uint32_t x3) {
  const uint32_t wv[2] = {w0, w1};
  const uint32_t xv[4] = {x0, x1, x2, x3};
  float d = 0.0f;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int8_t wi = (int8_t)(wv[i >> 2] >> (8 * (i & 3)));
    const float xf = h2f((uint16_t)((i & 1) ? (xv[i >> 1] >> 16) : (xv[i >> 1] & 0xffffu)));
    const float prod = (float)wi * xf;  // exact: 8-bit x 11-bit significands
    d = (i == 0) ? prod : d + prod;
  }
  return d;
}

}  // namespace

// PG: per-group scales; VEC: how the weights load.  kFull: K % 256 == 0 and
// 16-byte aligned w and x.  kChunks: K % 16 == 0, 16-byte aligned w, x in LDS:
// the same loads, clamped to the row's last chunk in a part-filled last block,
// where the staged x is zero (N=4096 K=4160: 32.8 us bytewise, 10.2 so).  kBytes:
// anything else, bytewise with bounds.
// XLDS: x staged in LDS (K <= kMaxLdsK); otherwise read from global.
enum MvLoad { kBytes, kChunks, kFull };

template <bool PG, int VEC, bool XLDS, int U>
__global__ __launch_bounds__(256) void mv_kernel(
    const uint16_t* __restrict__ x, const int8_t* __restrict__ w,
    const float* __restrict__ sw, const uint16_t* __restrict__ bias,
    uint16_t* __restrict__ y, int N, int K, int gs, int rows_per_wg) {
  extern __shared__ __attribute__((aligned(16))) uint8_t dyn[];
  const int nb = (K + 255) / 256;
  const int kp = nb * 256;  // padded K
  uint16_t* xs = reinterpret_cast<uint16_t*>(dyn);
  const int G = PG ? K / gs : 0;
  float* sws = reinterpret_cast<float*>(dyn + (XLDS ? (size_t)kp * 2 : 0));

  const int tid = threadIdx.x, nthr = blockDim.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rg = lane >> 4, j = lane & 15;
  const int row_in_wg = wave * 4 + rg;
  const int n0 = blockIdx.x * rows_per_wg;
  const int n = n0 + row_in_wg;
  const bool live = n < N;
  const int8_t* wr = w + (int64_t)(live ? n : 0) * K;

  // weight slice of block b for this lane (16 bytes at 256 b + 16 j)
  auto load_w = [&](int b, i32x4& v) {
    if constexpr (VEC == kChunks) {
      v = ld16_nt(wr + min(min(b, nb - 1) * 256 + 16 * j, K - 16));
      return;
    }
    if constexpr (VEC == kFull) {
      // branch-free: a block index past the end re-reads the last block (its
      // value is never consumed), so every load is issued unconditionally and
      // the compiler can count outstanding loads exactly
      v = ld16_nt(wr + min(b, nb - 1) * 256 + 16 * j);
      return;
    }
    const int k = b * 256 + 16 * j;
    if (live && b < nb) {
      {
        uint32_t t[4] = {0u, 0u, 0u, 0u};
        for (int i = 0; i < 16; ++i)
          if (k + i < K) t[i >> 2] |= (uint32_t)(uint8_t)wr[k + i] << (8 * (i & 3));
        v = i32x4{(int)t[0], (int)t[1], (int)t[2], (int)t[3]};
      }
    } else {
      v = i32x4{0, 0, 0, 0};
    }
  };
  // ---- stage x (and the per-group scales of this workgroup's rows).
  // Order of issue: the x chunks (and scales) of this thread first, then the
  // first 2U weight blocks, then the LDS stores.  Vector loads return in
  // order, so the stores wait only for the short x reads, while the weight
  // stream, the only HBM traffic, is already in flight across the barrier.
  constexpr int XR = 4;  // x chunks (8 halves each) per thread held in registers
  constexpr int SR = 4;  // per-group scales per thread held in registers
  const int nchunk = kp / 8;
  auto load_x = [&](int e) -> i32x4 {
    const int k = 8 * e;
    if (VEC == kFull || (k + 8 <= K && (((uintptr_t)(x + k) & 15) == 0))) return ld16(x + k);
    uint32_t t[4] = {0u, 0u, 0u, 0u};
    for (int i = 0; i < 8; ++i)
      if (k + i < K) t[i >> 1] |= (uint32_t)x[k + i] << (16 * (i & 1));
    return i32x4{(int)t[0], (int)t[1], (int)t[2], (int)t[3]};
  };
  auto load_s = [&](int e) -> float {
    const int g = e / rows_per_wg, r = e % rows_per_wg;
    return (n0 + r < N) ? sw[(int64_t)g * N + n0 + r] : 0.0f;
  };
  i32x4 xr[XR];
  float sr[SR];
  if constexpr (XLDS) {
#pragma unroll
    for (int q = 0; q < XR; ++q) {
      const int e = tid + q * nthr;
      if (VEC == kFull)
        xr[q] = ld16(x + 8 * min(e, nchunk - 1));  // unconditional, stored only if e < nchunk
      else if (e < nchunk)
        xr[q] = load_x(e);
    }
  }
  if constexpr (PG) {
#pragma unroll
    for (int q = 0; q < SR; ++q) {
      const int e = tid + q * nthr;
      if (e < G * rows_per_wg) sr[q] = load_s(e);
    }
  }
  i32x4 wa[U], wb[U];
#pragma unroll
  for (int u = 0; u < U; ++u) load_w(u, wa[u]);
  // VEC loads are unconditional (a branch here lets the compiler sink them
  // past the staging barrier); the scalar path loads only what exists
  if (VEC != kBytes || U < nb) {
#pragma unroll
    for (int u = 0; u < U; ++u) load_w(U + u, wb[u]);
  }
  if constexpr (XLDS) {
#pragma unroll
    for (int q = 0; q < XR; ++q) {
      const int e = tid + q * nthr;
      if (e < nchunk) *reinterpret_cast<i32x4*>(xs + 8 * e) = xr[q];
    }
    for (int e = tid + XR * nthr; e < nchunk; e += nthr)
      *reinterpret_cast<i32x4*>(xs + 8 * e) = load_x(e);
  }
  if constexpr (PG) {
#pragma unroll
    for (int q = 0; q < SR; ++q) {
      const int e = tid + q * nthr;
      if (e < G * rows_per_wg) sws[e] = sr[q];
    }
    for (int e = tid + SR * nthr; e < G * rows_per_wg; e += nthr) sws[e] = load_s(e);
  }
  if (XLDS || PG) __syncthreads();

  float r0 = 0.0f, r1 = 0.0f;  // chains of reference lanes 2j and 2j+1
  auto consume = [&](int b0, const i32x4 (&wv)[U]) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (b0 + u >= nb) break;
      const int k = (b0 + u) * 256 + 16 * j;
      i32x4 xa, xb;
      if constexpr (XLDS) {
        xa = *reinterpret_cast<const i32x4*>(xs + k);
        xb = *reinterpret_cast<const i32x4*>(xs + k + 8);
      } else {
        uint32_t t[8] = {0u, 0u, 0u, 0u, 0u, 0u, 0u, 0u};
        for (int i = 0; i < 16; ++i)
          if (k + i < K) t[i >> 1] |= (uint32_t)x[k + i] << (16 * (i & 1));
        xa = i32x4{(int)t[0], (int)t[1], (int)t[2], (int)t[3]};
        xb = i32x4{(int)t[4], (int)t[5], (int)t[6], (int)t[7]};
      }
      const float d0 = dot8((uint32_t)wv[u][0], (uint32_t)wv[u][1], (uint32_t)xa[0],
                            (uint32_t)xa[1], (uint32_t)xa[2], (uint32_t)xa[3]);
      const float d1 = dot8((uint32_t)wv[u][2], (uint32_t)wv[u][3], (uint32_t)xb[0],
                            (uint32_t)xb[1], (uint32_t)xb[2], (uint32_t)xb[3]);
      if constexpr (PG) {
        // reference lanes past K (d == 0) use the last group's scale, as the
        // padded blocks of the reference would; never an index past G
        const int g0 = min(k / gs, G - 1), g1 = min((k + 8) / gs, G - 1);
        const float t0 = sws[g0 * rows_per_wg + row_in_wg] * d0;
        const float t1 = sws[g1 * rows_per_wg + row_in_wg] * d1;
        r0 = r0 + t0;
        r1 = r1 + t1;
      } else {
        r0 = r0 + d0;
        r1 = r1 + d1;
      }
    }
  };
  // two register buffers: while one set of U blocks reduces, the other loads
  for (int b = 0; b < nb; b += 2 * U) {
    consume(b, wa);
    if (b + U >= nb) break;
    if (b + 2 * U < nb) {
#pragma unroll
      for (int u = 0; u < U; ++u) load_w(b + 2 * U + u, wa[u]);
    }
    consume(b + U, wb);
    if (b + 3 * U < nb) {
#pragma unroll
      for (int u = 0; u < U; ++u) load_w(b + 3 * U + u, wb[u]);
    }
  }
  // butterfly over reference lanes: offsets 16, 8, 4, 2 are physical 8, 4, 2, 1
#pragma unroll
  for (int off = 8; off >= 1; off >>= 1) {
    r0 = r0 + __shfl_xor(r0, off, kLanesPerRow);
    r1 = r1 + __shfl_xor(r1, off, kLanesPerRow);
  }
  const float R = r0 + r1;  // offset 1
  if (j == 0 && live) {
    float v;
    if constexpr (PG) {
      v = bias ? R + h2f(bias[n]) : R;
    } else {
      v = sw[n] * R;
      if (bias) v = v + h2f(bias[n]);
    }
    y[n] = f2h(v);
  }
}

// ---------------------------------------------------------------------------
// Wide-row variant for full blocks (K % 256 == 0, K <= kMaxF32K, aligned):
// one physical lane per reference lane (32 lanes per row, two rows per wave),
// so each block costs a lane one 8-byte weight load, and the grid has twice
// the waves of the 16-lane layout (more weight bytes in flight on short-N
// shapes).  x is staged in LDS as fp32, converted once per workgroup, which
// leaves three VALU operations per weight element (byte -> f32, multiply,
// add) in the loop.  Same reduction order as mv_kernel and the reference:
// lane l's chain over blocks, then the xor butterfly 16, 8, 4, 2, 1.
// ---------------------------------------------------------------------------
constexpr int kMaxF32K = 16384;  // fp32 x in LDS up to 64 KB

__device__ __forceinline__ float dot8f(uint32_t w0, uint32_t w1, const f32x4& xa,
                                       const f32x4& xb) {
  float d = (float)(int8_t)(w0 & 0xffu) * xa[0];
  d = d + (float)(int8_t)((w0 >> 8) & 0xffu) * xa[1];
  d = d + (float)(int8_t)((w0 >> 16) & 0xffu) * xa[2];
  d = d + (float)(int8_t)(w0 >> 24) * xa[3];
  d = d + (float)(int8_t)(w1 & 0xffu) * xb[0];
  d = d + (float)(int8_t)((w1 >> 8) & 0xffu) * xb[1];
  d = d + (float)(int8_t)((w1 >> 16) & 0xffu) * xb[2];
  d = d + (float)(int8_t)(w1 >> 24) * xb[3];
  return d;
}

// Producer run inside the x staging of the M == 1 linear (XM):
//   XM_PLAIN   x is the fp16 input row;
//   XM_NORM    x' = RMSNorm(x) with weight nw (fused.hip's rmsnorm order);
//   XM_ADDNORM h = x + add (fp16), written to hsum by workgroup 0, x' = RMSNorm(h);
//   XM_SWIGLU  x is a [gate | up] row of 2K, x' = h(h(silu(gate)) * up).
// Thread t stages the 8-element chunks t, t + 256, ... as the producer
// kernels do (the RMSNorm sum of squares in that order, then block_sum4), so
// x' is bit-identical to what the producer kernel writes.
template <bool PG, int U, int XM = XM_PLAIN>
__global__ __launch_bounds__(256) void mv_wide_kernel(
    const uint16_t* __restrict__ x, const int8_t* __restrict__ w,
    const float* __restrict__ sw, const uint16_t* __restrict__ bias,
    uint16_t* __restrict__ y, int N, int K, int gs, MvProducer pp) {
  constexpr int kRows = 8;  // rows per workgroup: 2 per wave
  extern __shared__ __attribute__((aligned(16))) uint8_t dyn[];
  float* xs = reinterpret_cast<float*>(dyn);
  const int nb = K >> 8;
  const int G = PG ? K / gs : 0;
  float* sws = xs + K;  // per-group scales [G][kRows]

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rl = lane & 31;                 // reference lane
  const int row_in_wg = wave * 2 + (lane >> 5);
  const int n0 = blockIdx.x * kRows;
  const int n = n0 + row_in_wg;
  const bool live = n < N;
  const int8_t* wr = w + (int64_t)(live ? n : 0) * K + 8 * rl;

  // branch-free: a block past the end re-reads the last one (never consumed)
  auto load_w = [&](int b) -> i32x2 { return ld8_nt(wr + (int64_t)min(b, nb - 1) * 256); };

  // ---- stage x as fp32 (and the group scales); x reads first, then the
  // first 2U weight blocks, then the conversions and LDS stores
  // fused modes hold the whole row: ceil(K / 2048) chunks per thread (U <= 4:
  // K <= 2048; U <= 8: K <= 4096; U <= 12: K <= 6144; U == 16: K <= 16384)
  constexpr int XR = XM == XM_PLAIN ? 4 : (U <= 4 ? 1 : U <= 8 ? 2 : U <= 12 ? 3 : 8);
  const int nchunk = K >> 3;
  i32x4 xr[XR];
  float ss = 0.0f;  // XM_NORM / XM_ADDNORM: the sum of squares of this thread's chunks
#pragma unroll
  for (int q = 0; q < XR; ++q) {
    const int e = min(tid + q * 256, nchunk - 1);
    if constexpr (XM == XM_SWIGLU) {
      xr[q] = swiglu8(ld16(x + 8 * e), ld16(x + K + 8 * e));
    } else {
      xr[q] = ld16(x + 8 * e);
      if constexpr (XM == XM_ADDNORM) xr[q] = add8(xr[q], ld16(pp.add + 8 * e));
    }
  }
  constexpr int SR = 4;
  float sr[SR];
  auto load_s = [&](int e) -> float {
    const int g = e / kRows, r = e % kRows;
    return (n0 + r < N) ? sw[(int64_t)g * N + n0 + r] : 0.0f;
  };
  if constexpr (PG) {
#pragma unroll
    for (int q = 0; q < SR; ++q) {
      const int e = tid + q * 256;
      if (e < G * kRows) sr[q] = load_s(e);
    }
  }
  i32x2 wa[U], wb[U];
#pragma unroll
  for (int u = 0; u < U; ++u) wa[u] = load_w(u);
#pragma unroll
  for (int u = 0; u < U; ++u) wb[u] = load_w(U + u);

  if constexpr (XM == XM_NORM || XM == XM_ADDNORM) {
    // whole row in registers (XR * 256 chunks cover K <= 16384): the sum of
    // squares in chunk order, h written out once, then the normalisation
#pragma unroll
    for (int q = 0; q < XR; ++q) {
      const int e = tid + q * 256;
      if (e < nchunk) {
        if constexpr (XM == XM_ADDNORM)
          if (blockIdx.x == 0) *reinterpret_cast<i32x4*>(pp.hsum + 8 * e) = xr[q];
        ss = sumsq8(xr[q], ss);
      }
    }
    __shared__ float red[4];
    ss = block_sum4(ss, red);
    const float r = 1.0f / sqrtf(ss / (float)K + pp.eps);
#pragma unroll
    for (int q = 0; q < XR; ++q) {
      const int e = tid + q * 256;
      if (e < nchunk) xr[q] = norm8(xr[q], ld16(pp.nw + 8 * e), r);
    }
  }
  auto store_x = [&](int e, i32x4 v) {
    f32x4 lo, hi;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      lo[2 * i] = h2f((uint16_t)((uint32_t)v[i] & 0xffffu));
      lo[2 * i + 1] = h2f((uint16_t)((uint32_t)v[i] >> 16));
      hi[2 * i] = h2f((uint16_t)((uint32_t)v[2 + i] & 0xffffu));
      hi[2 * i + 1] = h2f((uint16_t)((uint32_t)v[2 + i] >> 16));
    }
    *reinterpret_cast<f32x4*>(xs + 8 * e) = lo;
    *reinterpret_cast<f32x4*>(xs + 8 * e + 4) = hi;
  };
#pragma unroll
  for (int q = 0; q < XR; ++q) {
    const int e = tid + q * 256;
    if (e < nchunk) store_x(e, xr[q]);
  }
  if constexpr (XM == XM_PLAIN)
    for (int e = tid + XR * 256; e < nchunk; e += 256) store_x(e, ld16(x + 8 * e));
  if constexpr (PG) {
#pragma unroll
    for (int q = 0; q < SR; ++q) {
      const int e = tid + q * 256;
      if (e < G * kRows) sws[e] = sr[q];
    }
    for (int e = tid + SR * 256; e < G * kRows; e += 256) sws[e] = load_s(e);
  }
  __syncthreads();

  float r = 0.0f;  // the chain of reference lane rl
  auto consume = [&](int b0, const i32x2 (&wv)[U]) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (b0 + u >= nb) break;
      const int k = (b0 + u) * 256 + 8 * rl;
      const f32x4 xa = *reinterpret_cast<const f32x4*>(xs + k);
      const f32x4 xb = *reinterpret_cast<const f32x4*>(xs + k + 4);
      const float d = dot8f((uint32_t)wv[u][0], (uint32_t)wv[u][1], xa, xb);
      if constexpr (PG) {
        const float t = sws[(k / gs) * kRows + row_in_wg] * d;
        r = r + t;
      } else {
        r = r + d;
      }
    }
  };
  for (int b = 0; b < nb; b += 2 * U) {
    consume(b, wa);
    if (b + U >= nb) break;
    if (b + 2 * U < nb) {
#pragma unroll
      for (int u = 0; u < U; ++u) wa[u] = load_w(b + 2 * U + u);
    }
    consume(b + U, wb);
    if (b + 3 * U < nb) {
#pragma unroll
      for (int u = 0; u < U; ++u) wb[u] = load_w(b + 3 * U + u);
    }
  }
#pragma unroll
  for (int off = 16; off >= 1; off >>= 1) r = r + __shfl_xor(r, off, 32);
  if (rl == 0 && live) {
    float v;
    if constexpr (PG) {
      v = bias ? r + h2f(bias[n]) : r;
    } else {
      v = sw[n] * r;
      if (bias) v = v + h2f(bias[n]);
    }
    y[n] = f2h(v);
  }
}

namespace {

constexpr int kMaxLdsK = 32768;  // x staged in LDS up to 64 KB

template <bool PG, bool XLDS, int U>
hipError_t run_mv(const uint16_t* x, const int8_t* w, const float* sw, const uint16_t* bias,
                  uint16_t* y, int N, int K, int gs, int vec, int rows, size_t lds,
                  hipStream_t s) {
  const dim3 grid((N + rows - 1) / rows), block(rows * kLanesPerRow);
  if (vec == kFull) {
    mv_kernel<PG, kFull, XLDS, U><<<grid, block, lds, s>>>(x, w, sw, bias, y, N, K, gs, rows);
    return hipGetLastError();
  }
  if constexpr (XLDS) {
    if (vec == kChunks) {
      mv_kernel<PG, kChunks, XLDS, U><<<grid, block, lds, s>>>(x, w, sw, bias, y, N, K, gs, rows);
      return hipGetLastError();
    }
  }
  mv_kernel<PG, kBytes, XLDS, U><<<grid, block, lds, s>>>(x, w, sw, bias, y, N, K, gs, rows);
  return hipGetLastError();
}

template <bool PG, bool XLDS>
hipError_t pick_u(const uint16_t* x, const int8_t* w, const float* sw, const uint16_t* bias,
                  uint16_t* y, int N, int K, int gs, int vec, int rows, size_t lds,
                  hipStream_t s) {
  // the prologue requests 2U blocks: U = ceil(nb / 2) up to 8 puts the whole
  // row of a short-K shape in flight at once with no redundant loads
  const int nb = (K + 255) / 256;
  if (nb <= 8) return run_mv<PG, XLDS, 4>(x, w, sw, bias, y, N, K, gs, vec, rows, lds, s);
  if (nb <= 10) return run_mv<PG, XLDS, 5>(x, w, sw, bias, y, N, K, gs, vec, rows, lds, s);
  if (nb <= 12) return run_mv<PG, XLDS, 6>(x, w, sw, bias, y, N, K, gs, vec, rows, lds, s);
  return run_mv<PG, XLDS, 8>(x, w, sw, bias, y, N, K, gs, vec, rows, lds, s);
}

}  // namespace

namespace {

template <bool PG, int U, int XM = XM_PLAIN>
hipError_t run_wide(const uint16_t* x, const int8_t* w, const float* sw, const uint16_t* bias,
                    uint16_t* y, int N, int K, int gs, size_t lds, hipStream_t s,
                    const MvProducer& pp = MvProducer{}) {
  mv_wide_kernel<PG, U, XM><<<(N + 7) / 8, 256, lds, s>>>(x, w, sw, bias, y, N, K, gs, pp);
  return hipGetLastError();
}

template <bool PG>
hipError_t pick_wide(const uint16_t* x, const int8_t* w, const float* sw, const uint16_t* bias,
                     uint16_t* y, int N, int K, int gs, size_t lds, hipStream_t s) {
  const int nb = K >> 8;
  if (nb <= 8) return run_wide<PG, 4>(x, w, sw, bias, y, N, K, gs, lds, s);
  if (nb <= 10) return run_wide<PG, 5>(x, w, sw, bias, y, N, K, gs, lds, s);
  if (nb <= 12) return run_wide<PG, 6>(x, w, sw, bias, y, N, K, gs, lds, s);
  if (nb <= 16) return run_wide<PG, 8>(x, w, sw, bias, y, N, K, gs, lds, s);
  if (nb <= 24) return run_wide<PG, 12>(x, w, sw, bias, y, N, K, gs, lds, s);
  return run_wide<PG, 16>(x, w, sw, bias, y, N, K, gs, lds, s);
}

}  // namespace

namespace {

template <int XM>
hipError_t pick_producer(const uint16_t* x, const int8_t* w, const float* sw,
                         const uint16_t* bias, uint16_t* y, int N, int K, size_t lds,
                         hipStream_t s, const MvProducer& pp) {
  const int nb = K >> 8;
  if (nb <= 8) return run_wide<false, 4, XM>(x, w, sw, bias, y, N, K, 0, lds, s, pp);
  if (nb <= 10) return run_wide<false, 5, XM>(x, w, sw, bias, y, N, K, 0, lds, s, pp);
  if (nb <= 12) return run_wide<false, 6, XM>(x, w, sw, bias, y, N, K, 0, lds, s, pp);
  if (nb <= 16) return run_wide<false, 8, XM>(x, w, sw, bias, y, N, K, 0, lds, s, pp);
  if (nb <= 24) return run_wide<false, 12, XM>(x, w, sw, bias, y, N, K, 0, lds, s, pp);
  return run_wide<false, 16, XM>(x, w, sw, bias, y, N, K, 0, lds, s, pp);
}

}  // namespace

bool mv_producer_supported(const void* x, const void* w, int K) {
  return K % 256 == 0 && K <= kMaxF32K && (((uintptr_t)w & 15) == 0) &&
         (((uintptr_t)x & 15) == 0);
}

hipError_t launch_mv_producer(int xm, const uint16_t* x, const uint16_t* add, uint16_t* hsum,
                              const uint16_t* nw, float eps, const int8_t* w, const float* sw,
                              const uint16_t* bias, uint16_t* y, int N, int K, hipStream_t s) {
  MvProducer pp;
  pp.add = add;
  pp.hsum = hsum;
  pp.nw = nw;
  pp.eps = eps;
  // the same kernel choice as launch_mv, so a fused launch equals the
  // producer launch followed by launch_mv bit for bit
  if (mv_stream_supported(x, w, sw, K, 0))
    return launch_mv_stream(xm, x, w, sw, bias, y, N, K, 0, pp, s);
  const size_t lds = (size_t)K * sizeof(float);
  switch (xm) {
    case XM_NORM: return pick_producer<XM_NORM>(x, w, sw, bias, y, N, K, lds, s, pp);
    case XM_ADDNORM: return pick_producer<XM_ADDNORM>(x, w, sw, bias, y, N, K, lds, s, pp);
    case XM_SWIGLU: return pick_producer<XM_SWIGLU>(x, w, sw, bias, y, N, K, lds, s, pp);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_mv(const uint16_t* x, const int8_t* w, const float* sw,
                     const uint16_t* bias, uint16_t* y, int N, int K, int gs,
                     hipStream_t s, bool bf) {
  if (mv_stream_supported(x, w, sw, K, gs)) {
    MvProducer pp;
    pp.bf16 = bf;
    return launch_mv_stream(XM_PLAIN, x, w, sw, bias, y, N, K, gs, pp, s);
  }
  if (bf) return hipErrorNotSupported;
  return launch_mv_lanes(x, w, sw, bias, y, N, K, gs, s);
}

hipError_t launch_mv_lanes(const uint16_t* x, const int8_t* w, const float* sw,
                           const uint16_t* bias, uint16_t* y, int N, int K, int gs,
                           hipStream_t s) {
  if (K % 256 == 0 && K <= kMaxF32K && (((uintptr_t)w & 15) == 0) &&
      (((uintptr_t)x & 15) == 0)) {
    const int G = gs > 0 ? K / gs : 0;
    const size_t lds = (size_t)K * sizeof(float) + (size_t)G * 8 * sizeof(float);
    if (gs > 0) return pick_wide<true>(x, w, sw, bias, y, N, K, gs, lds, s);
    return pick_wide<false>(x, w, sw, bias, y, N, K, gs, lds, s);
  }
  // Rows per workgroup: 16 (4 waves) when N is large, down to 4 (one wave)
  // so that short-N shapes still launch >= 512 workgroups.
  int rows = 16;
  while (rows > 4 && (N + rows - 1) / rows < 512) rows >>= 1;
  const int nb = (K + 255) / 256;
  const bool xlds = K <= kMaxLdsK;
  const int G = gs > 0 ? K / gs : 0;
  const size_t lds = (xlds ? (size_t)nb * 256 * 2 : 0) + (size_t)G * rows * sizeof(float);
  if (lds > 160 * 1024) return hipErrorInvalidValue;
  const bool wal = ((uintptr_t)w & 15) == 0;
  const int vec = K % 256 == 0 && wal && ((uintptr_t)x & 15) == 0 ? kFull
                  : K % 16 == 0 && K > 0 && wal && xlds           ? kChunks
                                                                  : kBytes;
  if (gs > 0) {
    if (xlds) return pick_u<true, true>(x, w, sw, bias, y, N, K, gs, vec, rows, lds, s);
    return pick_u<true, false>(x, w, sw, bias, y, N, K, gs, vec, rows, lds, s);
  }
  if (xlds) return pick_u<false, true>(x, w, sw, bias, y, N, K, gs, vec, rows, lds, s);
  return pick_u<false, false>(x, w, sw, bias, y, N, K, gs, vec, rows, lds, s);
}

}  // namespace cider
