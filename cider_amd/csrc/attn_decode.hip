// Single-query (decode) attention over a KV cache, grouped-query heads.
//
//   for query head h = j * G + r of KV head j (G = H / KV):
//     s_t = scale * sum_d f32(q[h,d]) * f32(K[j,t,d])        t < n
//     o   = sum_t softmax(s)_t * f32(V[j,t,d])               -> fp16 [H, D]
// with both caches [KV, T, D] (position-major, 256 bytes per position); n,
// the number of valid positions, is read from device memory so a captured
// decode step replays unchanged while the sequence grows.  All arithmetic is
// fp32 with one rounding per operation, each sum in ascending order (the
// reference's models call MLX's fused SDPA here, whose accumulation order is
// not specified; parity is against an fp32 softmax attention, within a
// tolerance).
//
// MI355X design (split-K "flash decoding"):
//   * the cache is cut into chunks of 128 positions; workgroup (chunk c, KV
//     head j) computes, for all G query heads of j at once, the chunk's
//     scores, its max m_c, sum l_c and unnormalised output o_c (fp32) and
//     writes them to a workspace; a second kernel merges the chunks with the
//     usual max-rescaling.  Each K / V byte is read once for all G heads.
//   * scores: a thread owns 4 consecutive positions and 8 of the 128
//     dimensions (one 16-byte K load per position); the 16 dimension slices
//     are summed through LDS.
//   * P.V: a thread owns 4 dimensions (one 8-byte V load per position) and
//     8 positions; the 16 position slices are summed through LDS.
//   * What bounds a chunk once its loads are in is VALU issue, so both products
//     take as few operations as their roundings allow: v_fma_mix_f32 widens its
//     fp16 operands in place.  A score's term is one of them (the product of two
//     fp16 is exact in fp32, so the fused add rounds as a multiply and an add
//     do); a term of P.V is one for the rounded product and an add.
//     v_dot2_f32_f16 and a fused P.V would be half the operations, in another
//     rounding: the logits of a whole model move by 0.5 %, and their error
//     against 64 bits from 0.00574 to 0.00596.
//   * eight waves, two per SIMD, issue them at twice the rate of four with the
//     same sums in the same order: Qwen3-8B-shaped decode step 2313 -> 2257 us
//     (2252 with four waves in that other rounding, 2545 before fma_mix), 32
//     heads at n = 2112 10.5 us (10.9, 11.9), at n = 32000 51.1 (50.4, 54.6).
//   * the grid covers the cache capacity T; chunks at or past n exit at once
//     (n is clamped to T).
//   * with more than 4 query heads per KV head, the heads are split over
//     several workgroups that each read that KV head's chunk.
#include "common.hpp"
#include "kernels.hpp"
#include "norm_common.hpp"

namespace cider {

namespace {

constexpr int kD = 128;      // head dimension
constexpr int kChunk = 128;  // positions per workgroup
constexpr int kThreads = 512;  // per workgroup

__device__ __forceinline__ float wave_max_f(float v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v = fmaxf(v, __shfl_xor(v, off));
  return v;
}

__device__ __forceinline__ float wave_sum_f(float v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v = v + __shfl_xor(v, off);
  return v;
}

// element i of a vector of fp16
template <typename V>
__device__ __forceinline__ float elem(V v, int i) {
  const uint32_t w = (uint32_t)v[i / 2];
  return h2f((uint16_t)(i & 1 ? w >> 16 : w & 0xffffu));
}

// The products of two vectors of 8 fp16 (exact in fp32), added in order.
__device__ __forceinline__ float dot8(i32x4 a, i32x4 b) {
  float s = 0.0f;
#pragma unroll
  for (int j = 0; j < 8; ++j) s = __builtin_fmaf(elem(a, j), elem(b, j), s);
  return s;
}

// A workgroup serves G query heads of one KV head (G <= 4: the LDS slices
// below hold G * 8 KB); R = (H / KV) / G workgroups share a KV head.
// workspace layout per (head block y, chunk c): G * (kD + 2) floats:
// o_c[G][kD], m_c[G], l_c[G]
//
// ROPE: q is the token's fused projection [q heads | k heads | v heads], and
// each workgroup norms and rotates its G query heads itself (eight lanes per
// head, the arithmetic of qk_norm_rope_kernel, so the same bits), from LDS; the
// workgroup whose chunk holds the token's slot does the same for the KV head's
// key, writes key and value to the caches and attends the values it computed
// instead of the cache rows it loaded meanwhile.  One launch less per layer; the
// loads of the projection run beside those of the chunk.
template <int G, int R, bool ROPE>
__global__ __launch_bounds__(kThreads) void attn_chunk_kernel(
    const uint16_t* __restrict__ q, uint16_t* kc, uint16_t* vc,
    const int64_t* __restrict__ n_ptr, float scale, float* __restrict__ ws, int64_t T, int nchunk,
    const DecodeRope rp) {
  __shared__ __attribute__((aligned(16))) uint16_t qs[G][kD];
  __shared__ float part[16][G][kChunk];  // dimension / position slices
  __shared__ float ps[G][kChunk];        // scores, then probabilities
  __shared__ float ml[G][2];

  const int c = blockIdx.x, y = blockIdx.y, j = y / R, tid = threadIdx.x;
  const int64_t nn = *n_ptr;
  const int64_t n = nn < T ? nn : T;
  const int64_t c0 = (int64_t)c * kChunk;
  const int64_t p = ROPE ? *rp.slot : -1;
  const bool mine = ROPE && p >= c0 && p < c0 + kChunk && p < T;
  // uniform: nothing of this chunk is valid (nor written)
  if (c0 >= n && !mine) return;
  [[maybe_unused]] __shared__ __attribute__((aligned(16))) uint16_t new_kv[2][kD];

  // Issue every load of the chunk first (K for the scores, V for P.V: neither
  // depends on the other), so the chunk costs one memory latency.  Positions
  // past n (within T) are loaded and never used; 8-position groups wholly
  // past n re-load group 0 of the chunk (always valid).
  const int tq = tid & 31, dq = tid >> 5;  // scores: 4 positions x 8 dimensions
  const int dv = tid & 31, ts = tid >> 5;  // P.V: 4 dimensions x 8 positions
  const int64_t tk0 = c0 + 4 * tq, tv0 = c0 + 8 * ts;
  i32x4 kv[4];
  i32x2 vv[8];
  {
    const uint16_t* kp = kc + ((int64_t)j * T + (tk0 < n ? tk0 : c0)) * kD + 8 * dq;
#pragma unroll
    for (int i = 0; i < 4; ++i) kv[i] = ld16(kp + (int64_t)i * kD);
    const uint16_t* vp = vc + ((int64_t)j * T + (tv0 < n ? tv0 : c0)) * kD + 4 * dv;
#pragma unroll
    for (int i = 0; i < 8; ++i) vv[i] = ld8(vp + (int64_t)i * kD);
  }
  if constexpr (ROPE) {
    // threads 8r .. 8r+7: query head r; 64 .. 71: the key; 128 .. 135: the value
    const int j8 = tid & 7, hr = tid >> 3;
    const bool is_q = hr < G, is_k = mine && hr == 8, is_v = mine && hr == 16;
    if (is_q || is_k || is_v) {
      const int KV = rp.KV, H = G * R * KV;
      const int hh = is_q ? y * G + hr : is_k ? H + j : H + KV + j;
      const uint16_t* src = q + (int64_t)hh * kD + 8 * j8;
      i32x4 o0 = ld16(src), o1 = ld16(src + 64);
      const int64_t rr = *rp.rope_row;
      const bool has_row = rr >= 0 && rr < rp.P;
      if (!is_v) {
        const int64_t rc = (has_row ? rr : 0) * kD + 8 * j8;
        const uint16_t* wn = (is_q ? rp.qw : rp.kw) + 8 * j8;
        const i32x4 x0 = o0, x1 = o1;
        norm_rope8(x0, x1, ld16(wn), ld16(wn + 64), ld16(rp.cos_t + rc), ld16(rp.cos_t + rc + 64),
                   ld16(rp.sin_t + rc), ld16(rp.sin_t + rc + 64), head_sumsq(x0, x1), rp.eps, o0,
                   o1);
      }
      if (is_q && !has_row) {  // as qk_norm_rope: quiet NaN
        o0 = i32x4{0x7E007E00, 0x7E007E00, 0x7E007E00, 0x7E007E00};
        o1 = o0;
      }
      uint16_t* const dst = is_q ? qs[hr] : new_kv[is_v];
      uint16_t* const row = (is_v ? vc : kc) + ((int64_t)j * T + p) * kD;
      if (is_k && !has_row) {  // no key is written: what the cache holds stays
        o0 = ld16(row + 8 * j8);
        o1 = ld16(row + 8 * j8 + 64);
      } else if (!is_q && y % R == 0) {
        *reinterpret_cast<i32x4*>(row + 8 * j8) = o0;
        *reinterpret_cast<i32x4*>(row + 8 * j8 + 64) = o1;
      }
      *reinterpret_cast<i32x4*>(dst + 8 * j8) = o0;
      *reinterpret_cast<i32x4*>(dst + 8 * j8 + 64) = o1;
    }
    __syncthreads();
    if (c0 >= n) return;  // uniform: only the write was due
    if (mine) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        if (i < 4 && tk0 + i == p) kv[i % 4] = *reinterpret_cast<const i32x4*>(&new_kv[0][8 * dq]);
        if (tv0 + i == p) vv[i] = *reinterpret_cast<const i32x2*>(&new_kv[1][4 * dv]);
      }
    }
  } else {
    for (int e = tid; e < G * kD / 8; e += kThreads)
      *reinterpret_cast<i32x4*>(&qs[0][8 * e]) = ld16(q + (int64_t)y * G * kD + 8 * e);
    __syncthreads();
  }

  // ---- scores: thread (dq, tq) sums dimensions 8dq..8dq+7 for positions
  // c0 + 4tq .. +3
  {
    const int64_t t0 = tk0;
    float acc[G][4];
#pragma unroll
    for (int r = 0; r < G; ++r) {
      const i32x4 qv = *reinterpret_cast<const i32x4*>(&qs[r][8 * dq]);
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[r][i] = t0 < n ? dot8(kv[i], qv) : 0.0f;
    }
#pragma unroll
    for (int r = 0; r < G; ++r)
#pragma unroll
      for (int i = 0; i < 4; ++i) part[dq][r][4 * tq + i] = acc[r][i];
  }
  __syncthreads();
  for (int e = tid; e < G * kChunk; e += kThreads) {
    const int r = e / kChunk, t = e % kChunk;
    float s = 0.0f;
#pragma unroll
    for (int dq = 0; dq < 16; ++dq) s = s + part[dq][r][t];
    ps[r][t] = (c0 + t < n) ? s * scale : -INFINITY;
  }
  __syncthreads();

  // ---- chunk softmax statistics: wave w handles head w
  {
    const int wave = tid >> 6, lane = tid & 63;
    for (int r = wave; r < G; r += kThreads / 64) {
      const float a = ps[r][lane], b = ps[r][lane + 64];
      const float m = wave_max_f(fmaxf(a, b));  // finite: position c0 < n is valid
      const float pa = expf(a - m), pb = expf(b - m);
      ps[r][lane] = pa;
      ps[r][lane + 64] = pb;
      const float l = wave_sum_f(pa + pb);
      if (lane == 0) {
        ml[r][0] = m;
        ml[r][1] = l;
      }
    }
  }
  __syncthreads();

  // ---- P.V: thread (ts, dv) sums positions 8ts..8ts+7 for dimensions
  // 4dv..4dv+3
  {
    float acc[G][4];
#pragma unroll
    for (int r = 0; r < G; ++r)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[r][i] = 0.0f;
    const int64_t t0 = tv0;
    if (t0 < n) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        if (t0 + i >= n) break;  // invalid positions may hold anything
#pragma unroll
        for (int r = 0; r < G; ++r) {
          const float p = ps[r][8 * ts + i];
#pragma unroll
          for (int d = 0; d < 4; ++d)  // the product rounded, then the sum
            acc[r][d] = acc[r][d] + __builtin_fmaf(p, elem(vv[i], d), 0.0f);
        }
      }
    }
    __syncthreads();  // every thread is done reading ps before part is reused
#pragma unroll
    for (int r = 0; r < G; ++r)
#pragma unroll
      for (int d = 0; d < 4; ++d) part[ts][r][4 * dv + d] = acc[r][d];
  }
  __syncthreads();
  float* out = ws + ((int64_t)y * nchunk + c) * G * (kD + 2);
  for (int e = tid; e < G * kD; e += kThreads) {
    const int r = e / kD, d = e % kD;
    float o = 0.0f;
#pragma unroll
    for (int ts = 0; ts < 16; ++ts) o = o + part[ts][r][d];
    out[e] = o;
  }
  if (tid < G) {
    out[G * kD + tid] = ml[tid][0];
    out[G * kD + G + tid] = ml[tid][1];
  }
}

// One wave per query head merges the chunks that hold valid positions: lane c
// reads chunk c's max and sum (64 chunks per pass), then every lane
// accumulates its two output dimensions over the chunks with the weights
// broadcast from the owning lane.
template <int G>
__global__ __launch_bounds__(64) void attn_merge_kernel(const float* __restrict__ ws,
                                                        const int64_t* __restrict__ n_ptr,
                                                        uint16_t* __restrict__ out, int nchunk,
                                                        int64_t T) {
  const int h = blockIdx.x, lane = threadIdx.x;
  const int j = h / G, r = h % G;  // j: head block
  const int64_t nn = *n_ptr;
  const int64_t n = nn < T ? nn : T;
  const int nc = (int)((n + kChunk - 1) / kChunk);
  const int last = nc < nchunk ? nc : nchunk;
  uint16_t* o = out + (int64_t)h * kD;
  if (last <= 0) {
    o[lane] = 0;
    o[lane + 64] = 0;
    return;
  }
  const float* base = ws + (int64_t)j * nchunk * G * (kD + 2);
  constexpr int kStride = G * (kD + 2);
  float m = -INFINITY;
  for (int c = lane; c < last; c += 64) m = fmaxf(m, base[(int64_t)c * kStride + G * kD + r]);
  m = wave_max_f(m);
  float l = 0.0f, a0 = 0.0f, a1 = 0.0f;
  for (int c0 = 0; c0 < last; c0 += 64) {
    const int c = c0 + lane;
    float f = 0.0f;
    if (c < last) {
      const float* p = base + (int64_t)c * kStride;
      f = expf(p[G * kD + r] - m);
      l = l + f * p[G * kD + G + r];
    }
    const int cnt = last - c0 < 64 ? last - c0 : 64;
    int i = 0;
    for (; i + 4 <= cnt; i += 4) {  // four chunks' loads in flight
      float fi[4], x0[4], x1[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const float* p = base + (int64_t)(c0 + i + u) * kStride + r * kD;
        fi[u] = __shfl(f, i + u);
        x0[u] = p[lane];
        x1[u] = p[lane + 64];
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        a0 = a0 + fi[u] * x0[u];
        a1 = a1 + fi[u] * x1[u];
      }
    }
    for (; i < cnt; ++i) {
      const float* p = base + (int64_t)(c0 + i) * kStride + r * kD;
      const float fi = __shfl(f, i);
      a0 = a0 + fi * p[lane];
      a1 = a1 + fi * p[lane + 64];
    }
  }
  l = wave_sum_f(l);
  o[lane] = f2h(a0 / l);
  o[lane + 64] = f2h(a1 / l);
}

template <int G, int R>
hipError_t run_attn(const uint16_t* q, uint16_t* kc, uint16_t* vc, const int64_t* n, float scale,
                    float* ws, uint16_t* out, int KV, int64_t T, const DecodeRope* rp,
                    hipStream_t s) {
  const int nchunk = (int)((T + kChunk - 1) / kChunk);
  const dim3 grid(nchunk, KV * R);
  if (rp)
    attn_chunk_kernel<G, R, true><<<grid, kThreads, 0, s>>>(q, kc, vc, n, scale, ws, T, nchunk, *rp);
  else
    attn_chunk_kernel<G, R, false><<<grid, kThreads, 0, s>>>(q, kc, vc, n, scale, ws, T, nchunk,
                                                         DecodeRope{});
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  attn_merge_kernel<G><<<KV * R * G, 64, 0, s>>>(ws, n, out, nchunk, T);
  return hipGetLastError();
}

}  // namespace

size_t attn_decode_ws_floats(int H, int64_t T) {
  const int64_t nchunk = (T + kChunk - 1) / kChunk;
  return (size_t)(nchunk * H * (kD + 2));
}

hipError_t launch_attn_decode(const uint16_t* q, const uint16_t* kc, const uint16_t* vc,
                              const int64_t* n, float scale, float* ws, uint16_t* out, int H,
                              int KV, int64_t T, hipStream_t s) {
  // written only with rotary arguments
  return launch_attn_decode_rope(q, const_cast<uint16_t*>(kc), const_cast<uint16_t*>(vc), n,
                                 scale, ws, out, H, KV, T, nullptr, s);
}

hipError_t launch_attn_decode_rope(const uint16_t* q, uint16_t* kc, uint16_t* vc,
                                   const int64_t* n, float scale, float* ws, uint16_t* out, int H,
                                   int KV, int64_t T, const DecodeRope* rp, hipStream_t s) {
  switch (H / KV) {
    case 1: return run_attn<1, 1>(q, kc, vc, n, scale, ws, out, KV, T, rp, s);
    case 2: return run_attn<2, 1>(q, kc, vc, n, scale, ws, out, KV, T, rp, s);
    case 4: return run_attn<4, 1>(q, kc, vc, n, scale, ws, out, KV, T, rp, s);
    case 8: return run_attn<4, 2>(q, kc, vc, n, scale, ws, out, KV, T, rp, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace cider
