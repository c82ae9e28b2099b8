// Per-token activation quantization (fp16 [M,K] -> int8 [M,K] + fp32 [M]).
//
// Semantics of cider/kernels/w8a8_quantize.metal:33-86:
//   amax = max_k |x[m,k]|        (fmax: NaN never wins)
//   s    = amax / 127, s == 0 -> 1
//   inv  = 1 / s
//   q    = clamp(round_half_away(x * inv), -128, 127)   (NaN -> -128)
//
// MI355X design: one 64-lane wavefront owns one row, so the absmax is a pure
// cross-lane reduction (no LDS, no barrier); a workgroup of 4 waves handles 4
// rows.  Up to 64 rows (decode-sized batches) get a 1024-thread workgroup per
// row instead, and rows of 2048 to 16384 elements a 256-thread one, except
// at M >= 2048 with rows of at most 3072 elements.  A row stays in registers between the absmax and the quantize pass
// (each element is read from HBM once); rows past 16384 elements are re-read,
// which hits in L2.
#include "common.hpp"
#include "kernels.hpp"
#include "quant_common.hpp"

namespace cider {

namespace {

// Vector e (8 elements) of a quantized row.  il = 32 or 16: every il consecutive
// elements are stored as those of even index, then those of odd index (K % il
// == 0), the orders the int4 GEMMs take (gemm_pp.hip 32, gemm_dma_pg.hip 16).
__device__ __forceinline__ void store_q8(int8_t* qr, int e, i32x2 v, int il) {
  if (!il) {
    *reinterpret_cast<i32x2*>(qr + 8 * e) = v;
    return;
  }
  const int m = il / 8 - 1, half = il / 2;  // vectors per block - 1, bytes of the evens
  int8_t* const d = qr + 8 * (e & ~m) + 4 * (e & m);
  *reinterpret_cast<int32_t*>(d) =
      (int32_t)__builtin_amdgcn_perm((uint32_t)v[1], (uint32_t)v[0], 0x06040200u);
  *reinterpret_cast<int32_t*>(d + half) =
      (int32_t)__builtin_amdgcn_perm((uint32_t)v[1], (uint32_t)v[0], 0x07050301u);
}

}  // namespace

// bf: x is bf16, rounded to fp16 first (three VALU operations per two
// elements, instead of a cast kernel that reads and writes x).  PLAIN: neither
// that nor another order; the common case does not test for them (5 x
// 12288 3.33 -> 3.23 us, 400 x 12288 4.69 -> 4.51, 4096 x 2560 6.77 -> 6.62).
//
// Vectorized rows: K % 8 == 0, x 16-byte and q 8-byte aligned.  NV > 0 keeps
// NV 16-byte vectors per lane in registers; NV == 0 streams the row twice.
template <int NV, bool PLAIN>
__global__ __launch_bounds__(256) void quantize_vec_kernel(
    const uint16_t* __restrict__ x, int8_t* __restrict__ q,
    float* __restrict__ sa, int M, int K, int il_, int bf_) {
  const int il = PLAIN ? 0 : il_;
  const bool bf = !PLAIN && bf_;
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= M) return;  // uniform per wave
  const uint16_t* xr = x + row * K;
  int8_t* qr = q + row * K;
  const int nvec = K >> 3;
  float amax = 0.0f;
  if constexpr (NV > 0) {
    // every load first, unconditional (clamped: a lane past the row re-reads
    // its last vector, which leaves the max unchanged), as a load under a
    // lane mask makes the compiler wait for each before the next: M=4096
    // K=2560 5.99 -> 5.79 us, M=2048 K=4096 5.37 -> 4.98 us (M=8192 level)
    i32x4 v[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) v[i] = ld16(xr + 8 * min(lane + i * kWave, nvec - 1));
    if (bf) {
#pragma unroll
      for (int i = 0; i < NV; ++i) v[i] = bf16x8_to_f16(v[i]);
    }
#pragma unroll
    for (int i = 0; i < NV; ++i) amax = absmax8(v[i], amax);
    amax = wave_max(amax);
    const float s = row_scale(amax);
    const float inv = 1.0f / s;
    if (lane == 0) sa[row] = s;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int e = lane + i * kWave;
      if (e < nvec) store_q8(qr, e, quant8(v[i], inv), il);
    }
  } else {
    auto ldv = [&](int e) {
      const i32x4 v = ld16(xr + 8 * e);
      return bf ? bf16x8_to_f16(v) : v;
    };
    for (int e = lane; e < nvec; e += kWave) amax = absmax8(ldv(e), amax);
    amax = wave_max(amax);
    const float s = row_scale(amax);
    const float inv = 1.0f / s;
    if (lane == 0) sa[row] = s;
    for (int e = lane; e < nvec; e += kWave)
      store_q8(qr, e, quant8(ldv(e), inv), il);
  }
}

// A workgroup of NT threads per row: few rows (M <= 64, NT = 1024: sixteen
// waves share a row's loads and conversions, where a single wave per row
// leaves the row's VALU work serial: about 8 us at K = 12288) and long rows
// (NT = 256); the absmax goes through LDS in wave order.  Vectorized rows
// only; NV 16-byte vectors per thread.
template <bool PLAIN, int NV, int NT = 1024>
__global__ __launch_bounds__(NT) void quantize_row_kernel(
    const uint16_t* __restrict__ x, int8_t* __restrict__ q,
    float* __restrict__ sa, int K, int il_, int bf_) {
  const int il = PLAIN ? 0 : il_;
  const bool bf = !PLAIN && bf_;
  constexpr int NWV = NT / 64;
  __shared__ float red[NWV];
  const int tid = threadIdx.x;
  const int64_t row = blockIdx.x;
  const uint16_t* xr = x + row * K;
  int8_t* qr = q + row * K;
  const int nvec = K >> 3;
  i32x4 v[NV];
  float amax = 0.0f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int e = tid + i * NT;
    v[i] = e < nvec ? ld16(xr + 8 * e) : i32x4{0, 0, 0, 0};
  }
  if (bf) {
#pragma unroll
    for (int i = 0; i < NV; ++i) v[i] = bf16x8_to_f16(v[i]);
  }
#pragma unroll
  for (int i = 0; i < NV; ++i) amax = absmax8(v[i], amax);
  amax = wave_max(amax);
  if ((tid & 63) == 0) red[tid >> 6] = amax;
  __syncthreads();
  amax = red[0];
#pragma unroll
  for (int w = 1; w < NWV; ++w) amax = fmaxf(amax, red[w]);
  const float s = row_scale(amax);
  const float inv = 1.0f / s;
  if (tid == 0) sa[row] = s;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int e = tid + i * NT;
    if (e < nvec) store_q8(qr, e, quant8(v[i], inv), il);
  }
}

// Any K and alignment: element-wise, two passes.  IL: the order store_q8 writes
// (K % IL == 0).  The type and the order are template arguments: with a test of the
// type in the loops the M=137 N=2560 K=10240 int4 linear on such x took 105 us, 93 so.
template <bool BF, int IL>
__global__ __launch_bounds__(256) void quantize_scalar_kernel(
    const uint16_t* __restrict__ x, int8_t* __restrict__ q,
    float* __restrict__ sa, int M, int K) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= M) return;
  const uint16_t* xr = x + row * K;
  int8_t* qr = q + row * K;
  auto ldx = [&](int k) {
    if constexpr (BF) return h2f(f2h(__builtin_bit_cast(float, (uint32_t)xr[k] << 16)));
    return h2f(xr[k]);
  };
  auto at = [](int k) {
    if constexpr (IL == 0) return k;
    return (k & ~(IL - 1)) + (k & 1) * (IL / 2) + ((k & (IL - 1)) >> 1);
  };
  float amax = 0.0f;
  for (int k = lane; k < K; k += kWave) amax = fmaxf(amax, fabsf(ldx(k)));
  amax = wave_max(amax);
  const float s = row_scale(amax);
  const float inv = 1.0f / s;
  if (lane == 0) sa[row] = s;
  for (int k = lane; k < K; k += kWave) qr[at(k)] = quant1(ldx(k), inv);
}

template <bool BF>
hipError_t run_scalar(const uint16_t* x, int8_t* q, float* sa, int M, int K, int il,
                      hipStream_t s) {
  const dim3 grid((M + 3) / 4), block(256);
  if (il == 0)
    quantize_scalar_kernel<BF, 0><<<grid, block, 0, s>>>(x, q, sa, M, K);
  else if (il == 16 && K % 16 == 0)
    quantize_scalar_kernel<BF, 16><<<grid, block, 0, s>>>(x, q, sa, M, K);
  else if (il == 32 && K % 32 == 0)
    quantize_scalar_kernel<BF, 32><<<grid, block, 0, s>>>(x, q, sa, M, K);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

template <bool PLAIN>
hipError_t run_vec(const uint16_t* x, int8_t* q, float* sa, int M, int K, int il, bool bf,
                   hipStream_t s) {
  const dim3 grid((M + 3) / 4), block(256);
  const int nvec = K >> 3;
  if (M <= 64 && nvec > 64 && nvec <= 8 * 1024) {
    // a row per 1024-thread workgroup (max(a, b) is exact, so the absmax does
    // not depend on how the row is split)
    if (nvec <= 1024)
      quantize_row_kernel<PLAIN, 1><<<M, 1024, 0, s>>>(x, q, sa, K, il, bf);
    else if (nvec <= 2048)
      quantize_row_kernel<PLAIN, 2><<<M, 1024, 0, s>>>(x, q, sa, K, il, bf);
    else if (nvec <= 4096)
      quantize_row_kernel<PLAIN, 4><<<M, 1024, 0, s>>>(x, q, sa, K, il, bf);
    else
      quantize_row_kernel<PLAIN, 8><<<M, 1024, 0, s>>>(x, q, sa, K, il, bf);
    return hipGetLastError();
  }
  const int per_lane = (nvec + kWave - 1) / kWave;
  // Many rows of up to 3072 elements: one wave per row, the row in at most 6
  // vectors per lane (4096 x 2560: 7.5 -> 6.4 us, 8192 x 2560: 13.0 -> 11.4
  // us, 4096 x 2048: 6.8 -> 5.4 us against the 256-thread row workgroups;
  // level at M <= 1024).
  const bool wave_rows = M >= 2048 && per_lane <= 6;
  if (!wave_rows && nvec >= 256 && nvec <= 8 * 256) {
    // Rows of 2048 .. 16384 elements at any M: a 256-thread workgroup per
    // row, its four waves' maxima meeting in LDS.  One wave per row held up
    // to 32 16-byte vectors per lane and ran at few waves per SIMD (4096 x
    // 10240: 36.3 -> 21.7 us; 4096 x 4096: 10.8 -> 9.7 us).
    const int nv = (nvec + 255) / 256;
    if (nv <= 2) quantize_row_kernel<PLAIN, 2, 256><<<M, 256, 0, s>>>(x, q, sa, K, il, bf);
    else if (nv <= 3) quantize_row_kernel<PLAIN, 3, 256><<<M, 256, 0, s>>>(x, q, sa, K, il, bf);
    else if (nv <= 4) quantize_row_kernel<PLAIN, 4, 256><<<M, 256, 0, s>>>(x, q, sa, K, il, bf);
    else if (nv <= 5) quantize_row_kernel<PLAIN, 5, 256><<<M, 256, 0, s>>>(x, q, sa, K, il, bf);
    else if (nv <= 6) quantize_row_kernel<PLAIN, 6, 256><<<M, 256, 0, s>>>(x, q, sa, K, il, bf);
    else quantize_row_kernel<PLAIN, 8, 256><<<M, 256, 0, s>>>(x, q, sa, K, il, bf);
    return hipGetLastError();
  }
  if (per_lane <= 1)
    quantize_vec_kernel<1, PLAIN><<<grid, block, 0, s>>>(x, q, sa, M, K, il, bf);
  else if (per_lane <= 2)
    quantize_vec_kernel<2, PLAIN><<<grid, block, 0, s>>>(x, q, sa, M, K, il, bf);
  else if (per_lane <= 4)
    quantize_vec_kernel<4, PLAIN><<<grid, block, 0, s>>>(x, q, sa, M, K, il, bf);
  else if (per_lane <= 5)
    quantize_vec_kernel<5, PLAIN><<<grid, block, 0, s>>>(x, q, sa, M, K, il, bf);
  else if (per_lane <= 6)
    quantize_vec_kernel<6, PLAIN><<<grid, block, 0, s>>>(x, q, sa, M, K, il, bf);
  else if (per_lane <= 8)
    quantize_vec_kernel<8, PLAIN><<<grid, block, 0, s>>>(x, q, sa, M, K, il, bf);
  else if (per_lane <= 16)
    quantize_vec_kernel<16, PLAIN><<<grid, block, 0, s>>>(x, q, sa, M, K, il, bf);
  else if (per_lane <= 32)
    quantize_vec_kernel<32, PLAIN><<<grid, block, 0, s>>>(x, q, sa, M, K, il, bf);
  else
    quantize_vec_kernel<0, PLAIN><<<grid, block, 0, s>>>(x, q, sa, M, K, il, bf);
  return hipGetLastError();
}

hipError_t launch_quantize(const uint16_t* x, int8_t* q, float* sa, int M,
                           int K, hipStream_t s, int il, bool bf) {
  const bool vec = (K % 8 == 0) && (((uintptr_t)x & 15) == 0) &&
                   (((uintptr_t)q & 7) == 0);
  if (!vec)
    return bf ? run_scalar<true>(x, q, sa, M, K, il, s) : run_scalar<false>(x, q, sa, M, K, il, s);
  return il || bf ? run_vec<false>(x, q, sa, M, K, il, bf, s)
                  : run_vec<true>(x, q, sa, M, K, 0, false, s);
}

}  // namespace cider
