// Persistent ping-pong int8 GEMM, the main path for M > 64 or so: int8 weights
// (int32 and per-channel epilogues) and int4 weights (per-channel, the
// reference W4A8), K % 128 == 0, N % 8 == 0 and >= 256.
//
// Reference semantics are those of gemm.hip (same epilogues, same fp32
// operation order, bit-identical results):
//   EPI_I32 cider/kernels/w8a8_matmul.metal:301-453
//   EPI_PC  cider/kernels/w8a8_matmul.metal:63-81
//   int4    cider/kernels/w4a8_matmul.metal:47-89,189-246 (no bias)
//
// What bounds it: power.  Under a random int8 load the part lowers its clock
// until the chip fits its power limit, so what counts is energy per product.
// M=8192 N=10240 K=2560: the MFMAs are busy 62 % of the cycles at 2.00 GHz
// (the 32x32x32 tiles of gemm_dma.hip that this kernel replaced: 58 % at 1.90
// GHz); v_mfma_i32_16x16x64_i8 alone, all operands in registers, holds 2.00
// GHz.  Kernel times before and after, same box, outputs bit-identical:
//   M=4096 N=10240 K=2560   100.4 ->  93.3 us (2301 TOPS)
//   M=8192 N=10240 K=2560   196   -> 169   us (2540 TOPS)
//   M=2048 N=24576 K=4096   174   -> 152   us (2717 TOPS)
//   M=2048 N=4096  K=12288   92   ->  81   us
//   M=4096 N=2560  K=10240   99   ->  87   us
//
// Design
//   * A workgroup of 8 waves, one per CU, computes BM x 256 tiles, BM = 64 MB
//     for MB = 1 .. 4.  Wave (wr, wc), wr = wave / 4: columns [64 wc, +64),
//     and rows [16 MB wr, +16 MB) of each half of the tile's rows, as 4 x 2 MB
//     blocks of v_mfma_i32_16x16x64_i8, weights as the A operand.
//   * Ping-pong: waves w and w + 4 share a SIMD, and the set wr = 1 runs one
//     barrier behind the set wr = 0 (one extra s_barrier at the start; the set
//     0 pays it at the end).  A 128-k stage is two phases, A (upper rows) and
//     B (lower rows), each a load slot (fragment reads, DMA issue, waits) and
//     an MFMA slot (8 MB MFMAs back to back) between barriers; so one wave of
//     a SIMD loads while the other multiplies.  The same loop without the
//     extra barrier, both sets in step: M=8192 N=10240 203 us against 179.
//   * The ring holds two stages of 64 KB (W rows, then X rows).  Load slot A(t)
//     reads W(t), and issues the upper X rows of stage t+2 and the lower X
//     rows of t+1; B(t) reads the lower X rows of t and the upper ones of
//     t+1, and issues W(t+2).  A slot's reads are complete (lgkmcnt 0) before
//     its barrier, so what slot p read may be overwritten from slot p+1 on by
//     either set, and what slot p reads was issued three slots (6 barriers)
//     before, each wave waiting for its own loads (vmcnt, in order) one
//     barrier earlier.
//   * Persistent: workgroup g takes tiles g, g + 256, ..  The load cursor runs
//     two stages ahead across tile boundaries, so the next tile's operands and
//     scales land while this tile's epilogue runs (no prologue per tile: 181
//     -> 174 us at M=8192), and the epilogue stores straight from registers,
//     so it never waits for LDS.
//   * MFMA A block a takes tile columns 64 wc + 32 (a / 2) + 8 g + 4 (a % 2) +
//     r (g = lane / 16): a lane then holds 8 consecutive columns per block
//     pair, one 16-byte store, and four lanes one 64-byte piece of a row.
//   * The order of the MFMAs is serpentine: consecutive ones share an operand
//     also where the other one changes row, which toggles fewer bits (171.3 ->
//     169.1 us at M=8192, 153.0 -> 151.3 us at M=4096 N=12288 K=4096).
//   * Tiles at the lower and right edge are moved inside (their first row or
//     column min(m0, M - BM)), so no load or store needs a bound; the rows or
//     columns two tiles then share get the same values from both.
//   * LDS rows are 128 bytes, 16-byte chunks XOR-swizzled so that the 16 lanes
//     LDS serves together hit 16 distinct bank groups; the DMA lane picks the
//     global chunk of the slot it writes (SQ_LDS_BANK_CONFLICT 0).
//   * int4 weights: x comes with every 32 consecutive k reordered (the 16 even
//     ones, then the 16 odd ones; launch_quantize writes it so).  A lane's 16
//     bytes of nibbles then unpack by (w << 4) & 0xF0.. and w & 0xF0.. into the
//     operands of two MFMAs, 3 VALU operations per 8 weights instead of 19, as
//     16 times the weight; the factor 16 leaves with sa / 16 (exact: powers of
//     two, sa >= 2^-24 / 127 stays normal), so the fp32 products are the same.
#include "common.hpp"
#include "dma_common.hpp"
#include "kernels.hpp"

#include <type_traits>

namespace cider {

namespace {

constexpr int kStageBytes = 64 * 1024;   // W 32 KB (int4: 16), X up to 32 KB
constexpr int kXBase = 32 * 1024;
constexpr int kSclBytes = 3 * 1024;      // sw 1 KB, bias 512 B (1 KB written), sa 1 KB
// Scale buffers: the cursor is two stages ahead and takes a tile's scales as it
// reaches the tile, before the epilogue of the one being computed: at K = 128,
// one stage per tile, four tiles' scales are held at once.
constexpr int kSclBufs = 4;
constexpr int kPpSmem = 2 * kStageBytes + kSclBufs * kSclBytes;

__device__ __forceinline__ void pp_bar() { asm volatile("s_barrier" ::: "memory"); }
__device__ __forceinline__ void pp_lgkm0() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// W rows are read as r = 64 wc + 8 (i / 4) + i % 4 + (multiples of 4 and 32),
// i = lane % 16: chunk XOR for rows of 128 (64) bytes.
template <int WF>
__device__ __forceinline__ int swz_w(int r) {
  return WF == W_I4 ? (r >> 3) & 3 : ((r >> 1) & 1) | (((r >> 3) & 3) << 1);
}

// Tiles wg, wg + nwg, .. < ntiles of the region rows [m_lo, m_hi), columns
// [n_lo, n_hi) in BM x 256 tiles.  m_hi >= BM, n_hi >= 256.
struct PpRegion {
  int ntiles, m_lo, m_hi, n_lo, n_hi;
};

template <int MB, int EPI, int WF>
__device__ __forceinline__ void pp_run(const GemmArgs& p, int8_t* __restrict__ smem, const int wg,
                                       const int nwg, const PpRegion& rg) {
  constexpr int BM = 64 * MB, BN = 256, BK = 128;
  constexpr bool W4 = WF == W_I4;
  constexpr int WB = W4 ? BK / 2 : BK;  // weight bytes per row and stage
  constexpr int WI = W4 ? 2 : 4;        // W DMA instructions per wave and stage
  constexpr int RPW = 1024 / WB;        // W rows per DMA instruction
  constexpr int STORES = EPI == EPI_I32 ? 8 * MB : 4 * MB;  // per wave and tile
  const int ntiles = rg.ntiles;
  if (wg >= ntiles) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = wave >> 2, wc = wave & 3;
  const int N = p.N, K = p.K, nk = K / BK;
  const int64_t ldw = W4 ? (K >> 1) : K;
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane(
      (uint32_t)(uintptr_t)(__attribute__((address_space(3))) int8_t*)smem);

  // DMA: a piece is 1 KB of consecutive LDS rows; piece i of this wave holds X
  // rows (8 i + wave) * 8 + [0, 8) and W rows (8 i + wave) * RPW + [0, RPW).
  // The swizzles do not change from one i to the next, so one lane offset
  // serves every piece and the scalar base advances.
  const int xrow = wave * 8 + (lane >> 3);
  const uint32_t xoff = (uint32_t)(xrow * K + (((lane & 7) ^ ((xrow >> 1) & 7)) << 4));
  constexpr int LPW = WB / 16;  // lanes per W row
  const int wrow = wave * RPW + lane / LPW;
  const uint32_t woff = (uint32_t)(wrow * (int)ldw + (((lane % LPW) ^ swz_w<WF>(wrow)) << 4));
  const int64_t xstep = (int64_t)64 * K, wstep = (int64_t)8 * RPW * ldw;

  // fragment reads
  const int lr = lane & 15, g = lane >> 4;
  const int fw = wc * 64 + 8 * (lr >> 2) + (lr & 3);
  const int fx = wr * 16 * MB + lr;
  const int sx = (lr >> 1) & 7, sw = swz_w<WF>(fw);
  // int8: k chunk 4 j + g of MFMA j; int4: one chunk g of nibbles for both
  // MFMAs, whose x are chunks 2 g + j
  int waddr0 = fw * WB + ((g ^ sw) << 4);
  int waddr1 = fw * WB + (((W4 ? g : 4 + g) ^ sw) << 4);
  int xaddr0 = kXBase + fx * BK + (((W4 ? 2 * g : g) ^ sx) << 4);
  int xaddr1 = kXBase + fx * BK + (((W4 ? 2 * g + 1 : 4 + g) ^ sx) << 4);
  i32x4 wf[2][4], x0[2][MB], x1[2][MB], acc[4][2 * MB];
  i32x4 raw[4];
  auto read_w = [&]() {
#pragma unroll
    for (int j = 0; j < (W4 ? 1 : 2); ++j)
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        const i32x4 v = *reinterpret_cast<const i32x4*>(smem + (j ? waddr1 : waddr0) +
                                                        ((a & 1) * 4 + (a >> 1) * 32) * WB);
        if constexpr (W4)
          raw[a] = v;
        else
          wf[j][a] = v;
      }
  };
  auto read_x = [&](int half, i32x4 (&x)[2][MB]) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int q = 0; q < MB; ++q)
        x[j][q] = *reinterpret_cast<const i32x4*>(smem + (j ? xaddr1 : xaddr0) +
                                                  half * (BM / 2) * BK + q * 16 * BK);
  };
  auto zero_acc = [&]() {
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int q = 0; q < 2 * MB; ++q) acc[a][q] = i32x4{0, 0, 0, 0};
  };

  auto coords = [&](int t, int& m0, int& n0) {
    int m, n;
    tile_coords<BM, BN>(xcd_remap(t, ntiles), rg.m_hi - rg.m_lo, rg.n_lo, rg.n_hi, m, n);
    m0 = __builtin_amdgcn_readfirstlane(min(rg.m_lo + m, rg.m_hi - BM));
    n0 = __builtin_amdgcn_readfirstlane(min(n, rg.n_hi - BN));
  };
  int m0, n0;  // the tile being computed
  coords(wg, m0, n0);

  // Load cursor: tile lt, stage lk; lx1 is the X pointer of the stage before.
  int lt = wg, lk = 0, lbuf = 0, lm0 = m0, ln0 = n0;
  const int8_t* const wp = reinterpret_cast<const int8_t*>(p.w);
  const int8_t* lw = wp + ln0 * ldw;
  const int8_t* lx = p.x + (int64_t)lm0 * K;
  const int8_t* lx1 = lx;
  // The scales of the cursor's tile, into the next scale buffer.  Extra loads of
  // some waves only make those waves' counted waits stricter.  A bias that is not
  // 16-byte aligned goes through registers, 4 elements per lane; the wait for it
  // drains wave 1's loads once per tile (M=4096 N=10240 K=2560 linear 95.6
  // us, on an aligned one 95.2; in LDS-DMA tiles 153).
  auto dma_scales = [&]() {
    if constexpr (EPI == EPI_PC) {
      const uint32_t sb =
          __builtin_amdgcn_readfirstlane(lds0 + 2 * kStageBytes + lbuf * kSclBytes);
      if (wave == 0) dma16s(reinterpret_cast<const float*>(p.sw) + ln0, lane * 16, sb);
      if (wave == 1 && p.bias) {
        if (W4 || ((uintptr_t)p.bias & 15) == 0) {
          dma16s(p.bias + ln0, (lane & 31) * 16, sb + 1024);
        } else {
          const uint16_t* const bp = p.bias + ln0 + 4 * lane;
          *reinterpret_cast<i32x2*>(smem + 2 * kStageBytes + lbuf * kSclBytes + 1024 + 8 * lane) =
              i32x2{(int)(bp[0] | (uint32_t)bp[1] << 16), (int)(bp[2] | (uint32_t)bp[3] << 16)};
        }
      }
      if (wave >= 4 && wave < 4 + MB)
        dma4s(p.sa + lm0, ((wave - 4) * 64 + lane) * 4, sb + 2048 + (wave - 4) * 256);
    }
  };
  // past the last stage of the last tile the cursor stays (reloads into slots
  // that nobody reads), so every slot issues the same loads
  auto advance = [&]() {
    lx1 = lx;
    if (lk + 1 < nk) {
      ++lk;
      lw += WB;
      lx += BK;
    } else if (lt + nwg < ntiles) {
      lt += nwg;
      lk = 0;
      lbuf = (lbuf + 1) % kSclBufs;
      coords(lt, lm0, ln0);
      lw = wp + ln0 * ldw;
      lx = p.x + (int64_t)lm0 * K;
      dma_scales();
    }
  };
  // the X pieces of one phase A: upper rows (the first BM / 16 pieces) of the
  // cursor's stage into buffer b, lower rows of the stage before into b ^ 1
  auto dma_x = [&](int b, bool upper_only) {
#pragma unroll
    for (int i = 0; i < MB; ++i) {
      const int piece = i * 8 + wave;
      const bool up = piece < BM / 16;
      if (upper_only && !up) continue;
      const uint32_t sb = __builtin_amdgcn_readfirstlane(
          lds0 + (uint32_t)((up ? b : b ^ 1) * kStageBytes) + kXBase + piece * 1024);
      dma16s((up ? lx : lx1) + i * xstep, xoff, sb);
    }
  };
  auto dma_w = [&](int b) {
#pragma unroll
    for (int i = 0; i < WI; ++i)
      dma16s(lw + i * wstep, woff,
             __builtin_amdgcn_readfirstlane(lds0 + (uint32_t)(b * kStageBytes) +
                                            (i * 8 + wave) * 1024));
  };

  // stage 0 whole but for its lower X rows, then as phases A(-1), B(-1) issue
  dma_scales();
  dma_x(0, true);
  dma_w(0);
  advance();
  dma_x(1, false);
  dma_w(1);
  advance();
  wait_vmcnt<WI + MB>();
  pp_bar();
  read_x(0, x0);
  pp_lgkm0();
  __builtin_amdgcn_sched_barrier(0);
  pp_bar();
  if (wr == 1) pp_bar();
  __builtin_amdgcn_sched_barrier(0);
  zero_acc();

  // End of a load slot: what the next slot reads was issued before the last
  // WI + MB loads.  In the first stage after an epilogue its stores are still
  // in flight and younger than those loads (lax).
  auto end_load = [&](bool lax) {
    if (lax)
      wait_vmcnt<WI + MB + STORES>();
    else
      wait_vmcnt<WI + MB>();
    pp_lgkm0();
    __builtin_amdgcn_sched_barrier(0);
    pp_bar();
    __builtin_amdgcn_sched_barrier(0);
  };
  auto mfmas = [&](auto halfc, const i32x4 (&x)[2][MB]) {
    constexpr int Q0 = decltype(halfc)::value * MB;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int i = 0; i < MB; ++i) {
          const int q = (a & 1) ? MB - 1 - i : i;
          acc[a][Q0 + q] = mfma_i8(wf[j][a], x[j][q], acc[a][Q0 + q]);
        }
    __builtin_amdgcn_sched_barrier(0);
  };
  auto stage = [&](int b, bool lax) {
    read_w();
    __builtin_amdgcn_sched_barrier(0);
    waddr0 ^= kStageBytes;
    waddr1 ^= kStageBytes;
    dma_x(b, false);
    if constexpr (W4) {
#pragma unroll
      for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          wf[0][a][c] = (int)(((uint32_t)raw[a][c] << 4) & 0xF0F0F0F0u);
          wf[1][a][c] = (int)((uint32_t)raw[a][c] & 0xF0F0F0F0u);
        }
    }
    end_load(lax);
    mfmas(std::integral_constant<int, 0>{}, x0);
    pp_bar();
    __builtin_amdgcn_sched_barrier(0);
    read_x(1, x1);
    xaddr0 ^= kStageBytes;
    xaddr1 ^= kStageBytes;
    read_x(0, x0);
    __builtin_amdgcn_sched_barrier(0);
    dma_w(b);
    end_load(lax);
    mfmas(std::integral_constant<int, 1>{}, x1);
    advance();
    pp_bar();
    __builtin_amdgcn_sched_barrier(0);
  };

  int buf = 0, b = 0;
  for (int t = wg; t < ntiles; t += nwg) {
    for (int kt = 0; kt < nk; ++kt) {
      stage(b, kt == 0 && t != wg);
      b ^= 1;
    }
    // Epilogue.  The lane index is opaque here: the store offsets it gives do
    // not change from tile to tile, and hoisted out of the loop they spilled.
    int le = lane;
    asm volatile("" : "+v"(le));
    const int er = wr * 16 * MB + (le & 15), ec = wc * 64 + 8 * (le >> 4);
    if constexpr (EPI == EPI_PC) {
      const int8_t* const sc = smem + 2 * kStageBytes + buf * kSclBytes;
      const float* const ssw = reinterpret_cast<const float*>(sc) + ec;
      const uint16_t* const sbi = reinterpret_cast<const uint16_t*>(sc + 1024) + ec;
      const float* const ssa = reinterpret_cast<const float*>(sc + 2048) + er;
      uint16_t* const yb = reinterpret_cast<uint16_t*>(p.y) + (int64_t)m0 * N + n0;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const f32x4 s0 = *reinterpret_cast<const f32x4*>(ssw + 32 * h);
        const f32x4 s1 = *reinterpret_cast<const f32x4*>(ssw + 32 * h + 4);
        auto convert = [&](auto biasc, auto bfc) {
          constexpr bool BIAS = decltype(biasc)::value, BF = decltype(bfc)::value;
          float bv[8];
          if constexpr (BIAS) {
            const i32x4 bb = *reinterpret_cast<const i32x4*>(sbi + 32 * h);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              bv[2 * r] = h2f((uint16_t)((uint32_t)bb[r] & 0xffffu));
              bv[2 * r + 1] = h2f((uint16_t)((uint32_t)bb[r] >> 16));
            }
          }
#pragma unroll
          for (int q = 0; q < 2 * MB; ++q) {
            const int ro = (q / MB) * (BM / 2) + (q % MB) * 16;
            float sa = ssa[ro];
            if constexpr (W4) sa = sa * 0.0625f;
            float o[8];
#pragma unroll
            for (int r = 0; r < 8; ++r) {
              // opaque: the conversions stay inside this path
              int iv = acc[2 * h + r / 4][q][r % 4];
              asm volatile("" : "+v"(iv));
              float v = (float)iv * sa;
              v = v * (r < 4 ? s0[r & 3] : s1[r & 3]);
              if constexpr (BIAS) v = v + bv[r];
              o[r] = v;
            }
            *reinterpret_cast<i32x4*>(yb + (uint32_t)((er + ro) * N + ec + 32 * h)) =
                i32x4{(int)f2o2(o[0], o[1], BF), (int)f2o2(o[2], o[3], BF),
                      (int)f2o2(o[4], o[5], BF), (int)f2o2(o[6], o[7], BF)};
          }
        };
        if (p.y_bf16) {
          if (p.bias)
            convert(std::true_type{}, std::true_type{});
          else
            convert(std::false_type{}, std::true_type{});
        } else if (p.bias) {
          convert(std::true_type{}, std::false_type{});
        } else {
          convert(std::false_type{}, std::false_type{});
        }
      }
    } else {
      int32_t* const yb = reinterpret_cast<int32_t*>(p.y) + (int64_t)m0 * N + n0;
#pragma unroll
      for (int q = 0; q < 2 * MB; ++q) {
        const int ro = (q / MB) * (BM / 2) + (q % MB) * 16;
#pragma unroll
        for (int a = 0; a < 4; ++a)
          *reinterpret_cast<i32x4*>(yb + (uint32_t)((er + ro) * N + ec + 32 * (a >> 1) +
                                                    4 * (a & 1))) = acc[a][q];
      }
    }
    zero_acc();
    buf = (buf + 1) % kSclBufs;
    __builtin_amdgcn_sched_barrier(0);
    if (t + nwg < ntiles) coords(t + nwg, m0, n0);
  }
  if (wr == 0) pp_bar();
  wait_vmcnt<0>();  // no DMA may land after the ring is given up
  pp_bar();
}

// Big tiles (BM = 64 MB) of one region and small ones (64 MS) of another:
// workgroup g takes big tiles g, g + G, .. and, from workgroup s0 on, small
// tiles g - s0, g - s0 + (G - s0), ..  Where every workgroup has both (s0 ==
// 0), every other one of an XCD takes its small ones first, so the halves of
// the chip run their epilogues at different times (M=4096 N=10240 K=2560,
// two 256-row tiles and one of 128 rows each: 92.1 -> 90.1 us).
template <int MB, int MS, int EPI, int WF>
__global__ __launch_bounds__(512, 2) void gemm_pp_kernel(const GemmArgs p, const PpRegion big,
                                                         const PpRegion small, const int s0) {
  __shared__ __attribute__((aligned(1024))) int8_t smem[kPpSmem];
  const int g = blockIdx.x, G = gridDim.x;
  const int big_pass = s0 == 0 ? (g >> 3) & 1 : 0;
  for (int pass = 0; pass < 2; ++pass) {
    if (pass == big_pass)
      pp_run<MB, EPI, WF>(p, smem, g, G, big);
    else if (g >= s0)
      pp_run<MS, EPI, WF>(p, smem, g - s0, G - s0, small);
  }
}

template <int EPI, int WF>
hipError_t run_pp(const GemmArgs& a, const PpPlan& pl, hipStream_t s) {
  const PpRegion big{pl.nbig, 0, pl.m_split, 0, pl.n_split};
  PpRegion small{0, 0, a.M, 0, a.N};
  if (pl.nsmall > 0) {
    small.ntiles = pl.nsmall;
    if (pl.m_split < a.M)
      small.m_lo = pl.m_split;
    else
      small.n_lo = pl.n_split;
  }
  const dim3 grid(pl.grid), block(512);
#define CIDER_PP(MB, MS)                                                                 \
  if (pl.mb == MB && pl.ms == MS) {                                                      \
    gemm_pp_kernel<MB, MS, EPI, WF><<<grid, block, 0, s>>>(a, big, small, pl.s0);        \
    return hipGetLastError();                                                            \
  }
  CIDER_PP(4, 2)
  CIDER_PP(4, 1)
  CIDER_PP(3, 2)
  CIDER_PP(3, 1)
  CIDER_PP(2, 1)
  CIDER_PP(1, 1)
#undef CIDER_PP
  return hipErrorInvalidValue;
}

// Estimated time (us) of a plan whose workgroups have at most (b, s) big and
// small tiles each.  Fitted to the measured times of some 1500 plans (M = 300
// .. 4096, the (N, K) of two transformer models and the 10240 x 2560 pair;
// rms error 3 %): a tile of 64 m rows costs stage[m] per 128-k stage and
// fill[m] besides while few workgroups run, and a full chip is held to `full`
// per stage of 256 x 256 per CU by its power limit.  The two meet in the
// fourth-power mean.
struct PpCost {
  double stage[5], fill[5], full, extra, launch;
};
constexpr PpCost kCostI8 = {{0, 0.559, 0.597, 0.776, 1.033}, {0, 2.32, 5.25, 7.52, 9.0},
                            1.281, 0.374, 6.4};
constexpr PpCost kCostI4 = {{0, 0.645, 0.696, 0.828, 1.014}, {0, 4.04, 5.79, 7.51, 9.0},
                            1.243, 0.551, 5.4};

double plan_cost(const PpCost& c, const PpPlan& pl, int nk, int cus) {
  const double tb = nk * c.stage[pl.mb] + c.fill[pl.mb];
  const double ts = nk * c.stage[pl.ms] + c.fill[pl.ms];
  const int f = pl.nbig / pl.grid, r = pl.nbig % pl.grid, w = pl.grid - pl.s0;
  const double small = (double)((pl.nsmall + w - 1) / w) * ts;
  // workgroups below s0 (= r) have f + 1 big tiles and no small ones
  const double crit = pl.s0 > 0 ? fmax((f + (r > 0)) * tb, f * tb + small)
                                : (f + (r > 0)) * tb + small;
  const double work = (pl.nbig * (pl.mb + c.extra) + pl.nsmall * (pl.ms + c.extra)) / (4.0 * cus);
  const double power = work * c.full * nk + c.launch;
  const double c2 = crit * crit, p2 = power * power;
  return sqrt(sqrt(c2 * c2 + p2 * p2));
}

}  // namespace

bool pp_supported(const GemmArgs& a, int epi, int wf) {
  // 32-bit element offsets within a tile of the output; the DMA of the weight
  // scales and the stores move 16 bytes per lane; 16 times the int4 weights' sums fit int32
  return a.M >= 64 && a.N >= 256 && a.N % 8 == 0 && a.N <= (1 << 22) && a.K >= 128 &&
         a.K % 128 == 0 && (wf == W_I8 ? epi != EPI_PG : epi == EPI_PC && a.K < (1 << 17)) &&
         (((uintptr_t)a.y | (uintptr_t)a.sw | (wf == W_I4 ? (uintptr_t)a.bias : 0)) & 15) == 0;
}

// The cheapest of: one tile height throughout; the rows below the last whole
// big tile in small ones; and as many whole tile columns of big tiles as fill
// whole rounds of the CUs, the columns right of them in small ones.  One or two
// k-stages are mostly stores: for fp16 results tiles of 128 rows then, if there is
// more than one round, so that a tile's stores run beside the next one's loads
// (linears, int8 / int4: M=N=8192 K=256 256 rows 60.4 / 60.0, 128 rows 45.1 / 44.1 us;
// M=4096 N=10240 K=128 64 rows 31.5 / -, 256 rows - / 32.0, 128 rows 26.9 / 26.9).
// int32 results were split: M=N=8192 82 -> 62 us, but M=2048 N=12288 26.4 -> 29.9.
double pp_plan(int M, int N, int K, int wf, int epi, PpPlan& best) {
  const PpCost& c = wf == W_I4 ? kCostI4 : kCostI8;
  const int cus = num_cus(), nk = K / 128, tn = (N + 255) / 256;
  auto ceil_div = [](int x, int y) { return (x + y - 1) / y; };
  double best_cost = 1e300;
  auto offer = [&](int mb, int ms, int nbig, int nsmall, int m_split, int n_split) {
    PpPlan pl{mb, ms, nbig, nsmall, m_split, n_split, 0, 0};
    pl.grid = nbig + nsmall < cus ? nbig + nsmall : cus;
    // small tiles go to the workgroups with one big tile less, if there are any
    pl.s0 = nsmall > 0 ? nbig % pl.grid : 0;
    const double cost = plan_cost(c, pl, nk, cus);
    if (cost < best_cost) {
      best_cost = cost;
      best = pl;
    }
  };
  for (int mb = 1; mb <= 4; ++mb) {
    const int bm = 64 * mb, tm = ceil_div(M, bm);
    if (M < bm) continue;
    if (epi == EPI_PC && nk < 3 && mb != 2 && M >= 128 && tm * tn > cus) continue;
    offer(mb, mb > 2 ? 2 : 1, tm * tn, 0, M, N);
    if (mb < 3) continue;
    const int rows = M / bm, rest = M - rows * bm;
    for (int ms = 1; ms <= 2; ++ms)
      if (rest > 0) offer(mb, ms, rows * tn, ceil_div(rest, 64 * ms) * tn, rows * bm, N);
    const int full = tm * tn / cus;  // whole rounds
    for (int f = full > 1 ? full - 1 : 1; f <= full; ++f) {
      const int cols = f * cus / tm;
      if (cols > 0 && cols < tn)
        offer(mb, 2, tm * cols, ceil_div(M, 128) * (tn - cols), M, cols * 256);
    }
  }
  return best_cost;
}

hipError_t launch_gemm_pp(const GemmArgs& a, int epi, int wf, const PpPlan& pl, hipStream_t s) {
  if (wf == W_I4) return run_pp<EPI_PC, W_I4>(a, pl, s);
  if (epi == EPI_I32) return run_pp<EPI_I32, W_I8>(a, pl, s);
  return run_pp<EPI_PC, W_I8>(a, pl, s);
}

}  // namespace cider
