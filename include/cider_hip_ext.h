/*
 * cider_hip_ext.h - entry points of libcider_hip.so beside those of
 * cider_hip.h (same conventions): the linears on bfloat16 activations, and
 * longer fusions of the decode step.
 */
#ifndef CIDER_HIP_EXT_H
#define CIDER_HIP_EXT_H

#include "cider_hip.h"

#ifdef __cplusplus
extern "C" {
#endif

/* The linears of cider_hip.h (op: CIDER_OP_PERCHANNEL, _PERGROUP, _W4A8 or
 * _W4A8_PERGROUP; w and scale as there) on bfloat16 activations with a
 * bfloat16 result: x is rounded to fp16 as it is read, and y is the fp16
 * result rounded once more to bf16, the same values as casting around the fp16
 * entry gives (the reference casts too: cider/ops.py:136-148), without the two
 * cast kernels. group_size is read by the per-group ops; bias fp16 or NULL
 * (NULL for _W4A8). Workspace as for the fp16 entries. M == 1 on int8 weights
 * is CIDER_E_UNSUPPORTED for a K that the streaming MV does not take (1024 <=
 * K <= 16384, K % 256 == 0 with a whole number of 1 KB wave loads, x and w
 * 16-byte aligned): cast around the fp16 entry there. */
int cider_linear_bf16(int op, const void* x_bf16, const void* w, const void* scale,
                      const void* bias_f16, void* y_bf16, void* ws, size_t ws_bytes,
                      int64_t M, int64_t N, int64_t K, int group_size, void* stream);

/* Whether it takes such a call (1) or answers CIDER_E_UNSUPPORTED (0); asked
 * before the result and the workspace are allocated. Reads no memory. */
int cider_linear_bf16_supported(int op, const void* x_bf16, const void* w, const void* scale,
                                int64_t M, int64_t K, int group_size);

/* The tiles of the GEMM that cider_perchannel_gemm (op CIDER_OP_PERCHANNEL), or
 * cider_w4a8_linear after its quantization (op CIDER_OP_W4A8), run on 16-byte
 * aligned operands at M > 64: tiles[0] 1 for the
 * ping-pong kernel and 0 for the LDS-DMA tiles, tiles[1] x tiles[2] rows x columns
 * of a tile, tiles[3] rows of the ping-pong kernel's small tiles beside those
 * (0: none). CIDER_E_UNSUPPORTED for a shape that runs neither. The per-channel
 * linear runs the same where it does not split K, cider_int8_matmul_int32 from K =
 * 384 on. Launches nothing. */
int cider_gemm_tiles(int op, int64_t M, int64_t N, int64_t K, int tiles[4]);

/* The MLP's first half in one decode (M == 1) launch: y [I] = SwiGLU of the
 * fused gate + up projection w [2I, K] (gate rows first), exactly as
 * cider_rmsnorm_mv (norm_w non-NULL; with add and sum as there) or
 * cider_perchannel_linear at M == 1 (norm_w NULL) on w, followed by
 * cider_silu_mul_quantize's y. Bit-identical to that pair. K a multiple of 1024
 * up to 8192, x and w 16-byte aligned; else CIDER_E_UNSUPPORTED (use the two
 * calls). y must not overlap any input; sum must not overlap x or add. */
int cider_gate_up_mv(const void* x_f16, const void* add_f16, void* sum_f16,
                     const void* norm_w_f16, float eps, const int8_t* w,
                     const float* scale_w, const void* bias_f16, void* y_f16,
                     int64_t I, int64_t K, void* stream);

/* cider_qk_norm_rope of one token (L == 1) and cider_attn_decode on its query
 * heads in one call, two launches instead of three: qkv [(H + 2 KV) * 128] is
 * the token's fused projection; its key and value go to cache row *slot as
 * there (nothing is written for a slot outside [0, T), and no key for a
 * *rope_row outside [0, P), which makes the output NaN), and the attention runs
 * over the first min(*n_valid, T) rows, the written one among them.
 * Bit-identical to the two calls. Requirements of both; every fp16 array
 * 16-byte aligned. */
int cider_attn_decode_rope(const void* qkv_f16, const void* q_norm_w_f16,
                           const void* k_norm_w_f16, float eps, const void* cos_f16,
                           const void* sin_f16, int64_t P, const int64_t* rope_row,
                           const int64_t* slot, void* k_cache_f16, void* v_cache_f16,
                           const int64_t* n_valid, float scale, void* ws, size_t ws_bytes,
                           void* out_f16, int64_t H, int64_t KV, int64_t D, int64_t T,
                           void* stream);

#ifdef __cplusplus
}
#endif

#endif /* CIDER_HIP_EXT_H */
