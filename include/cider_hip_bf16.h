/*
 * cider_hip_bf16.h - the linears of cider_hip.h on bfloat16 activations
 * (libcider_hip.so; conventions as in cider_hip.h).
 */
#ifndef CIDER_HIP_BF16_H
#define CIDER_HIP_BF16_H

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

#ifdef __cplusplus
}
#endif

#endif /* CIDER_HIP_BF16_H */
