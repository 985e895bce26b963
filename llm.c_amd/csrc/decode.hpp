// What the generation loop (driver/gpt2.cpp) asks of the kernels beyond the public launchers: the forward pass of the last
// row of one sequence, with the same bits as the full forward pass gives that row.
#pragma once
#include <hip/hip_runtime.h>

namespace llmk {
// out[OC] = x[C] . weight[OC][C]^T + bias, then gelu (pre_gelu != nullptr: receives the pre-activation) or + residual (residual !=
// nullptr): llmk_matmul_forward and llmk_matmul_forward_residual, bit for bit. x is the row inp, or, with ln_weight, its LayerNorm:
// llmk_layernorm_forward, bit for bit (ln: room for it, which may stay unwritten).
void decode_matmul(void* out, void* ln, const void* inp, const void* ln_weight, const void* ln_bias, const void* weight, const void* bias,
                   void* pre_gelu, const void* residual, int C, int OC, hipStream_t st);
void decode_attention(void* out, const void* qkv, int t0, int T, int NH, int C, hipStream_t st);
}  // namespace llmk
