// What the generation loop (driver/gpt2.cpp) asks of the kernels beyond the public launchers: the forward pass of the few
// rows at the end of one sequence, with the same bits as the full forward pass gives those rows.
#pragma once
#include <hip/hip_runtime.h>

namespace llmk {
// out[M][OC] = inp[M][C] . weight[OC][C]^T + bias, then gelu (pre_gelu != nullptr: receives the pre-activation) or + residual
// (residual != nullptr), M at most 32: llmk_matmul_forward and llmk_matmul_forward_residual, bit for bit.
void decode_matmul(void* out, const void* inp, const void* weight, const void* bias, void* pre_gelu, const void* residual, int M,
                   int C, int OC, hipStream_t st);
void decode_attention(void* out, const void* qkv, int t0, int T, int NH, int C, hipStream_t st);
}  // namespace llmk
