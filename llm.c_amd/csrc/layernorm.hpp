// LayerNorm backward in two parts for the driver: the rows of one LayerNorm, and the sums of several at once.
// llmk_layernorm_backward is the two for one, with the same bits.
#pragma once
#include <hip/hip_runtime.h>

namespace llmk {
// where the sums of up to 2 * layers + 1 LayerNorms go: the first `layers` of them at [0] + i * C, the next `layers` at [1] + i * C,
// the last at [2]
struct LnGrads {
    void* dweight[3];
    void* dbias[3];
    int layers;
};
// dinp += the input gradient; partial[layernorm_backward_partials(N, C)][2][C]: what N rows add to dweight and dbias
int layernorm_backward_partials(int N, int C);
void layernorm_backward_rows(void* dinp, float* partial, const void* dout, const void* inp, const void* weight, const float* mean,
                             const float* rstd, int N, int C, hipStream_t st);
// dweight, dbias += the partials of `count` LayerNorms, which lie one after the other: [count][blocks][2][C]
void layernorm_backward_reduce(const LnGrads& grads, int count, const float* partial, int blocks, int C, hipStream_t st);
}  // namespace llmk
