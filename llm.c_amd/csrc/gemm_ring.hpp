// The GEMM for launches that the persistent 256 x 256 kernel (gemm_pipelined.hpp) leaves half the chip idle in: fewer than
// one such tile per CU. Declarations; the kernel and what bounds it are in gemm_ring.hip.
#pragma once
#include "gemm_pipelined.hpp"

namespace gemmk {

enum { PERSISTENT_BIG = -1, PERSISTENT_SMALL = -2 };     // 256 x 256 and 128 x 128 tiles of gemm_pipelined.hpp
struct GemmPlan {
    int kernel = PERSISTENT_BIG;         // or a tile configuration of gemm_ring.hip, from 0
    int splits = 1;                      // pieces of K, each an fp32 partial product
    int k_per_split = 0;
    double us = 1e30;                    // estimated time of the launch and of the pass over its partial products
};
constexpr int RING_K = 128 / (int)sizeof(floatX);       // K of a stage: 128 bytes of a row
// What C[M][N] over K takes. layout: 0 forward, 1 dinp (K multiples of RING_K), 2 dweight (any K; persistent_us is then the
// estimate of the other way, persistent_tn_us, or infinity where there is none). max_splits: most pieces of K; small_tiles: the
// 128 x 128 persistent kernel has the epilogue. Arithmetic on the shape alone.
GemmPlan plan_gemm(int layout, int M, int N, int K, int max_splits, bool small_tiles, double persistent_us, int num_cu);
double persistent_tn_us(int M, int N, int K, int splits, bool big, int num_cu);
// epi: any of the epilogues of gemm_pipelined.hpp. EPI_PARTIAL_ROWSUM leaves one row sum per split ([splits][M]); rowvec (EPI_ACCUM
// with both operands K-major, or nullptr): rowvec[m] += sum over k of A(m, k).
void launch_ring(const GemmPlan& plan, GemmArgs g, bool a_t, bool b_t, int epi, floatX* rowvec, hipStream_t st);

}  // namespace gemmk
