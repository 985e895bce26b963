// Matrix products of at most 32 rows for the generation loop: out[M][OC] = inp[M][C] . weight[OC][C]^T, with the bits of the
// library's other forward kernels (K added up sixteen at a time, first to last, by the same matrix instruction; one rounding
// after the bias, one more after the residual). CPU definition train_gpt2.c:163-190.
//
// What bounds it: the weights are read once for 32 rows, so memory should, but 768 columns of a 3072-long product are only 24
// tiles of 32 with 192 dependent matrix instructions each, and a CU that has one tile has to keep enough bytes in flight by
// itself. So a workgroup is one wave that multiplies and four that do nothing but request: a ring of DEC_RING 64-wide stages
// in LDS filled by direct-to-LDS loads of whole 128-byte lines, one barrier per stage, operands read one step ahead.
// Measured, weights not in L2, us: C = 3072, OC = 768 10.1 (the 192 dependent matrix instructions are 6 of it), C = 768,
// OC = 768 4.6, OC = 3072 4.9, OC = 50304 20. The same wave requesting for itself: 19 and 6.2; operands straight from memory to
// registers in the matrix layout, 32 bytes of a line at a time: 20 and 6.5. The 128 x 128 tile that 256 rows take: 23 and 8.4.
#include "common.hpp"
#include "gelu.hpp"
#include "decode.hpp"
#include "gemm_pipelined.hpp"
#include "../../include/llmk.h"

#if !defined(LLMK_FP32)
namespace {
using namespace gemmk;

enum { DEC_PLAIN = 0, DEC_GELU = 1, DEC_RES = 2 };
constexpr int DEC_RING = 6;                                        // 48 KiB: three workgroups to a CU where there are that many
constexpr int DEC_STAGE = 64 * 128;                                // 32 rows of the activations, 32 of the weights, 64 of K

template <int MODE>
__global__ void __launch_bounds__(320)
decode_matmul_kernel(floatX* __restrict__ out, const floatX* __restrict__ inp, const floatX* __restrict__ weight,
                     const floatX* __restrict__ bias, floatX* __restrict__ pre_gelu, const floatX* __restrict__ residual, int M, int C, int OC) {
#if defined(__HIP_DEVICE_COMPILE__)
    extern __shared__ __attribute__((aligned(1024))) char lds[];
    typedef __attribute__((address_space(3))) const char* lds_cptr;
    const unsigned lds0 = (unsigned)(size_t)(lds_cptr)lds;
    const int lane = threadIdx.x & 63, idx = lane & 31, half = lane >> 5, n0 = blockIdx.x * 32;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nst = C / 64;
    if (wave < 4) {                                                // rows 8 wave .. 8 wave + 7 of both tiles, every stage
        const int row = wave * 8 + (lane >> 3), c = (lane & 7) ^ ((row >> 1) & 7);
        const unsigned off_a = ((unsigned)min(row, M - 1) * (unsigned)C + c * 8) * 2u;
        const unsigned off_b = ((unsigned)min(row, OC - 1 - n0) * (unsigned)C + c * 8) * 2u;
        const unsigned long long pa = (unsigned long long)(size_t)inp, pb = (unsigned long long)(size_t)(weight + (size_t)n0 * C);
        auto issue = [&](int st, int buf) {
            const unsigned dst = lds0 + buf * DEC_STAGE + wave * 1024;
            unsigned saved;
            asm volatile("s_mov_b32 %0, m0\n\t"
                         "s_mov_b32 m0, %1\n\t"
                         "global_load_lds_dwordx4 %3, %4\n\t"
                         "s_add_u32 m0, m0, 0x1000\n\t"
                         "global_load_lds_dwordx4 %2, %5\n\t"
                         "s_mov_b32 m0, %0"
                         : "=&s"(saved) : "s"(dst), "v"(off_b), "v"(off_a), "s"(pa + (size_t)st * 128), "s"(pb + (size_t)st * 128) : "memory", "scc");
        };
#pragma unroll
        for (int st = 0; st < DEC_RING; st++)
            if (st < nst) issue(st, st);
        int buf = DEC_RING - 1;                                    // the buffer of stage st - 1
        for (int st = 0; st < nst; st++) {
            const int younger = min(st == 0 ? DEC_RING - 1 : DEC_RING - 2, nst - 1 - st);    // requested behind stage st
            static_for<DEC_RING>([&](auto y) {
                if (younger == decltype(y)::value) wait_vmcnt<2 * decltype(y)::value>();
            });
            barrier_no_fence();                                    // stage st is there, stage st - 1 has been read
            if (st > 0 && st - 1 + DEC_RING < nst) issue(st - 1 + DEC_RING, buf);
            buf = buf + 1 == DEC_RING ? 0 : buf + 1;
        }
        return;
    }
    const unsigned arow = lds0 + idx * 128 + ((((idx >> 1) & 7) ^ half) << 4);
    auto frag = [&](unsigned base, int s) -> bf16x8 {
        return *reinterpret_cast<const __attribute__((address_space(3))) bf16x8*>((size_t)(base ^ (unsigned)(s << 5)));
    };
    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = 0.f;
    bf16x8 fa[4], fb[4];
    auto read = [&](int buf) {
#pragma unroll
        for (int s = 0; s < 4; s++) { fa[s] = frag(arow + buf * DEC_STAGE, s); fb[s] = frag(arow + buf * DEC_STAGE + 4096, s); }
    };
    barrier_no_fence();
    read(0);
    int buf = 0;
    for (int st = 0; st < nst; st++) {
        bf16x8 ca[4], cb[4];
#pragma unroll
        for (int s = 0; s < 4; s++) { ca[s] = fa[s]; cb[s] = fb[s]; }
        buf = buf + 1 == DEC_RING ? 0 : buf + 1;
        if (st + 1 < nst) {
            __builtin_amdgcn_s_waitcnt(0xC07F);                    // lgkmcnt(0): stage st is in registers
            barrier_no_fence();
            read(buf);
        }
#pragma unroll
        for (int s = 0; s < 4; s++) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(cb[s], ca[s], acc, 0, 0, 0);
    }
    if (idx >= M) return;
#pragma unroll
    for (int q = 0; q < 4; q++) {                                  // four consecutive columns of row idx
        const int n = n0 + 8 * q + 4 * half;
        if (n >= OC) continue;
        const size_t o = (size_t)idx * OC + n;
        bf16x4 y;
        if (bias) {
            const bf16x4 b = *reinterpret_cast<const bf16x4*>(bias + n);
#pragma unroll
            for (int e = 0; e < 4; e++) y[e] = (__bf16)(acc[4 * q + e] + (float)b[e]);
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++) y[e] = (__bf16)acc[4 * q + e];
        }
        if (MODE == DEC_GELU) {
            *reinterpret_cast<bf16x4*>(pre_gelu + o) = y;
#pragma unroll
            for (int e = 0; e < 4; e++) y[e] = (__bf16)gelu_f((float)y[e]);
        } else if (MODE == DEC_RES) {
            const bf16x4 r = *reinterpret_cast<const bf16x4*>(residual + o);
#pragma unroll
            for (int e = 0; e < 4; e++) y[e] = (__bf16)((float)y[e] + (float)r[e]);
        }
        *reinterpret_cast<bf16x4*>(out + o) = y;
    }
#endif
}
}  // namespace
#endif

namespace llmk {
void decode_matmul(void* out, const void* inp, const void* weight, const void* bias, void* pre_gelu, const void* residual, int M,
                   int C, int OC, hipStream_t st) {
    if (failed()) return;
#if !defined(LLMK_FP32)
    auto al = [](const void* p, uintptr_t a) { return ((uintptr_t)p % a) == 0; };
    if (M <= 32 && C % 64 == 0 && OC % 4 == 0 && al(inp, 16) && al(weight, 16) && al(out, 8) && al(bias, 8) && al(pre_gelu, 8) && al(residual, 8)) {
        auto run = [&](auto kern) {
            kern<<<CEIL_DIV(OC, 32), 320, DEC_RING * DEC_STAGE, st>>>((floatX*)out, (const floatX*)inp, (const floatX*)weight, (const floatX*)bias, (floatX*)pre_gelu,
                                                  (const floatX*)residual, M, C, OC);
        };
        if (pre_gelu) run(decode_matmul_kernel<DEC_GELU>);
        else if (residual) run(decode_matmul_kernel<DEC_RES>);
        else run(decode_matmul_kernel<DEC_PLAIN>);
        LAUNCH_CHECK();
        return;
    }
#endif
    llmk_matmul_forward(out, inp, weight, bias, 1, M, C, OC, st, pre_gelu, 1);
    if (residual) llmk_residual_forward(out, residual, out, M * OC, st);
}
}  // namespace llmk
