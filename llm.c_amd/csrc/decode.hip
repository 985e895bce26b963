// The products of one row for the generation loop: out[OC] = (LayerNorm of) inp[C] . weight[OC][C]^T, with the bits of the library's
// other forward kernels (K added up sixteen at a time, first to last, by the same matrix instruction; one rounding after the
// bias, one more after the residual; the LayerNorm as layernorm.hip forms it). CPU definitions train_gpt2.c:78-118, :163-190.
//
// What bounds it: reading the weights should, but 768 columns of a 3072-long product are only 24 tiles of 32 with 192
// dependent matrix instructions each, and a CU that has one tile has to keep enough bytes in flight by itself. So a
// workgroup is one wave that multiplies and four that do nothing but request weights: a ring of stages in LDS
// filled by direct-to-LDS loads of whole 128-byte lines, one barrier per stage, operands read one step ahead. The row sits in LDS,
// normalized by the multiplying wave of every workgroup while the first weights are on their way: a launch of its own for the
// LayerNorm of one row takes 3.8 us, most of it start and end.
// Measured, us, against a block of 32 rows whose activations went through the ring as well: C = 3072, OC = 768 12.5 -> 11.5 (the
// chain of matrix instructions, 43 ns each, is 8 of it), 768, 768 5.3 -> 5.0, LayerNorm + 768, 2304 9.0 -> 5.5, LayerNorm + 768,
// 3072 9.6 -> 6.5, LayerNorm + 768, 50304 18.7 -> 18.8. Tiles of 16 columns and stages of 128 against 32 and 64: 10.7 / 11.8 at
// 3072, 768; 6.0 / 6.2 at 768, 3072; the LM head 47 / 35, weights out of cache.
#include "common.hpp"
#include "gelu.hpp"
#include "decode.hpp"
#include "gemm_pipelined.hpp"
#include "../../include/llmk.h"

#if !defined(LLMK_FP32)
namespace {
using namespace gemmk;

enum { DEC_PLAIN = 0, DEC_GELU = 1, DEC_RES = 2 };
constexpr int DEC_RING_BYTES = 48 * 1024;                          // three workgroups to a CU where there are that many
constexpr int DEC_FEW = 2;                                         // workgroups per CU up to which tiles are 16 columns wide
constexpr int DEC_LN_VECS = 4;                                     // vectors of a lane: LayerNorm rows up to 2048
constexpr int DEC_MAX_C = 8192;                                    // 16 KiB of row

// the row as layernorm.hip normalizes it: the sums in the same order, the same roundings
__device__ __forceinline__ void normalize_row(char* to, const floatX* inp, const floatX* weight, const floatX* bias, int C, int lane) {
    const int nvec = C / 8;
    vecX x[DEC_LN_VECS], w[DEC_LN_VECS], b[DEC_LN_VECS];
#pragma unroll
    for (int i = 0; i < DEC_LN_VECS; i++) {
        const int v = lane + i * 64;
        if (v < nvec) { x[i] = ld_vec(inp + (size_t)v * 8); w[i] = ld_vec(weight + (size_t)v * 8); b[i] = ld_vec(bias + (size_t)v * 8); }
    }
    const float invC = 1.0f / (float)C;
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < DEC_LN_VECS; i++)
        if (lane + i * 64 < nvec) {
#pragma unroll
            for (int k = 0; k < 8; k++) s += to_f32(x[i][k]);
        }
    const float m = wave_sum(s) * invC;
    float q = 0.f;
#pragma unroll
    for (int i = 0; i < DEC_LN_VECS; i++)
        if (lane + i * 64 < nvec) {
#pragma unroll
            for (int k = 0; k < 8; k++) { float d = to_f32(x[i][k]) - m; q += d * d; }
        }
    const float var = wave_sum(q) * invC;
    const float r = 1.0f / sqrtf(var + 1e-5f);
#pragma unroll
    for (int i = 0; i < DEC_LN_VECS; i++) {
        const int v = lane + i * 64;
        if (v < nvec) {
            vecX o;
#pragma unroll
            for (int k = 0; k < 8; k++) o[k] = from_f32<floatX>(r * (to_f32(x[i][k]) - m) * to_f32(w[i][k]) + to_f32(b[i][k]));
            *reinterpret_cast<vecX*>(to + v * 16) = o;
        }
    }
}

// NC columns of the output per workgroup, stages of KS of K. LDS of a stage: [KS / 64][NC] rows of 128 bytes.
// (Registers: five waves to a workgroup, so four a SIMD - 128 registers - for the three workgroups a CU's LDS has room for, three for
// two. With neither the LM head ran one to a CU: 29 us.)
template <int MODE, bool LN, int NC, int KS>
__global__ void __launch_bounds__(320, NC == 32 ? 4 : 3)
decode_matmul_kernel(floatX* __restrict__ out, const floatX* __restrict__ inp, const floatX* __restrict__ ln_weight,
                     const floatX* __restrict__ ln_bias, const floatX* __restrict__ weight, const floatX* __restrict__ bias,
                     floatX* __restrict__ pre_gelu, const floatX* __restrict__ residual, int C, int OC) {
#if defined(__HIP_DEVICE_COMPILE__)
    constexpr int STAGE = NC * KS * 2, RING = DEC_RING_BYTES / STAGE, CHUNKS = STAGE / 1024, CPW = CHUNKS / 4, BLOCKS = KS / 64;
    static_assert(CHUNKS % 4 == 0 && (RING - 1) * CPW <= 63, "four requesting waves, a 6-bit counter");
    extern __shared__ __attribute__((aligned(1024))) char lds[];
    typedef __attribute__((address_space(3))) const char* lds_cptr;
    const unsigned lds0 = (unsigned)(size_t)(lds_cptr)lds;
    const int lane = threadIdx.x & 63, idx = lane & 31, half = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nst = CEIL_DIV(C, KS), n0 = blockIdx.x * NC;
    if (wave < 4) {                                                // chunk i: 8 rows of one 64-wide block of the stage
        unsigned off[CPW];
#pragma unroll
        for (int i = 0; i < CPW; i++) {
            const int chunk = wave + 4 * i, row = chunk % (NC / 8) * 8 + (lane >> 3), c = (lane & 7) ^ ((row >> 1) & 7);
            off[i] = ((unsigned)min(row, OC - 1 - n0) * (unsigned)C + c * 8) * 2u;
        }
        auto issue = [&](int st, int buf) {
            unsigned saved;
            asm volatile("s_mov_b32 %0, m0" : "=s"(saved));
#pragma unroll
            for (int i = 0; i < CPW; i++) {
                const int chunk = wave + 4 * i, k = st * KS + chunk / (NC / 8) * 64;       // (a block past the end of K is not used: any address)
                asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2"
                             :: "s"(lds0 + buf * STAGE + chunk * 1024), "v"(off[i]),
                                "s"((unsigned long long)(size_t)(weight + (size_t)n0 * C + (k < C ? k : 0))) : "memory");
            }
            asm volatile("s_mov_b32 m0, %0" :: "s"(saved));
        };
#pragma unroll
        for (int st = 0; st < RING; st++)
            if (st < nst) issue(st, st);
        int buf = RING - 1;                                        // the buffer of stage st - 1
        for (int st = 0; st < nst; st++) {
            const int younger = min(st == 0 ? RING - 1 : RING - 2, nst - 1 - st);          // requested behind stage st
            static_for<RING>([&](auto y) {
                if (younger == decltype(y)::value) wait_vmcnt<decltype(y)::value * CPW>();
            });
            barrier_no_fence();                                    // stage st is there, stage st - 1 has been read
            if (st > 0 && st - 1 + RING < nst) issue(st - 1 + RING, buf);
            buf = buf + 1 == RING ? 0 : buf + 1;
        }
        return;
    }
    char* row = lds + RING * STAGE;
    if constexpr (LN) normalize_row(row, inp, ln_weight, ln_bias, C, lane);
    else {
#pragma unroll 4
        for (int v = lane; v < C / 8; v += 64) *reinterpret_cast<vecX*>(row + v * 16) = ld_vec(inp + (size_t)v * 8);
    }
    const int brow_at = idx % NC;                                  // (with fewer than 32 columns the rest repeats them)
    const unsigned brow = lds0 + brow_at * 128 + ((((brow_at >> 1) & 7) ^ half) << 4);
    f32x16 acc;                                                    // rows: the tile's columns; every column the same product
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = 0.f;
    struct Frags { bf16x8 a[KS / 16], b[KS / 16]; } f0, f1;
    auto read = [&](Frags& f, int st, int buf) {
#pragma unroll
        for (int s = 0; s < KS / 16; s++) {
            f.a[s] = *reinterpret_cast<const bf16x8*>(row + min(st * KS + s * 16, C - 16) * 2 + half * 16);
            f.b[s] = *reinterpret_cast<const __attribute__((address_space(3))) bf16x8*>((size_t)((brow ^ (unsigned)((s & 3) << 5)) + buf * STAGE + (s >> 2) * (NC * 128)));
        }
    };
    barrier_no_fence();
    read(f0, 0, 0);
    int buf = 0;
    // (two sets of fragments by turns: copying one set to another costs as much as a third of the multiplications)
    auto step = [&](int st, const Frags& f, Frags& next) {
        buf = buf + 1 == RING ? 0 : buf + 1;
        if (st + 1 < nst) {
            __builtin_amdgcn_s_waitcnt(0xC07F);                    // lgkmcnt(0): stage st is in registers
            barrier_no_fence();
            read(next, st + 1, buf);
        }
#pragma unroll
        for (int k = 0; k < KS / 64; k++)
            if (KS == 64 || st * KS + k * 64 < C) {
#pragma unroll
                for (int s = 4 * k; s < 4 * k + 4; s++) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.b[s], f.a[s], acc, 0, 0, 0);
            }
    };
    for (int st = 0; st < nst; st += 2) {
        step(st, f0, f1);
        if (st + 1 < nst) step(st + 1, f1, f0);
    }
    if (idx > 0) return;
#pragma unroll
    for (int q = 0; q < NC / 8; q++) {                             // four consecutive columns
        const int n = n0 + 8 * q + 4 * half;
        if (n >= OC) continue;
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
            *reinterpret_cast<bf16x4*>(pre_gelu + n) = y;
#pragma unroll
            for (int e = 0; e < 4; e++) y[e] = (__bf16)gelu_f((float)y[e]);
        } else if (MODE == DEC_RES) {
            const bf16x4 r = *reinterpret_cast<const bf16x4*>(residual + n);
#pragma unroll
            for (int e = 0; e < 4; e++) y[e] = (__bf16)((float)y[e] + (float)r[e]);
        }
        *reinterpret_cast<bf16x4*>(out + n) = y;
    }
#endif
}
}  // namespace
#endif

namespace llmk {
void decode_matmul(void* out, void* ln, const void* inp, const void* ln_weight, const void* ln_bias, const void* weight, const void* bias,
                   void* pre_gelu, const void* residual, int C, int OC, hipStream_t st) {
    if (failed()) return;
#if !defined(LLMK_FP32)
    auto al = [](const void* p, uintptr_t a) { return ((uintptr_t)p % a) == 0; };
    if (C % 64 == 0 && C <= (ln_weight ? DEC_LN_VECS * 512 : DEC_MAX_C) && OC % 4 == 0 && al(inp, 16) && al(ln_weight, 16) && al(ln_bias, 16) &&
        al(weight, 16) && al(out, 8) && al(bias, 8) && al(pre_gelu, 8) && al(residual, 8)) {
        // Every workgroup normalizes the row for itself, which pays while all of them run at once; with more (the LM head) the row is
        // normalized by a launch of its own and read as it is.
        const bool few = CEIL_DIV(OC, 16) <= DEC_FEW * device_info().num_cu;
        if (!few && ln_weight) {
            llmk_layernorm_forward(ln, nullptr, nullptr, inp, ln_weight, ln_bias, 1, 1, C, st);
            inp = ln;
            ln_weight = nullptr;
        }
        auto run = [&](auto kern, int nc) {
            kern<<<CEIL_DIV(OC, nc), 320, DEC_RING_BYTES + C * 2, st>>>((floatX*)out, (const floatX*)inp, (const floatX*)ln_weight,
                (const floatX*)ln_bias, (const floatX*)weight, (const floatX*)bias, (floatX*)pre_gelu, (const floatX*)residual, C, OC);
        };
        auto mode = [&](auto ln_here, auto nc, auto ks) {
            constexpr bool LN = decltype(ln_here)::value;
            constexpr int NC = decltype(nc)::value, KS = decltype(ks)::value;
            if (pre_gelu) run(decode_matmul_kernel<DEC_GELU, LN, NC, KS>, NC);
            else if (residual) run(decode_matmul_kernel<DEC_RES, LN, NC, KS>, NC);
            else run(decode_matmul_kernel<DEC_PLAIN, LN, NC, KS>, NC);
        };
        using std::integral_constant;
        if (!few) mode(std::false_type{}, integral_constant<int, 32>{}, integral_constant<int, 64>{});
        else if (ln_weight) mode(std::true_type{}, integral_constant<int, 16>{}, integral_constant<int, 128>{});
        else mode(std::false_type{}, integral_constant<int, 16>{}, integral_constant<int, 128>{});
        LAUNCH_CHECK();
        return;
    }
#endif
    if (ln_weight) {
        llmk_layernorm_forward(ln, nullptr, nullptr, inp, ln_weight, ln_bias, 1, 1, C, st);
        inp = ln;
    }
    llmk_matmul_forward(out, inp, weight, bias, 1, 1, C, OC, st, pre_gelu, 1);
    if (residual) llmk_residual_forward(out, residual, out, OC, st);
}
}  // namespace llmk
