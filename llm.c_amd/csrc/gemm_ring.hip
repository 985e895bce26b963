// GEMM for launches of few output tiles: small batches, narrow layers, short sequences.
#include "common.hpp"
#include "gelu.hpp"
#include "gemm_ring.hpp"
#include <algorithm>
#include <limits>
#include "../../include/llmk.h"

namespace gemmk {
namespace {

// What a stage past the end of K is read from (both operands K-major, K not a multiple of RING_K)
__device__ const u32x4 g_zero_chunk = {0, 0, 0, 0};

// One output tile (and one piece of K) per workgroup; K in stages of RING_K through a ring of NST LDS buffers, NST - 1 of them
// in flight. A launch of few tiles has nothing to hide memory latency behind but its own lookahead: with the two buffers of
// the persistent kernel a stage costs a trip to HBM. Operand layouts, swizzles, fragment reads and the order of every sum are the
// persistent kernel's, so that a forward pass has the same bits whichever of the two ran it. The finished tile goes through
// LDS in fp32 once and leaves in rows of 16-byte stores, whatever the epilogue.
// What bounds it: a lone workgroup draws 25 bytes a clock from L2 whatever its tile and however deep the ring, so few tiles want
// to be many small ones (the fourfold traffic of 64 x 64 is spread over more CUs); a full chip wants 256 x 128, whose 96 KiB of
// stages in flight leave no epilogue to overlap with, which is why the persistent kernel keeps launches of many tiles.
// Wave tiles are 64 x 32 or 32 x 64 (32 x 32 in the two smallest): twice the waves of 64 x 64 ones read half as much again from LDS
// and hide its latency and the loads' issue from each other: 3885 x 1024 over 4096 40.8 -> 37.0 us, dweight 2048 x 2048 over 4096
// 48.6 -> 41.8, 3000 x 1536 over 4608 60 -> 53.
// Measured, weights from HBM, us, the persistent kernel's better tile against this: 256 x 768 over K = 3072 29.6 / 15.0 (one
// piece), 9.9 (four, with the pass over the partials), over K = 50304 613 / 42; 4096 x 2048 over 8192 156 / 124; 3000 x 1536 over
// 6144 120 / 80; dweight 3072 x 768 over 256 rows 19.7 / 7.1, 4608 x 1536 over 3000 rows (no persistent kernel) 83 / 52.
// The fp32 library has the same kernel with the fp32 matrix instruction, 16 of which make a stage of 32: the matrix cores bound
// it (2048 x 50304 over 768: 119 TFLOP/s of 157) as soon as every CU has a tile, so what counts is tiles small enough for that.
constexpr int CE = 16 / (int)sizeof(floatX);     // elements of a 16-byte chunk
#if defined(LLMK_FP32)
typedef f32x4 frag_t;                            // eight of K: lane half h holds 4 h .. 4 h + 3
#else
typedef bf16x8 frag_t;                           // sixteen of K
#endif

template <int BM, int BN, int WGM, int WGN, int NST, bool A_T, bool B_T>
__global__ void __launch_bounds__(WGM * WGN * 64)
gemm_ring_kernel(GemmArgs g, int epi, floatX* rowvec) {
#if defined(__HIP_DEVICE_COMPILE__)
    constexpr int NW = WGM * WGN, NT = NW * 64;
    constexpr int WTM = BM / WGM, WTN = BN / WGN, TM = WTM / 32, TN = WTN / 32;
    constexpr int A_STAGE = BM * 128, B_STAGE = BN * 128, STAGE = A_STAGE + B_STAGE, X = (int)sizeof(floatX);
    constexpr int A_CHUNKS = A_STAGE / 1024, B_CHUNKS = B_STAGE / 1024, CPW = (A_CHUNKS + B_CHUNKS) / NW;
    static_assert(A_CHUNKS % NW == 0 && B_CHUNKS % NW == 0, "each load slot of a wave is all-A or all-B");
    static_assert(NST >= 2 && (NST - 2) * CPW <= 63, "vmcnt is a 6-bit counter");
    static_assert(BM * BN * 4 <= NST * STAGE && BN >= 64, "the fp32 tile reuses the ring");
    constexpr bool K_TAIL = A_T && B_T;
    extern __shared__ __attribute__((aligned(1024))) char lds[];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WGN, wn = wave % WGN;
    const int idx = lane & 31, half = lane >> 5;
    const int tiles_m = CEIL_DIV(g.M, BM), tiles_n = CEIL_DIV(g.N, BN), num_tiles = tiles_m * tiles_n;

    // workgroups are dealt round-robin over the 8 XCDs: XCD x takes a contiguous share of the list, so that tiles which share
    // operand panels (and the same piece of K) sit behind one L2
    const int total = gridDim.x, xcd = blockIdx.x & 7, local = blockIdx.x >> 3;
    const int id = (total >> 3) * xcd + min(xcd, total & 7) + local;
    int tile_m, tile_n;
    tile_of(id % num_tiles, tiles_m, tiles_n, tile_m, tile_n);
    const int split = id / num_tiles;
    const int m0 = tile_m * BM, n0 = tile_n * BN;
    const int kbeg = split * g.k_per_split, kend = min(g.K, kbeg + g.k_per_split);
    const int nst = CEIL_DIV(kend - kbeg, RING_K);
    const int tail = K_TAIL && (kend - kbeg) % RING_K ? nst - 1 : -1;      // the stage that reaches past K

    typedef __attribute__((address_space(3))) const char* lds_cptr;
    const unsigned lds0 = (unsigned)(size_t)(lds_cptr)lds;
    const char* base_a = reinterpret_cast<const char*>(A_T ? g.A + (size_t)kbeg * g.lda + m0 : g.A + (size_t)m0 * g.lda + kbeg);
    const char* base_b = reinterpret_cast<const char*>(B_T ? g.B + (size_t)kbeg * g.ldb + n0 : g.B + (size_t)n0 * g.ldb + kbeg);
    const size_t step_a = (A_T ? (size_t)RING_K * g.lda : (size_t)RING_K) * X;
    const size_t step_b = (B_T ? (size_t)RING_K * g.ldb : (size_t)RING_K) * X;
    // K-major tiles [k][rows]: which 16-byte chunk of row k a lane fetches, so that the reads - of four consecutive k by the
    // transposing read, of k and k + 4 by the two half-waves in fp32 - meet no bank twice
    auto swz_t = [](int rows, int k) { return X == 4 ? 8 * ((k >> 2) & 1) : rows >= 128 ? 4 * (k & 3) : 4 * ((k >> 1) & 1); };
    unsigned voff[CPW];
    int krow_of[K_TAIL ? CPW : 1];
#pragma unroll
    for (int i = 0; i < CPW; i++) {
        const bool isA = i * NW < A_CHUNKS;
        const int cc = isA ? wave + i * NW : wave + i * NW - A_CHUNKS;
        const int ld = isA ? g.lda : g.ldb, r0 = isA ? m0 : n0, rmax = isA ? g.M : g.N, R = isA ? BM : BN;
        if (!(isA ? A_T : B_T)) {
            const int row = cc * 8 + (lane >> 3), c = (lane & 7) ^ ((row >> 1) & 7);
            voff[i] = ((unsigned)min(row, rmax - 1 - r0) * (unsigned)ld + c * CE) * (unsigned)X;
        } else {
            const int byte = cc * 1024 + lane * 16, krow = byte / (R * X), cn = ((byte % (R * X)) >> 4) ^ swz_t(R, krow);
            voff[i] = ((unsigned)krow * (unsigned)ld + (r0 + cn * CE < rmax ? cn * CE : 0)) * (unsigned)X;
            if (K_TAIL) krow_of[i] = krow;
        }
    }
    auto issue = [&](int st, int buf) {
        const unsigned stage = lds0 + buf * STAGE;
        const unsigned long long pa = (unsigned long long)(size_t)(base_a + (size_t)st * step_a);
        const unsigned long long pb = (unsigned long long)(size_t)(base_b + (size_t)st * step_b);
        unsigned saved;
        asm volatile("s_mov_b32 %0, m0" : "=s"(saved));
        if (K_TAIL && st == tail) {                               // rows past K are zeros
#pragma unroll
            for (int i = 0; i < CPW; i++) {
                const bool in = kbeg + st * RING_K + krow_of[K_TAIL ? i : 0] < kend;
                const unsigned long long p = in ? (i * NW < A_CHUNKS ? pa : pb) + voff[i] : (unsigned long long)(size_t)&g_zero_chunk;
                asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, off" :: "s"(stage + (wave + i * NW) * 1024), "v"(p) : "memory");
            }
        } else {
#pragma unroll
            for (int i = 0; i < CPW; i++)
                asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2"
                             :: "s"(stage + (wave + i * NW) * 1024), "v"(voff[i]), "s"(i * NW < A_CHUNKS ? pa : pb) : "memory");
        }
        asm volatile("s_mov_b32 m0, %0" :: "s"(saved));
    };

    auto frag_base = [&](bool trans, int region, int rows, int row0) -> unsigned {
        if (!trans) {
            const int row = row0 + idx;
            return region + row * 128 + ((((row >> 1) & 7) ^ half) << 4);
        }
        if (X == 4) {                                             // row 4 half + e of eight, column idx
            const int col = row0 + idx;
            return region + 4 * half * (rows * 4) + ((col >> 2) ^ swz_t(rows, 4 * half)) * 16 + (col & 3) * 4;
        }
        const int s16 = lane & 15, grp = lane >> 4;
        const int krow = 8 * (grp >> 1) + (s16 >> 2), col = row0 + (grp & 1) * 16 + 4 * (s16 & 3);
        return region + krow * (rows * 2) + ((col >> 3) ^ swz_t(rows, krow)) * 16 + (col & 7) * 2;
    };
    unsigned abase[TM], bbase[TN];
#pragma unroll
    for (int i = 0; i < TM; i++) abase[i] = lds0 + frag_base(A_T, 0, BM, wm * WTM + i * 32);
#pragma unroll
    for (int j = 0; j < TN; j++) bbase[j] = lds0 + frag_base(B_T, A_STAGE, BN, wn * WTN + j * 32);
    auto frag = [&](bool trans, unsigned base, unsigned buf, int s, int rows) -> frag_t {
        if (!trans)
            return *reinterpret_cast<const __attribute__((address_space(3))) frag_t*>((size_t)((base ^ (unsigned)(s << 5)) + buf));
#if defined(LLMK_FP32)
        frag_t v;
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = *reinterpret_cast<const __attribute__((address_space(3))) float*>((size_t)(base + buf + (8 * s + e) * rows * 4));
        return v;
#else
        typedef s16x4 __attribute__((address_space(3))) * lp;
        union { struct { s16x4 a, b; } p; bf16x8 v; } u;
        u.p.a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lp)(size_t)(base + buf + s * 16 * rows * 2));
        u.p.b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lp)(size_t)(base + buf + (s * 16 + 4) * rows * 2));
        return u.v;
#endif
    };
    auto read_frags = [&](int b, int s, frag_t (&fa)[TM], frag_t (&fb)[TN]) {
        const unsigned buf = (unsigned)b * STAGE;
#pragma unroll
        for (int i = 0; i < TM; i++) fa[i] = frag(A_T, abase[i], buf, s, BM);
#pragma unroll
        for (int j = 0; j < TN; j++) fb[j] = frag(B_T, bbase[j], buf, s, BN);
    };
    f32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;
    // row sums of A, from the fragments (as in the persistent kernel): the column waves take the 16-wide steps in turn
    const bool rowsum = A_T && tile_n == 0 && (epi == EPI_PARTIAL_ROWSUM || (epi == EPI_ACCUM && rowvec != nullptr));
    float rsum[A_T ? TM : 1];
#pragma unroll
    for (int i = 0; i < (A_T ? TM : 1); i++) rsum[i] = 0.f;
    auto mma = [&](const frag_t (&fa)[TM], const frag_t (&fb)[TN], int s) {
#if defined(LLMK_FP32)
#pragma unroll
        for (int e = 0; e < 4; e++)
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fb[j][e], fa[i][e], acc[i][j], 0, 0, 0);
#else
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[j], fa[i], acc[i][j], 0, 0, 0);
#endif
        if constexpr (A_T) {
            if (rowsum && s % WGN == wn) {
#if defined(LLMK_FP32)
#pragma unroll
                for (int i = 0; i < TM; i++) rsum[i] += (fa[i][0] + fa[i][1]) + (fa[i][2] + fa[i][3]);
#else
                typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
                const bf16x2 ones = {(__bf16)1.0f, (__bf16)1.0f};
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const bf16x2 p = {fa[i][2 * e], fa[i][2 * e + 1]};
                        rsum[i] = __builtin_amdgcn_fdot2_f32_bf16(p, ones, rsum[i], false);
                    }
#endif
            }
        }
    };
    // stage st has landed for this wave: the stages behind it in the ring (at most NST - 2) may be on the way
    auto wait_stage = [&](int st) {
        const int behind = nst - 1 - st;
        if (behind >= NST - 2) wait_vmcnt<(NST - 2) * CPW>();
        else if (NST > 4 && behind == 2) wait_vmcnt<2 * CPW>();
        else if (NST > 3 && behind == 1) wait_vmcnt<CPW>();
        else wait_vmcnt<0>();
    };
#pragma unroll
    for (int s = 0; s < NST - 1; s++)
        if (s < nst) issue(s, s);
    frag_t fa0[TM], fb0[TN], fa1[TM], fb1[TN];
    wait_stage(0);
    barrier_no_fence();
    if (NST - 1 < nst) issue(NST - 1, NST - 1);
    read_frags(0, 0, fa0, fb0);
    int buf = 0;
    for (int st = 0; st < nst; st++) {
        read_frags(buf, 1, fa1, fb1);
        mma(fa0, fb0, 0);
        read_frags(buf, 2, fa0, fb0);
        mma(fa1, fb1, 1);
        read_frags(buf, 3, fa1, fb1);
        mma(fa0, fb0, 2);
        const int done = buf;
        buf = buf + 1 == NST ? 0 : buf + 1;
        if (st + 1 < nst) {
            __builtin_amdgcn_s_waitcnt(0xC07F);                   // lgkmcnt(0): this wave has read its last of stage st
            // (behind stage st + 1: what was issued up to now, stages st + 2 .. st + NST - 1)
            wait_stage(st + 1);
            barrier_no_fence();                                   // ... and so has everyone; stage st + 1 is there
            if (st + NST < nst) issue(st + NST, done);
            read_frags(buf, 0, fa0, fb0);
        }
        mma(fa1, fb1, 3);
    }
    __builtin_amdgcn_s_waitcnt(0xC07F);
    barrier_no_fence();                                           // the ring is free

    if constexpr (A_T) {
        if (rowsum) {                                             // uniform over the workgroup
            float* rs = reinterpret_cast<float*>(lds);
#pragma unroll
            for (int i = 0; i < TM; i++) {
                const float s = rsum[i] + __shfl_xor(rsum[i], 32, 64);
                if (half == 0) rs[wn * BM + wm * WTM + i * 32 + idx] = s;
            }
            __syncthreads();
            for (int r = tid; r < BM && m0 + r < g.M; r += NT) {
                float s = 0.f;
#pragma unroll
                for (int w = 0; w < WGN; w++) s += rs[w * BM + r];
                if (epi == EPI_ACCUM) rowvec[m0 + r] = from_f32<floatX>(to_f32(rowvec[m0 + r]) + s);
                else g.rowsum[(size_t)split * g.M + m0 + r] = s;
            }
            __syncthreads();
        }
    }
    // the tile in LDS, fp32: 16-byte chunk c of row r at chunk c ^ (r & 15)
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int row = wm * WTM + i * 32 + idx, c = (wn * WTN + j * 32 + 8 * q + 4 * half) >> 2;
                const f32x4 o = {acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
                *reinterpret_cast<f32x4*>(lds + row * (BN * 4) + ((c ^ (row & 15)) << 4)) = o;
            }
    __syncthreads();
    for (int v = tid; v < BM * (BN / 8); v += NT) {
        const int row = v / (BN / 8), c8 = v % (BN / 8);
        const int m = m0 + row, n = n0 + c8 * 8;
        if (m >= g.M || n >= g.N) continue;
        float x[8];
        *reinterpret_cast<f32x4*>(x) = *reinterpret_cast<const f32x4*>(lds + row * (BN * 4) + (((2 * c8) ^ (row & 15)) << 4));
        *reinterpret_cast<f32x4*>(x + 4) = *reinterpret_cast<const f32x4*>(lds + row * (BN * 4) + (((2 * c8 + 1) ^ (row & 15)) << 4));
        const size_t o = (size_t)m * g.ldc + n;
        if (epi == EPI_PARTIAL || epi == EPI_PARTIAL_ROWSUM) {
            float* p = g.partial + ((size_t)split * g.M + m) * g.N + n;
            *reinterpret_cast<f32x4*>(p) = *reinterpret_cast<f32x4*>(x);
            *reinterpret_cast<f32x4*>(p + 4) = *reinterpret_cast<f32x4*>(x + 4);
            continue;
        }
        // eight columns in storage type: 16 bytes, or 32 in fp32
        struct alignas(CE == 8 ? 16 : 32) V { floatX h[8]; };
        auto load8 = [](const floatX* p) {
            V v;
#pragma unroll
            for (int k = 0; k < 8 / CE; k++) reinterpret_cast<u32x4*>(&v)[k] = reinterpret_cast<const u32x4*>(p)[k];
            return v;
        };
        auto store8 = [](floatX* p, const V& v) {
#pragma unroll
            for (int k = 0; k < 8 / CE; k++) reinterpret_cast<u32x4*>(p)[k] = reinterpret_cast<const u32x4*>(&v)[k];
        };
        if (g.bias) {                                             // (the callers give one to the epilogues that have one)
            typedef floatX half_t __attribute__((ext_vector_type(8 / (int)sizeof(floatX))));      // 8 bytes: the alignment asked of a bias
#pragma unroll
            for (int k = 0; k < X; k++) {
                const half_t b = reinterpret_cast<const half_t*>(g.bias + n)[k];
#pragma unroll
                for (int e = 0; e < 8 / X; e++) x[8 / X * k + e] += (float)b[e];
            }
        }
        V y, a;
        if (epi == EPI_ACCUM) {
            a = load8(g.C + o);
#pragma unroll
            for (int e = 0; e < 8; e++) y.h[e] = (floatX)((float)a.h[e] + x[e]);
        } else {
#pragma unroll
            for (int e = 0; e < 8; e++) y.h[e] = (floatX)x[e];
            if (epi_gelu_fwd(epi)) {
                a = y;
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    if (epi == EPI_BIAS_GELU) y.h[e] = (floatX)gelu_f((float)y.h[e]);
                    else { float gr; y.h[e] = (floatX)gelu_with_grad_f((float)y.h[e], gr); a.h[e] = (floatX)gr; }
                }
                store8(g.aux + o, a);
            } else if (epi_reads_aux(epi)) {
                a = load8(g.aux + o);
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const float p = (float)a.h[e], d = (float)y.h[e];
                    y.h[e] = (floatX)(epi == EPI_BIAS_RES ? d + p : (epi == EPI_DGELU_D ? p : gelu_grad_f(p)) * d);
                }
            }
        }
        store8(g.C + o, y);
    }
#endif
}

template <int BM, int BN, int WGM, int WGN, int NST, bool A_T, bool B_T>
void launch_cfg(const GemmArgs& g, int epi, floatX* rowvec, hipStream_t st) {
    constexpr int SMEM = NST * (BM + BN) * 128;
    auto kern = gemm_ring_kernel<BM, BN, WGM, WGN, NST, A_T, B_T>;
    static bool attr_set = false;
    if (!attr_set) {
        HIP_CHECK(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, SMEM));
        attr_set = true;
    }
    kern<<<CEIL_DIV(g.M, BM) * CEIL_DIV(g.N, BN) * g.splits, WGM * WGN * 64, SMEM, st>>>(g, epi, rowvec);
    LAUNCH_CHECK();
}
template <bool A_T, bool B_T>
void launch_layout(int cfg, const GemmArgs& g, int epi, floatX* rowvec, hipStream_t st) {
    switch (cfg) {
        case 0: launch_cfg<256, 128, 4, 4, 3, A_T, B_T>(g, epi, rowvec, st); break;
        case 1: launch_cfg<128, 128, 2, 4, 2, A_T, B_T>(g, epi, rowvec, st); break;
        case 2: launch_cfg<128, 128, 4, 2, 4, A_T, B_T>(g, epi, rowvec, st); break;
        case 3: launch_cfg<128, 64, 4, 2, 3, A_T, B_T>(g, epi, rowvec, st); break;
        case 4: launch_cfg<64, 64, 2, 2, 3, A_T, B_T>(g, epi, rowvec, st); break;
        default: LLMK_REQUIRE(false, "launch_ring: no configuration %d", cfg);
    }
}

// ---- which kernel a product takes -----------------------------------------------------------------------------------------
// Estimated microseconds, from timing every configuration over the projections of all model sizes at 256 to 4096 rows, the
// weights not in cache. A stage (64 of K) of one workgroup alone on its CU takes `alone`, of a workgroup on a full chip `full`
// (the CUs then share L2 and HBM, and a workgroup its CU's LDS with its neighbours); between, in proportion to the load.
struct TileCost { int bm, bn, per_cu; double alone, full[3], fixed; };      // full: forward, dinp, dweight
constexpr int RING_CFGS = 5;
#if defined(LLMK_FP32)
constexpr TileCost RING_COST[RING_CFGS] = {
    {256, 128, 1, 3.75, {3.9, 3.9, 4.1}, 7.0},
    {128, 128, 2, 1.95, {3.9, 3.9, 4.1}, 6.0},
    {128, 128, 1, 1.95, {2.0, 2.0, 2.1}, 6.0},
    {128, 64, 2, 1.0, {1.95, 1.95, 2.05}, 5.0},
    {64, 64, 3, 0.52, {1.5, 1.5, 1.55}, 4.0},
};
#else
constexpr TileCost RING_COST[RING_CFGS] = {
    {256, 128, 1, 0.72, {0.94, 0.92, 1.05}, 5.0},
    {128, 128, 2, 0.46, {0.95, 1.02, 1.05}, 4.2},
    {128, 128, 1, 0.45, {0.57, 0.53, 0.60}, 4.2},
    {128, 64, 2, 0.32, {0.61, 0.61, 0.70}, 3.4},
    {64, 64, 3, 0.29, {0.58, 0.58, 0.64}, 2.8},
};
#endif
constexpr TileCost PERSISTENT_COST[2] = {{256, 256, 1, 1.07, {1.70, 1.62, 1.62}, 3.5}, {128, 128, 1, 0.57, {0.70, 0.70, 0.70}, 2.8}};
double launch_us(const TileCost& c, int layout, int M, int N, int K, int splits, double per_round, int num_cu) {
    const int wgs = CEIL_DIV(M, c.bm) * CEIL_DIV(N, c.bn) * splits, slots = num_cu * c.per_cu;
    const int nst = CEIL_DIV(CEIL_DIV(K, RING_K), splits), rest = wgs % slots;
    double stages = (wgs / slots) * c.full[layout];
    if (rest) stages += c.alone + (c.full[layout] - c.alone) * rest / slots;
    const double bytes = ((double)M * K + (double)N * K + (double)M * N * (layout == 2 ? 2 : 1)) * sizeof(floatX);
    return std::max(c.fixed + nst * stages + per_round * wgs / slots, 4.0 + bytes / 3.5e6);
}
// writing and adding up the fp32 partial products
double reduce_us(int M, int N, int splits) { return 3.5 + (double)M * N * 8.0 * splits / 5e6; }
constexpr int MIN_STAGES = 4;            // fewest stages of a piece of K
// What a ring launch's estimate has to come down to before it replaces the persistent kernel. Where the weight gradients of the two
// are estimated within a tenth the persistent kernel was as good or better (dinp and dweight, us, persistent / ring: 1024 x 1024 over
// 16384 rows, estimated at 0.91, 94.1 / 95.0; 768 x 768 over 32768, 0.96, 120.4 / 121.9; on the other side 1280 x 1280 over 8192,
// 0.90, 107 / 87; 768 x 768 over 24576, 0.87, 102.7 / 99.7 and over 16384, 0.82, 83.6 / 69.5).
constexpr double STAY = 0.96, STAY_DWEIGHT = 0.905;
}  // namespace

GemmPlan plan_gemm(int layout, int M, int N, int K, int max_splits, bool small_tiles, double persistent_us, int num_cu) {
    GemmPlan best;
    best.kernel = PERSISTENT_BIG;
    best.k_per_split = CEIL_DIV(K, RING_K) * RING_K;
    const size_t big_tiles = (size_t)CEIL_DIV(M, 256) * CEIL_DIV(N, 256);
    if (layout == 2) best.us = persistent_us;
    else if (sizeof(floatX) == 4) best.us = std::numeric_limits<double>::infinity();      // no persistent kernel
    else {
        if (big_tiles >= 4 * (size_t)num_cu) return best;         // the last round's share is small whatever it is
        best.us = launch_us(PERSISTENT_COST[0], layout, M, N, K, 1, 0.8, num_cu);
        if (small_tiles) {
            const double us = launch_us(PERSISTENT_COST[1], layout, M, N, K, 1, 0.8, num_cu);
            if (us < best.us) { best.us = us; best.kernel = PERSISTENT_SMALL; }
        }
    }
    const int stages = CEIL_DIV(K, RING_K);
    double least = best.us * (layout == 2 ? STAY_DWEIGHT : STAY);
    for (int c = 0; c < RING_CFGS; c++) {
        const size_t tiles = (size_t)CEIL_DIV(M, RING_COST[c].bm) * CEIL_DIV(N, RING_COST[c].bn);
        if (tiles > (size_t)num_cu * 4096) continue;                // (a grid of 32 bits)
        for (int s = 1; s <= max_splits && s * MIN_STAGES <= std::max(stages, MIN_STAGES); s++) {
            if (s > 1 && (tiles * s > (size_t)num_cu * 4 || CEIL_DIV(stages, CEIL_DIV(stages, s)) != s)) continue;
            const double us = launch_us(RING_COST[c], layout, M, N, K, s, 2.2, num_cu) + (s > 1 ? reduce_us(M, N, s) : 0.0);
            if (us < least) {
                least = us;
                best.kernel = c; best.splits = s; best.us = us; best.k_per_split = CEIL_DIV(stages, s) * RING_K;
            }
        }
    }
    return best;
}
double persistent_tn_us(int M, int N, int K, int splits, bool big, int num_cu) {
    return launch_us(PERSISTENT_COST[big ? 0 : 1], 2, M, N, K, splits, 0.8, num_cu) + reduce_us(M, N, splits);
}

void launch_ring(const GemmPlan& plan, GemmArgs g, bool a_t, bool b_t, int epi, floatX* rowvec, hipStream_t st) {
    if (llmk::failed()) return;
    g.splits = plan.splits;
    g.k_per_split = plan.k_per_split;
    if (a_t) launch_layout<true, true>(plan.kernel, g, epi, rowvec, st);
    else if (b_t) launch_layout<false, true>(plan.kernel, g, epi, rowvec, st);
    else launch_layout<false, false>(plan.kernel, g, epi, rowvec, st);
}
}  // namespace gemmk
