// Causal self-attention, forward and backward, as fused flash-style kernels for gfx950.
// Replaces the reference's cuDNN path (llmc/cudnn_att.cpp:222 forward, :256 backward):
// QKV is read in place as (B,T,3,NH,hs), the output is (B,T,NH,hs), and the only thing kept for
// backward is one fp32 log-sum-exp per (b,h,t). CPU definition: train_gpt2.c:271-405.
//
// bf16 build (head sizes 64, 80, 96, 128). Everything is computed "transposed" so that no softmax statistic
// ever has to cross lanes. A 32x32 MFMA accumulator gives each lane ONE column and 16 rows;
// by computing S^T = K.Q^T the lane's column is a query, so the running max / sum / rescale
// of the online softmax are per-lane scalars (one cross-half exchange per tile for the max).
// The probabilities never leave registers: an accumulator, converted to bf16, already has the
// MFMA B-operand layout (lane = non-contracted index, 8 contracted values), provided the other
// operand is fetched in the same key order — which the transposing LDS read
// (ds_read_b64_tr_b16) does for free. The same identity drives backward:
//   dK/dV kernel: S = Q.K^T (lane = key), P and dS feed dV^T = dO^T.P and dK^T = Q^T.dS
//   dQ kernel:    S^T = K.Q^T (lane = query), dS^T feeds dQ^T = K^T.dS^T
// Two kernels instead of one with atomics: every output element has exactly one owner, so the
// result is deterministic, as the reference requests from cuDNN (cudnn_att.cpp:187-189).
//
// fp32 build: the same on the fp32 matrix instruction for heads of 32, 64, 96 and 128; other head sizes of either build take
// one-wave-per-row kernels (lanes = head dimensions).
#include "common.hpp"
#include "decode.hpp"
#include <type_traits>
#include <utility>
#include "../../include/llmk.h"

namespace {

#if !defined(LLMK_FP32)
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(4))) short s16x4;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;

constexpr float LOG2E = 1.4426950408889634f;

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// accumulator registers r = 8*s2 .. 8*s2+7 as a bf16 operand
__device__ __forceinline__ bf16x8 pack_acc(const f32x16& a, int s2) {
    bf16x8 o;
#pragma unroll
    for (int e = 0; e < 8; e++) o[e] = (__bf16)a[8 * s2 + e];
    return o;
}
// What the rounding to bf16 left over, itself a bf16 operand: hi + lo carries a probability to 2^-17. The heads of 80, 96 and
// 128 contract P and dS in both parts (two MFMAs on one fragment of the other operand): their results, which used to be
// formed in fp32 throughout, keep that precision. A head size of 64 rounds P and dS to bf16, as it always has.
__device__ __forceinline__ bf16x8 pack_acc_low(const f32x16& a, int s2, const bf16x8& hi) {
    bf16x8 o;
#pragma unroll
    for (int e = 0; e < 8; e++) o[e] = (__bf16)(a[8 * s2 + e] - (float)hi[e]);
    return o;
}
// The lane id as a value the compiler cannot trace back: what is derived from it (row offsets, per-lane pointers) is then
// formed where it is used and dies there, instead of being carried in registers through the tile loops of kernels that
// have none to spare.
__device__ __forceinline__ int fresh_lane(int lane) {
    asm volatile("" : "+v"(lane));
    return lane;
}
// max of a value with the one held by the lane 32 away (the other 16 keys of each 32-key block): one lane swap inside
// the vector ALU instead of a trip through the LDS crossbar, which sits in every step's dependent chain
__device__ __forceinline__ float fa_max_with_other_half(float v) {
    // As an instruction, not through __builtin_amdgcn_permlane32_swap: this compiler hands back the first result for both
    // elements of the builtin's pair, which silently drops the maximum (and overflows the exponentials as soon as scores
    // are large). The two wait states are the ones the compiler puts between a vector write and this instruction.
    unsigned a = __builtin_bit_cast(unsigned, v), b = a;
    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b));
    return fmaxf(__builtin_bit_cast(float, a), __builtin_bit_cast(float, b));
}
// row index (within a 32-row block) of accumulator register r for this lane
__device__ __forceinline__ int acc_row(int r, int lane) { return (r >> 2) * 8 + (lane >> 5) * 4 + (r & 3); }

// The causal mask of a 32 x 32 block on the diagonal (its first row and its first column are the same position; the
// direct-to-LDS kernels meet no other kind, all their blocks start at multiples of 32). Register r of lane l is row
// acc_row(r, l) against column l % 32, so WHICH LANES are masked in register r is a constant of r: a 64-bit lane mask
// that lives in scalar registers, and one select per element - where the per-lane form took an add, a compare and a
// select each, with wait states between them, a tenth of the forward loop's vector instructions at T = 1024.
// ROW_GT: rows past the column are masked (rows are keys: forward, dQ); else rows before it (rows are queries: dK/dV).
template <int R, bool ROW_GT>
constexpr unsigned long long fa_diag_lanes() {
    unsigned long long m = 0;
    for (int l = 0; l < 64; l++) {
        const int row = (R >> 2) * 8 + (l >> 5) * 4 + (R & 3), col = l & 31;
        if (ROW_GT ? row > col : row < col) m |= 1ull << l;
    }
    return m;
}
template <int R, bool ROW_GT>
__device__ __forceinline__ float fa_mask_one(float x, float fill) {
    // (the builtin, not the instruction in asm: x comes straight out of an MFMA, and the wait states between a matrix
    // instruction and a vector instruction that reads its result are the compiler's to insert - it does not look into asm)
    return __builtin_amdgcn_inverse_ballot_w64(fa_diag_lanes<R, ROW_GT>()) ? fill : x;
}
template <bool ROW_GT, int... R>
__device__ __forceinline__ void fa_mask_diag_seq(f32x16& a, float fill, std::integer_sequence<int, R...>) {
    ((a[R] = fa_mask_one<R, ROW_GT>(a[R], fill)), ...);
}
template <bool ROW_GT>
__device__ __forceinline__ void fa_mask_diag(f32x16& a, float fill) {
    fa_mask_diag_seq<ROW_GT>(a, fill, std::make_integer_sequence<int, 16>{});
}

// 4 consecutive head-dim values of one row -> 8-byte store
__device__ __forceinline__ void store4(floatX* p, float a, float b, float c, float d) {
    bf16x4 o;
    o[0] = (__bf16)a; o[1] = (__bf16)b; o[2] = (__bf16)c; o[3] = (__bf16)d;
    *reinterpret_cast<bf16x4*>(p) = o;
}

// ---- tiles filled by direct-to-LDS loads ---------------------------------------------------------
// A tile of 64 rows x HD columns (HD = the head size: 64, 80, 96 or 128) stored without padding; the 16-byte chunk c of
// row r sits at chunk c ^ swz(r). A direct-to-LDS load deposits a wave's 64 x 16 B linearly, so the swizzle is applied
// on the global side (the lane that fills slot p of a row fetches chunk p ^ swz(row)). swz is chosen so that 16 consecutive
// rows read at one chunk (MFMA operand along rows) and 4 rows x 64 B (transposing reads) both spread over all banks, a
// bank row being 16 chunks:
//   64  (8 chunks a row):  the three bits of row >> 1 in reverse order. Rows 2 apart (the ones a transposing read takes
//       from the same half of the banks in one cycle) land 64 bytes apart, and the 8 even (odd) rows of a 16-row column
//       read get 8 different chunks.
//   128 (16 chunks, every row starts at bank 0): the four bits of row in reverse order, for the same reason.
//   96  (12 chunks): rows r .. r + 3 already start 64 bytes apart; rows 4 apart, which start at the same bank, differ in
//       the low two bits of the chunk.
//   80  (10 chunks): 8 consecutive rows start at 8 different even chunks; rows 8 apart differ in the low bit.
template <int HD>
__device__ __forceinline__ int fa_swz(int row) {
    if constexpr (HD == 64) return (((row >> 1) & 1) << 2) | (((row >> 2) & 1) << 1) | ((row >> 3) & 1);
    else if constexpr (HD == 128) return ((row & 1) << 3) | ((row & 2) << 1) | ((row & 4) >> 1) | ((row & 8) >> 3);
    else if constexpr (HD == 96) return (row >> 2) & 3;
    else return (row >> 3) & 1;
}
template <int HD> struct FaTile {
    static constexpr int CPR = HD / 8, PITCH = HD * 2, BYTES = 64 * PITCH;
    static constexpr bool SPLIT = HD != 64;               // P and dS as two bf16 parts, see pack_acc_low
    static constexpr int KS = HD / 16;                    // 16-wide steps of a contraction over the head dimension
    static constexpr int NB = (HD + 31) / 32;             // 32-wide blocks of an output over it (80: the last one half used)
    static constexpr int NLD = (CPR + 3) / 4;             // 1 KiB pieces of a tile that one of four waves brings in
    // a 32-column read of the last block of 80 runs 32 bytes past the row: of the last row, past the tile
    static constexpr int SLOT = BYTES + (HD == 80 ? 1024 : 0);
    static constexpr float SCALE = HD == 64 ? 0.125f : HD == 80 ? 0.11180339887498949f : HD == 96 ? 0.10206207261596575f : 0.08838834764831845f;
};
constexpr int SW_TILE = FaTile<64>::BYTES;
typedef __attribute__((address_space(3))) void* fa_lds_ptr;
template <int HD>
struct FaLane {
    unsigned rowb;          // frag along rows: byte offset of (row = lane%32, K step 0); see fa_rows_off for step s
    unsigned colb0, colb1;  // transposing reads: byte offsets of this lane's two 8-byte pieces for (kbase 0, column block 0)
    unsigned ld_off[FaTile<HD>::NLD];   // staging: byte offset inside the global tile of this lane's 16 bytes of piece i (row stride given at init)
    __device__ __forceinline__ void init(int lane, int wave, size_t row_stride) {
        const int idx = lane & 31, half = lane >> 5;
        rowb = idx * FaTile<HD>::PITCH + ((half ^ fa_swz<HD>(idx)) << 4);
        const int s16 = lane & 15, grp = lane >> 4;
        const int r = 4 * (grp >> 1) + (s16 >> 2), col = (grp & 1) * 16 + 4 * (s16 & 3);
        colb0 = r * FaTile<HD>::PITCH + (((col >> 3) ^ fa_swz<HD>(r)) << 4) + (col & 7) * 2;
        colb1 = (r + 8) * FaTile<HD>::PITCH + (((col >> 3) ^ fa_swz<HD>(r + 8)) << 4) + (col & 7) * 2;
#pragma unroll
        for (int i = 0; i < FaTile<HD>::NLD; i++) ld_off[i] = piece_off(lane, wave, i, 63, row_stride);
    }
    // a 4-wave workgroup: wave w deposits the 1 KiB pieces w, w + 4, ... Rows past last_row (the end of the sequence in a
    // ragged tile) are replaced by that row: readable, and what is computed from them is masked.
    static __device__ __forceinline__ unsigned piece_off(int lane, int wave, int i, int last_row, size_t row_stride) {
        const int slot = (wave + 4 * i) * 64 + lane, row = slot / FaTile<HD>::CPR, p = slot % FaTile<HD>::CPR;
        return (unsigned)((size_t)min(row, last_row) * row_stride + ((p ^ fa_swz<HD>(row)) * 8)) * (unsigned)sizeof(floatX);
    }
};
// A wave-uniform pointer, stated as such: pointer arithmetic that follows stays in scalar registers, which is where
// fa_tile_request needs the tile address. (The builtin returns int: the halves are widened as unsigned.)
template <typename T>
__device__ __forceinline__ const T* fa_uniform(const T* p) {
    const unsigned long long v = (unsigned long long)(size_t)p;
    const unsigned hi = (unsigned)__builtin_amdgcn_readfirstlane((int)(v >> 32));
    const unsigned lo = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)v);
    return reinterpret_cast<const T*>((size_t)(((unsigned long long)hi << 32) | (unsigned long long)lo));
}
// Request this wave's pieces of the tile whose first row is at `gtile` (off: the lane's offsets inside it). The loads are
// issued from inline asm, M0 (the LDS destination) included: when the compiler knows of a direct-to-LDS load in
// flight it makes every later LDS read wait for it, whatever the read's address, which would turn the prefetch into
// a synchronous copy. The kernel waits for its loads explicitly (fa_tiles_landed) before the barrier that publishes them.
template <int HD>
__device__ __forceinline__ void fa_request_pieces(const unsigned (&off)[FaTile<HD>::NLD], const floatX* gtile, unsigned lds_tile, int wave) {
    const unsigned long long g = (unsigned long long)(size_t)gtile;
    const unsigned dst = lds_tile + wave * 1024;
    unsigned saved;
    if constexpr (FaTile<HD>::NLD == 2) {
        asm volatile("s_mov_b32 %0, m0\n\t"
                     "s_mov_b32 m0, %1\n\t"
                     "global_load_lds_dwordx4 %3, %2\n\t"
                     "s_add_u32 m0, m0, 0x1000\n\t"
                     "global_load_lds_dwordx4 %4, %2\n\t"
                     "s_mov_b32 m0, %0"
                     : "=&s"(saved) : "s"(dst), "s"(g), "v"(off[0]), "v"(off[1]) : "memory", "scc");
    } else if constexpr (FaTile<HD>::NLD == 3) {
        asm volatile("s_mov_b32 %0, m0\n\t"
                     "s_mov_b32 m0, %1\n\t"
                     "global_load_lds_dwordx4 %3, %2\n\t"
                     "s_add_u32 m0, m0, 0x1000\n\t"
                     "global_load_lds_dwordx4 %4, %2\n\t"
                     "s_mov_b32 m0, %0"
                     : "=&s"(saved) : "s"(dst), "s"(g), "v"(off[0]), "v"(off[1]) : "memory", "scc");
        if (FaTile<HD>::CPR == 12 || wave < 2)            // 80: ten pieces, the last two are waves 0 and 1's (wave-uniform)
            asm volatile("s_mov_b32 %0, m0\n\t"
                         "s_mov_b32 m0, %1\n\t"
                         "global_load_lds_dwordx4 %3, %2\n\t"
                         "s_mov_b32 m0, %0"
                         : "=&s"(saved) : "s"(dst + 0x2000u), "s"(g), "v"(off[2]) : "memory", "scc");
    } else {
        asm volatile("s_mov_b32 %0, m0\n\t"
                     "s_mov_b32 m0, %1\n\t"
                     "global_load_lds_dwordx4 %3, %2\n\t"
                     "s_add_u32 m0, m0, 0x1000\n\t"
                     "global_load_lds_dwordx4 %4, %2\n\t"
                     "s_add_u32 m0, m0, 0x1000\n\t"
                     "global_load_lds_dwordx4 %5, %2\n\t"
                     "s_add_u32 m0, m0, 0x1000\n\t"
                     "global_load_lds_dwordx4 %6, %2\n\t"
                     "s_mov_b32 m0, %0"
                     : "=&s"(saved) : "s"(dst), "s"(g), "v"(off[0]), "v"(off[1]), "v"(off[2]), "v"(off[3]) : "memory", "scc");
    }
}
template <int HD>
__device__ __forceinline__ void fa_tile_request(const FaLane<HD>& a, const floatX* gtile, unsigned lds_tile, int wave) {
    fa_request_pieces<HD>(a.ld_off, gtile, lds_tile, wave);
}
// The same for a tile that may end past the sequence (RAGGED; the kernels for whole tiles do not ask): rows_left > 0 rows
// of it exist.
template <int HD, bool RAGGED>
__device__ __forceinline__ void fa_tile_request(const FaLane<HD>& a, const floatX* gtile, unsigned lds_tile, int wave, int rows_left,
                                                size_t row_stride, int lane) {
    if (RAGGED && rows_left < 64) {                       // wave-uniform, at most once per tile of the last kind
        unsigned off[FaTile<HD>::NLD];
        const int ln = fresh_lane(lane);
#pragma unroll
        for (int i = 0; i < FaTile<HD>::NLD; i++) off[i] = FaLane<HD>::piece_off(ln, wave, i, rows_left - 1, row_stride);
        fa_request_pieces<HD>(off, gtile, lds_tile, wave);
    } else {
        fa_request_pieces<HD>(a.ld_off, gtile, lds_tile, wave);
    }
}
__device__ __forceinline__ void fa_tiles_landed() {
    __builtin_amdgcn_s_waitcnt(0x0F70);     // vmcnt(0), other counters untouched; as a builtin, so that the compiler also knows its own loads are done
    asm volatile("" ::: "memory");
}
// LDS reads of these tiles go through integer addresses: a read the compiler can trace to the array that a
// direct-to-LDS load is filling is preceded by a wait for every load in flight, which would undo the prefetch.
__device__ __forceinline__ unsigned fa_lds_addr(const void* p) {
    return (unsigned)(size_t)(__attribute__((address_space(3))) const char*)p;
}
// step s of a lane's operand along rows / column block d of a transposing read, from the address of step (block) 0: an
// XOR where the swizzle reaches those bits of the chunk, else an addition, which the read takes as its immediate offset
template <int HD>
__device__ __forceinline__ unsigned fa_rows_off(unsigned rowb, int s) {
    if constexpr (HD == 64 || HD == 128) return rowb ^ (unsigned)(s << 5);
    else if constexpr (HD == 96) return (rowb ^ (unsigned)((s & 1) << 5)) + (unsigned)((s >> 1) << 6);
    else return rowb + (unsigned)(s << 5);
}
template <int HD>
__device__ __forceinline__ unsigned fa_cols_off(unsigned colb, int d) {
    if constexpr (HD == 64 || HD == 128) return colb ^ (unsigned)(d << 6);
    else return colb + (unsigned)(d << 6);
}
template <int HD>
__device__ __forceinline__ bf16x8 fa_frag_rows(unsigned tile, const FaLane<HD>& a, int row0, int s) {
    return *reinterpret_cast<const __attribute__((address_space(3))) bf16x8*>((size_t)(tile + row0 * FaTile<HD>::PITCH + fa_rows_off<HD>(a.rowb, s)));
}
// The same reads for a kernel short of registers: the swizzled address of each step is formed at the read (one
// xor-add) rather than held for the life of the kernel.
// (lane ^ X) + tile as ONE vector instruction issued where it is written: stated in asm, the compiler neither hoists the
// four (eight) variants of an address into registers of their own nor copies the lane part first to protect it. X has to
// be an inline constant (0, 32, 64); 96 takes a xor and an add. `tile` is wave-uniform (a scalar register).
template <int X>
__device__ __forceinline__ unsigned fa_xad(unsigned lane_part, unsigned tile) {
    unsigned r;
    if constexpr (X == 0) asm volatile("v_add_u32 %0, %2, %1" : "=v"(r) : "v"(lane_part), "s"(tile));
    else if constexpr (X <= 64) asm volatile("v_xad_u32 %0, %1, %2, %3" : "=v"(r) : "v"(lane_part), "n"(X), "s"(tile));
    else asm volatile("v_xor_b32 %0, %2, %1\n\tv_add_u32 %0, %3, %0" : "=&v"(r) : "v"(lane_part), "n"(X), "s"(tile));
    return r;
}
template <int S>
__device__ __forceinline__ bf16x8 fa_frag_rows_lean(unsigned tile, const FaLane<64>& a, int row0) {
    return *reinterpret_cast<const __attribute__((address_space(3))) bf16x8*>((size_t)(fa_xad<(S << 5)>(a.rowb, tile) + (unsigned)(row0 * 128)));
}
__device__ __forceinline__ f32x4 fa_lds_f32x4(unsigned addr) {
    return *reinterpret_cast<const __attribute__((address_space(3))) f32x4*>((size_t)addr);
}
// Transposed operand of a swizzled tile: lane (idx = lane&31, half = lane>>5) receives, for e = 0..7,
//   tile[kbase + 8*(e/4) + 4*half + e%4][32*d + idx]
// i.e. the contracted index runs over tile ROWS, in exactly the order in which a 32x32 accumulator's registers
// r = 8*s2 .. 8*s2+7 enumerate its rows. Two transposing 8-byte reads.
template <int HD>
__device__ __forceinline__ bf16x8 fa_frag_cols(unsigned tile, const FaLane<HD>& a, int kbase, int d) {
    typedef s16x4 __attribute__((address_space(3))) * lds_ptr;
    const unsigned t = tile + kbase * FaTile<HD>::PITCH;
    s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(size_t)(t + fa_cols_off<HD>(a.colb0, d)));
    s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(size_t)(t + fa_cols_off<HD>(a.colb1, d)));
    union { struct { s16x4 a, b; } s; bf16x8 v; } u;
    u.s.a = lo; u.s.b = hi;
    return u.v;
}

template <int COL0>
__device__ __forceinline__ bf16x8 fa_frag_cols_lean(unsigned tile, const FaLane<64>& a, int kbase) {
    typedef s16x4 __attribute__((address_space(3))) * lds_ptr;
    constexpr int X = COL0 ? 64 : 0;
    const unsigned off = (unsigned)(kbase * 128);
    s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(size_t)(fa_xad<X>(a.colb0, tile) + off));
    s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(size_t)(fa_xad<X>(a.colb1, tile) + off));
    union { struct { s16x4 a, b; } s; bf16x8 v; } u;
    u.s.a = lo; u.s.b = hi;
    return u.v;
}

// Which (tile along T, batch*head) a workgroup works on. The grid is (tiles, B*NH) with x fastest, and workgroups
// are dealt round-robin over the 8 XCDs, each with its own L2: taken literally, the tiles of one head would land
// on 8 different XCDs and each would pull that head's K and V through its own L2. Instead XCD x takes the heads
// x, x+8, ... and walks all tiles of a head with consecutive workgroups, so a head's K/V cross HBM once.
__device__ __forceinline__ void fa_block_coords(int& tile, int& bh) {
    const int nt = gridDim.x, nbh = gridDim.y;
    tile = blockIdx.x; bh = blockIdx.y;
    if ((nbh & 7) == 0) {
        const int lin = blockIdx.y * nt + blockIdx.x;
        const int xcd = lin & 7, slot = lin >> 3;
        bh = (slot / nt) * 8 + xcd;
        tile = slot % nt;
    }
}

// The running reference point m of a row (log2 units) only has to stay near the row's maximum, not at it: the
// probabilities are exp2(s - m) and the final division by their sum takes m out again. Moving m costs 48 multiplies
// per lane (output and row-sum accumulators), a fifth of the loop's vector work, and with m at the exact maximum some
// row of the 32 moves in most steps. So a row's m follows its maximum only once a score exceeds m by FA_MAX_SLACK;
// until then probabilities may reach 2^FA_MAX_SLACK instead of 1, which neither bf16 nor the fp32 sums mind.
constexpr float FA_MAX_SLACK = 8.0f;

// ---- forward ----------------------------------------------------------------------------------
// 256 threads: wave w owns queries [128*qt + 32w, +32) and walks the key tiles up to its diagonal, 64 keys at a time, K and
// V brought in by direct-to-LDS loads. The loop is bound by the vector ALU at a head size of 64 (one exp2 per score costs as
// much as the two MFMAs that score takes part in; wider heads do more matrix work per score), so everything else per score
// is kept to a minimum: the first MFMA of a block starts from a constant zero instead of a cleared accumulator, maxima are
// taken three at a time. Without staging registers the kernel for 64 fits 128 VGPRs, four waves per SIMD; the wider ones hold
// an output of HD x 32 per wave and fit two. With the loads issued from inline asm the reads of the tile in use do not wait
// for the tile in flight.
// RAGGED: T is not a multiple of 128, so the last tiles of a head are cut (see fa_tile_request); the same arithmetic in
// the same order, so a row's bits do not depend on which of the two it went through.
// Workgroups take one query tile or two (nq tiles per head): see fa_tiles_paired.
// Measured against the one-wave-per-row kernels that the heads of 80, 96 and 128 used to take, whose every score is a 64-lane
// reduction on the vector ALU (2 x 2048 x 16 heads of 128, us): forward 15348 -> 92 (375 TFLOP/s of the causal half), dQ
// 15684 -> 114, dK/dV 17177 -> 189; 3 x 1000 x 16 heads of 96: 4705 -> 43, 4845 -> 52, 5708 -> 65. What bounds them now: two
// waves per SIMD (registers), a third of the matrix work being the low parts of P and dS.
template <int HD, bool RAGGED>
__global__ void __launch_bounds__(256, HD == 64 ? 4 : 2)
fa_forward_dma_kernel(floatX* __restrict__ out, float* __restrict__ stats, const floatX* __restrict__ qkv, int T, int NH, int nq, bool paired) {
    constexpr int NWAVES = 4;
    constexpr int KS = FaTile<HD>::KS, NB = FaTile<HD>::NB;
    __shared__ __attribute__((aligned(1024))) char sK[2][FaTile<HD>::BYTES];
    __shared__ __attribute__((aligned(1024))) char sV[2][FaTile<HD>::SLOT];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int tile_x, bh;
    fa_block_coords(tile_x, bh);
    // A workgroup takes TWO tiles of 128 queries of its head, nq - 1 - x and then x (one when they coincide): together
    // they walk nq + 1 pairs of key tiles whatever x is, so every workgroup of the launch does the same work, and the
    // second tile's first keys are already on their way when the first tile is stored. Launches too small for that take
    // one, the longest first.
    const int qt_first = nq - 1 - tile_x, qt_second = tile_x;
    const int nphase = qt_first == qt_second || !paired ? 1 : 2;
    const int b = bh / NH, h = bh % NH;
    const int C = NH * HD;
    const size_t C3 = 3 * (size_t)C;
    const floatX* base = qkv + (size_t)b * T * C3 + h * HD;
    // the first K and V tiles are requested before anything else: they travel while the wave fetches its own rows
    const int uwave = __builtin_amdgcn_readfirstlane(wave);
    FaLane<HD> la;
    la.init(lane, uwave, C3);
    const floatX* kbase = fa_uniform(base + C);
    const floatX* vbase = fa_uniform(base + 2 * C);
    fa_tile_request<HD, RAGGED>(la, kbase, fa_lds_addr(sK[0]), uwave, T, C3, lane);
    fa_tile_request<HD, RAGGED>(la, vbase, fa_lds_addr(sV[0]), uwave, T, C3, lane);
    constexpr int GQ = 32 * NWAVES;                       // queries per tile
    const float c = FaTile<HD>::SCALE * LOG2E;            // 1/sqrt(HD) folded into the exp2 argument
    const f32x16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    bf16x8 ones;
#pragma unroll
    for (int e = 0; e < 8; e++) ones[e] = (__bf16)1.0f;

    for (int phase = 0; phase < nphase; phase++) {
        const int qt = phase == 0 ? qt_first : qt_second;
        const int qw0 = qt * GQ + uwave * 32;             // wave-uniform
        bf16x8 qf[KS];
        {
            const int ln = fresh_lane(lane), idx = ln & 31, half = ln >> 5, my_q = qw0 + idx;
#pragma unroll
        for (int s = 0; s < KS; s++) {
            if (my_q < T) qf[s] = *reinterpret_cast<const bf16x8*>(base + (size_t)my_q * C3 + 16 * s + 8 * half);
            else
#pragma unroll
                for (int e = 0; e < 8; e++) qf[s][e] = (__bf16)0.f;
        }
        }
        f32x16 o[NB];
#pragma unroll
        for (int d = 0; d < NB; d++)
#pragma unroll
            for (int r = 0; r < 16; r++) o[d][r] = 0.f;
        float m = -INFINITY;
        // The softmax denominator is accumulated by the matrix cores, which have cycles to spare here: a ones operand
        // in place of V makes every row of this accumulator the sum over keys of the (bf16-rounded) probabilities of
        // the lane's query - the same rounded values that multiply V.
        f32x16 lacc = zero;

        const int n_kt = 2 * qt + 2;                          // (RAGGED: the last of them may start past the end: nobody's keys)
        // the wave's own rows have arrived (and, for the first tile, the first keys; the second tile's first keys were
        // awaited by the step that ended the first tile): after this the only loads in flight are tile requests
        fa_tiles_landed();
        if (phase == 0) __syncthreads();

        // One step = one tile of 64 keys. The buffer is a compile-time constant (the loop below alternates two copies of
        // the step), so a fragment's LDS address is a lane register plus an immediate: no vector add per read.
        auto step = [&](int j, auto bufc) {
            constexpr int BUF = decltype(bufc)::value;
            const unsigned tk = fa_lds_addr(sK[BUF]), tv = fa_lds_addr(sV[BUF]);
            constexpr int buf = BUF ^ 1;
            if (j + 1 < n_kt) {                          // the other buffer was last read before the barrier that ended the previous step
                const int left = T - 64 * (j + 1);
                if (!RAGGED || left > 0) {
                    fa_tile_request<HD, RAGGED>(la, kbase + (size_t)(64 * (j + 1)) * C3, fa_lds_addr(sK[buf]), uwave, left, C3, lane);
                    fa_tile_request<HD, RAGGED>(la, vbase + (size_t)(64 * (j + 1)) * C3, fa_lds_addr(sV[buf]), uwave, left, C3, lane);
                }
            } else if (phase + 1 < nphase) {             // the second tile starts over at the head's first keys
                fa_tile_request<HD, RAGGED>(la, kbase, fa_lds_addr(sK[buf]), uwave, T, C3, lane);
                fa_tile_request<HD, RAGGED>(la, vbase, fa_lds_addr(sV[buf]), uwave, T, C3, lane);
            }
            auto kfrag = [&](int row0, int s) -> bf16x8 { return fa_frag_rows(tk, la, row0, s); };
            auto vfrag = [&](int kb, int d) -> bf16x8 { return fa_frag_cols(tv, la, kb, d); };
            if (64 * j <= qw0 + 31 && (!RAGGED || 64 * j < T)) {   // else: every key of this tile is in the future of this wave (past the end)
                // S^T for both 32-key blocks, the two accumulation chains interleaved
                f32x16 sacc[2];
                sacc[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kfrag(0, 0), qf[0], zero, 0, 0, 0);
                sacc[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kfrag(32, 0), qf[0], zero, 0, 0, 0);
#pragma unroll
                for (int s = 1; s < KS; s++) {
                    sacc[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kfrag(0, s), qf[s], sacc[0], 0, 0, 0);
                    sacc[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kfrag(32, s), qf[s], sacc[1], 0, 0, 0);
                }
                if (64 * j + 63 > qw0) {                      // diagonal tile: some (key, query) pairs are masked (wave-uniform test)
                    asm volatile("" ::: "memory");            // keep this a branch: off the diagonal the selects are pure overhead
                    // qw0 - 64 j is 0 (the first 32 keys are the wave's diagonal block, the other 32 all in the future) or 32
                    // (the first 32 all visible, the other 32 the diagonal block)
                    if (qw0 == 64 * j) {
                        fa_mask_diag<true>(sacc[0], -INFINITY);
#pragma unroll
                        for (int r = 0; r < 16; r++) sacc[1][r] = -INFINITY;
                    } else {
                        fa_mask_diag<true>(sacc[1], -INFINITY);
                    }
                }
                float mx = fmaxf(sacc[0][0], sacc[1][0]);
#pragma unroll
                for (int r = 1; r < 16; r++) mx = fmaxf(fmaxf(mx, sacc[0][r]), sacc[1][r]);     // v_max3_f32
                mx = fa_max_with_other_half(mx);
                const float m_top = fmaxf(m, mx * c);
                const bool outgrown = m_top > m + FA_MAX_SLACK;
                if (__builtin_amdgcn_ballot_w64(outgrown) != 0) {   // some row's scores outgrew its reference point: rescale
                    asm volatile("" ::: "memory");
                    // every row decides for itself, so that what a row computes depends on that row's scores alone
                    const float m_new = outgrown ? m_top : m;
                    const float alpha = fast_exp2(m - m_new);
                    m = m_new;
#pragma unroll
                    for (int r = 0; r < 16; r++) lacc[r] *= alpha;
#pragma unroll
                    for (int d = 0; d < NB; d++)
#pragma unroll
                        for (int r = 0; r < 16; r++) o[d][r] *= alpha;
                }
#pragma unroll
                for (int kb = 0; kb < 2; kb++)
#pragma unroll
                    for (int r = 0; r < 16; r++)
                        sacc[kb][r] = fast_exp2(fmaf(sacc[kb][r], c, -m));
#pragma unroll
                for (int s2 = 0; s2 < 4; s2++) {
                    const bf16x8 pf = pack_acc(sacc[s2 >> 1], s2 & 1);
                    lacc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ones, pf, lacc, 0, 0, 0);       // every row: sum over keys of P
                    if constexpr (FaTile<HD>::SPLIT) {
                        const bf16x8 pl = pack_acc_low(sacc[s2 >> 1], s2 & 1, pf);
                        lacc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ones, pl, lacc, 0, 0, 0);
#pragma unroll
                        for (int d = 0; d < NB; d++) {
                            const bf16x8 vf = vfrag(16 * s2, d);
                            o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, pf, o[d], 0, 0, 0);
                            o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, pl, o[d], 0, 0, 0);
                        }
                    } else {
#pragma unroll
                        for (int d = 0; d < NB; d++)
                            o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vfrag(16 * s2, d), pf, o[d], 0, 0, 0);
                    }
                }
            }
            fa_tiles_landed();
            __syncthreads();
        };
        for (int j = 0; j < n_kt; j += 2) {             // n_kt is even: a tile of 128 queries ends on a multiple of 128 keys
            step(j, std::integral_constant<int, 0>{});
            step(j + 1, std::integral_constant<int, 1>{});
        }

        const float l = lacc[0];                              // complete: the MFMA already summed over all 32 keys of both halves
        const int ln = fresh_lane(lane), idx = ln & 31, half = ln >> 5, my_q = qw0 + idx;
        if (my_q < T) {
            const float inv = 1.0f / l;
            floatX* dst = out + ((size_t)b * T + my_q) * C + h * HD;
#pragma unroll
            for (int d = 0; d < NB; d++)
#pragma unroll
                for (int g = 0; g < 4; g++)
                    if (32 * d + 8 * g < HD) store4(dst + 32 * d + 8 * g + 4 * half, o[d][4 * g] * inv, o[d][4 * g + 1] * inv, o[d][4 * g + 2] * inv, o[d][4 * g + 3] * inv);
            if (stats && half == 0) stats[((size_t)b * NH + h) * T + my_q] = (m + __log2f(l)) * 0.6931471805599453f;
        }
    }
}

// ---- backward: dK, dV --------------------------------------------------------------------------------
// wave w owns keys [128*kt + 32w, +32) and walks all later query tiles; Q and dO tiles come in by direct-to-LDS loads.
// RAGGED: T is not a multiple of 64. LDS_STATS: the per-query statistics of a head fit in LDS beside the tiles (T up to 4096
// at least); else they are read from memory where they are used.
template <int HD, bool RAGGED, bool LDS_STATS>
__global__ void __launch_bounds__(256, HD == 64 ? 1 : 2)
fa_backward_dkdv_dma_kernel(floatX* __restrict__ dqkv, const floatX* __restrict__ dout, const floatX* __restrict__ qkv,
                        const float* __restrict__ stats, const float* __restrict__ Dsum, int T, int NH, int nk, bool paired) {
    constexpr int KS = FaTile<HD>::KS, NB = FaTile<HD>::NB;
    constexpr int SLOT = HD == 64 ? SW_TILE : 2 * SW_TILE;       // the power of two that holds a tile
    static_assert(FaTile<HD>::SLOT <= SLOT, "a tile fits its slot");
    // Q tiles in sT[0..1], dO tiles in sT[2..3]. One array, aligned to twice the tile pair: the buffer in use is one bit of an
    // LDS address, and the dO tile of a buffer is a constant 2 * SLOT behind its Q tile.
    __shared__ __attribute__((aligned(4 * SLOT))) char sT[4][SLOT];
    extern __shared__ __attribute__((aligned(16))) float sStat[];   // [2][T rounded up to 64]: log-sum-exp (in log2 units) and -rowsum(dO*O) of every query of this head
    const int Tp = RAGGED ? (T + 63) & ~63 : T;
    float* sLall = sStat;
    float* sDall = sStat + Tp;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int tile_x, bh;
    fa_block_coords(tile_x, bh);
    // Two tiles of 128 keys per workgroup, x (the one with more queries after it) and then nk - 1 - x (one when they
    // coincide): equal work for every workgroup of the launch, and the second tile's first queries are on their way
    // when the first tile is stored. Launches too small for that take one.
    const int kt_first = tile_x, kt_second = nk - 1 - tile_x;
    const int nphase = kt_first == kt_second || !paired ? 1 : 2;
    const int b = bh / NH, h = bh % NH;
    const int C = NH * HD;
    const size_t C3 = 3 * (size_t)C;
    const floatX* base = qkv + (size_t)b * T * C3 + h * HD;      // reassigned below, stated uniform
    const floatX* dobase = dout + (size_t)b * T * C + h * HD;
    const float* lbase = stats + ((size_t)b * NH + h) * T;
    const float* dbase = Dsum + ((size_t)b * NH + h) * T;
    const float c = FaTile<HD>::SCALE * LOG2E;
    // the first Q and dO tiles are requested before anything else: they travel while the wave fetches its own rows
    const int q_end = CEIL_DIV(T, 64);
    const int uwave = __builtin_amdgcn_readfirstlane(wave);
    FaLane<HD> laq, lado;
    laq.init(lane, uwave, C3);
    lado.init(lane, uwave, (size_t)C);
    base = fa_uniform(base);
    dobase = fa_uniform(dobase);
    {
        const int q_first = (kt_first * 128) / 64;
        fa_tile_request<HD, RAGGED>(laq, base + (size_t)(64 * q_first) * C3, fa_lds_addr(sT[0]), uwave, T - 64 * q_first, C3, lane);
        fa_tile_request<HD, RAGGED>(lado, dobase + (size_t)(64 * q_first) * C, fa_lds_addr(sT[2]), uwave, T - 64 * q_first, (size_t)C, lane);
        // the per-query statistics of the head go to LDS once (the first tile's queries include the second's): no global
        // loads besides the tiles inside the loops. A query past the end gets an infinite log-sum-exp: its probabilities are 0.
        if (LDS_STATS) {
            for (int q = 64 * q_first + tid; q < T; q += 256) { sLall[q] = lbase[q] * LOG2E; sDall[q] = -dbase[q]; }    // negated: see below
            if (RAGGED && tid < Tp - T) { sLall[T + tid] = INFINITY; sDall[T + tid] = 0.f; }
        }
    }
    int buf = 0;
    // LDS addresses of this lane's operand pieces in the Q tile of the buffer in use. Everything that is the same for all
    // lanes about a read (the 32-query block, the 16-query step, the dO tile, and the K step or column block where the tile
    // layout adds it) is an immediate offset, and the change of buffer is one XOR per register and iteration: no address
    // arithmetic at the reads themselves (it was a vector add per read, a quarter of the loop's vector instructions at 64).
    // Where the layout XORs a K step or column block in, there is a register for each at 64; at 128 that would be sixteen of
    // a kernel that has none to spare, and the XOR is done at the read.
    constexpr int NAR = HD == 64 ? 4 : HD == 96 ? 2 : 1, NAC = HD == 64 ? 2 : 1;
    unsigned ar[NAR], ac[2 * NAC];
    {
        const unsigned t0 = fa_lds_addr(sT[0]);
#pragma unroll
        for (int s = 0; s < NAR; s++) ar[s] = t0 + (laq.rowb ^ (unsigned)(s << 5));
#pragma unroll
        for (int d = 0; d < NAC; d++) { ac[2 * d] = t0 + (laq.colb0 ^ (unsigned)(d << 6)); ac[2 * d + 1] = t0 + (laq.colb1 ^ (unsigned)(d << 6)); }
    }
    typedef const __attribute__((address_space(3))) bf16x8* lds_frag_ptr;
    typedef s16x4 __attribute__((address_space(3))) * lds_tr_ptr;
    auto rows_frag = [&](bool of_do, int qb, int s) -> bf16x8 {
        const unsigned a = HD == 64 ? ar[s % NAR] : HD == 96 ? ar[s % NAR] + (unsigned)((s >> 1) << 6) : fa_rows_off<HD>(ar[0], s);
        return *reinterpret_cast<lds_frag_ptr>((size_t)(a + (unsigned)(32 * qb * FaTile<HD>::PITCH + (of_do ? 2 * SLOT : 0))));
    };
    auto cols_frag = [&](bool of_do, int kbase, int d) -> bf16x8 {
        const unsigned off = (unsigned)(kbase * FaTile<HD>::PITCH + (of_do ? 2 * SLOT : 0));
        const unsigned lo = HD == 64 ? ac[2 * (d % NAC)] : fa_cols_off<HD>(ac[0], d), hi = HD == 64 ? ac[2 * (d % NAC) + 1] : fa_cols_off<HD>(ac[1], d);
        union { struct { s16x4 a, b; } s; bf16x8 v; } u;
        u.s.a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr_ptr)(size_t)(lo + off));
        u.s.b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr_ptr)(size_t)(hi + off));
        return u.v;
    };

    for (int phase = 0; phase < nphase; phase++) {
        const int kt = phase == 0 ? kt_first : kt_second;
        const int kw0 = kt * 128 + uwave * 32;           // wave-uniform
        const int q_first = (kt * 128) / 64;
        bf16x8 kf[KS], vf[KS];
        {
        const int ln = fresh_lane(lane), idx = ln & 31, half = ln >> 5, my_k = kw0 + idx;
#pragma unroll
        for (int s = 0; s < KS; s++) {
            if (my_k < T) {
                kf[s] = *reinterpret_cast<const bf16x8*>(base + C + (size_t)my_k * C3 + 16 * s + 8 * half);
                vf[s] = *reinterpret_cast<const bf16x8*>(base + 2 * C + (size_t)my_k * C3 + 16 * s + 8 * half);
            } else {
#pragma unroll
                for (int e = 0; e < 8; e++) { kf[s][e] = (__bf16)0.f; vf[s][e] = (__bf16)0.f; }
            }
        }
        }
        f32x16 dv[NB], dk[NB];
#pragma unroll
        for (int d = 0; d < NB; d++)
#pragma unroll
            for (int r = 0; r < 16; r++) { dv[d][r] = 0.f; dk[d][r] = 0.f; }
        fa_tiles_landed();                               // the wave's own rows (and, first time, the first tiles and the statistics)
        if (phase == 0) __syncthreads();

        // this lane's four statistics of a 16-query group: one address register per table, advanced by a tile per iteration
        unsigned stat_l = fa_lds_addr(sLall + 64 * q_first) + (unsigned)(lane >> 5) * 16u;
        unsigned stat_d = fa_lds_addr(sDall + 64 * q_first) + (unsigned)(lane >> 5) * 16u;
        for (int qi = q_first; qi < q_end; qi++) {
            buf ^= 1;
            if (qi + 1 < q_end) {
                const int left = T - 64 * (qi + 1);
                fa_tile_request<HD, RAGGED>(laq, base + (size_t)(64 * (qi + 1)) * C3, fa_lds_addr(sT[buf]), uwave, left, C3, lane);
                fa_tile_request<HD, RAGGED>(lado, dobase + (size_t)(64 * (qi + 1)) * C, fa_lds_addr(sT[2 + buf]), uwave, left, (size_t)C, lane);
            } else if (phase + 1 < nphase) {             // the second tile's first queries
                const int qn = (kt_second * 128) / 64;
                fa_tile_request<HD, RAGGED>(laq, base + (size_t)(64 * qn) * C3, fa_lds_addr(sT[buf]), uwave, T - 64 * qn, C3, lane);
                fa_tile_request<HD, RAGGED>(lado, dobase + (size_t)(64 * qn) * C, fa_lds_addr(sT[2 + buf]), uwave, T - 64 * qn, (size_t)C, lane);
            }
            // statistics of the 4 queries of group g of block qb: from LDS, or (very long sequences) from memory
            auto stat4 = [&](bool of_d, int qb, int g) -> f32x4 {
                if constexpr (LDS_STATS) {
                    return fa_lds_f32x4((of_d ? stat_d : stat_l) + (32 * qb + g * 8) * 4);
                } else {
                    f32x4 v;
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const int q = 64 * qi + 32 * qb + g * 8 + (lane >> 5) * 4 + e;
                        if (of_d) v[e] = q < T ? -dbase[q] : 0.f;
                        else v[e] = q < T ? lbase[q] * LOG2E : INFINITY;
                    }
                    return v;
                }
            };
#pragma unroll
            for (int qb = 0; qb < 2; qb++) {
                const int q0 = 64 * qi + 32 * qb;
                if (q0 + 31 < kw0) continue;                 // all 32 queries precede every key of this wave
                // dP - rowsum(dO*O) comes out of the matrix cores: the accumulator of dO.V^T starts from -rowsum(dO*O) of its
                // 16 queries (an accumulator register is a query here), which takes a subtraction per score off the vector ALU
                f32x16 sacc, pacc;
#pragma unroll
                for (int r = 0; r < 16; r++) sacc[r] = 0.f;
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    const f32x4 d4 = stat4(true, qb, g);
#pragma unroll
                    for (int e = 0; e < 4; e++) pacc[4 * g + e] = d4[e];
                }
                // one chain after the other, S first: its exponentials then run under the dP chain's matrix instructions, and
                // the -rowsum(dO*O) values have the S chain's time to arrive from LDS (measured against the two chains
                // interleaved step by step: -9 %). Written as ONE loop on purpose: two loops are fused by the
                // compiler, which puts the chains back side by side.
                constexpr int LAG = KS;                          // steps by which the dP chain runs behind the S chain
#pragma unroll
                for (int s = 0; s < KS + LAG; s++) {
                    if (s < KS) sacc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(rows_frag(false, qb, s), kf[s], sacc, 0, 0, 0);
                    if (s >= LAG) pacc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(rows_frag(true, qb, s - LAG), vf[s - LAG], pacc, 0, 0, 0);
                }
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    const f32x4 l4 = stat4(false, qb, g);
#pragma unroll
                    for (int e = 0; e < 4; e++) sacc[4 * g + e] = fast_exp2(fmaf(sacc[4 * g + e], c, -l4[e]));
                }
                if (q0 < kw0 + 31) {                             // diagonal block (wave-uniform test; rows past the end have no weight, see above)
                    asm volatile("" ::: "memory");                // keep this a branch: off the diagonal the selects are pure overhead
                    fa_mask_diag<false>(sacc, 0.f);               // q0 == kw0: query q0 + acc_row(r) against key kw0 + idx
                }
#pragma unroll
                for (int r = 0; r < 16; r++) pacc[r] = sacc[r] * pacc[r];
                // dV needs only P, dK needs dS: the dV matrix instructions go first and run under the vector work that forms dS
#pragma unroll
                for (int s2 = 0; s2 < 2; s2++) {
                    const bf16x8 pf = pack_acc(sacc, s2);
                    bf16x8 pl;
                    if constexpr (FaTile<HD>::SPLIT) pl = pack_acc_low(sacc, s2, pf);
#pragma unroll
                    for (int d = 0; d < NB; d++) {
                        const bf16x8 gf = cols_frag(true, 32 * qb + 16 * s2, d);
                        dv[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(gf, pf, dv[d], 0, 0, 0);
                        if constexpr (FaTile<HD>::SPLIT) dv[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(gf, pl, dv[d], 0, 0, 0);
                    }
                }
#pragma unroll
                for (int s2 = 0; s2 < 2; s2++) {
                    const bf16x8 dsf = pack_acc(pacc, s2);
                    bf16x8 dsl;
                    if constexpr (FaTile<HD>::SPLIT) dsl = pack_acc_low(pacc, s2, dsf);
#pragma unroll
                    for (int d = 0; d < NB; d++) {
                        const bf16x8 qf = cols_frag(false, 32 * qb + 16 * s2, d);
                        dk[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(qf, dsf, dk[d], 0, 0, 0);
                        if constexpr (FaTile<HD>::SPLIT) dk[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(qf, dsl, dk[d], 0, 0, 0);
                    }
                }
            }
#pragma unroll
            for (int s = 0; s < NAR; s++) ar[s] ^= (unsigned)SLOT;    // the other buffer
#pragma unroll
            for (int s = 0; s < 2 * NAC; s++) ac[s] ^= (unsigned)SLOT;
            // (in asm: as a plain addition the compiler re-bases the reads on the advanced value, with negative offsets that
            // a read cannot encode, and is back to an add per read)
            asm volatile("v_add_u32 %0, 0x100, %0\n\tv_add_u32 %1, 0x100, %1" : "+v"(stat_l), "+v"(stat_d));
            fa_tiles_landed();
            __syncthreads();
        }

        const int ln = fresh_lane(lane), idx = ln & 31, half = ln >> 5, my_k = kw0 + idx;
        if (my_k < T) {
            floatX* dkp = dqkv + ((size_t)b * T + my_k) * C3 + C + h * HD;
            floatX* dvp = dqkv + ((size_t)b * T + my_k) * C3 + 2 * C + h * HD;
#pragma unroll
            for (int d = 0; d < NB; d++)
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    const int col = 32 * d + 8 * g + 4 * half;
                    if (32 * d + 8 * g >= HD) continue;
                    constexpr float sc = FaTile<HD>::SCALE;
                    store4(dkp + col, dk[d][4 * g] * sc, dk[d][4 * g + 1] * sc, dk[d][4 * g + 2] * sc, dk[d][4 * g + 3] * sc);
                    store4(dvp + col, dv[d][4 * g], dv[d][4 * g + 1], dv[d][4 * g + 2], dv[d][4 * g + 3]);
                }
        }
    }
}

// ---- backward: dQ ---------------------------------------------------------------------------------------
// wave w owns queries [128*qt + 32w, +32) and walks the key tiles up to the diagonal, brought in by direct-to-LDS loads like
// the forward kernel's: no staging registers, at 64 four waves per SIMD. It also produces D = rowsum(dO * O) itself and
// writes it out, which saves a pass over dO and O: it runs before the dK/dV kernel. RAGGED: T is not a multiple of 64.
template <int HD, bool RAGGED>
__global__ void __launch_bounds__(256, HD == 64 ? 4 : 2)
fa_backward_dq_dma_kernel(floatX* __restrict__ dqkv, const floatX* __restrict__ dout, const floatX* __restrict__ qkv,
                          const floatX* __restrict__ o, const float* __restrict__ stats, float* __restrict__ Dsum, int T, int NH,
                          int nq, bool paired) {
    constexpr int KS = FaTile<HD>::KS, NB = FaTile<HD>::NB;
    __shared__ __attribute__((aligned(1024))) char sK[2][FaTile<HD>::SLOT];
    __shared__ __attribute__((aligned(1024))) char sV[2][FaTile<HD>::BYTES];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int tile_x, bh;
    fa_block_coords(tile_x, bh);
    // two query tiles per workgroup, nq - 1 - x and then x, as in fa_forward_dma_kernel: equal work for every workgroup (or one)
    const int qt_first = nq - 1 - tile_x, qt_second = tile_x;
    const int nphase = qt_first == qt_second || !paired ? 1 : 2;
    const int b = bh / NH, h = bh % NH;
    const int C = NH * HD;
    const size_t C3 = 3 * (size_t)C;
    const floatX* base = qkv + (size_t)b * T * C3 + h * HD;
    // the first K and V tiles are requested before anything else: they travel while the wave fetches its own rows
    const int uwave = __builtin_amdgcn_readfirstlane(wave);
    FaLane<HD> la;
    la.init(lane, uwave, C3);
    const floatX* kbase = fa_uniform(base + C);
    const floatX* vbase = fa_uniform(base + 2 * C);
    fa_tile_request<HD, RAGGED>(la, kbase, fa_lds_addr(sK[0]), uwave, T, C3, lane);
    fa_tile_request<HD, RAGGED>(la, vbase, fa_lds_addr(sV[0]), uwave, T, C3, lane);
    const float c = FaTile<HD>::SCALE * LOG2E;
    int buf = 0;

    for (int phase = 0; phase < nphase; phase++) {
        const int qt = phase == 0 ? qt_first : qt_second;
        const int qw0 = qt * 128 + uwave * 32;           // wave-uniform
        bf16x8 qf[KS], dof[KS];
        float lse2, dsum = 0.f;
        {
        const int ln = fresh_lane(lane), idx = ln & 31, half = ln >> 5, my_q = qw0 + idx;
#pragma unroll
        for (int s = 0; s < KS; s++) {
            if (my_q < T) {
                qf[s] = *reinterpret_cast<const bf16x8*>(base + (size_t)my_q * C3 + 16 * s + 8 * half);
                dof[s] = *reinterpret_cast<const bf16x8*>(dout + ((size_t)b * T + my_q) * C + h * HD + 16 * s + 8 * half);
            } else {
#pragma unroll
                for (int e = 0; e < 8; e++) { qf[s][e] = (__bf16)0.f; dof[s][e] = (__bf16)0.f; }
            }
        }
        lse2 = my_q < T ? stats[((size_t)b * NH + h) * T + my_q] * LOG2E : 0.f;
        // D = rowsum(dO * O) of the lane's query from the dO values it already holds: the two halves of the wave own
        // half of the head dimensions each. The dK/dV kernel, launched after this one, reads D from memory.
        if (my_q < T) {
#pragma unroll
            for (int s = 0; s < KS; s++) {
                const bf16x8 of = *reinterpret_cast<const bf16x8*>(o + ((size_t)b * T + my_q) * C + h * HD + 16 * s + 8 * half);
#pragma unroll
                for (int e = 0; e < 8; e++) dsum = fmaf((float)dof[s][e], (float)of[e], dsum);
            }
        }
        dsum += __shfl_xor(dsum, 32, WAVE);
        if (my_q < T && half == 0) Dsum[((size_t)b * NH + h) * T + my_q] = dsum;
        }
        f32x16 dq[NB];
#pragma unroll
        for (int d = 0; d < NB; d++)
#pragma unroll
            for (int r = 0; r < 16; r++) dq[d][r] = 0.f;

        const int last_q = min(qt * 128 + 127, T - 1);
        const int n_kt = last_q / 64 + 1;
        fa_tiles_landed();                               // the wave's own rows (and the first keys of the first tile)
        if (phase == 0) __syncthreads();

        for (int j = 0; j < n_kt; j++) {
            const unsigned tk = fa_lds_addr(sK[buf]), tv = fa_lds_addr(sV[buf]);
            buf ^= 1;
            if (j + 1 < n_kt) {                          // the other buffer was last read before the barrier that ended the previous step
                const int left = T - 64 * (j + 1);
                fa_tile_request<HD, RAGGED>(la, kbase + (size_t)(64 * (j + 1)) * C3, fa_lds_addr(sK[buf]), uwave, left, C3, lane);
                fa_tile_request<HD, RAGGED>(la, vbase + (size_t)(64 * (j + 1)) * C3, fa_lds_addr(sV[buf]), uwave, left, C3, lane);
            } else if (phase + 1 < nphase) {             // the second tile starts over at the head's first keys
                fa_tile_request<HD, RAGGED>(la, kbase, fa_lds_addr(sK[buf]), uwave, T, C3, lane);
                fa_tile_request<HD, RAGGED>(la, vbase, fa_lds_addr(sV[buf]), uwave, T, C3, lane);
            }
#pragma unroll
            for (int kb = 0; kb < 2; kb++) {
                const int k0 = 64 * j + 32 * kb;
                if (k0 > qw0 + 31) continue;
                f32x16 sacc, pacc;
#pragma unroll
                for (int r = 0; r < 16; r++) { sacc[r] = 0.f; pacc[r] = 0.f; }
                if constexpr (HD == 64) {
                    sacc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa_frag_rows_lean<0>(tk, la, 32 * kb), qf[0], sacc, 0, 0, 0);
                    sacc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa_frag_rows_lean<1>(tk, la, 32 * kb), qf[1], sacc, 0, 0, 0);
                    sacc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa_frag_rows_lean<2>(tk, la, 32 * kb), qf[2], sacc, 0, 0, 0);
                    sacc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa_frag_rows_lean<3>(tk, la, 32 * kb), qf[3], sacc, 0, 0, 0);
                    pacc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa_frag_rows_lean<0>(tv, la, 32 * kb), dof[0], pacc, 0, 0, 0);
                    pacc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa_frag_rows_lean<1>(tv, la, 32 * kb), dof[1], pacc, 0, 0, 0);
                    pacc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa_frag_rows_lean<2>(tv, la, 32 * kb), dof[2], pacc, 0, 0, 0);
                    pacc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa_frag_rows_lean<3>(tv, la, 32 * kb), dof[3], pacc, 0, 0, 0);
                } else {
#pragma unroll
                    for (int s = 0; s < KS; s++) sacc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa_frag_rows(tk, la, 32 * kb, s), qf[s], sacc, 0, 0, 0);
#pragma unroll
                    for (int s = 0; s < KS; s++) pacc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa_frag_rows(tv, la, 32 * kb, s), dof[s], pacc, 0, 0, 0);
                }
#pragma unroll
                for (int r = 0; r < 16; r++) sacc[r] = fast_exp2(fmaf(sacc[r], c, -lse2));
                if (k0 + 31 > qw0) {                              // diagonal block (wave-uniform test)
                    asm volatile("" ::: "memory");                // keep this a branch: off the diagonal the selects are pure overhead
                    fa_mask_diag<true>(sacc, 0.f);                // k0 == qw0: key k0 + acc_row(r) against query qw0 + idx
                }
#pragma unroll
                for (int r = 0; r < 16; r++) pacc[r] = sacc[r] * (pacc[r] - dsum);
#pragma unroll
                for (int s2 = 0; s2 < 2; s2++) {
                    const bf16x8 dsf = pack_acc(pacc, s2);
                    if constexpr (HD == 64) {
                        dq[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa_frag_cols_lean<0>(tk, la, 32 * kb + 16 * s2), dsf, dq[0], 0, 0, 0);
                        dq[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa_frag_cols_lean<32>(tk, la, 32 * kb + 16 * s2), dsf, dq[1], 0, 0, 0);
                    } else {
                        const bf16x8 dsl = pack_acc_low(pacc, s2, dsf);
#pragma unroll
                        for (int d = 0; d < NB; d++) {
                            const bf16x8 kf = fa_frag_cols(tk, la, 32 * kb + 16 * s2, d);
                            dq[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, dsf, dq[d], 0, 0, 0);
                            dq[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, dsl, dq[d], 0, 0, 0);
                        }
                    }
                }
            }
            fa_tiles_landed();
            __syncthreads();
        }
        const int ln = fresh_lane(lane), idx = ln & 31, half = ln >> 5, my_q = qw0 + idx;
        if (my_q < T) {
            floatX* dqp = dqkv + ((size_t)b * T + my_q) * C3 + h * HD;
#pragma unroll
            for (int d = 0; d < NB; d++)
#pragma unroll
                for (int g = 0; g < 4; g++)
                    if (32 * d + 8 * g < HD) {
                        constexpr float sc = FaTile<HD>::SCALE;
                        store4(dqp + 32 * d + 8 * g + 4 * half, dq[d][4 * g] * sc, dq[d][4 * g + 1] * sc, dq[d][4 * g + 2] * sc, dq[d][4 * g + 3] * sc);
                    }
        }
    }
}

#endif  // !LLMK_FP32

// =============================================================================================
// Any head size up to 128, either storage type: one wavefront per row, lane l holds head dimensions l and l + 64
// (EPL = 2) or l alone (EPL = 1, hs <= 64). All arithmetic in fp32. For the head sizes
// that the MFMA kernels do not cover (none of the descriptors', train_gpt2.cu:519-559).
// =============================================================================================
template <int EPL>
__global__ void __launch_bounds__(256)
att_forward_rows_kernel(floatX* __restrict__ out, float* __restrict__ stats, const floatX* __restrict__ qkv, int B, int T,
                        int NH, int hs, int t0) {
    const int lane = threadIdx.x & 63, nt = T - t0;                       // positions t0 .. T - 1 of every head
    const size_t row = (size_t)blockIdx.x * 4 + (threadIdx.x >> 6);       // (b, h, t)
    if (row >= (size_t)B * NH * nt) return;
    const int t = t0 + (int)(row % nt), h = (int)((row / nt) % NH), b = (int)(row / ((size_t)nt * NH));
    const int C = NH * hs;
    const size_t C3 = 3 * (size_t)C;
    const floatX* base = qkv + (size_t)b * T * C3 + h * hs;
    const float scale = 1.0f / sqrtf((float)hs);
    bool act[EPL];
    float q[EPL], acc[EPL];
#pragma unroll
    for (int e = 0; e < EPL; e++) {
        act[e] = lane + 64 * e < hs;
        q[e] = act[e] ? to_f32(base[(size_t)t * C3 + lane + 64 * e]) : 0.f;
        acc[e] = 0.f;
    }
    float m = -INFINITY, l = 0.f;
    for (int t2 = 0; t2 <= t; t2++) {
        float qk = 0.f, v[EPL];
#pragma unroll
        for (int e = 0; e < EPL; e++) {
            const float k = act[e] ? to_f32(base[(size_t)t2 * C3 + C + lane + 64 * e]) : 0.f;
            v[e] = act[e] ? to_f32(base[(size_t)t2 * C3 + 2 * C + lane + 64 * e]) : 0.f;
            qk = e == 0 ? q[e] * k : qk + q[e] * k;
        }
        const float s = wave_sum(qk) * scale;
        const float m_new = fmaxf(m, s);
        const float alpha = expf(m - m_new), p = expf(s - m_new);
#pragma unroll
        for (int e = 0; e < EPL; e++) acc[e] = acc[e] * alpha + p * v[e];
        l = l * alpha + p;
        m = m_new;
    }
#pragma unroll
    for (int e = 0; e < EPL; e++)
        if (act[e]) out[((size_t)b * T + t) * C + h * hs + lane + 64 * e] = from_f32<floatX>(acc[e] / l);
    if (stats && lane == 0) stats[((size_t)b * NH + h) * T + t] = m + logf(l);
}

// dQ: one wave per query row
template <int EPL>
__global__ void __launch_bounds__(256)
att_backward_dq_rows_kernel(floatX* __restrict__ dqkv, const floatX* __restrict__ dout, const floatX* __restrict__ qkv,
                            const floatX* __restrict__ o, const float* __restrict__ stats, int B, int T, int NH, int hs) {
    const int lane = threadIdx.x & 63;
    const size_t row = (size_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= (size_t)B * NH * T) return;
    const int t = (int)(row % T), h = (int)((row / T) % NH), b = (int)(row / ((size_t)T * NH));
    const int C = NH * hs;
    const size_t C3 = 3 * (size_t)C;
    const floatX* base = qkv + (size_t)b * T * C3 + h * hs;
    const float scale = 1.0f / sqrtf((float)hs);
    const size_t orow = ((size_t)b * T + t) * C + h * hs;
    bool act[EPL];
    float q[EPL], go[EPL], dq[EPL], go_o = 0.f;
#pragma unroll
    for (int e = 0; e < EPL; e++) {
        const int d = lane + 64 * e;
        act[e] = d < hs;
        q[e] = act[e] ? to_f32(base[(size_t)t * C3 + d]) : 0.f;
        go[e] = act[e] ? to_f32(dout[orow + d]) : 0.f;
        const float prod = act[e] ? go[e] * to_f32(o[orow + d]) : 0.f;
        go_o = e == 0 ? prod : go_o + prod;
        dq[e] = 0.f;
    }
    const float dsum = wave_sum(go_o);
    const float lse = stats[((size_t)b * NH + h) * T + t];
    for (int t2 = 0; t2 <= t; t2++) {
        float k[EPL], qk = 0.f, gv = 0.f;
#pragma unroll
        for (int e = 0; e < EPL; e++) {
            const int d = lane + 64 * e;
            k[e] = act[e] ? to_f32(base[(size_t)t2 * C3 + C + d]) : 0.f;
            const float v = act[e] ? to_f32(base[(size_t)t2 * C3 + 2 * C + d]) : 0.f;
            qk = e == 0 ? q[e] * k[e] : qk + q[e] * k[e];
            gv = e == 0 ? go[e] * v : gv + go[e] * v;
        }
        const float s = wave_sum(qk) * scale;
        const float dp = wave_sum(gv);
        const float p = expf(s - lse);
#pragma unroll
        for (int e = 0; e < EPL; e++) dq[e] += p * (dp - dsum) * scale * k[e];
    }
#pragma unroll
    for (int e = 0; e < EPL; e++)
        if (act[e]) dqkv[((size_t)b * T + t) * C3 + h * hs + lane + 64 * e] = from_f32<floatX>(dq[e]);
}

// dK, dV: one wave per key row
template <int EPL>
__global__ void __launch_bounds__(256)
att_backward_dkdv_rows_kernel(floatX* __restrict__ dqkv, const floatX* __restrict__ dout, const floatX* __restrict__ qkv,
                              const floatX* __restrict__ o, const float* __restrict__ stats, int B, int T, int NH, int hs) {
    const int lane = threadIdx.x & 63;
    const size_t row = (size_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= (size_t)B * NH * T) return;
    const int t2 = (int)(row % T), h = (int)((row / T) % NH), b = (int)(row / ((size_t)T * NH));
    const int C = NH * hs;
    const size_t C3 = 3 * (size_t)C;
    const floatX* base = qkv + (size_t)b * T * C3 + h * hs;
    const float scale = 1.0f / sqrtf((float)hs);
    bool act[EPL];
    float k[EPL], v[EPL], dk[EPL], dv[EPL];
#pragma unroll
    for (int e = 0; e < EPL; e++) {
        const int d = lane + 64 * e;
        act[e] = d < hs;
        k[e] = act[e] ? to_f32(base[(size_t)t2 * C3 + C + d]) : 0.f;
        v[e] = act[e] ? to_f32(base[(size_t)t2 * C3 + 2 * C + d]) : 0.f;
        dk[e] = dv[e] = 0.f;
    }
    for (int t = t2; t < T; t++) {
        const size_t orow = ((size_t)b * T + t) * C + h * hs;
        float q[EPL], go[EPL], go_o = 0.f, qk = 0.f, gv = 0.f;
#pragma unroll
        for (int e = 0; e < EPL; e++) {
            const int d = lane + 64 * e;
            q[e] = act[e] ? to_f32(base[(size_t)t * C3 + d]) : 0.f;
            go[e] = act[e] ? to_f32(dout[orow + d]) : 0.f;
            const float prod = act[e] ? go[e] * to_f32(o[orow + d]) : 0.f;
            go_o = e == 0 ? prod : go_o + prod;
            qk = e == 0 ? q[e] * k[e] : qk + q[e] * k[e];
            gv = e == 0 ? go[e] * v[e] : gv + go[e] * v[e];
        }
        const float dsum = wave_sum(go_o);
        const float s = wave_sum(qk) * scale;
        const float dp = wave_sum(gv);
        const float p = expf(s - stats[((size_t)b * NH + h) * T + t]);
#pragma unroll
        for (int e = 0; e < EPL; e++) {
            dv[e] += p * go[e];
            dk[e] += p * (dp - dsum) * scale * q[e];
        }
    }
#pragma unroll
    for (int e = 0; e < EPL; e++)
        if (act[e]) {
            dqkv[((size_t)b * T + t2) * C3 + C + h * hs + lane + 64 * e] = from_f32<floatX>(dk[e]);
            dqkv[((size_t)b * T + t2) * C3 + 2 * C + h * hs + lane + 64 * e] = from_f32<floatX>(dv[e]);
        }
}

#if defined(LLMK_FP32)
// =============================================================================================
// fp32 build, heads of 32, 64, 96 and 128: the same two-kernel
// scheme as the bf16 build on v_mfma_f32_32x32x2_f32, true fp32 multiply-adds. A wave owns 32 queries (forward, dQ) or 32 keys
// (dK/dV), two waves share the 32-row tiles of the other side in LDS; the next tile is on its way in registers meanwhile.
//   * The contraction over head dimensions may take them in any order as long as both operands agree: lane half h holds dims
//     8 j + 4 h .. + 3 of its row, one 16-byte read for four matrix instructions.
//   * A 32 x 32 accumulator gives lane l column l % 32 and rows 8 g + 4 (l / 32) + e: as the second operand of the next product, its
//     register 4 g + e is the k pair (8 g + e, 8 g + 4 + e), so probabilities go from one product into the next without moving.
//   * Probabilities of masked positions are zeros that are multiplied like any other, as in the bf16 kernels.
// What bounds it: one dependent chain of matrix instructions per wave (64 cycles each) with the exponentials between; the
// one-wave-per-row kernels it replaces spend two 64-lane reductions per score.
// =============================================================================================
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) float f32x4;
constexpr int F_ROWS = 64, F_THREADS = 128;                       // rows of a workgroup (32 per wave)

// 32 rows x HD floats of a matrix with `ld` floats between rows, rows past the last one repeating it
template <int HD>
struct F32Tile {
    static constexpr int PITCH = HD + 4;                          // 16 rows' 16-byte reads cover all banks
    static constexpr int FLOATS = 32 * PITCH, N = 32 * HD / 4 / F_THREADS;
    f32x4 reg[N];
    __device__ __forceinline__ void load(const float* base, size_t ld, int r0, int rows) {
#pragma unroll
        for (int i = 0; i < N; i++) {
            const int q = (int)threadIdx.x + i * F_THREADS, row = q / (HD / 4), c = q % (HD / 4);
            reg[i] = *reinterpret_cast<const f32x4*>(base + (size_t)min(r0 + row, rows - 1) * ld + c * 4);
        }
    }
    __device__ __forceinline__ void store(float* lds) const {
#pragma unroll
        for (int i = 0; i < N; i++) {
            const int q = (int)threadIdx.x + i * F_THREADS, row = q / (HD / 4), c = q % (HD / 4);
            *reinterpret_cast<f32x4*>(lds + row * PITCH + c * 4) = reg[i];
        }
    }
};
template <int HD> using F32Row = f32x4[HD / 8];
template <int HD>
__device__ __forceinline__ void f32_row(F32Row<HD>& r, const float* row, int half) {
#pragma unroll
    for (int j = 0; j < HD / 8; j++) r[j] = *reinterpret_cast<const f32x4*>(row + 8 * j + 4 * half);
}
// rows of the LDS tile (accumulator rows) against this lane's row (accumulator column)
template <int HD>
__device__ __forceinline__ f32x16 f32_scores(const float* tile, const F32Row<HD>& mine, int lane) {
    const float* row = tile + (lane & 31) * F32Tile<HD>::PITCH + 4 * (lane >> 5);
    f32x16 a;
#pragma unroll
    for (int r = 0; r < 16; r++) a[r] = 0.f;
#pragma unroll
    for (int j = 0; j < HD / 8; j++) {
        const f32x4 t = *reinterpret_cast<const f32x4*>(row + 8 * j);
#pragma unroll
        for (int e = 0; e < 4; e++) a = __builtin_amdgcn_mfma_f32_32x32x2f32(t[e], mine[j][e], a, 0, 0, 0);
    }
    return a;
}
// acc[d] (rows: head dims 32 d ..) += tile^T . p, contracted over the tile's 32 rows
template <int HD>
__device__ __forceinline__ void f32_accumulate(f32x16 (&acc)[HD / 32], const float* tile, const f32x16& p, int lane) {
    const float* at = tile + 4 * (lane >> 5) * F32Tile<HD>::PITCH + (lane & 31);
#pragma unroll
    for (int r = 0; r < 16; r++)
#pragma unroll
        for (int d = 0; d < HD / 32; d++)
            acc[d] = __builtin_amdgcn_mfma_f32_32x32x2f32(at[(8 * (r >> 2) + (r & 3)) * F32Tile<HD>::PITCH + 32 * d], p[r], acc[d], 0, 0, 0);
}
// the lane's column of an accumulator over head dims to its row in memory
template <int HD>
__device__ __forceinline__ void f32_store(float* row, const f32x16 (&acc)[HD / 32], float denominator, int half) {
#pragma unroll
    for (int d = 0; d < HD / 32; d++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const f32x4 o = {acc[d][4 * g] / denominator, acc[d][4 * g + 1] / denominator, acc[d][4 * g + 2] / denominator, acc[d][4 * g + 3] / denominator};
            *reinterpret_cast<f32x4*>(row + 32 * d + 8 * g + 4 * half) = o;
        }
}

// queries q_first + 64 x ..; blocks of the later ones, which have more keys, are dealt first
template <int HD>
__global__ void __launch_bounds__(F_THREADS)
att_forward_f32_kernel(float* __restrict__ out, float* __restrict__ stats, const float* __restrict__ qkv, int T, int NH, int q_first) {
    __shared__ __attribute__((aligned(16))) float sk[F32Tile<HD>::FLOATS], sv[F32Tile<HD>::FLOATS];
    const int lane = threadIdx.x & 63, half = lane >> 5, wave = threadIdx.x >> 6;
    const int b = blockIdx.y / NH, h = blockIdx.y % NH, C = NH * HD;
    const size_t C3 = 3 * (size_t)C;
    const float* base = qkv + (size_t)b * T * C3 + h * HD;
    const int w0 = q_first + (int)(gridDim.x - 1 - blockIdx.x) * F_ROWS, q0 = w0 + wave * 32, q = q0 + (lane & 31);
    const float scale = 1.0f / sqrtf((float)HD);
    F32Row<HD> mine;
    f32_row<HD>(mine, base + (size_t)min(q, T - 1) * C3, half);
    f32x16 acc[HD / 32];
#pragma unroll
    for (int d = 0; d < HD / 32; d++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[d][r] = 0.f;
    float m = -INFINITY, l = 0.f;
    const int kend = min(w0 + F_ROWS, T);                         // keys of the workgroup's last query
    F32Tile<HD> tk, tv;
    tk.load(base + C, C3, 0, T);
    tv.load(base + 2 * C, C3, 0, T);
    for (int k0 = 0; k0 < kend; k0 += 32) {
        __syncthreads();
        tk.store(sk);
        tv.store(sv);
        __syncthreads();
        if (k0 + 32 < kend) {
            tk.load(base + C, C3, k0 + 32, T);
            tv.load(base + 2 * C, C3, k0 + 32, T);
        }
        if (k0 > q0) continue;                                    // the first wave is done a block earlier
        f32x16 s = f32_scores<HD>(sk, mine, lane);
        float top = m;
#pragma unroll
        for (int r = 0; r < 16; r++) {
            s[r] *= scale;
            if (k0 == q0 && (r >> 2) * 8 + 4 * half + (r & 3) > (lane & 31)) s[r] = -INFINITY;
            top = fmaxf(top, s[r]);
        }
        top = fmaxf(top, __shfl_xor(top, 32, 64));
        const float alpha = expf(m - top);
        float sum = 0.f;
#pragma unroll
        for (int r = 0; r < 16; r++) { s[r] = expf(s[r] - top); sum += s[r]; }
        l = l * alpha + (sum + __shfl_xor(sum, 32, 64));
        m = top;
#pragma unroll
        for (int d = 0; d < HD / 32; d++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[d][r] *= alpha;
        f32_accumulate<HD>(acc, sv, s, lane);
    }
    if (q >= T) return;
    f32_store<HD>(out + ((size_t)b * T + q) * C + h * HD, acc, l, half);
    if (stats && half == 0) stats[((size_t)b * NH + h) * T + q] = m + logf(l);
}

template <int HD>
__global__ void __launch_bounds__(F_THREADS)
att_backward_dq_f32_kernel(float* __restrict__ dqkv, const float* __restrict__ dout, const float* __restrict__ qkv,
                           const float* __restrict__ o, const float* __restrict__ stats, int T, int NH) {
    __shared__ __attribute__((aligned(16))) float sk[F32Tile<HD>::FLOATS], sv[F32Tile<HD>::FLOATS];
    const int lane = threadIdx.x & 63, half = lane >> 5, wave = threadIdx.x >> 6;
    const int b = blockIdx.y / NH, h = blockIdx.y % NH, C = NH * HD;
    const size_t C3 = 3 * (size_t)C;
    const float* base = qkv + (size_t)b * T * C3 + h * HD;
    const int w0 = (int)(gridDim.x - 1 - blockIdx.x) * F_ROWS, q0 = w0 + wave * 32, q = q0 + (lane & 31), qc = min(q, T - 1);
    const float scale = 1.0f / sqrtf((float)HD);
    const size_t orow = ((size_t)b * T + qc) * C + h * HD;
    F32Row<HD> mine, go;
    f32_row<HD>(mine, base + (size_t)qc * C3, half);
    f32_row<HD>(go, dout + orow, half);
    float dsum = 0.f;
    {
        F32Row<HD> fo;
        f32_row<HD>(fo, o + orow, half);
#pragma unroll
        for (int j = 0; j < HD / 8; j++)
#pragma unroll
            for (int e = 0; e < 4; e++) dsum += go[j][e] * fo[j][e];
        dsum += __shfl_xor(dsum, 32, 64);
    }
    const float lse = stats[((size_t)b * NH + h) * T + qc];
    f32x16 acc[HD / 32];
#pragma unroll
    for (int d = 0; d < HD / 32; d++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[d][r] = 0.f;
    const int kend = min(w0 + F_ROWS, T);
    F32Tile<HD> tk, tv;
    tk.load(base + C, C3, 0, T);
    tv.load(base + 2 * C, C3, 0, T);
    for (int k0 = 0; k0 < kend; k0 += 32) {
        __syncthreads();
        tk.store(sk);
        tv.store(sv);
        __syncthreads();
        if (k0 + 32 < kend) {
            tk.load(base + C, C3, k0 + 32, T);
            tv.load(base + 2 * C, C3, k0 + 32, T);
        }
        if (k0 > q0) continue;
        f32x16 p = f32_scores<HD>(sk, mine, lane);
        const f32x16 dp = f32_scores<HD>(sv, go, lane);
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const bool masked = k0 == q0 && (r >> 2) * 8 + 4 * half + (r & 3) > (lane & 31);
            p[r] = masked ? 0.f : expf(p[r] * scale - lse) * (dp[r] - dsum) * scale;
        }
        f32_accumulate<HD>(acc, sk, p, lane);
    }
    if (q < T) f32_store<HD>(dqkv + ((size_t)b * T + q) * C3 + h * HD, acc, 1.0f, half);
}

template <int HD>
__global__ void __launch_bounds__(F_THREADS)
att_backward_dkdv_f32_kernel(float* __restrict__ dqkv, const float* __restrict__ dout, const float* __restrict__ qkv,
                             const float* __restrict__ o, const float* __restrict__ stats, int T, int NH) {
    __shared__ __attribute__((aligned(16))) float sq[F32Tile<HD>::FLOATS], sg[F32Tile<HD>::FLOATS], sl[32], sd[32];
    const int lane = threadIdx.x & 63, half = lane >> 5, wave = threadIdx.x >> 6;
    const int b = blockIdx.y / NH, h = blockIdx.y % NH, C = NH * HD;
    const size_t C3 = 3 * (size_t)C;
    const float* base = qkv + (size_t)b * T * C3 + h * HD;
    const float *gbase = dout + (size_t)b * T * C + h * HD, *obase = o + (size_t)b * T * C + h * HD;
    const float* lbase = stats + ((size_t)b * NH + h) * T;
    const int w0 = (int)blockIdx.x * F_ROWS, k0 = w0 + wave * 32, k = k0 + (lane & 31), kc = min(k, T - 1);
    const float scale = 1.0f / sqrtf((float)HD);
    F32Row<HD> mk, mv;
    f32_row<HD>(mk, base + C + (size_t)kc * C3, half);
    f32_row<HD>(mv, base + 2 * C + (size_t)kc * C3, half);
    f32x16 dk[HD / 32], dv[HD / 32];
#pragma unroll
    for (int d = 0; d < HD / 32; d++)
#pragma unroll
        for (int r = 0; r < 16; r++) dk[d][r] = dv[d][r] = 0.f;
    F32Tile<HD> tq, tg;
    tq.load(base, C3, w0, T);
    tg.load(gbase, C, w0, T);
    float lse = 0.f, dsum = 0.f;
    auto load_rows = [&](int t0) {                                // D = rowsum(dO * O): four threads to a row
        const int row = (int)threadIdx.x >> 2, part = threadIdx.x & 3;
        const size_t at = (size_t)min(t0 + row, T - 1) * C + part * (HD / 4);
        float s = 0.f;
#pragma unroll
        for (int c = 0; c < HD / 4; c += 4) {
            const f32x4 x = *reinterpret_cast<const f32x4*>(gbase + at + c), y = *reinterpret_cast<const f32x4*>(obase + at + c);
#pragma unroll
            for (int e = 0; e < 4; e++) s += x[e] * y[e];
        }
        s += __shfl_xor(s, 1, 64);
        dsum = s + __shfl_xor(s, 2, 64);
        lse = lbase[min(t0 + row, T - 1)];
    };
    load_rows(w0);
    for (int t0 = w0; t0 < T; t0 += 32) {
        __syncthreads();
        tq.store(sq);
        tg.store(sg);
        if ((threadIdx.x & 3) == 0) { sl[threadIdx.x >> 2] = lse; sd[threadIdx.x >> 2] = dsum; }
        __syncthreads();
        if (t0 + 32 < T) {
            tq.load(base, C3, t0 + 32, T);
            tg.load(gbase, C, t0 + 32, T);
            load_rows(t0 + 32);
        }
        if (t0 < k0) continue;                                    // the second wave starts a block later
        f32x16 p = f32_scores<HD>(sq, mk, lane), ds = f32_scores<HD>(sg, mv, lane);
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int row = (r >> 2) * 8 + 4 * half + (r & 3);
            const bool out_of_it = (t0 == k0 && row < (lane & 31)) || t0 + row >= T;
            p[r] = out_of_it ? 0.f : expf(p[r] * scale - sl[row]);
            ds[r] = out_of_it ? 0.f : p[r] * (ds[r] - sd[row]) * scale;
        }
        f32_accumulate<HD>(dv, sg, p, lane);
        f32_accumulate<HD>(dk, sq, ds, lane);
    }
    if (k < T) {
        float* row = dqkv + ((size_t)b * T + k) * C3 + h * HD;
        f32_store<HD>(row + C, dk, 1.0f, half);
        f32_store<HD>(row + 2 * C, dv, 1.0f, half);
    }
}

template <class F>
bool with_f32_head(int hs, F f) {
    switch (hs) {
        case 32: f(std::integral_constant<int, 32>{}); return true;
        case 64: f(std::integral_constant<int, 64>{}); return true;
        case 96: f(std::integral_constant<int, 96>{}); return true;
        case 128: f(std::integral_constant<int, 128>{}); return true;
        default: return false;
    }
}
bool f32_aligned(const void* a, const void* b, const void* c, const void* d) {
    return (((uintptr_t)a | (uintptr_t)b | (uintptr_t)c | (uintptr_t)d) % 16) == 0;
}
#endif

void launch_forward_rows(floatX* out, float* stats, const floatX* qkv, int B, int T, int NH, int hs, int t0, hipStream_t st) {
#if defined(LLMK_FP32)
    if (t0 % 32 == 0 && B * NH <= 65535 && f32_aligned(out, qkv, nullptr, nullptr) && with_f32_head(hs, [&](auto hd) {
            att_forward_f32_kernel<decltype(hd)::value><<<dim3(CEIL_DIV(T - t0, F_ROWS), B * NH), F_THREADS, 0, st>>>(out, stats, qkv, T, NH, t0);
        })) return;
#endif
    const unsigned blocks = (unsigned)CEIL_DIV((size_t)B * NH * (T - t0), (size_t)4);
    if (hs <= 64) att_forward_rows_kernel<1><<<blocks, 256, 0, st>>>(out, stats, qkv, B, T, NH, hs, t0);
    else att_forward_rows_kernel<2><<<blocks, 256, 0, st>>>(out, stats, qkv, B, T, NH, hs, t0);
}
void launch_backward_rows(floatX* dqkv, const floatX* dout, const floatX* qkv, const floatX* o, const float* stats, int B,
                          int T, int NH, int hs, hipStream_t st) {
#if defined(LLMK_FP32)
    if (B * NH <= 65535 && f32_aligned(dqkv, dout, qkv, o) && with_f32_head(hs, [&](auto hd) {
            const dim3 grid(CEIL_DIV(T, F_ROWS), B * NH);
            att_backward_dq_f32_kernel<decltype(hd)::value><<<grid, F_THREADS, 0, st>>>(dqkv, dout, qkv, o, stats, T, NH);
            att_backward_dkdv_f32_kernel<decltype(hd)::value><<<grid, F_THREADS, 0, st>>>(dqkv, dout, qkv, o, stats, T, NH);
        })) return;
#endif
    const unsigned blocks = (unsigned)CEIL_DIV((size_t)B * NH * T, (size_t)4);
    if (hs <= 64) {
        att_backward_dq_rows_kernel<1><<<blocks, 256, 0, st>>>(dqkv, dout, qkv, o, stats, B, T, NH, hs);
        att_backward_dkdv_rows_kernel<1><<<blocks, 256, 0, st>>>(dqkv, dout, qkv, o, stats, B, T, NH, hs);
    } else {
        att_backward_dq_rows_kernel<2><<<blocks, 256, 0, st>>>(dqkv, dout, qkv, o, stats, B, T, NH, hs);
        att_backward_dkdv_rows_kernel<2><<<blocks, 256, 0, st>>>(dqkv, dout, qkv, o, stats, B, T, NH, hs);
    }
}


// ---- scratch that needs no allocation ------------------------------------------------------------------------------
// Device memory that exists from the moment the code object is loaded: the rowsum(dO*O) vector of
// llmk_attention_backward_static. Each GPU holds its own copy at its own address; in host code the array's name is
// only a handle for hipGetSymbolAddress, never an address to hand to a kernel.
constexpr size_t STATIC_SCRATCH_FLOATS = (size_t)1 << 20;        // 4 MiB: B*NH*T up to 1048576 (GPT-2 124M at B=64, T=1024 needs 786432)
static __device__ __align__(256) float scratch[STATIC_SCRATCH_FLOATS];
constexpr int MAX_DEVICES = 64;
float* g_static_scratch[MAX_DEVICES];                             // per device, filled by static_scratch_setup()

float* static_scratch_setup() {
    int dev = -1;
    HIP_CHECK(hipGetDevice(&dev));
    if (dev < 0 || dev >= MAX_DEVICES) { llmk::fail(__FILE__, __LINE__, "device index %d out of range", dev); return nullptr; }
    if (!g_static_scratch[dev]) {
        void* p = nullptr;
        hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            llmk::fail(__FILE__, __LINE__, "hipGetSymbolAddress(scratch) on device %d: %s", dev, hipGetErrorString(e));
            return nullptr;
        }
        g_static_scratch[dev] = (float*)p;
    }
    return g_static_scratch[dev];
}
float* static_scratch_ptr() { return static_scratch_setup(); }    // the current device's copy (looked up once per device)

#if !defined(LLMK_FP32)
// One or two tiles of 128 rows per workgroup. Two even the work out (a tile near the end of a head has more keys than one at
// its start: a pair of nt tiles walks nt + 1 tiles' worth whatever pair it is) and save a start-up; one per workgroup ends
// sooner where every workgroup gets a CU to itself (the longest walks nt), and where an odd number of tiles leaves the middle
// one alone beside pairs of nt + 1, unless nt is large. Forward, us, two against one: 4 x 1024 x 12 heads of 64 20.0 / 22.4,
// 2 x 2048 x 16 of 128 63.5 / 84.2, 32 x 512 x 12 29.9 / 33.3, 16 x 1920 x 12 121.8 / 126.7; other side: 2 x 1024 x 12
// 19.6 / 16.4 (192 tiles for 256 CUs), 64 x 384 x 12 43.6 / 36.5 (3 tiles), 5 x 777 x 16 26.1 / 22.1 (7), 32 x 256 x 12 15.7 / 14.4 (2).
bool fa_tiles_paired(int ntiles, int nbh) {
    return ntiles > 2 && (ntiles % 2 == 0 || ntiles > 8) && (size_t)ntiles * nbh > (size_t)llmk::device_info().num_cu;
}

template <int HD, bool RAGGED>
void launch_fa_forward(floatX* out, float* stats, const floatX* qkv, int B, int T, int NH, hipStream_t st) {
    const int nq = CEIL_DIV(T, 128);
    const bool paired = fa_tiles_paired(nq, B * NH);
    const int gx = paired ? (nq + 1) / 2 : nq;
    fa_forward_dma_kernel<HD, RAGGED><<<dim3(gx, B * NH), 256, 0, st>>>(out, stats, qkv, T, NH, nq, paired);
}
template <int HD, bool RAGGED>
void launch_fa_dq(floatX* dqkv, const floatX* dout, const floatX* qkv, const floatX* o, const float* stats, float* Dsum, int B, int T,
                  int NH, hipStream_t st) {
    const int nq = CEIL_DIV(T, 128);
    const bool paired = fa_tiles_paired(nq, B * NH);
    const int gx = paired ? (nq + 1) / 2 : nq;
    fa_backward_dq_dma_kernel<HD, RAGGED><<<dim3(gx, B * NH), 256, 0, st>>>(dqkv, dout, qkv, o, stats, Dsum, T, NH, nq, paired);
}
template <int HD, bool RAGGED>
void launch_fa_dkdv(floatX* dqkv, const floatX* dout, const floatX* qkv, const float* stats, const float* Dsum, int B, int T, int NH,
                    hipStream_t st) {
    const int nk = CEIL_DIV(T, 128);
    const bool paired = fa_tiles_paired(nk, B * NH);
    const int gx = paired ? (nk + 1) / 2 : nk;
    const dim3 grid(gx, B * NH);
    if (T <= 4096) {                              // 2 T floats of statistics (32 KiB at most) beside the 32 or 64 KiB of tiles
        const size_t dyn = 2 * (size_t)CEIL_DIV(T, 64) * 64 * sizeof(float);
        static bool attr_set = false;
        auto kern = fa_backward_dkdv_dma_kernel<HD, RAGGED, true>;
        if (!attr_set) {
            HIP_CHECK(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, 2 * 4096 * (int)sizeof(float)));
            attr_set = true;
        }
        kern<<<grid, 256, dyn, st>>>(dqkv, dout, qkv, stats, Dsum, T, NH, nk, paired);
    } else {
        fa_backward_dkdv_dma_kernel<HD, RAGGED, false><<<grid, 256, 0, st>>>(dqkv, dout, qkv, stats, Dsum, T, NH, nk, paired);
    }
}
// the head sizes of the GPT-2 and GPT-3 models run on the matrix cores (the direct-to-LDS loads and the stores of a lane need
// 16- and 8-byte rows); anything else takes the one-wave-per-row kernels
bool fa_head_size(int hs) { return hs == 64 || hs == 80 || hs == 96 || hs == 128; }
#endif

// Dsum_static: device memory for the B*NH*T floats of rowsum(dO*O), or nullptr to take them from the library workspace
// (which may allocate). With Dsum_static nothing on this path allocates: no workspace, no timing events.
void attention_backward_impl(void* dqkvr, const void* dout, const void* qkvr, const void* o, const float* stats,
                             int B, int T, int NH, int C, void* stream, float* Dsum_static) {
    if (llmk::failed()) return;
    LLMK_REQUIRE(NH > 0 && C % NH == 0, "attention_backward: C=%d not divisible by NH=%d", C, NH);
    LLMK_REQUIRE(stats != nullptr, "attention_backward: stats from the forward pass are required");
    const int hs = C / NH;
    if ((size_t)B * T == 0) return;
    hipStream_t st = (hipStream_t)stream;
    LLMK_REQUIRE(hs <= 128, "attention_backward: head size %d unsupported (up to 128)", hs);
#if !defined(LLMK_FP32)
    auto aligned = [](const void* p, uintptr_t n) { return ((uintptr_t)p % n) == 0; };
    if (hs == 64 || (fa_head_size(hs) && aligned(dqkvr, 8) && aligned(dout, 16) && aligned(qkvr, 16) && aligned(o, 16))) {
        float* Dsum = Dsum_static ? Dsum_static : (float*)llmk::workspace((size_t)B * NH * T * sizeof(float));
        const double fwd_flops = 4.0 * B * NH * hs * ((double)T * (T + 1) / 2);
        floatX* dq = (floatX*)dqkvr;
        const floatX *go = (const floatX*)dout, *qkv = (const floatX*)qkvr, *fo = (const floatX*)o;
        // dQ first: it also leaves D = rowsum(dO * O) for dK/dV. Algorithmic backward work is 2.5x forward (5 contractions
        // vs 2); booked 1.5x on dK/dV, 1.0x on dQ.
        {
            llmk::ProfScope prof(Dsum_static != nullptr, "attention_backward_dq", 1.0 * fwd_flops, 6.0 * B * T * C * sizeof(floatX), st);
            if (hs == 64 && T % 64 == 0) launch_fa_dq<64, false>(dq, go, qkv, fo, stats, Dsum, B, T, NH, st);
            else if (hs == 64) launch_fa_dq<64, true>(dq, go, qkv, fo, stats, Dsum, B, T, NH, st);
            else if (hs == 80) launch_fa_dq<80, true>(dq, go, qkv, fo, stats, Dsum, B, T, NH, st);
            else if (hs == 96) launch_fa_dq<96, true>(dq, go, qkv, fo, stats, Dsum, B, T, NH, st);
            else launch_fa_dq<128, true>(dq, go, qkv, fo, stats, Dsum, B, T, NH, st);
            LAUNCH_CHECK();
        }
        llmk::ProfScope prof(Dsum_static != nullptr, "attention_backward_dkdv", 1.5 * fwd_flops, 6.0 * B * T * C * sizeof(floatX), st);
        if (hs == 64 && T % 64 == 0) launch_fa_dkdv<64, false>(dq, go, qkv, stats, Dsum, B, T, NH, st);
        else if (hs == 64) launch_fa_dkdv<64, true>(dq, go, qkv, stats, Dsum, B, T, NH, st);
        else if (hs == 80) launch_fa_dkdv<80, true>(dq, go, qkv, stats, Dsum, B, T, NH, st);
        else if (hs == 96) launch_fa_dkdv<96, true>(dq, go, qkv, stats, Dsum, B, T, NH, st);
        else launch_fa_dkdv<128, true>(dq, go, qkv, stats, Dsum, B, T, NH, st);
        LAUNCH_CHECK();
        return;
    }
#endif
    llmk::ProfScope prof(Dsum_static != nullptr, "attention_backward_rows", 2.5 * 4.0 * B * NH * hs * ((double)T * (T + 1) / 2), 6.0 * B * T * C * sizeof(floatX), st);
    launch_backward_rows((floatX*)dqkvr, (const floatX*)dout, (const floatX*)qkvr, (const floatX*)o, stats, B, T, NH, hs, st);
    LAUNCH_CHECK();
}

}  // namespace

namespace llmk {
void attention_static_scratch_init() { (void)static_scratch_setup(); }

// One sequence, query T - 1 against keys 0 .. T - 1, with the bits that a sampled token has always depended on; t0: T - 1 rounded
// down to a multiple of 32. Heads of 64, and fp32: the matrix-core kernels run the query tile that holds the row, one workgroup
// per head; the rows of that tile before it come out again as they were. Others: one wave per head.
void decode_attention(void* out, const void* qkv, int t0, int T, int NH, int C, hipStream_t st) {
    if (failed()) return;
    const int hs = C / NH;
#if !defined(LLMK_FP32)
    if (hs == 64) {
        fa_forward_dma_kernel<64, true><<<dim3(1, NH), 256, 0, st>>>((floatX*)out, nullptr, (const floatX*)qkv, T, NH, CEIL_DIV(T, 128), false);
        LAUNCH_CHECK();
        return;
    }
    t0 = T - 1;
#endif
    launch_forward_rows((floatX*)out, nullptr, (const floatX*)qkv, 1, T, NH, hs, t0, st);
    LAUNCH_CHECK();
}
}  // namespace llmk

extern "C" {

void llmk_attention_forward(void* out, float* stats, const void* inp, int B, int T, int NH, int C, void* stream) {
    if (llmk::failed()) return;
    LLMK_REQUIRE(NH > 0 && C % NH == 0, "attention_forward: C=%d not divisible by NH=%d", C, NH);
    const int hs = C / NH;
    if ((size_t)B * T == 0) return;
    hipStream_t st = (hipStream_t)stream;
    const double fwd_flops = 4.0 * B * NH * hs * ((double)T * (T + 1) / 2);
    llmk::ProfScope prof("attention_forward", fwd_flops, 4.0 * B * T * C * sizeof(floatX), st);
    LLMK_REQUIRE(hs <= 128, "attention_forward: head size %d unsupported (up to 128)", hs);
#if !defined(LLMK_FP32)
    const bool aligned = ((uintptr_t)inp % 16) == 0 && ((uintptr_t)out % 8) == 0;
    LLMK_REQUIRE(hs != 64 || aligned, "attention_forward: misaligned buffers");
    if (fa_head_size(hs) && aligned) {
        floatX* o = (floatX*)out;
        const floatX* qkv = (const floatX*)inp;
        if (hs == 64 && T % 128 == 0) launch_fa_forward<64, false>(o, stats, qkv, B, T, NH, st);
        else if (hs == 64) launch_fa_forward<64, true>(o, stats, qkv, B, T, NH, st);
        else if (hs == 80) launch_fa_forward<80, true>(o, stats, qkv, B, T, NH, st);
        else if (hs == 96) launch_fa_forward<96, true>(o, stats, qkv, B, T, NH, st);
        else launch_fa_forward<128, true>(o, stats, qkv, B, T, NH, st);
        LAUNCH_CHECK();
        return;
    }
#endif
    launch_forward_rows((floatX*)out, stats, (const floatX*)inp, B, T, NH, hs, 0, st);
    LAUNCH_CHECK();
}

size_t llmk_attention_backward_workspace_bytes(int B, int T, int NH) {
    return (size_t)B * NH * T * sizeof(float);                   // rowsum(dO * O), one float per (batch, head, query)
}

void llmk_attention_backward(void* dqkvr, const void* dout, const void* qkvr, const void* o, const float* stats,
                             int B, int T, int NH, int C, void* stream) {
    attention_backward_impl(dqkvr, dout, qkvr, o, stats, B, T, NH, C, stream, nullptr);
}

// The reference's launchers for builds without cuDNN (llmc/attention.cuh:195, :239) keep a permuted copy of Q, K, V and
// the (B,NH,T,T) probabilities between the passes. Here the same buffers carry what the flash kernels need instead: qkvr
// holds Q, K, V as they came (B,T,3,NH,hs), and the first B*NH*T*4 bytes of att hold the fp32 log-sum-exp of every row.
void llmk_attention_forward_fallback(void* out, void* qkvr, void* att, void* inp, int B, int T, int C, int NH, void* stream) {
    if (llmk::failed()) return;
    if ((size_t)B * T == 0) return;
    LLMK_REQUIRE((size_t)T * sizeof(floatX) >= sizeof(float), "attention_forward: T=%d too short for the statistics to fit the att buffer", T);
    LLMK_REQUIRE(((uintptr_t)att % 4) == 0, "attention_forward: att must be 4-byte aligned");
    HIP_CHECK(hipMemcpyAsync(qkvr, inp, (size_t)B * T * 3 * C * sizeof(floatX), hipMemcpyDeviceToDevice, (hipStream_t)stream));
    llmk_attention_forward(out, (float*)att, qkvr, B, T, NH, C, stream);
}

void llmk_attention_backward_fallback(void* dinp, void* dqkvr, void* datt, void* scratch, const void* dout, const void* qkvr,
                                      const void* att, int B, int T, int C, int NH, void* stream) {
    if (llmk::failed()) return;
    (void)dqkvr; (void)datt;                                     // the flash kernels need neither
    if ((size_t)B * T == 0) return;
    // the output of the forward pass is not among the arguments: it is formed again, in scratch (B*T*C elements)
    llmk_attention_forward(scratch, nullptr, qkvr, B, T, NH, C, stream);
    llmk_attention_backward(dinp, dout, qkvr, scratch, (const float*)att, B, T, NH, C, stream);
}

void llmk_attention_backward_static(void* dqkvr, const void* dout, const void* qkvr, const void* o, const float* stats,
                                    int B, int T, int NH, int C, void* stream) {
    if (llmk::failed()) return;
    LLMK_REQUIRE((size_t)B * (size_t)max(NH, 0) * (size_t)T <= STATIC_SCRATCH_FLOATS,
                 "attention_backward_static: B*NH*T = %zu exceeds the %zu floats of static scratch; use llmk_attention_backward",
                 (size_t)B * NH * T, STATIC_SCRATCH_FLOATS);
    float* ptr = static_scratch_ptr();
    if (!ptr) return;                                            // the failure is recorded
    attention_backward_impl(dqkvr, dout, qkvr, o, stats, B, T, NH, C, stream, ptr);
}

}  // extern "C"
