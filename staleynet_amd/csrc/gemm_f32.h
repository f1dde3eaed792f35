// fp32 matrix products on the bf16 matrix cores: the tile engine behind every
// tiled fp32 product (gemm_f32.hip launches it, gemm_f32_unaligned.hip holds
// the instantiations for operands that 16-byte loads cannot serve). It is the
// role of the reference's default kernel, matmul_blocked
// (crates/staleynet-cuda/src/kernels/matmul.rs:283-355), behind the same
// contract: any operand storage, strided batches, overwrite or accumulate,
// zero padding of partial tiles, row-major output with row stride N.
//
// Arithmetic. An fp32 value is the exact sum of three bf16 values: hi, the
// value rounded to bf16; mid, the rest rounded to bf16; lo, what that leaves
// (at most 7 bits, so exact). A product of two such sums has nine terms, each
// exact in fp32 (8 x 8 bits); six are accumulated in fp32 by
// v_mfma_f32_32x32x16_bf16, smallest first, for every 16 k: lo hi, hi lo, mid
// mid, mid hi, hi mid, hi hi. The three left out are together under 2^-24 of
// the product, of either sign. (With hi truncated they reached 2^-22, and
// single products were off by 4.1e-8 rms and 4.3 x 2^-24 at worst.) Per 16 k
// that is 6 roundings of an output where v_mfma_f32_32x32x2_f32 rounds 16
// times. Relative 2-norm error on N(0, 1) operands at K = 4 / 64 / 768 / 3072 /
// 16384: 3.2e-8 / 1.10e-7 / 2.41e-7 / 2.52e-7 / 3.6e-7 against 4.0e-8 /
// 1.45e-7 / 2.89e-7 / 2.94e-7 / 3.8e-7 for the fp32 instruction, and 0.8 to 0.99
// of it on positive and on widely spread operands (the larger K split over
// workgroups as launched). Up to three products the fp32 instruction's few
// roundings are the better ones (2.5e-8 for one), so it computes those
// (kFewProducts). A row with a single nonzero entry among more keeps the
// split's own error of one product: 3.5e-8 rms, 2.6 x 2^-24 at worst (0 where
// one factor has 8 bits, a power of two or a small whole number).
//  * Range. The split holds zeros and every finite operand from 2^-110 on
//    (split_bf16.h) up to 2^-9 under the largest float. The values of a step
//    are looked at before they are split (note_set); a workgroup that has met
//    a smaller one computes its tile again with the fp32 instruction from the
//    operands in memory (recompute_f32), and so does a wave whose outputs are
//    not finite (an infinite, NaN or largest operand, or an overflow). The
//    operands decide, not the outputs: a tiny operand with a huge partner
//    gives outputs of any size, and subnormal ones can leave 0. The look
//    costs 1.7 % of a large product (32768 x 768 x 2304, a Linear step: 1860
//    -> 1893 us), 3.5 % of the smallest tiled ones (it waits for a step's
//    loads at once) and 3 % more where operands hold zeros (each value's
//    range then); three instructions per pair as each is split, which zeros
//    do not slow, cost 3 to 4 %. A tile computed again takes 3.5 times as
//    long (4096 cubed with one such operand in each tile 865 -> 2995 us).
//  * Six bf16 MFMAs do the work of eight fp32 ones (16 k of a 32 x 32 block)
//    in 192 matrix-core cycles instead of 512. What bounds the kernel is
//    power: on random operands six products' worth of MFMAs alone run at
//    305-312 TFLOP/s (the clock falls from 2.38 to 1.75 GHz; zeros run at
//    2.37), 269-276 with the conversions, 234-241 with the LDS traffic and
//    216-226 with the operand loads besides. The large layer's products run
//    at 170-190 (the fp32 instruction: 136-140) with the matrix cores busy 58
//    to 60 % of the cycles at 1.65 GHz, so less work beside the
//    MFMAs is what would make it faster; deeper prefetch and other issue
//    orders changed cycles and clock by the same factor.
//
// Schedule. A workgroup of four waves owns a BM x BN tile, a wave FM x FN
// blocks of 32 x 32. Operand tiles of 32 k go through registers: a thread
// loads its 16-byte pieces three K-steps ahead (two register sets), splits
// each once and writes the three bf16 parts to one LDS stage; every wave then
// reads its fragments from there (splitting fragments as each wave reads them
// would convert every value twice: 169 TFLOP/s against 190).
//  * A step's two 16-deep chunks: chunk 0's fragments are read first, chunk
//    1's under chunk 0's MFMAs; a barrier after the first MFMAs of chunk 1
//    (every wave then holds all its fragments) frees the stage, and under the
//    other MFMAs of chunk 1 the next step's registers are split and written
//    to it, a few vector instructions after each MFMA. A second barrier ends
//    the step. Both wait on LDS only; loads in flight are waited for by
//    count where their registers are used.
//  * Two workgroups per CU (four of the 64 x 64 tile): one's barriers and
//    first reads run under the other's MFMAs.
//
// LDS. Per operand and part (hi, mid, lo): four k-octets of ROWS + 4 slots of
// 16 bytes, slot (o, p) holding k = 8 o .. 8 o + 7 of the row at position p.
// A fragment is one ds_read_b128 per block and part (32 consecutive slots;
// lane half h of chunk c reads octet 2 c + h). Writes are 8 bytes (four k):
// the four-slot pad puts the octets of a 16-lane write phase 64 bytes apart,
// so 8 k-groups x 2 rows (K-contiguous) or 2 groups x 8 row blocks
// (row-contiguous) fall on distinct banks of that phase (counted over all LDS
// instructions, two conflict cycles each remain). Where a wave has two blocks on a
// side their rows interleave (block i's position q holds row 2 q + i of the
// wave's 64): a row-contiguous loader's block of four rows then writes
// slots two apart, and a lane's two columns are adjacent in the output (one
// 8-byte store; TileMap in gemm_common.h).
#pragma once

#include "gemm_common.h"

namespace sn {
namespace gemm {

// How an operand is loaded.
//  kLoadVector: 16-byte buffer loads; the contiguous dimension, leading
//    dimension and base are multiples of 4 floats, so a vector is inside the
//    matrix or outside as a whole.
//  kLoadDword: the same loads at 4-byte alignment where a whole step (or the
//    whole row range) is inside, single floats on the edges.
//  kLoadPointer: single floats by 64-bit address, for operands whose offsets
//    within a step do not fit the buffer's 31 bits.
constexpr int kLoadVector = 0;
constexpr int kLoadDword = 1;
constexpr int kLoadPointer = 2;

// A thread index the compiler cannot trace, so that what is derived from it
// on a rare path is formed there and not held in registers across the loop.
__device__ __forceinline__ int fresh(int tid) {
    asm volatile("" : "+v"(tid));
    return tid;
}

// LDS geometry of one operand's stage.
template <int ROWS>
struct SplitStage {
    static constexpr int PLANE = ROWS + 4;        // slots per k-octet
    static constexpr int PART = 4 * PLANE * 16;   // bytes of one part
    static constexpr int BYTES = kParts * PART;
};

// The row a stage position holds (PAIRED: two blocks per wave interleaved).
template <bool PAIRED>
__device__ __forceinline__ constexpr int row_at(int position) {
    return PAIRED ? position / 64 * 64 + 2 * (position % 32) + position % 64 / 32 : position;
}

// K-contiguous operand: vector v of a thread is k-group tid % 8 (4 k) of the
// row at position tid / 8 + 32 v, so 8 lanes read a row's 128 bytes.
template <int ROWS, int THREADS, bool PAIRED, int MODE>
struct SplitLoaderK {
    static constexpr int N = ROWS * 8 / THREADS;  // vectors a thread holds
    static constexpr int PIECES = 6 * N;          // of the split: two pairs a vector
    using Stage = SplitStage<ROWS>;
    f32x4 reg[N];
    uint32_t part[kParts][2];  // the vector being split
    int32_t offset[N];         // bytes from the step's origin; kOutOfRange past the last row

    __device__ __forceinline__ static int group(int tid) { return tid % 8; }
    __device__ __forceinline__ static int row(int tid, int v) { return row_at<PAIRED>(tid / 8 + v * (THREADS / 8)); }

    __device__ __forceinline__ void init(int64_t ld, int64_t row0, int64_t rows, int tid) {
        if constexpr (MODE != kLoadPointer) {
#pragma unroll
            for (int v = 0; v < N; ++v) {
                const int r = row(tid, v);
                offset[v] = row0 + r < rows ? int32_t((r * ld + 4 * group(tid)) * 4) : kOutOfRange;
            }
        }
    }
    // k = k0 .. k0 + 31 of the rows from row0; zeros from k_end on. `origin`
    // is the operand's element (row0, k = 0).
    __device__ __forceinline__ void load(const float* origin, int64_t ld, int64_t row0, int64_t rows, int64_t k0,
                                         int64_t k_end, int tid) {
        const int left = int(min(max(k_end - k0, int64_t(0)), int64_t(32))) - 4 * group(tid);
        if constexpr (MODE == kLoadPointer) {
#pragma unroll
            for (int v = 0; v < N; ++v)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    reg[v][e] = row0 + row(tid, v) < rows && e < left
                                    ? origin[row(tid, v) * ld + k0 + 4 * group(tid) + e]
                                    : 0.f;
        } else {
            const __amdgpu_buffer_rsrc_t rsrc = buffer_of(origin + k0);
            if (MODE == kLoadVector || k0 + 32 <= k_end || k0 >= k_end) {
                const int32_t outside = (left - 1) & kOutOfRange;
#pragma unroll
                for (int v = 0; v < N; ++v) reg[v] = buffer_load4(rsrc, offset[v] | outside);
            } else {
#pragma unroll
                for (int v = 0; v < N; ++v)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        reg[v][e] = buffer_load1(rsrc, (offset[v] + 4 * e) | (offset[v] & kOutOfRange) |
                                                           ((left - 1 - e) & kOutOfRange));
            }
        }
    }
    // Zeroes elements (r, k) with k > r + query_offset (r = query, k = key).
    __device__ __forceinline__ void mask_keys_after_query(int64_t row0, int64_t k0, int64_t query_offset, int thread) {
        const int tid = fresh(thread);
#pragma unroll
        for (int v = 0; v < N; ++v)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (k0 + 4 * group(tid) + e > row0 + row(tid, v) + query_offset) reg[v][e] = 0.f;
    }
    // f(x0, x1) of every pair of values held.
    template <class F>
    __device__ __forceinline__ void pairs(F&& f) const {
#pragma unroll
        for (int v = 0; v < N; ++v) {
            f(reg[v][0], reg[v][1]);
            f(reg[v][2], reg[v][3]);
        }
    }
    __device__ __forceinline__ static int store_base(int tid) {
        return (group(tid) / 2 * Stage::PLANE + tid / 8) * 16 + 8 * (group(tid) % 2);
    }
    // Piece p of the split (in place); the last piece of a vector writes its
    // parts to the stage.
    __device__ __forceinline__ void piece(int p, uint32_t upper, char* stage, int base) {
        const int v = p / 6, pair = p % 6 / 3;
        float x0 = reg[v][2 * pair], x1 = reg[v][2 * pair + 1];
        split_piece(p % 3, x0, x1, upper, part[0][pair], part[1][pair], part[2][pair]);
        reg[v][2 * pair] = x0;
        reg[v][2 * pair + 1] = x1;
        if (p % 6 == 5) {
#pragma unroll
            for (int q = 0; q < kParts; ++q)
                *reinterpret_cast<u32x2*>(stage + base + q * Stage::PART + v * (THREADS / 8) * 16) =
                    u32x2{part[q][0], part[q][1]};
        }
    }
};

// Row-contiguous operand: a thread holds a block of N consecutive rows x 4 k,
// k-octet tid / 64, half tid % 2, rows N (tid % 64 / 2) .. + N - 1: a wave's
// load instruction reads two k-rows over the tile's whole width.
template <int ROWS, int THREADS, bool PAIRED, int MODE>
struct SplitLoaderR {
    static constexpr int N = ROWS * 8 / THREADS;
    static constexpr int PIECES = 6 * N;
    static_assert(THREADS == 256 && (N == 2 || N == 4), "a wave per octet, two or four rows a thread");
    using Stage = SplitStage<ROWS>;
    float reg[4][N];
    uint32_t part[kParts][2];
    int32_t offset;  // of the block's first element; kOutOfRange past the last row

    __device__ __forceinline__ static int first_row(int tid) { return N * (tid % 64 / 2); }
    __device__ __forceinline__ static int first_k(int tid) { return 8 * (tid / 64) + 4 * (tid % 2); }

    __device__ __forceinline__ void init(int64_t ld, int64_t row0, int64_t rows, int tid) {
        if constexpr (MODE != kLoadPointer)
            offset = row0 + first_row(tid) < rows ? int32_t((first_k(tid) * ld + first_row(tid)) * 4) : kOutOfRange;
    }
    __device__ __forceinline__ void load(const float* origin, int64_t ld, int64_t row0, int64_t rows, int64_t k0,
                                         int64_t k_end, int tid) {
        const int left = int(min(max(k_end - k0, int64_t(0)), int64_t(32))) - first_k(tid);
        if constexpr (MODE == kLoadPointer) {
#pragma unroll
            for (int kk = 0; kk < 4; ++kk)
#pragma unroll
                for (int e = 0; e < N; ++e)
                    reg[kk][e] = row0 + first_row(tid) + e < rows && kk < left
                                     ? origin[(k0 + first_k(tid) + kk) * ld + first_row(tid) + e]
                                     : 0.f;
        } else {
            const __amdgpu_buffer_rsrc_t rsrc = buffer_of(origin + k0 * ld);
            const int32_t ld_bytes = int32_t(ld * 4);
            const int32_t row_outside = offset & kOutOfRange;
            if (MODE == kLoadVector || row0 + ROWS <= rows) {
#pragma unroll
                for (int kk = 0; kk < 4; ++kk) {
                    const int32_t o = (offset + kk * ld_bytes) | row_outside | ((left - 1 - kk) & kOutOfRange);
                    if constexpr (N == 4) {
                        const f32x4 x = buffer_load4(rsrc, o);
#pragma unroll
                        for (int e = 0; e < N; ++e) reg[kk][e] = x[e];
                    } else {
                        const f32x2 x = __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(rsrc, o, 0, 0));
#pragma unroll
                        for (int e = 0; e < N; ++e) reg[kk][e] = x[e];
                    }
                }
            } else {
#pragma unroll
                for (int kk = 0; kk < 4; ++kk)
#pragma unroll
                    for (int e = 0; e < N; ++e) {
                        const bool inside = kk < left && row0 + first_row(tid) + e < rows;
                        reg[kk][e] = buffer_load1(rsrc, inside ? offset + kk * ld_bytes + 4 * e : kOutOfRange);
                    }
            }
        }
    }
    // Zeroes elements (r, k) with r > k + query_offset (r = key, k = query).
    __device__ __forceinline__ void mask_keys_after_query(int64_t row0, int64_t k0, int64_t query_offset, int thread) {
        const int tid = fresh(thread);
#pragma unroll
        for (int kk = 0; kk < 4; ++kk)
#pragma unroll
            for (int e = 0; e < N; ++e)
                if (row0 + first_row(tid) + e > k0 + first_k(tid) + kk + query_offset) reg[kk][e] = 0.f;
    }
    template <class F>
    __device__ __forceinline__ void pairs(F&& f) const {
#pragma unroll
        for (int e = 0; e < N; ++e) {
            f(reg[0][e], reg[1][e]);
            f(reg[2][e], reg[3][e]);
        }
    }
    __device__ __forceinline__ static int store_base(int tid) {
        const int r = first_row(tid);
        return (tid / 64 * Stage::PLANE + (PAIRED ? r / 64 * 64 + r % 64 / 2 : r)) * 16 + 8 * (tid % 2);
    }
    __device__ __forceinline__ void piece(int p, uint32_t upper, char* stage, int base) {
        const int e = p / 6, pair = p % 6 / 3;
        float x0 = reg[2 * pair][e], x1 = reg[2 * pair + 1][e];
        split_piece(p % 3, x0, x1, upper, part[0][pair], part[1][pair], part[2][pair]);
        reg[2 * pair][e] = x0;
        reg[2 * pair + 1][e] = x1;
        if (p % 6 == 5) {
            const int position = PAIRED ? 32 * (e & 1) + (e >> 1) : e;
#pragma unroll
            for (int q = 0; q < kParts; ++q)
                *reinterpret_cast<u32x2*>(stage + base + q * Stage::PART + position * 16) =
                    u32x2{part[q][0], part[q][1]};
        }
    }
};

// Barrier for the LDS stage: this wave's LDS accesses complete (lgkmcnt(0)),
// the global loads in flight stay in flight.
__device__ __forceinline__ void split_barrier() {
    __builtin_amdgcn_s_waitcnt(0xC07F);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// A wave's fragments of one 16-deep chunk.
template <class T>
struct SplitFragments {
    bf16x8 a[kParts][T::FM], b[kParts][T::FN];
};

// The registers and LDS addresses of a workgroup's tile, and its K-step.
template <class T, bool A_K, bool B_K, int MODE>
struct SplitEngine {
    static constexpr bool PAIR_M = T::FM == 2, PAIR_N = T::FN == 2;
    using LA = typename std::conditional<A_K, SplitLoaderK<T::BM, T::THREADS, PAIR_M, MODE>,
                                         SplitLoaderR<T::BM, T::THREADS, PAIR_M, MODE>>::type;
    using LB = typename std::conditional<B_K, SplitLoaderK<T::BN, T::THREADS, PAIR_N, MODE>,
                                         SplitLoaderR<T::BN, T::THREADS, PAIR_N, MODE>>::type;
    using SA = SplitStage<T::BM>;
    using SB = SplitStage<T::BN>;
    static constexpr int MFMAS = kTerms * T::FM * T::FN;  // of one chunk

    LA la[2];  // set j holds the steps s with s % 2 == j, loaded three ahead
    LB lb[2];
    f32x16 acc[T::FM][T::FN];
    char* stage_a;
    char* stage_b;
    int a_store, b_store, a_read, b_read;
    uint32_t upper;
    uint32_t* mark;  // this wave's word in LDS: 1 once it has split a value the split does not hold

    __device__ __forceinline__ void init(char* sa, char* sb, uint32_t* marks, int tid, int64_t lda, int64_t ldb, int64_t m0, int64_t m,
                                         int64_t n0, int64_t n) {
        stage_a = sa;
        stage_b = sb;
        const int lane = tid & 63, wave = tid >> 6;
        a_store = LA::store_base(tid);
        b_store = LB::store_base(tid);
        a_read = ((lane >> 5) * SA::PLANE + wave / T::WAVES_N * T::WTM + (lane & 31)) * 16;
        b_read = ((lane >> 5) * SB::PLANE + wave % T::WAVES_N * T::WTN + (lane & 31)) * 16;
        upper = upper_half_mask();
        mark = marks + wave;
        *mark = 0;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            la[q].init(lda, m0, m, tid);
            lb[q].init(ldb, n0, n, tid);
        }
    }
    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int i = 0; i < T::FM; ++i)
#pragma unroll
            for (int j = 0; j < T::FN; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
    }
    // Marks this wave if set Q holds a value that the split does not.
    template <int Q>
    __device__ __forceinline__ void note_set() {
        if (out_of_range([&](auto f) __attribute__((always_inline)) {
                la[Q].pairs(f);
                lb[Q].pairs(f);
            }))
            *mark = 1;
    }
    // Splits set Q into the stage (the first step, before any MFMA).
    template <int Q>
    __device__ __forceinline__ void stage_set() {
        note_set<Q>();
#pragma unroll
        for (int p = 0; p < LA::PIECES; ++p) la[Q].piece(p, upper, stage_a, a_store);
#pragma unroll
        for (int p = 0; p < LB::PIECES; ++p) lb[Q].piece(p, upper, stage_b, b_store);
    }
    // Fragment x of the left operand in the order the terms need them.
    __device__ __forceinline__ void read_a(int chunk, int x, SplitFragments<T>& f) const {
        const int q = x / T::FM == 0 ? 2 : x / T::FM - 1, i = x % T::FM;
        f.a[q][i] = *reinterpret_cast<const bf16x8*>(stage_a + a_read + q * SA::PART + 2 * chunk * SA::PLANE * 16 +
                                                     512 * i);
    }
    __device__ __forceinline__ void read_b(int chunk, int j, int x, SplitFragments<T>& f) const {
        const int q = x == 0 ? 0 : 3 - x;
        f.b[q][j] = *reinterpret_cast<const bf16x8*>(stage_b + b_read + q * SB::PART + 2 * chunk * SB::PLANE * 16 +
                                                     512 * j);
    }
    // MFMA x of a chunk: column block x / (6 FM), term, row block.
    __device__ __forceinline__ void mfma(int x, const SplitFragments<T>& f) {
        const int j = x / (kTerms * T::FM), t = x / T::FM % kTerms, i = x % T::FM;
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.a[term_left(t)][i], f.b[term_right(t)][j], acc[i][j], 0,
                                                            0, 0);
    }
    // One K-step from the stage. NEXT: also splits set Q (the next step) into
    // the stage as soon as every wave holds this step's fragments; `before`
    // runs on the set's values first, `reload` issues its next loads after.
    template <int Q, bool NEXT, class Before, class Reload>
    __device__ __forceinline__ void step(Before&& before, Reload&& reload) {
        SplitFragments<T> f0, f1;
#pragma unroll
        for (int x = 0; x < 3; ++x) {
#pragma unroll
            for (int i = 0; i < T::FM; ++i) read_a(0, x * T::FM + i, f0);
            read_b(0, 0, x, f0);
        }
#pragma unroll
        for (int j = 1; j < T::FN; ++j)
#pragma unroll
            for (int x = 0; x < 3; ++x) read_b(0, j, x, f0);
        __builtin_amdgcn_sched_barrier(0);
        // Chunk 1's left fragments and its first column block's are read
        // under chunk 0's MFMAs, the others when chunk 0's are done with.
#pragma unroll
        for (int x = 0; x < MFMAS; ++x) {
            mfma(x, f0);
            if (x < 3 * T::FM) read_a(1, x, f1);
            else if (x >= 6 * T::FM && x < 6 * T::FM + 3) read_b(1, 0, x - 6 * T::FM, f1);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int j = T::FN == 1 ? 0 : 1; j < T::FN; ++j)
#pragma unroll
            for (int x = 0; x < 3; ++x) read_b(1, j, x, f1);
        constexpr int FIRST = 2 * T::FM;  // MFMAs before the barrier
        constexpr int PIECES = LA::PIECES + LB::PIECES;
#pragma unroll
        for (int x = 0; x < FIRST; ++x) {
            mfma(x, f1);
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (NEXT) {
            split_barrier();  // every wave holds both chunks' fragments
            before();
            note_set<Q>();
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int x = FIRST; x < MFMAS; ++x) {
            mfma(x, f1);
            if constexpr (NEXT) {
#pragma unroll
                for (int p = (x - FIRST) * PIECES / (MFMAS - FIRST); p < (x - FIRST + 1) * PIECES / (MFMAS - FIRST);
                     ++p) {
                    if (p < LA::PIECES) la[Q].piece(p, upper, stage_a, a_store);
                    else lb[Q].piece(p - LA::PIECES, upper, stage_b, b_store);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (NEXT) {
            reload();
            split_barrier();
        }
    }
};

// Products per output (of a K slice) up to which the fp32 instruction's few
// roundings err less than the split.
constexpr int kFewProducts = 3;

// Whether a wave's accumulators hold a value that is not finite.
template <class T>
__device__ __forceinline__ bool not_finite(const f32x16 (&acc)[T::FM][T::FN]) {
    float poison = 0.f;
#pragma unroll
    for (int i = 0; i < T::FM; ++i)
#pragma unroll
        for (int j = 0; j < T::FN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) poison = __builtin_fmaf(acc[i][j][r], 0.f, poison);  // NaN from then on
    return __any(poison != 0.f);
}

// Whether a wave of the workgroup has split a value the split does not hold
// (after the barrier that follows the last split).
template <class T>
__device__ __forceinline__ bool marked(const uint32_t (&marks)[T::THREADS / 64]) {
    uint32_t any = 0;
#pragma unroll
    for (int w = 0; w < T::THREADS / 64; ++w) any |= marks[w];
    return __builtin_amdgcn_readfirstlane(any) != 0;
}

// A wave's blocks again, by v_mfma_f32_32x32x2_f32 on the operands as they
// are in memory (a and b: the matrix's first elements). Single-float loads,
// no LDS and no barrier: only the waves whose outputs ask for it run it.
template <class T, bool A_K, bool B_K>
__device__ __forceinline__ void recompute_f32(const Args& args, const float* a, const float* b, int64_t m0, int64_t n0,
                                              int64_t k_begin, int64_t k_end, int wave_m, int wave_n, int lane,
                                              f32x16 (&acc)[T::FM][T::FN]) {
    const bool left_causal = args.mask == int(SN_MASK_CAUSAL_LEFT);
    const int q = lane & 31, half = lane >> 5;
#pragma unroll
    for (int i = 0; i < T::FM; ++i)
#pragma unroll
        for (int j = 0; j < T::FN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
    constexpr int DEEP = 4;  // MFMAs whose loads are in flight together
    for (int64_t k2 = k_begin; k2 < k_end; k2 += 2 * DEEP) {
        float av[DEEP][T::FM], bv[DEEP][T::FN];
#pragma unroll
        for (int d = 0; d < DEEP; ++d) {
            const int64_t k = k2 + 2 * d + half;
#pragma unroll
            for (int i = 0; i < T::FM; ++i) {
                const int64_t row = m0 + wave_m * T::WTM + (T::FM == 2 ? 2 * q + i : 32 * i + q);
                bool use = row < args.m && k < k_end;
                if (left_causal) use = use && (A_K ? k <= row + args.query_offset : row <= k + args.query_offset);
                av[d][i] = use ? a[A_K ? row * args.lda + k : k * args.lda + row] : 0.f;
            }
#pragma unroll
            for (int j = 0; j < T::FN; ++j) {
                const int64_t col = n0 + wave_n * T::WTN + (T::FN == 2 ? 2 * q + j : 32 * j + q);
                bv[d][j] = col < args.n && k < k_end ? b[B_K ? col * args.ldb + k : k * args.ldb + col] : 0.f;
            }
        }
#pragma unroll
        for (int d = 0; d < DEEP; ++d)
#pragma unroll
            for (int i = 0; i < T::FM; ++i)
#pragma unroll
                for (int j = 0; j < T::FN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[d][i], bv[d][j], acc[i][j], 0, 0, 0);
    }
}

// One output tile per workgroup. COLSUM: the workgroups of the first tile row
// also add the right operand's columns over K (row-contiguous), from the
// registers before they are split.
template <class T, bool A_K, bool B_K, int MODE, bool COLSUM>
__device__ __forceinline__ void split_tile(const Args& args) {
    static_assert(!COLSUM || !B_K, "column sums of a row-contiguous right operand");
    using Engine = SplitEngine<T, A_K, B_K, MODE>;
    using LB = typename Engine::LB;
    __shared__ __attribute__((aligned(16))) char stage_a[Engine::SA::BYTES];
    __shared__ __attribute__((aligned(16))) char stage_b[Engine::SB::BYTES];
    __shared__ __attribute__((aligned(16))) uint32_t marks[T::THREADS / 64];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int wave_m = wave / T::WAVES_N;
    const int wave_n = wave % T::WAVES_N;

    int batch_local, split, tm, tn;
    tile_coordinates(blockIdx.x, gridDim.x, args.tiles_m, args.tiles_n, args.splits, batch_local, split, tm, tn);
    const int64_t batch = args.batch_base + batch_local;
    const int64_t m0 = int64_t(tm) * T::BM;
    const int64_t n0 = int64_t(tn) * T::BN;
    const int64_t row_last = min(m0 + T::BM, args.m) - 1;
    const bool left_causal = args.mask == int(SN_MASK_CAUSAL_LEFT);
    float* c_batch = args.c + batch * args.stride_c;
    if (args.mask == int(SN_MASK_CAUSAL_OUTPUT) && n0 > row_last + args.query_offset) {
        // Every output of this tile is masked: the product is 0 there.
        if (!args.accumulate) zero_tile<T>(args, c_batch, m0, n0, tid);
        return;
    }
    int64_t k_begin = int64_t(split) * args.k_per_split;
    int64_t k_end = min(args.k, k_begin + args.k_per_split);
    if (left_causal) {
        if (A_K) {
            k_end = min(k_end, row_last + args.query_offset + 1);
        } else {
            const int64_t first = m0 - args.query_offset;
            if (first > k_begin) k_begin = first / T::BK * T::BK;
        }
    }
    const float* a = args.a + batch * args.stride_a;
    const float* b = args.b + batch * args.stride_b;
    const float* a_origin = a + (A_K ? m0 * args.lda : m0);
    const float* b_origin = b + (B_K ? n0 * args.ldb : n0);

    Engine e;
    e.init(stage_a, stage_b, marks, tid, args.lda, args.ldb, m0, args.m, n0, args.n);
    e.clear();
    auto load = [&](auto set, int64_t k0) __attribute__((always_inline)) {
        constexpr int Q = decltype(set)::value;
        e.la[Q].load(a_origin, args.lda, m0, args.m, k0, k_end, tid);
        e.lb[Q].load(b_origin, args.ldb, n0, args.n, k0, k_end, tid);
    };
    // Column sums (COLSUM, first tile row): a thread adds its block's columns
    // over each step's k in order; the eight threads of a column meet at the
    // end in a fixed order.
    const bool colsum_tile = COLSUM && tm == 0;  // uniform over the workgroup
    float colsum[LB::N];
#pragma unroll
    for (int c = 0; c < LB::N; ++c) colsum[c] = 0.f;
    // On a set's values before they are split: the causal left mask (on the
    // K-steps that reach the diagonal) and the column sums.
    auto before = [&](auto set, int64_t k0) __attribute__((always_inline)) {
        constexpr int Q = decltype(set)::value;
        if (left_causal && (A_K ? k0 + T::BK - 1 > m0 + args.query_offset : k0 + args.query_offset < row_last))
            e.la[Q].mask_keys_after_query(m0, k0, args.query_offset, tid);
        if constexpr (COLSUM) {
            if (colsum_tile) {
#pragma unroll
                for (int kk = 0; kk < 4; ++kk)
#pragma unroll
                    for (int c = 0; c < LB::N; ++c) colsum[c] = colsum[c] + e.lb[Q].reg[kk][c];
            }
        }
    };
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    const int steps = k_end > k_begin ? int((k_end - k_begin + T::BK - 1) / T::BK) : 0;
    if (steps > 0) {
        load(I0{}, k_begin);
        load(I1{}, k_begin + T::BK);
        before(I0{}, k_begin);
        e.template stage_set<0>();
        load(I0{}, k_begin + 2 * T::BK);
        split_barrier();
        // Step s splits set (s + 1) % 2 and reloads it with step s + 3 (past
        // the last step: out of range, no memory traffic).
        int64_t k0 = k_begin;
        int s = 0;
        for (; s + 2 < steps; s += 2, k0 += 2 * T::BK) {
            e.template step<1, true>([&] { before(I1{}, k0 + T::BK); }, [&] { load(I1{}, k0 + 3 * T::BK); });
            e.template step<0, true>([&] { before(I0{}, k0 + 2 * T::BK); }, [&] { load(I0{}, k0 + 4 * T::BK); });
        }
        if (s + 1 < steps) e.template step<1, true>([&] { before(I1{}, k0 + T::BK); }, [&] {});
        e.template step<0, false>([&] {}, [&] {});
    }
    if (marked<T>(marks) || k_end - k_begin <= kFewProducts || not_finite<T>(e.acc))
        recompute_f32<T, A_K, B_K>(args, a, b, m0, n0, k_begin, k_end, wave_m, wave_n, lane, e.acc);

    const bool partial = args.splits > 1;
    if constexpr (COLSUM) {
        if (colsum_tile) {
            float* parts = reinterpret_cast<float*>(stage_a);
            split_barrier();  // every wave is done with the stage
#pragma unroll
            for (int c = 0; c < LB::N; ++c) {
                colsum[c] = colsum[c] + __shfl_xor(colsum[c], 1);
                if ((tid & 1) == 0) parts[wave * T::BN + LB::first_row(tid) + c] = colsum[c];
            }
            split_barrier();
            if (tid < T::BN) {
                float total = parts[tid];
#pragma unroll
                for (int q = 1; q < T::THREADS / 64; ++q) total = total + parts[q * T::BN + tid];
                const int64_t c = n0 + tid;
                if (c < args.n) {
                    if (partial)
                        args.ws[int64_t(args.splits) * args.m * args.n + int64_t(split) * args.n + c] = total;
                    else
                        args.column_sums[c] = args.column_sums[c] + total;
                }
            }
        }
    }
    float* out = partial ? args.ws + ((batch_local * int64_t(args.splits) + split) * args.m) * args.n : c_batch;
    constexpr bool BUF = MODE != kLoadPointer;
    if (args.streaming_output)
        write_tile<T, BUF, Engine::PAIR_M, Engine::PAIR_N, kStreaming>(args, e.acc, out, m0, n0, wave_m, wave_n, lane,
                                                                       partial);
    else
        write_tile<T, BUF, Engine::PAIR_M, Engine::PAIR_N>(args, e.acc, out, m0, n0, wave_m, wave_n, lane, partial);
}

// Waves per SIMD: 128 x 128 two (256 registers a lane; its LDS would allow
// three workgroups a CU), 128 x 64 three (two for the unaligned loads, whose
// edge paths spilled at 168 registers), 64 x 64 four.
template <class T, int MODE = kLoadVector>
constexpr int split_waves_per_eu() {
    return T::BN == 128 ? 2 : T::BM == 64 ? 4 : MODE == kLoadVector ? 3 : 2;
}

template <class T, bool A_K, bool B_K, int MODE>
__global__ __launch_bounds__(T::THREADS)
__attribute__((amdgpu_waves_per_eu(split_waves_per_eu<T, MODE>(), split_waves_per_eu<T, MODE>())))
void gemm_f32_kernel(Args args) {
    split_tile<T, A_K, B_K, MODE, false>(args);
}

using F32Square = Tile<128, 128, 32, 2, 2>;  // 4 waves of 64 x 64, 2 workgroups per CU
using F32Narrow = Tile<128, 64, 32, 4, 1>;   // 4 waves of 32 x 64, 3 per CU: N <= 64 (attention head dim)
using F32Small = Tile<64, 64, 32, 2, 2>;     // 4 waves of 32 x 32, 4 per CU

// The one-tile launch under `plan` (its split-K reduce included), for operands
// that take `MODE` loads.
template <class T, int MODE>
hipError_t launch_f32_tiles(const Problem& p, const Env& env, const Plan& plan, hipStream_t stream, bool streaming) {
    const LaunchShape shape = tiled_shape<T>(p, plan, SN_PATH_NONE);
    if (shape.batches_per_launch < 1) return hipErrorInvalidConfiguration;
    Args args = make_args<T>(p, env, plan);
    args.streaming_output = streaming ? 1 : 0;
    const int64_t per_batch = int64_t(plan.tiles_m) * plan.tiles_n * plan.splits;
    for (int64_t first = 0; first < p.batch; first += shape.batches_per_launch) {
        const int64_t count = std::min<int64_t>(shape.batches_per_launch, p.batch - first);
        args.batch_base = first;
        const dim3 grid(unsigned(count * per_batch)), block(T::THREADS);
        if (p.a_k_contiguous && p.b_k_contiguous)
            hipLaunchKernelGGL((gemm_f32_kernel<T, true, true, MODE>), grid, block, 0, stream, args);
        else if (p.a_k_contiguous)
            hipLaunchKernelGGL((gemm_f32_kernel<T, true, false, MODE>), grid, block, 0, stream, args);
        else if (p.b_k_contiguous)
            hipLaunchKernelGGL((gemm_f32_kernel<T, false, true, MODE>), grid, block, 0, stream, args);
        else
            hipLaunchKernelGGL((gemm_f32_kernel<T, false, false, MODE>), grid, block, 0, stream, args);
        const hipError_t err = hipGetLastError();
        if (err != hipSuccess) return err;
    }
    if (plan.splits > 1) return launch_splitk_reduce(p, env, plan.splits, stream);
    return hipSuccess;
}

// The unaligned instantiations (gemm_f32_unaligned.hip).
template <class T>
hipError_t launch_f32_unaligned(const Problem& p, const Env& env, const Plan& plan, hipStream_t stream);

}  // namespace gemm
}  // namespace sn
