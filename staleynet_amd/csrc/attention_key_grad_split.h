// The key kernel of the causal attention backward on the bf16 matrix cores
// (attention_backward.hip has the gradients, the launch and KeyGradArgs; head
// dims 32 and 64, with the dQ partial sums): every product as six bf16 products
// of exactly split fp32 values, accumulated in fp32 (split_bf16.h, gemm_f32.h).
//
//  * A workgroup of four waves owns 128 keys of a head, a wave 32; Q and dO come
//    in stages of 32 queries. K stays in LDS, the wave's V in registers, both
//    split.
//  * A stage's values are loaded into registers under the stage before, split
//    once and written to LDS as octets of h per row. S = Q K^T and dP = dO V^T
//    read their fragments from there as they are; dV^T += dO^T P, dK^T += Q^T dS
//    and dQ^T = K^T dS^T read the same bytes with the transposing LDS load
//    (transposed()), so nothing is held twice.
//  * S and dP leave a lane 16 queries of its key. Eight consecutive registers
//    are queries 4 half + 0..3 and 8 + 4 half + 0..3 of 16: split, P and dS are
//    right operands as they are, against the same queries read transposed.
//  * dQ: dS, split, goes to LDS as octets of keys per query, over the stage's
//    Q and dO (every wave is done with them); lane pairs swap words so that a
//    word holds two keys. Wave w then takes 16 queries x H / 2 columns over
//    the 128 keys.
//  * 79 KB of LDS at h = 64 (52 KB at 32): two workgroups a CU (three), so one's
//    barriers, exponentials and splits run under the other's MFMAs. Eight waves
//    with the rows stored in both orders (146 KB, one workgroup a CU, K and V in
//    registers) left each wave's phases one after the other: 2335 us for 192
//    heads x 2048 x 64 against 1540-1670 (the fp32 kernel 2525; 165 TFLOP/s of
//    its five products). LDS reads and MFMAs bound it about equally: 6900 and
//    7700 cycles a CU for eight waves' blocks.
//  * Range (split_bf16.h): threads look at the Q, K, V and dO they split. P and
//    dS are formed 2^64 times too large (the factor rides in the rows' 1 / l,
//    and the sums are divided by it, exactly), so that every normal fp32 P or
//    dS is one the split holds. A block with an operand outside the range, or
//    with a sum that is not finite, is computed again by the same workgroup
//    with the fp32 instruction from memory. (A backward whose every block is:
//    192 heads x 1024 x 64 557 -> 2070 us. Peaked scores and gradients of a mean
//    loss stay at 575. A launch of their own for such blocks cost every backward
//    2 to 9 us.)
#pragma once

#include "attention_common.h"
#include "split_bf16.h"

namespace sn {
namespace {

typedef float split_f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t split_u32x2 __attribute__((ext_vector_type(2)));

// Hides a lane's address from the compiler where it is used, so that what is
// derived from it is formed there and not held in registers across the loop.
__device__ __forceinline__ void hide(int& x) { asm volatile("" : "+v"(x)); }

constexpr int kSplitWaves = 4;
constexpr int kSplitQueries = 32;  // per stage
// Stages between two additions of the dV and dK accumulators to memory, so that
// no chain of sums is longer than 2048 queries.
constexpr int kFlushStages = 64;

// P and dS are formed this many times too large; 2^64 x 2^-64 = 1.
constexpr float kGradScale = 0x1p64f, kGradUnscale = 0x1p-64f;

// LDS of the kernel, in bytes. The planes' four spare slots put the octets a
// transposing load or an 8-byte write phase touches 64 bytes apart.
template <int H>
struct KeyGradStage {
    static constexpr int ROW_PLANE = kSplitQueries + 4;  // slots per octet of h (slot = query)
    static constexpr int ROW_PART = H / 8 * ROW_PLANE * 16;
    static constexpr int ROWS = kParts * ROW_PART;       // Q's; dO's follow
    static constexpr int DS_PLANE = kSplitQueries + 2;   // slots per octet of keys (slot = query)
    static constexpr int DS_PART = kKeyBlock / 8 * DS_PLANE * 16;
    static constexpr int BYTES = 2 * ROWS > kParts * DS_PART ? 2 * ROWS : kParts * DS_PART;
    static constexpr int K_PLANE = kKeyBlock + 4;        // slots per octet of h (slot = key)
    static constexpr int K_PART = H / 8 * K_PLANE * 16;
    static constexpr int DS_ROW = kSplitQueries + 1;     // floats per key of the recomputed dS
    static_assert(kKeyBlock * DS_ROW * 4 <= BYTES, "the recomputed dS fits the stage");
};

// Four rows x 16 columns of 16-bit values per 16 lanes, transposed: lane 4 i +
// s of the 16 points at columns 4 s .. + 3 of row i, and lane c receives column
// c of rows 0 .. 3. Two such loads make eight values of a fragment.
__device__ __forceinline__ bf16x8 transposed(const char* first, const char* second) {
    typedef short four __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) four* lds_four;
    const four a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_four)first);
    const four b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_four)second);
    return __builtin_bit_cast(bf16x8, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
}

// Four floats, split, to three parts `part_bytes` apart.
__device__ __forceinline__ void put_split(char* to, int part_bytes, split_f32x4 x, uint32_t upper) {
    uint32_t w[2][kParts];
    split_pair(x[0], x[1], upper, w[0][0], w[0][1], w[0][2]);
    split_pair(x[2], x[3], upper, w[1][0], w[1][1], w[1][2]);
#pragma unroll
    for (int p = 0; p < kParts; ++p) *reinterpret_cast<split_u32x2*>(to + p * part_bytes) = split_u32x2{w[0][p], w[1][p]};
}

template <int H, bool DQ>
__global__ __launch_bounds__(64 * kSplitWaves)
__attribute__((amdgpu_waves_per_eu(H == 32 ? 3 : 2, H == 32 ? 3 : 2)))
void attention_key_grad_split_kernel(KeyGradArgs a) {
#pragma clang fp contract(off)
    using S = KeyGradStage<H>;
    constexpr int CHUNKS = H / 16;   // 16-deep chunks over h
    constexpr int OBLOCKS = H / 32;  // 32-row accumulator blocks of dV^T and dK^T
    constexpr int G = H / 4;         // groups of 4 h
    __shared__ __attribute__((aligned(16))) char stage[S::BYTES];
    __shared__ __attribute__((aligned(16))) char k_lds[kParts * S::K_PART];
    __shared__ __attribute__((aligned(16))) float records[3 * kSplitQueries];
    // Per wave: 1 once its part of the block has to be computed again.
    __shared__ __attribute__((aligned(16))) uint32_t marks[kSplitWaves];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 31;
    const int half = lane >> 5;
    const uint32_t upper = upper_half_mask();
    marks[wave] = 0;

    const int64_t block = blockIdx.x;
    const int64_t head = block % a.heads;
    const int64_t k_block = block / a.heads;
    const int64_t k_first = k_block * kKeyBlock;
    const int64_t k_wave = k_first + 32 * wave;
    const int64_t key = k_wave + col;
    const bool key_ok = key < a.keys;
    const int64_t q_begin = stage_begin(k_block, a.query_offset);
    const int stages_total = q_begin < a.queries ? int((a.queries - q_begin + kSplitQueries - 1) / kSplitQueries) : 0;

    const int64_t plane = plane_of(a.queries);
    const float* r_head = a.rows + head * 3 * plane;
    const __amdgpu_buffer_rsrc_t k_rsrc = buffer_of(a.k + head * a.kv_stride + k_first * H);

    // A thread's vectors of a stage: the first half of the threads take Q's rows,
    // the other dO's; G consecutive threads read a row.
    constexpr int VECTORS = H / 16;
    constexpr int ROWS_APART = 32 * kSplitWaves / G;
    const int operand = wave / 2;
    const int hg = tid % G;
    const int row0 = tid % (32 * kSplitWaves) / G;
    const float* o_head = (operand == 0 ? a.q : a.d_out) + head * a.q_stride;
    split_f32x4 next[VECTORS];
    float next_record = 0.f;
    auto load = [&](int64_t q0) __attribute__((always_inline)) {
        // Rows past the last query read zeros.
        const int left = int(min(max(a.queries - q0, int64_t(0)), int64_t(kSplitQueries)));
        const __amdgpu_buffer_rsrc_t rsrc = buffer_of(o_head + q0 * H);
#pragma unroll
        for (int r = 0; r < VECTORS; ++r) {
            const int row = row0 + ROWS_APART * r;
            const int32_t off = row < left ? (row * H + 4 * hg) * 4 : kOutOfRange;
            next[r] = __builtin_bit_cast(split_f32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, off, 0, 0));
        }
        if (tid < 3 * kSplitQueries) {
            const int q = tid % kSplitQueries;
            next_record = q < left ? r_head[(tid / kSplitQueries) * plane + q0 + q] : 0.f;
        }
    };
    const int row_store = operand * S::ROWS + (hg / 2 * S::ROW_PLANE + row0) * 16 + 8 * (hg % 2);
    auto store = [&]() __attribute__((always_inline)) {
        if (out_of_range([&](auto f) __attribute__((always_inline)) {
#pragma unroll
                for (int r = 0; r < VECTORS; ++r) {
                    f(next[r][0], next[r][1]);
                    f(next[r][2], next[r][3]);
                }
            }))
            marks[wave] = 1;
#pragma unroll
        for (int r = 0; r < VECTORS; ++r) put_split(stage + row_store + ROWS_APART * r * 16, S::ROW_PART, next[r], upper);
        if (tid < 3 * kSplitQueries)
            records[tid] = tid / kSplitQueries == 1 ? next_record * kGradScale : next_record;  // 1 / l scaled
    };

    load(q_begin);
    {
        const int rows_left = int(min(a.keys - k_first, int64_t(kKeyBlock)));
        constexpr int KN = kKeyBlock * G / (64 * kSplitWaves);
        split_f32x4 x[KN];
#pragma unroll
        for (int u = 0; u < KN; ++u) {
            const int e = tid + u * 64 * kSplitWaves;
            const int32_t off = e / G < rows_left ? 16 * e : kOutOfRange;
            x[u] = __builtin_bit_cast(split_f32x4, __builtin_amdgcn_raw_buffer_load_b128(k_rsrc, off, 0, 0));
        }
        if (out_of_range([&](auto f) __attribute__((always_inline)) {
#pragma unroll
                for (int u = 0; u < KN; ++u) {
                    f(x[u][0], x[u][1]);
                    f(x[u][2], x[u][3]);
                }
            }))
            marks[wave] = 1;
#pragma unroll
        for (int u = 0; u < KN; ++u)
            put_split(k_lds + (hg / 2 * S::K_PLANE + tid / G + u * 64 * kSplitWaves / G) * 16 + 8 * (hg % 2), S::K_PART,
                      x[u], upper);
    }
    __builtin_amdgcn_sched_barrier(0);
    // V of this lane's key: chunk c holds h 16 c + 8 half + (0..7).
    SplitVector vs[CHUNKS];
    {
        float x[CHUNKS][8];
#pragma unroll
        for (int c = 0; c < CHUNKS; ++c) {
            const float* from = a.v + head * a.kv_stride + (key_ok ? key : 0) * H + 8 * half + 16 * c;
            const split_f32x4 lo = *reinterpret_cast<const split_f32x4*>(from);
            const split_f32x4 hi = *reinterpret_cast<const split_f32x4*>(from + 4);
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                x[c][s] = key_ok ? lo[s] : 0.f;
                x[c][4 + s] = key_ok ? hi[s] : 0.f;
            }
        }
        if (out_of_range([&](auto f) __attribute__((always_inline)) {
#pragma unroll
                for (int c = 0; c < CHUNKS; ++c)
#pragma unroll
                    for (int s = 0; s < 8; s += 2) f(x[c][s], x[c][s + 1]);
            }))
            marks[wave] = 1;
#pragma unroll
        for (int c = 0; c < CHUNKS; ++c) vs[c] = split_vector(x[c], upper);
    }
    f32x16 dv[OBLOCKS], dk[OBLOCKS];
    auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int b = 0; b < OBLOCKS; ++b)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                dv[b][r] = 0.f;
                dk[b][r] = 0.f;
            }
    };
    clear();

    // The stage's 32 queries (octets of h at `rows`) against this wave's keys,
    // whose chunk c right(c, part) gives. Each chunk's fragments are read under
    // the MFMAs of the chunk before (all at once they would spill). The right
    // factor's parts come first in the terms, as K's do in the forward, so that
    // S has the bits its row statistics were formed from.
    const int row_read = (half * S::ROW_PLANE + col) * 16;
    auto product = [&](const char* rows, auto right) __attribute__((always_inline)) {
        f32x16 acc;
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[r] = 0.f;
        bf16x8 f[2][kParts], g[2][kParts];
        auto read = [&](int c) __attribute__((always_inline)) {
#pragma unroll
            for (int p = 0; p < kParts; ++p) {
                f[c % 2][p] =
                    *reinterpret_cast<const bf16x8*>(rows + row_read + p * S::ROW_PART + 2 * c * S::ROW_PLANE * 16);
                g[c % 2][p] = right(c, p);
            }
        };
        read(0);
#pragma unroll
        for (int c = 0; c < CHUNKS; ++c) {
            if (c + 1 < CHUNKS) read(c + 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int t = 0; t < kTerms; ++t)
                acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[c % 2][term_right(t)], g[c % 2][term_left(t)], acc, 0,
                                                              0, 0);
        }
        return acc;
    };
    const int k_read = (half * S::K_PLANE + 32 * wave + col) * 16;
    auto k_fragment = [&](int c, int p) __attribute__((always_inline)) {
        return *reinterpret_cast<const bf16x8*>(k_lds + k_read + p * S::K_PART + 2 * c * S::K_PLANE * 16);
    };
    auto v_fragment = [&](int c, int p) __attribute__((always_inline)) { return vs[c].part[p]; };
    // acc^T += rows^T x over the queries of chunk c (x: registers 8 c .. + 7):
    // this lane points at query 4 half + lane % 16 / 4 (and 8 more), h 16 (lane / 16 % 2) + 4 (lane % 4).
    const int column_read = ((lane >> 4 & 1) * 2 + (lane >> 1 & 1)) * S::ROW_PLANE * 16 +
                            (4 * half + (lane >> 2 & 3)) * 16 + 8 * (lane & 1);
    auto add_columns = [&](const char* rows, int c, const SplitVector& x, f32x16 (&acc)[OBLOCKS])
                           __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int b = 0; b < OBLOCKS; ++b) {
            bf16x8 f[kParts];
#pragma unroll
            for (int p = 0; p < kParts; ++p) {
                const char* at = rows + column_read + p * S::ROW_PART + (4 * b * S::ROW_PLANE + 16 * c) * 16;
                f[p] = transposed(at, at + 8 * 16);
            }
            // The chunk's terms from zero, then one addition: the long sum is rounded once per 16 queries, not six
            // times (2048 queries against 64 bits: 7.4e-7 with six, 3.3e-7 so; the fp32 kernel 6.8e-7).
            f32x16 sum;
#pragma unroll
            for (int r = 0; r < 16; ++r) sum[r] = 0.f;
#pragma unroll
            for (int t = 0; t < kTerms; ++t)
                sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[term_left(t)], x.part[term_right(t)], sum, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[b][r] = acc[b][r] + sum[r];
        }
    };
    // This wave's block of the stage; dS split, register pairs (2 i, 2 i + 1), into ds.
    auto block_grad = [&](int64_t q0, uint32_t (&ds)[kParts][8]) __attribute__((always_inline)) {
        const f32x16 s = product(stage, k_fragment);
        __builtin_amdgcn_sched_barrier(0);
        const f32x16 dp = product(stage + S::ROWS, v_fragment);
        const float* rs = records + 4 * half;
        __builtin_amdgcn_sched_barrier(0);
        // This lane's key is seen from row `first` of the block on. Rows past the last query have 1 / l = 0. One
        // path for all blocks: a second one without the test cost more in spilled registers than the test.
        const int first =
            key_ok ? int(max(min(k_wave - a.query_offset - q0, int64_t(32)), int64_t(-32))) + col - 4 * half : 64;
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            float p[8], gr[8];
#pragma unroll
            for (int g = 0; g < 2; ++g) {
                const int at = 8 * (2 * c + g);
                const split_f32x4 m4 = *reinterpret_cast<const split_f32x4*>(rs + at);
                const split_f32x4 il4 = *reinterpret_cast<const split_f32x4*>(rs + kSplitQueries + at);
                const split_f32x4 d4 = *reinterpret_cast<const split_f32x4*>(rs + 2 * kSplitQueries + at);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float shifted = s[8 * c + 4 * g + j] * a.scale - m4[j];
                    const float pr = exp_of(shifted) * il4[j];
                    const float difference = dp[8 * c + 4 * g + j] - d4[j];
                    p[4 * g + j] = at + j >= first ? pr : 0.f;
                    gr[4 * g + j] = p[4 * g + j] * difference;  // NaN if dP is not finite: computed again
                }
            }
            add_columns(stage + S::ROWS, c, split_vector(p, upper), dv);
            __builtin_amdgcn_sched_barrier(0);
            const SplitVector gs = split_vector(gr, upper);
            add_columns(stage, c, gs, dk);
            __builtin_amdgcn_sched_barrier(0);
            typedef uint32_t words __attribute__((ext_vector_type(4)));
#pragma unroll
            for (int q = 0; q < kParts; ++q) {
                const words w = __builtin_bit_cast(words, gs.part[q]);
#pragma unroll
                for (int i = 0; i < 4; ++i) ds[q][4 * c + i] = w[i];
            }
        }
    };

    // dQ partial sums of this block: rows from its first stage's first query.
    int64_t rows_before = 0;
    for (int64_t b = 0; b < k_block; ++b) rows_before += block_queries(b, a.queries, a.query_offset);
    const __amdgpu_buffer_rsrc_t p_rsrc = buffer_of(DQ ? a.partials + (head * a.partial_rows + rows_before) * H : a.q);
    constexpr int HT = H / 32;  // 16-column tiles of a wave's share
    const int h_base = (wave / 2) * (H / 2);
    // Word (keys col & ~1, + 1) of query row 4 half + (lane & 1) + ...
    const int ds_store = ((4 * wave + col / 8) * S::DS_PLANE + 4 * half + (lane & 1)) * 16 + col % 8 / 2 * 4;
    const uint32_t pick = lane & 1 ? 0x03020706u : 0x05040100u;
    float poison = 0.f;
    auto look = [&](float x) __attribute__((always_inline)) {
        poison = __builtin_fmaf(x, 0.f, poison);  // NaN from the first non-finite value on
    };
    // dQ's 16 x 16 result: lane l's four h of query dq_row. Rows past the last query are dropped (out-of-range
    // offsets).
    auto store_partial = [&](int64_t q0, int dq_row, int lg, int t, split_f32x4 sum) __attribute__((always_inline)) {
        typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
        const int64_t q = q0 + dq_row;
        const int32_t off =
            q < a.queries ? int32_t(((q - q_begin) * H + h_base + 16 * t + 4 * lg) * 4) : kOutOfRange;
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, sum), p_rsrc, off, 0, 0);
    };
    auto dq_step = [&](int64_t q0) __attribute__((always_inline)) {
        int l = lane;
        hide(l);
        const int lq = l % 16, lg = l / 16;
        const int dq_row = 16 * (wave % 2) + lq;
        const int b_read = (lg * S::DS_PLANE + dq_row) * 16;
        // This lane points at key 8 lg + lq / 4 (and 4 more), h h_base + 4 (lq % 4).
        const int a_read = ((h_base / 8 + (lq >> 1 & 1)) * S::K_PLANE + 8 * lg + lq / 4) * 16 + 8 * (lq & 1);
        split_f32x4 acc[HT];
#pragma unroll
        for (int t = 0; t < HT; ++t) acc[t] = split_f32x4{0.f, 0.f, 0.f, 0.f};
        // Read a tile ahead, as in product().
        constexpr int TILES = kKeyBlock / 32 * HT;  // tile x: keys 32 (x / HT) .. + 31, column tile x % HT
        bf16x8 d[2][kParts], f[2][kParts];
        auto read = [&](int x) __attribute__((always_inline)) {
            const int u = x / HT, t = x % HT;
#pragma unroll
            for (int p = 0; p < kParts; ++p) {
                if (t == 0)
                    d[u % 2][p] = *reinterpret_cast<const bf16x8*>(stage + b_read + p * S::DS_PART +
                                                                   4 * u * S::DS_PLANE * 16);
                const char* at = k_lds + a_read + p * S::K_PART + (2 * t * S::K_PLANE + 32 * u) * 16;
                f[x % 2][p] = transposed(at, at + 4 * 16);
            }
        };
        read(0);
#pragma unroll
        for (int x = 0; x < TILES; ++x) {
            if (x + 1 < TILES) read(x + 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < kTerms; ++i)
                acc[x % HT] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    f[x % 2][term_left(i)], d[x / HT % 2][term_right(i)], acc[x % HT], 0, 0, 0);
        }
#pragma unroll
        for (int t = 0; t < HT; ++t) {
            split_f32x4 sum;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                look(acc[t][r]);
                sum[r] = acc[t][r] * kGradUnscale;
            }
            store_partial(q0, dq_row, lg, t, sum);
        }
    };

    // dV = (dV^T)^T and dK = (dK^T)^T: lane l holds h rows 32 b + 4 half + 8 g + (0..3) of its key, times
    // 1 / `unscale`. Adds to what an earlier flush left (`add`); the last one scales dK.
    auto flush = [&](bool add, bool last, float unscale) __attribute__((always_inline)) {
        if (!key_ok) return;
        float* vrow = a.v_grad + (head * a.keys + key) * H + 4 * half;
        float* krow = a.k_grad + (head * a.keys + key) * H + 4 * half;
        const float scale = last ? a.scale : 1.f;
#pragma unroll
        for (int b = 0; b < OBLOCKS; ++b)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                split_f32x4* vp = reinterpret_cast<split_f32x4*>(vrow + 32 * b + 8 * g);
                split_f32x4* kp = reinterpret_cast<split_f32x4*>(krow + 32 * b + 8 * g);
                split_f32x4 vo, ko;
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    vo[s] = dv[b][4 * g + s] * unscale;
                    ko[s] = dk[b][4 * g + s] * unscale;
                }
                if (add) {
                    const split_f32x4 v0 = *vp, k0 = *kp;
#pragma unroll
                    for (int s = 0; s < 4; ++s) {
                        vo[s] = v0[s] + vo[s];
                        ko[s] = k0[s] + ko[s];
                    }
                }
#pragma unroll
                for (int s = 0; s < 4; ++s) ko[s] = scale * ko[s];
                *vp = vo;
                *kp = ko;
            }
    };
    auto look_all = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int b = 0; b < OBLOCKS; ++b)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                look(dv[b][r]);
                look(dk[b][r]);
            }
    };

    for (int st = 0; st < stages_total; ++st) {
        const int64_t q0 = q_begin + int64_t(st) * kSplitQueries;
        if (st > 0 && st % kFlushStages == 0) {
            look_all();
            flush(st > kFlushStages, false, kGradUnscale);
            clear();
        }
        store();
        load(q0 + kSplitQueries);  // past the last query: zeros, no traffic
        lds_barrier();
        uint32_t ds[kParts][8];
#pragma unroll
        for (int q = 0; q < kParts; ++q)
#pragma unroll
            for (int i = 0; i < 8; ++i) ds[q][i] = 0;
        // Wave-uniform: skipped when none of the block's queries sees the wave's first key.
        if (q0 + 31 + a.query_offset >= k_wave && k_wave < a.keys) block_grad(q0, ds);
        lds_barrier();  // every wave is done with the stage
        if constexpr (!DQ) continue;
        int to_ds = ds_store;
        hide(to_ds);
#pragma unroll
        for (int q = 0; q < kParts; ++q)
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                // Queries 8 (i / 2) + 2 (i % 2) + 0, 1 of this lane's key: an even lane keeps the first, an odd
                // one the second, each with its neighbour's key beside it.
                const uint32_t other = uint32_t(__builtin_amdgcn_mov_dpp(int(ds[q][i]), 0xB1, 0xF, 0xF, true));
                *reinterpret_cast<uint32_t*>(stage + to_ds + q * S::DS_PART + (8 * (i / 2) + 2 * (i % 2)) * 16) =
                    __builtin_amdgcn_perm(other, ds[q][i], pick);
            }
        lds_barrier();  // the stage's dS is whole
        dq_step(q0);
        lds_barrier();  // and read
    }
    look_all();
    if (__any(poison != 0.f)) marks[wave] = 1;
    lds_barrier();
    static_assert(kSplitWaves == 4, "the waves' marks");
    if (__builtin_amdgcn_readfirstlane(marks[0] | marks[1] | marks[2] | marks[3]) == 0) {
        flush(stages_total > kFlushStages, true, kGradUnscale);
        return;
    }

    // The block again, operands from memory: a 32 x 32 block of S (block_scores) and dP per wave as above, P and dS as
    // they are, dS through LDS for dQ; the products with the fp32 instruction. Rare, and written for few registers.
    clear();
    bool k_outside = false;  // this lane's K is not what the split holds
#pragma unroll 1
    for (int c = 0; c < CHUNKS; ++c) {
        const float* from = a.k + head * a.kv_stride + (key_ok ? key : 0) * H + 8 * half + 16 * c;
        k_outside |= out_of_range([&](auto f) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < 8; i += 2) f(key_ok ? from[i] : 0.f, key_ok ? from[i + 1] : 0.f);
        });
    }
#pragma unroll 1
    for (int64_t q0 = q_begin; q0 < a.queries; q0 += kSplitQueries) {
        const float* q_head = a.q + head * a.q_stride;
        const float* d_head = a.d_out + head * a.q_stride;
        const bool row_ok = q0 + col < a.queries;
        const int64_t row = (row_ok ? q0 + col : 0) * H + 8 * half;
        const int64_t kv_row = head * a.kv_stride + (key_ok ? key : 0) * H + 8 * half;
        const f32x16 s = block_scores<H, false, 1>(
            [&](int c, float (&x)[8]) __attribute__((always_inline)) {
#pragma unroll
                for (int i = 0; i < 8; ++i) x[i] = row_ok ? q_head[row + 16 * c + i] : 0.f;
            },
            [&](int c, float (&y)[8]) __attribute__((always_inline)) {
#pragma unroll
                for (int i = 0; i < 8; ++i) y[i] = key_ok ? a.k[kv_row + 16 * c + i] : 0.f;
            },
            k_outside, upper);
        f32x16 dp;
#pragma unroll
        for (int r = 0; r < 16; ++r) dp[r] = 0.f;
#pragma unroll 1
        for (int c = 0; c < CHUNKS; ++c) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float x = d_head[row + 16 * c + i], y = a.v[kv_row + 16 * c + i];
                dp = __builtin_amdgcn_mfma_f32_32x32x2f32(row_ok ? x : 0.f, key_ok ? y : 0.f, dp, 0, 0, 0);
            }
        }
        float* ds_lds = reinterpret_cast<float*>(stage) + (32 * wave + col) * S::DS_ROW;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int at = 8 * (r / 4) + 4 * half + r % 4;
            const int64_t q = q0 + at;
            const bool visible = key_ok && q < a.queries && key <= q + a.query_offset;
            const float* record = r_head + (q < a.queries ? q : 0);
            const float shifted = s[r] * a.scale - record[0];
            const float p = exp_of(shifted) * record[plane];
            const float g = p * (dp[r] - record[2 * plane]);
            const float pr = visible ? p : 0.f, gr = visible ? g : 0.f;
            ds_lds[at] = gr;
            const float* qrow = q_head + (q < a.queries ? q : 0) * H + col;
            const float* drow = d_head + (q < a.queries ? q : 0) * H + col;
#pragma unroll
            for (int b = 0; b < OBLOCKS; ++b) {
                dv[b] = __builtin_amdgcn_mfma_f32_32x32x2f32(q < a.queries ? drow[32 * b] : 0.f, pr, dv[b], 0, 0, 0);
                dk[b] = __builtin_amdgcn_mfma_f32_32x32x2f32(q < a.queries ? qrow[32 * b] : 0.f, gr, dk[b], 0, 0, 0);
            }
        }
        if constexpr (DQ) {
            lds_barrier();  // the stage's dS is whole
            const int lq = lane % 16, lg = lane / 16;
            const int dq_row = 16 * (wave % 2) + lq;
#pragma unroll
            for (int t = 0; t < HT; ++t) {
                split_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
                for (int u = 0; u < kKeyBlock; u += 4) {
                    const bool ok = k_first + u + lg < a.keys;
                    const float kv = a.k[head * a.kv_stride + (ok ? k_first + u + lg : 0) * H + h_base + 16 * t + lq];
                    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(
                        ok ? kv : 0.f, reinterpret_cast<const float*>(stage)[(u + lg) * S::DS_ROW + dq_row], acc, 0, 0,
                        0);
                }
                store_partial(q0, dq_row, lg, t, acc);
            }
            lds_barrier();  // and read
        }
    }
    flush(false, true, 1.f);
}

}  // namespace
}  // namespace sn
