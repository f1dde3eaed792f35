// Fused causal attention forward: O = causal_softmax(scale * Q K^T) V per
// head, without writing the [queries, keys] score matrix. The reference
// computes it as three calls (layers/attention.rs:206-213): the scores
// product (MatmulSpec::new(T, T, h).right_transposed(), batched over the
// heads), causal_softmax (kernels/attention.rs:140-183) and the mix product
// (MatmulSpec::new(T, h, T)); the probabilities it keeps for the backward
// are written here on request, so the backward (attention.rs:220-267) can
// run unchanged.
//
// Layout: Q [heads][queries][h] and K, V [heads][keys][h] (head-major, rows
// q_stride / kv_stride floats apart per head), O [heads][queries][h], P
// [heads][queries][keys]. Query q of a head sees keys 0 ..= q +
// query_offset (as causal_softmax with `queries` rows per matrix).
//
// Design (gfx950; both products as six bf16 products of exactly split fp32
// values, split_bf16.h and gemm_f32.h: 192 matrix-core cycles per 32 x 32 x 16
// where v_mfma_f32_32x32x2f32 takes 512):
//  * A workgroup of 4 waves owns 128 queries of one head; a wave owns 32.
//    K and V stream through LDS in blocks of 64 keys: a thread loads its
//    pieces of the next block into registers under the current block's work,
//    splits them once and writes the three parts to the one LDS stage, K as
//    octets of h per key, V as octets of keys per h.
//  * A wave computes S^T = K Q^T for 32 keys at a time (keys along the
//    accumulator rows, its 32 queries along the columns, the split Q held in
//    registers). In the 32x32 accumulator, lane l holds column l % 32, so
//    every register of a lane belongs to the lane's query: the online
//    softmax (running max m, running sum l, O rescaled by exp(m_old -
//    m_new)) is per lane, with one exchange between the lane pair (l, l ^
//    32) that share a query. A lane's eight consecutive registers are keys
//    4 half + 0..3 and 8 + 4 half + 0..3 of 16: split, they are a B operand
//    of O^T += V^T P^T as they are, because V's octets hold those keys.
//  * Element arithmetic follows causal_softmax: s * scale, minus the
//    maximum, each rounded, then the exponential (as 2^(d log2 e) on the
//    transcendental unit); the sum is accumulated in a different order (per
//    32-key block, then rescaled), so parity is to the fp32 tolerance.
//  * Only the 32-key blocks on a wave's diagonal (or past the last key) test
//    keys against each query's horizon; the others skip the mask.
//  * Operands outside the split's range (split_bf16.h): each thread looks at the
//    K and V it splits, and a wave at its Q. A wave with such a value among its
//    operands, with an output or sum that is not finite or with no finite
//    score recomputes its queries straight from memory, P V and the scores of
//    the blocks that need it (block_scores) with the fp32 instruction. The softmax's own e^(x - m) need no look: the exponential unit
//    gives 0 under 2^-126 (as it did before the split), and the split is off by
//    2^-134 at most on the ones between that and 2^-110, against sums of 1 or
//    more. (The look costs 0.4 us of a prompt chunk's 20, and half a percent of
//    a long sequence's training step.)
//  * P (optional) takes a second pass over K with the final m and l: p =
//    e^(s * scale - m) * (1 / l), 0 past the diagonal, so it matches the
//    probabilities causal_softmax leaves to the fp32 tolerance.
//  * Query blocks are launched longest first across all heads (the last
//    queries see the most keys).
//  * Few query blocks (a prompt chunk of one sequence) leave most CUs idle:
//    the keys are then split over workgroups that leave O, m and l of their
//    range in the workspace, merged by a second kernel in range order.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <type_traits>

#include "attention_common.h"
#include "gemm_internal.h"
#include "split_bf16.h"

namespace sn {
namespace {

using namespace attn;

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

struct AttentionArgs {
    const float* q;
    const float* k;
    const float* v;
    float* o;
    float* p;      // null: no probabilities
    float* stats;  // null, or per query {m, l}: the maximum of its scaled visible scores and the sum of e^(x - m)
    // Split keys: workgroup `split` of a query block takes keys split *
    // keys_per_split .. and leaves unscaled O [split][head][query][h] and {m,
    // l} [split][head][query] here. keys_per_split 0: all keys, O as it is.
    float* partial_o;
    float* partial_stats;
    int64_t queries, keys;
    int64_t q_stride, kv_stride;  // floats between heads
    int64_t query_offset;
    int64_t heads;
    int64_t keys_per_split;
    int32_t query_blocks;
    float scale;
};

// LDS stage of kKeys keys. K: per part, h / 8 octets of K_PLANE slots (slot =
// key; the pad puts the octets a 16-lane write phase touches on distinct
// banks); V: per part, kKeys / 8 octets of h slots.
template <int H>
struct KvStage {
    static constexpr int K_PLANE = kKeys + (H == 32 ? 4 : 2);
    static constexpr int K_PART = H / 8 * K_PLANE * 16;
    static constexpr int V_PART = kKeys / 8 * H * 16;
};

// A thread's pieces of one stage. K: vectors of 4 h (consecutive threads read
// consecutive 16 bytes of the contiguous rows). V: blocks of 4 keys x VN h:
// wave w the 16 keys of chunk w, lane bit 0 and bit 5 the 4-key group (8 and 4
// keys apart), bits 1-4 the h: a load instruction reads four rows whole, and
// an 8-byte write phase falls on distinct banks.
template <int H>
struct KvLoader {
    using S = KvStage<H>;
    static constexpr int THREADS = 64 * kWaves;
    static constexpr int G = H / 4;            // K vectors a row
    static constexpr int KN = kKeys * G / THREADS;
    static constexpr int VN = H >= 64 ? 4 : 2;
    static constexpr int VB = H >= 64 ? H / 64 : 1;
    f32x4 k[KN];
    float v[VB][4][VN];

    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t k_rsrc, __amdgpu_buffer_rsrc_t v_rsrc, int64_t key0,
                                         int64_t key_end, int tid, bool with_v) {
        // Rows from key_end on read zeros.
        const int left = int(min(max(key_end - key0, int64_t(0)), int64_t(kKeys)));
        const int32_t base = int32_t(key0 * H * 4);
#pragma unroll
        for (int u = 0; u < KN; ++u) {
            const int e = tid + u * THREADS;
            k[u] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                                 k_rsrc, (base + 16 * e) | ((left - 1 - e / G) & kOutOfRange), 0, 0));
        }
        if (!with_v) return;
        const int lane = tid & 63;
        const int key = 16 * (tid >> 6) + 8 * (lane & 1) + 4 * (lane >> 5);
        const int h = VN * (lane >> 1 & 15);
#pragma unroll
        for (int b = 0; b < VB; ++b)
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) {
                const int32_t off =
                    (base + ((key + kk) * H + 64 * b + h) * 4) | ((left - 1 - key - kk) & kOutOfRange);
                if constexpr (VN == 4) {
                    const f32x4 x = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(v_rsrc, off, 0, 0));
#pragma unroll
                    for (int e = 0; e < VN; ++e) v[b][kk][e] = x[e];
                } else {
                    const f32x2 x = __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(v_rsrc, off, 0, 0));
#pragma unroll
                    for (int e = 0; e < VN; ++e) v[b][kk][e] = x[e];
                }
            }
    }
    // f(x0, x1) of every pair of values held.
    template <class F>
    __device__ __forceinline__ void pairs(F&& f, bool with_v) const {
#pragma unroll
        for (int u = 0; u < KN; ++u) {
            f(k[u][0], k[u][1]);
            f(k[u][2], k[u][3]);
        }
        if (!with_v) return;
#pragma unroll
        for (int b = 0; b < VB; ++b)
#pragma unroll
            for (int kk = 0; kk < 4; ++kk)
#pragma unroll
                for (int e = 0; e < VN; e += 2) f(v[b][kk][e], v[b][kk][e + 1]);
    }
    __device__ __forceinline__ void store(char* k_stage, char* v_stage, int tid, uint32_t upper, bool with_v) const {
        const int group = tid % G;
        char* kp = k_stage + (group / 2 * S::K_PLANE + tid / G) * 16 + 8 * (group % 2);
#pragma unroll
        for (int u = 0; u < KN; ++u) put(kp + u * (THREADS / G) * 16, S::K_PART, k[u][0], k[u][1], k[u][2], k[u][3], upper);
        if (!with_v) return;
        const int lane = tid & 63;
        const int hq = lane >> 1 & 15;
        char* vp = v_stage + ((2 * (tid >> 6) + (lane >> 5)) * H + 2 * hq) * 16 + 8 * (lane & 1);
#pragma unroll
        for (int b = 0; b < VB; ++b)
#pragma unroll
            for (int e = 0; e < VN; ++e)
                put(vp + (64 * b + (H >= 64 ? 32 * (e & 1) + (e >> 1) : e)) * 16, S::V_PART, v[b][0][e], v[b][1][e],
                    v[b][2][e], v[b][3][e], upper);
    }

private:
    __device__ __forceinline__ static void put(char* to, int part_bytes, float x0, float x1, float x2, float x3,
                                               uint32_t upper) {
        uint32_t w[2][kParts];
        split_pair(x0, x1, upper, w[0][0], w[0][1], w[0][2]);
        split_pair(x2, x3, upper, w[1][0], w[1][1], w[1][2]);
#pragma unroll
        for (int q = 0; q < kParts; ++q) *reinterpret_cast<u32x2*>(to + q * part_bytes) = u32x2{w[0][q], w[1][q]};
    }
};

// h of row q of O^T's block b: V's positions interleave the two blocks of 64 h.
template <int H>
__device__ __forceinline__ constexpr int h_of(int b, int q) {
    return H >= 64 ? 64 * (b / 2) + 2 * q + b % 2 : q;
}

// Waves per SIMD the kernel's registers are budgeted for.
constexpr int forward_waves_per_simd(int h) { return h <= 32 ? 3 : h == 64 ? 2 : 1; }

template <int H>
__global__ __launch_bounds__(64 * kWaves)
__attribute__((amdgpu_waves_per_eu(forward_waves_per_simd(H), forward_waves_per_simd(H))))
void causal_attention_kernel(AttentionArgs args) {
#pragma clang fp contract(off)
    using S = KvStage<H>;
    constexpr int CHUNKS = H / 16;   // 16-deep chunks over h
    constexpr int OBLOCKS = H / 32;  // 32-row accumulator blocks of O^T
    constexpr int SUBS = kKeys / 32;
    __shared__ __attribute__((aligned(16))) char k_stage[kParts * S::K_PART];
    __shared__ __attribute__((aligned(16))) char v_stage[kParts * S::V_PART];
    // Per wave: 1 once it has staged a value the split does not hold.
    __shared__ __attribute__((aligned(16))) uint32_t marks[kWaves];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 31;  // this lane's query within the wave
    const int half = lane >> 5;
    const uint32_t upper = upper_half_mask();

    // Longest query blocks first, over all heads: the heads' last query
    // blocks (which see the most keys), then the ones before, so that the
    // short blocks fill in at the end.
    const int64_t block = blockIdx.x;
    const int64_t head = block % args.heads;
    const int64_t query_block = args.query_blocks - 1 - block / args.heads;
    const int64_t q_first = query_block * kQueries;
    const int64_t q_wave = q_first + 32 * wave;
    const int64_t q = q_wave + col;
    // Keys of this workgroup's range it can see, and those this wave can (exclusive ends).
    const int64_t key_first = int64_t(blockIdx.y) * args.keys_per_split;
    const int64_t visible = min(args.keys, min(q_first + kQueries, args.queries) - 1 + args.query_offset + 1);
    const int64_t wg_keys = args.keys_per_split > 0 ? min(visible, key_first + args.keys_per_split) : visible;
    if (key_first >= wg_keys) return;  // the merge does not read this range
    const int64_t wave_keys = min(wg_keys, q_wave + 31 + args.query_offset + 1);
    const int stages_total = int((wg_keys - key_first + kKeys - 1) / kKeys);

    const float* kh = args.k + head * args.kv_stride;
    const float* vh = args.v + head * args.kv_stride;
    const __amdgpu_buffer_rsrc_t k_rsrc = buffer_of(kh);
    const __amdgpu_buffer_rsrc_t v_rsrc = buffer_of(vh);

    // Q of this lane's query (zeros past the last): chunk c holds h 16 c + 8 half + (0..7).
    auto load_query = [&](int c, float (&x)[8]) __attribute__((always_inline)) {
        const bool ok = q < args.queries;
        const float* qrow = args.q + head * args.q_stride + (ok ? q : 0) * H;
        const f32x4 lo = *reinterpret_cast<const f32x4*>(qrow + 16 * c + 8 * half);
        const f32x4 hi = *reinterpret_cast<const f32x4*>(qrow + 16 * c + 8 * half + 4);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            x[s] = ok ? lo[s] : 0.f;
            x[4 + s] = ok ? hi[s] : 0.f;
        }
    };
    marks[wave] = 0;
    float qv[CHUNKS][8];
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) load_query(c, qv[c]);
    KvLoader<H> kv;
    kv.load(k_rsrc, v_rsrc, key_first, wg_keys, tid, true);
    // Whether this lane's Q is not what the split holds.
    const bool outside = out_of_range([&](auto f) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < CHUNKS; ++c)
#pragma unroll
            for (int s = 0; s < 8; s += 2) f(qv[c][s], qv[c][s + 1]);
    });
    SplitVector qs[CHUNKS];
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) qs[c] = split_vector(qv[c], upper);

    // S^T for 32 keys (rows 32 sub .. +31 of the stage) against this wave's queries.
    const int k_read = (half * S::K_PLANE + col) * 16;
    const int v_read = (half * H + col) * 16;
    auto scores = [&](int sub) __attribute__((always_inline)) {
        f32x16 acc;
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[r] = 0.f;
#pragma unroll
        for (int c = 0; c < CHUNKS; ++c) {
            bf16x8 f[kParts];
#pragma unroll
            for (int p = 0; p < kParts; ++p)
                f[p] = *reinterpret_cast<const bf16x8*>(k_stage + k_read + p * S::K_PART +
                                                        (2 * c * S::K_PLANE + 32 * sub) * 16);
#pragma unroll
            for (int t = 0; t < kTerms; ++t)
                acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[term_left(t)], qs[c].part[term_right(t)], acc, 0, 0, 0);
        }
        return acc;
    };
    // Key of accumulator register r of this lane, within the 32-key sub-block.
    auto key_of = [&](int r) __attribute__((always_inline)) { return 4 * half + 8 * (r / 4) + (r % 4); };

    // Online softmax state of this lane's query, and O^T (rows h, column q).
    float m = -INFINITY, l = 0.f;
    f32x16 o[OBLOCKS];
    auto clear = [&]() __attribute__((always_inline)) {
        m = -INFINITY;
        l = 0.f;
#pragma unroll
        for (int b = 0; b < OBLOCKS; ++b)
#pragma unroll
            for (int r = 0; r < 16; ++r) o[b][r] = 0.f;
    };
    clear();

    // Last key of the 32-key block from sub0 that this lane's query sees, as
    // an offset within the block: -1 (none) .. 31 (all).
    auto visible_limit = [&](int64_t sub0) __attribute__((always_inline)) {
        const int64_t last = min(wg_keys - 1, q + args.query_offset) - sub0;
        return int(max(int64_t(-1), min(int64_t(31), last)));
    };
    // Online softmax of one 32-key block (scores acc; keys sub0 ..): the
    // probability numerators in x, O rescaled to the new maximum. MASKED is
    // false when the wave's first query sees the whole block (so every lane's
    // query does): no per-key test.
    auto softmax = [&](auto masked, const f32x16& acc, int64_t sub0, float (&x)[16]) __attribute__((always_inline)) {
        constexpr bool MASKED = decltype(masked)::value;
        float block_max = -INFINITY;
        const int limit = MASKED ? visible_limit(sub0) : 31;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            x[r] = acc[r] * args.scale;
            if (MASKED) x[r] = key_of(r) <= limit ? x[r] : -INFINITY;
            block_max = fmaxf(block_max, x[r]);
        }
        block_max = fmaxf(block_max, __shfl_xor(block_max, 32));
        const float m_new = fmaxf(m, block_max);
        // A query that has seen no key yet (a split range past its horizon) has no maximum to subtract.
        const float reference = MASKED && m_new == -INFINITY ? 0.f : m_new;
        const float alpha = exp_of(m - reference);
        float sum = 0.f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            x[r] = exp_of(x[r] - reference);
            sum = sum + x[r];
        }
        sum = sum + __shfl_xor(sum, 32);
        l = l * alpha + sum;
        m = m_new;
#pragma unroll
        for (int b = 0; b < OBLOCKS; ++b)
#pragma unroll
            for (int r = 0; r < 16; ++r) o[b][r] = o[b][r] * alpha;
    };
    // O^T += V^T P^T over the block: chunk c takes registers 8 c .. 8 c + 7.
    auto mix = [&](int sub, const float (&x)[16]) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            float part[8];
#pragma unroll
            for (int s = 0; s < 8; ++s) part[s] = x[8 * c + s];
            const SplitVector ps = split_vector(part, upper);
#pragma unroll
            for (int b = 0; b < OBLOCKS; ++b) {
                bf16x8 f[kParts];
#pragma unroll
                for (int p = 0; p < kParts; ++p)
                    f[p] = *reinterpret_cast<const bf16x8*>(v_stage + v_read + p * S::V_PART +
                                                            (2 * (2 * sub + c) * H + 32 * b) * 16);
#pragma unroll
                for (int t = 0; t < kTerms; ++t)
                    o[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[term_left(t)], ps.part[term_right(t)], o[b], 0, 0,
                                                                   0);
            }
        }
    };
    using Masked = std::true_type;
    using Whole = std::false_type;
    const int64_t wave_horizon = q_wave + args.query_offset;  // last key the wave's first query sees
    // A block is whole for the wave when its first query sees every key of it (wave-uniform).
    auto whole = [&](int64_t sub0) { return sub0 + 31 <= wave_horizon && sub0 + 32 <= wg_keys; };
    for (int st = 0; st < stages_total; ++st) {
        const int64_t key0 = key_first + int64_t(st) * kKeys;
        if (out_of_range([&](auto f) __attribute__((always_inline)) { kv.pairs(f, true); })) marks[wave] = 1;
        kv.store(k_stage, v_stage, tid, upper, true);
        kv.load(k_rsrc, v_rsrc, key0 + kKeys, wg_keys, tid, true);  // past the last key: zeros, no traffic
        lds_barrier();
#pragma unroll
        for (int sub = 0; sub < SUBS; ++sub) {
            const int64_t sub0 = key0 + 32 * sub;
            if (sub0 < wave_keys) {  // wave-uniform
                const f32x16 s = scores(sub);
                float x[16];
                if (whole(sub0)) softmax(Whole{}, s, sub0, x);
                else softmax(Masked{}, s, sub0, x);
                mix(sub, x);
            }
        }
        lds_barrier();
    }

    // The scores from memory, by the split or with the fp32 instruction (block_scores).
    auto scores_again = [&](int64_t sub0) __attribute__((always_inline)) {
        const int64_t key = sub0 + col;
        const float* krow = kh + (key < wg_keys ? key : 0) * H;
        return block_scores<H, true, 1>(
            [&](int c, float (&x)[8]) __attribute__((always_inline)) {
#pragma unroll
                for (int s = 0; s < 8; ++s) x[s] = key < wg_keys ? krow[16 * c + 8 * half + s] : 0.f;
            },
            load_query, outside, upper);
    };
    float poison = l * 0.f;
#pragma unroll
    for (int b = 0; b < OBLOCKS; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) poison = __builtin_fmaf(o[b][r], 0.f, poison);  // NaN from the first non-finite value on
    // A query that sees a key of the range has a finite maximum, unless its scores overflowed.
    const bool sees = q < args.queries && q + args.query_offset >= key_first;
    const bool marked = (marks[0] | marks[1] | marks[2] | marks[3]) != 0;
    static_assert(kWaves == 4, "the waves' marks");
    const bool redo = __any(outside || marked || poison != 0.f || (sees && m == -INFINITY));
    if (redo) {
        clear();
        for (int64_t sub0 = key_first; sub0 < wave_keys; sub0 += 32) {
            const f32x16 s = scores_again(sub0);
            float x[16];
            softmax(Masked{}, s, sub0, x);
#pragma unroll
            for (int b = 0; b < OBLOCKS; ++b)
#pragma unroll
                for (int t = 0; t < 16; ++t) {
                    const int64_t key = sub0 + key_of(t);
                    const float value = key < wg_keys ? vh[key * H + h_of<H>(b, col)] : 0.f;
                    o[b] = __builtin_amdgcn_mfma_f32_32x32x2f32(value, x[t], o[b], 0, 0, 0);
                }
        }
    }

    // Element r of block b in this lane is h = h_of(b, 8 (r / 4) + 4 half + r % 4) of its query: with
    // 64 h, blocks 2 c and 2 c + 1 together hold eight consecutive h per r / 4.
    auto write_rows = [&](float* row, auto value) __attribute__((always_inline)) {
        if constexpr (H >= 64) {
#pragma unroll
            for (int c = 0; c < OBLOCKS / 2; ++c)
#pragma unroll
                for (int g = 0; g < 4; ++g)
#pragma unroll
                    for (int p = 0; p < 2; ++p) {
                        const f32x4 out = {value(o[2 * c][4 * g + 2 * p]), value(o[2 * c + 1][4 * g + 2 * p]),
                                           value(o[2 * c][4 * g + 2 * p + 1]), value(o[2 * c + 1][4 * g + 2 * p + 1])};
                        *reinterpret_cast<f32x4*>(row + 64 * c + 16 * g + 8 * half + 4 * p) = out;
                    }
        } else {
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                f32x4 out;
#pragma unroll
                for (int s = 0; s < 4; ++s) out[s] = value(o[0][4 * g + s]);
                *reinterpret_cast<f32x4*>(row + 4 * half + 8 * g) = out;
            }
        }
    };
    const int64_t row = head * args.queries + q;
    if (args.keys_per_split > 0) {
        if (q < args.queries) {
            const int64_t at = int64_t(blockIdx.y) * args.heads * args.queries + row;
            write_rows(args.partial_o + at * H, [](float x) { return x; });
            if (half == 0) *reinterpret_cast<float2*>(args.partial_stats + 2 * at) = make_float2(m, l);
        }
        return;
    }
    // The row statistics the recomputing backward needs (both lanes of a query hold the same m, l).
    if (args.stats != nullptr && q < args.queries && half == 0)
        *reinterpret_cast<float2*>(args.stats + 2 * row) = make_float2(m, l);
    if (q < args.queries) write_rows(args.o + row * H, [&](float x) { return x / l; });
    if (args.p == nullptr) return;

    // Probabilities: a second pass over K with the final m and l; 0 past the diagonal.
    float* prow = args.p + row * args.keys;
    const bool row_ok = q < args.queries;
    const bool vector_rows = (args.keys & 3) == 0;
    const float inv_l = 1.f / l;
    kv.load(k_rsrc, v_rsrc, 0, wg_keys, tid, false);
    for (int st = 0; st < stages_total; ++st) {
        const int64_t key0 = int64_t(st) * kKeys;
        kv.store(k_stage, v_stage, tid, upper, false);
        kv.load(k_rsrc, v_rsrc, key0 + kKeys, wg_keys, tid, false);
        lds_barrier();
#pragma unroll
        for (int sub = 0; sub < SUBS; ++sub) {
            const int64_t sub0 = key0 + 32 * sub;
            if (sub0 >= args.keys) continue;
            f32x16 acc;
            if (sub0 < wave_keys) {
                acc = redo ? scores_again(sub0) : scores(sub);
            } else {
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[r] = 0.f;
            }
            const int limit = visible_limit(sub0);
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                float pv[4];
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    const float shifted = acc[4 * g + s] * args.scale - m;
                    pv[s] = key_of(4 * g + s) <= limit ? exp_of(shifted) * inv_l : 0.f;
                }
                const int64_t key = sub0 + 4 * half + 8 * g;
                if (row_ok) {
                    if (vector_rows && key + 4 <= args.keys) {
                        *reinterpret_cast<f32x4*>(prow + key) = f32x4{pv[0], pv[1], pv[2], pv[3]};
                    } else {
#pragma unroll
                        for (int s = 0; s < 4; ++s)
                            if (key + s < args.keys) prow[key + s] = pv[s];
                    }
                }
            }
        }
        lds_barrier();
    }
    // Keys past every query of the workgroup: zeros, each row filled by the
    // whole workgroup with contiguous stores.
    const int64_t zero_from = int64_t(stages_total) * kKeys;
    if (zero_from < args.keys) {
        const int64_t rows = min(int64_t(kQueries), args.queries - q_first);
        for (int64_t r = 0; r < rows; ++r) {
            float* zrow = args.p + (head * args.queries + q_first + r) * args.keys;
            if (vector_rows) {
                for (int64_t e = zero_from + 4 * tid; e < args.keys; e += 4 * 64 * kWaves)
                    *reinterpret_cast<f32x4*>(zrow + e) = f32x4{0.f, 0.f, 0.f, 0.f};
            } else {
                for (int64_t e = zero_from + tid; e < args.keys; e += 64 * kWaves) zrow[e] = 0.f;
            }
        }
    }
}

// Merges the key ranges of a query in order: m the largest m_s, l = sum of
// l_s e^(m_s - m), O = sum of O_s e^(m_s - m) / l. H / 4 lanes per query.
template <int H>
__global__ __launch_bounds__(256) void attention_merge_kernel(AttentionArgs args) {
#pragma clang fp contract(off)
    const int64_t rows = args.heads * args.queries;
    const int64_t e = int64_t(blockIdx.x) * 256 + threadIdx.x;
    const int64_t row = e / (H / 4);
    const int piece = int(e % (H / 4));
    if (row >= rows) return;
    const int64_t q_first = row % args.queries / kQueries * kQueries;
    const int64_t visible = min(args.keys, min(q_first + kQueries, args.queries) - 1 + args.query_offset + 1);
    const int splits = int((visible + args.keys_per_split - 1) / args.keys_per_split);
    float m = -INFINITY;
    for (int s = 0; s < splits; ++s) m = fmaxf(m, args.partial_stats[2 * (s * rows + row)]);
    float l = 0.f;
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
    for (int s = 0; s < splits; ++s) {
        const float2 ml = *reinterpret_cast<const float2*>(args.partial_stats + 2 * (s * rows + row));
        const float weight = exp_of(ml.x - m);
        l = l + ml.y * weight;
        const f32x4 part = *reinterpret_cast<const f32x4*>(args.partial_o + (s * rows + row) * H + 4 * piece);
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = o[i] + part[i] * weight;
    }
    f32x4 out;
#pragma unroll
    for (int i = 0; i < 4; ++i) out[i] = o[i] / l;
    *reinterpret_cast<f32x4*>(args.o + row * H + 4 * piece) = out;
}

// Keys per range of the launch for `a` (0: the keys are not split): enough
// ranges for two workgroups per CU, each of two stages or more, when the query
// blocks alone give fewer than one per CU and the records fit the workspace.
// Only for queries against a cache (query_offset > 0: a prompt chunk, where
// the keys outnumber the queries). A whole sequence's forward gives the bits it
// gives with the row statistics, which do not depend on the workspace; with the
// probabilities, their pass needs the merged maximum.
constexpr int64_t kSplitMinKeys = 2 * kKeys;

int64_t keys_per_split(const CausalAttentionArgs& a, int64_t query_blocks) {
    const int64_t workgroups = a.heads * query_blocks;
    const int64_t visible = std::min(a.keys, a.queries + a.query_offset);
    const int64_t cus = std::max(a.cu_count, 1);
    if (a.p != nullptr || a.stats != nullptr || a.query_offset == 0 || a.workspace == nullptr || workgroups >= cus) return 0;
    const int64_t want = std::min((2 * cus + workgroups - 1) / workgroups, visible / kSplitMinKeys);
    if (want < 2) return 0;
    const int64_t per_split = ((visible + want - 1) / want + kKeys - 1) / kKeys * kKeys;
    const int64_t splits = (visible + per_split - 1) / per_split;
    if (splits < 2 || splits > 65535 ||
        size_t(splits) * size_t(a.heads * a.queries) * size_t(a.head_dim + 2) * sizeof(float) > a.workspace_bytes)
        return 0;
    return per_split;
}

}  // namespace

hipError_t launch_query_block_attention(const CausalAttentionArgs& a, hipStream_t stream) {
    AttentionArgs args;
    args.q = a.q;
    args.k = a.k;
    args.v = a.v;
    args.o = a.o;
    args.p = a.p;
    args.stats = a.stats;
    args.queries = a.queries;
    args.keys = a.keys;
    args.q_stride = a.q_stride;
    args.kv_stride = a.kv_stride;
    args.query_offset = a.query_offset;
    args.heads = a.heads;
    args.query_blocks = int32_t((a.queries + kQueries - 1) / kQueries);
    args.scale = a.scale;
    args.keys_per_split = keys_per_split(a, args.query_blocks);
    const int64_t visible = std::min(a.keys, a.queries + a.query_offset);
    const int64_t splits = args.keys_per_split > 0 ? (visible + args.keys_per_split - 1) / args.keys_per_split : 1;
    args.partial_o = a.workspace;
    args.partial_stats = args.keys_per_split > 0 ? a.workspace + splits * a.heads * a.queries * a.head_dim : nullptr;
    const dim3 grid(unsigned(a.heads * args.query_blocks), unsigned(splits));
    auto launch = [&](auto h) {
        constexpr int H = decltype(h)::value;
        hipLaunchKernelGGL(causal_attention_kernel<H>, grid, dim3(64 * kWaves), 0, stream, args);
        const hipError_t err = hipGetLastError();
        if (err != hipSuccess || args.keys_per_split == 0) return err;
        const int64_t threads = a.heads * a.queries * (H / 4);
        hipLaunchKernelGGL(attention_merge_kernel<H>, dim3(unsigned((threads + 255) / 256)), dim3(256), 0, stream, args);
        return hipGetLastError();
    };
    switch (a.head_dim) {
        case 32: return launch(std::integral_constant<int, 32>{});
        case 64: return launch(std::integral_constant<int, 64>{});
        case 128: return launch(std::integral_constant<int, 128>{});
        default: return hipErrorInvalidValue;
    }
}

}  // namespace sn
