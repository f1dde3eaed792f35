// An fp32 value as the exact sum of three bf16 values, for products of fp32
// operands on the bf16 matrix cores (gemm_f32.h has the arithmetic and its
// error; the attention kernels use the same terms).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace sn {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// Two floats -> two bf16 in one 32-bit word (element 0 in the low half):
// gfx950's v_cvt_pk_bf16_f32, which rounds by the MODE register's f32
// rounding mode (round to nearest, ties to even, by default) and keeps NaN a
// quiet NaN. One instruction per pair instead of a shift/add/compare
// sequence per element.
__device__ __forceinline__ uint32_t pack2_bf16(float lo, float hi) {
    typedef float pair_f32 __attribute__((ext_vector_type(2)));
    typedef __bf16 pair_bf16 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(pair_f32{lo, hi}, pair_bf16));
}

constexpr int kParts = 3;  // hi, mid, lo: each the rest so far rounded to bf16

// The six terms of a product of two split values that are kept, smallest first
// (parts of the left and of the right factor). With hi within 2^-8 of the
// value's power of two, mid is at most 2^-8 and lo 2^-17 of it, so the three
// terms left out (mid lo, lo mid, lo lo) are together under 2^-24 of the
// product. (Splitting fp32 into bf16 parts for the matrix cores: Henry, Tang
// and Heinecke, "Leveraging the bfloat16 Artificial Intelligence Datatype For
// Higher-Precision Computations", 2019.)
constexpr int kTerms = 6;
__host__ __device__ constexpr int term_left(int t) { return t == 0 ? 2 : t == 2 || t == 3 ? 1 : 0; }
__host__ __device__ constexpr int term_right(int t) { return t == 1 ? 2 : t == 2 || t == 4 ? 1 : 0; }

// 0xffff0000 in a vector register (v_and with a literal or scalar operand
// runs at half the rate).
__device__ __forceinline__ uint32_t upper_half_mask() {
    uint32_t mask = 0xffff0000u;
    asm("" : "+v"(mask));
    return mask;
}

// The split is exact for zeros and from 2^-110 on: there a value's last bit is
// 2^-133 or more, bf16's smallest subnormal (the matrix cores keep subnormal
// factors, products and sums). range_key orders values by magnitude with zeros
// last, so that the least key of many tells whether the split holds them all.
constexpr float kSplitLeast = 0x1p-110f;
constexpr uint32_t kSplitLeastKey = 2 * (17u << 23) - 1;  // of kSplitLeast
__device__ __forceinline__ uint32_t range_key(float x) { return (__builtin_bit_cast(uint32_t, x) << 1) - 1; }
__device__ __forceinline__ void note_range(float x0, float x1, uint32_t& least) {
    least = min(min(least, range_key(x0)), range_key(x1));
    asm("" : "+v"(least));  // one running value: keys gathered first would take registers
}

// Whether this lane holds a value that the split does not; `pairs` calls its
// argument with every pair of values. The smallest magnitude first (half an
// instruction a value), each value's range only where a lane of the wave has
// one under the range, or 0.
template <class Pairs>
__device__ __forceinline__ bool out_of_range(Pairs&& pairs) {
    float m = 1.f;
    pairs([&](float x0, float x1) __attribute__((always_inline)) {
        m = fminf(fminf(m, fabsf(x0)), fabsf(x1));
        asm("" : "+v"(m));  // one running value, as in note_range
    });
    if (!__any(m < kSplitLeast)) return false;
    uint32_t least = ~0u;
    pairs([&](float x0, float x1) __attribute__((always_inline)) { note_range(x0, x1, least); });
    return least < kSplitLeastKey;
}

// One third of the split of a pair of values: piece 0 takes hi (the value
// rounded to nearest) and leaves the rests in x0 and x1, piece 1 takes mid (the
// rest rounded), piece 2 lo (what that leaves: at most 7 bits, exact). A value
// within 2^-9 of the largest float rounds to an infinite hi and leaves NaN.
__device__ __forceinline__ void split_piece(int piece, float& x0, float& x1, uint32_t upper, uint32_t& hi,
                                            uint32_t& mid, uint32_t& lo) {
    if (piece == 2) {
        x1 = x1 - __builtin_bit_cast(float, mid & upper);
        lo = pack2_bf16(x0, x1);
        return;
    }
    uint32_t& part = piece == 0 ? hi : mid;
    part = pack2_bf16(x0, x1);
    x0 = x0 - __builtin_bit_cast(float, part << 16);
    if (piece == 0) x1 = x1 - __builtin_bit_cast(float, part & upper);
}

__device__ __forceinline__ void split_pair(float x0, float x1, uint32_t upper, uint32_t& hi, uint32_t& mid,
                                           uint32_t& lo) {
#pragma unroll
    for (int piece = 0; piece < 3; ++piece) split_piece(piece, x0, x1, upper, hi, mid, lo);
}

// Eight consecutive k of a fragment, split.
struct SplitVector {
    bf16x8 part[kParts];
};
__device__ __forceinline__ SplitVector split_vector(const float (&x)[8], uint32_t upper) {
    typedef uint32_t words __attribute__((ext_vector_type(4)));
    words w[kParts];
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        uint32_t h, m, l;
        split_pair(x[2 * p], x[2 * p + 1], upper, h, m, l);
        w[0][p] = h;
        w[1][p] = m;
        w[2][p] = l;
    }
    SplitVector out;
#pragma unroll
    for (int q = 0; q < kParts; ++q) out.part[q] = __builtin_bit_cast(bf16x8, w[q]);
    return out;
}

}  // namespace sn
