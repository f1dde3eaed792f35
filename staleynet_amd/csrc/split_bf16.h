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

constexpr int kParts = 3;  // hi, mid, lo

// The terms of a product of two split values that reach 2^-24 of it, smallest
// first (parts of the left and of the right factor).
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

// One third of the split of a pair of values: piece 0 takes hi (the upper 16
// bits) and leaves the rests in x0 and x1, piece 1 takes mid (the rest
// rounded), piece 2 lo (what that leaves: at most 8 bits, exact).
__device__ __forceinline__ void split_piece(int piece, float& x0, float& x1, uint32_t upper, uint32_t& hi,
                                            uint32_t& mid, uint32_t& lo) {
    if (piece == 0) {
        const uint32_t b0 = __builtin_bit_cast(uint32_t, x0), b1 = __builtin_bit_cast(uint32_t, x1);
        hi = __builtin_amdgcn_perm(b1, b0, 0x07060302u);
        x0 = x0 - __builtin_bit_cast(float, b0 & upper);
        x1 = x1 - __builtin_bit_cast(float, b1 & upper);
    } else if (piece == 1) {
        mid = pack2_bf16(x0, x1);
        x0 = x0 - __builtin_bit_cast(float, mid << 16);
    } else {
        x1 = x1 - __builtin_bit_cast(float, mid & upper);
        lo = pack2_bf16(x0, x1);
    }
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
