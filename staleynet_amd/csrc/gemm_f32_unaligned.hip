// The fp32 tile engine's instantiations for operands that 16-byte loads cannot
// serve: a base that is not 16-byte aligned, or a contiguous dimension, leading
// dimension or batch stride that is not a multiple of 4 floats. Buffer loads
// need only 4-byte alignment, so whole steps still load 16 bytes a lane
// (kLoadDword); operands whose offsets within a step pass 31 bits are read by
// 64-bit address (kLoadPointer). A translation unit of its own, compiled
// beside gemm_f32.hip.
#include "gemm_f32.h"

namespace sn {
namespace gemm {
namespace {

// Whether every offset of a step, and of an output tile, fits the buffer
// instructions' range (buffer_ok without its alignment).
template <class T>
bool offsets_fit(const Problem& p) {
    auto span = [](bool k_contiguous, int64_t ld, int tile_rows) {
        return k_contiguous ? (int64_t(tile_rows) * ld + T::BK) * 4 : (int64_t(T::BK) * ld + tile_rows) * 4;
    };
    return span(p.a_k_contiguous, p.lda, T::BM) < kMaxBufferOffset &&
           span(p.b_k_contiguous, p.ldb, T::BN) < kMaxBufferOffset &&
           (int64_t(T::BM) * p.n + T::BN) * 4 < kMaxBufferOffset;
}

}  // namespace

template <class T>
hipError_t launch_f32_unaligned(const Problem& p, const Env& env, const Plan& plan, hipStream_t stream) {
    if (offsets_fit<T>(p)) return launch_f32_tiles<T, kLoadDword>(p, env, plan, stream, false);
    return launch_f32_tiles<T, kLoadPointer>(p, env, plan, stream, false);
}

template hipError_t launch_f32_unaligned<F32Square>(const Problem&, const Env&, const Plan&, hipStream_t);
template hipError_t launch_f32_unaligned<F32Narrow>(const Problem&, const Env&, const Plan&, hipStream_t);
template hipError_t launch_f32_unaligned<F32Small>(const Problem&, const Env&, const Plan&, hipStream_t);

}  // namespace gemm
}  // namespace sn
