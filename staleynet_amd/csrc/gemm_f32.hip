// Launches of the fp32 products (the tile engine: gemm_f32.h): the choice of
// tile, the persistent form, the product with the right operand's column
// sums, and the split-K reduce.
//
// Grid: blockIdx.x enumerates (batch, split, tile), remapped so each XCD (the
// dispatcher deals workgroups round-robin over 8 XCDs, each with its own L2)
// receives a contiguous run of whole matrices or whole K splits, each walked
// as a grouped raster. Split-K partial sums go to the context's workspace and
// a second kernel adds them in split order (deterministic).
#include "gemm_f32.h"

namespace sn {
namespace gemm {
namespace {

// The engine's K-steps as a persistent loop: each workgroup takes work items
// blockIdx.x, blockIdx.x + gridDim.x, ... (a work item is a matrix, K slice
// and tile, mapped by tile_coordinates as the one-tile kernel maps its
// workgroups) for unmasked products of whole tiles that read nothing back.
// The loads run three K-steps ahead across items, and a tile's last step
// splits the next item's first into LDS, so a tile's output stores go out
// behind the next one's first loads and drain under its first steps, where
// the one-tile kernel ends the workgroup and starts the next one's loads
// after them. Per tile the steps and MFMAs are the one-tile kernel's, and so
// are its outputs' bits.
template <class T, bool A_K, bool B_K>
__global__ __launch_bounds__(T::THREADS)
__attribute__((amdgpu_waves_per_eu(split_waves_per_eu<T>(), split_waves_per_eu<T>())))
void gemm_f32_persistent_kernel(Args args) {
    using Engine = SplitEngine<T, A_K, B_K, kLoadVector>;
    __shared__ __attribute__((aligned(16))) char stage_a[Engine::SA::BYTES];
    __shared__ __attribute__((aligned(16))) char stage_b[Engine::SB::BYTES];
    // Of the item being computed and of the next, by turns.
    __shared__ __attribute__((aligned(16))) uint32_t marks[2][T::THREADS / 64];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int wave_m = wave / T::WAVES_N;
    const int wave_n = wave % T::WAVES_N;
    const int items = args.persistent_items;
    const int stride = int(gridDim.x);

    struct Item {
        int tm, tn, batch_local, split;
    };
    auto item_of = [&](int w) {
        Item it;
        tile_coordinates(w, items, args.tiles_m, args.tiles_n, args.splits, it.batch_local, it.split, it.tm, it.tn);
        return it;
    };
    auto k_begin_of = [&](const Item& it) { return int64_t(it.split) * args.k_per_split; };
    auto k_end_of = [&](const Item& it) { return min(args.k, k_begin_of(it) + args.k_per_split); };
    int w = int(blockIdx.x);
    if (w >= items) return;

    Engine e;
    // Whole tiles only: the loaders' offsets are the same for every item.
    marks[1][wave] = 0;
    e.init(stage_a, stage_b, marks[0], tid, args.lda, args.ldb, 0, T::BM, 0, T::BN);
    // The next step to load: its item's tile origins, k and K end. Past the
    // workgroup's last item every load is out of range (k at the K end).
    int ld_w = w;
    const float* ld_a;
    const float* ld_b;
    int64_t ld_k, ld_end;
    auto open_item = [&](int v) __attribute__((always_inline)) {
        const Item it = item_of(v);
        const int64_t batch = args.batch_base + it.batch_local;
        const int64_t m0 = int64_t(it.tm) * T::BM, n0 = int64_t(it.tn) * T::BN;
        ld_a = args.a + batch * args.stride_a + (A_K ? m0 * args.lda : m0);
        ld_b = args.b + batch * args.stride_b + (B_K ? n0 * args.ldb : n0);
        ld_k = k_begin_of(it);
        ld_end = k_end_of(it);
    };
    open_item(w);
    auto load_next = [&](auto set) __attribute__((always_inline)) {
        constexpr int Q = decltype(set)::value;
        e.la[Q].load(ld_a, args.lda, 0, T::BM, ld_k, ld_end, tid);
        e.lb[Q].load(ld_b, args.ldb, 0, T::BN, ld_k, ld_end, tid);
        if (ld_k < ld_end) ld_k += T::BK;
        if (ld_k >= ld_end && ld_w + stride < items) {
            ld_w += stride;
            open_item(ld_w);
        }
    };
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    load_next(I0{});
    load_next(I1{});
    e.template stage_set<0>();
    load_next(I0{});
    split_barrier();
    for (int turn = 0;; turn ^= 1) {
        const Item cur = item_of(w);
        const int64_t k_begin = k_begin_of(cur), k_end = k_end_of(cur);
        const int steps = int((k_end - k_begin + T::BK - 1) / T::BK);  // even (checked on the host)
        e.clear();
        for (int s = 0; s < steps; s += 2) {
            e.template step<1, true>([] {},
                                     [&] {
                                         // Every wave is done with the item before: its words are the next one's.
                                         if (s == 0) marks[turn ^ 1][wave] = 0;
                                         load_next(I1{});
                                     });
            e.template step<0, true>([&] { e.mark = marks[s + 2 >= steps ? turn ^ 1 : turn] + wave; },
                                     [&] { load_next(I0{}); });
        }
        const int64_t batch = args.batch_base + cur.batch_local;
        const int64_t m0 = int64_t(cur.tm) * T::BM, n0 = int64_t(cur.tn) * T::BN;
        if (marked<T>(marks[turn]) || not_finite<T>(e.acc))
            recompute_f32<T, A_K, B_K>(args, args.a + batch * args.stride_a, args.b + batch * args.stride_b, m0, n0,
                                       k_begin, k_end, wave_m, wave_n, lane, e.acc);
        const bool partial = args.splits > 1;
        float* out = partial ? args.ws + ((cur.batch_local * int64_t(args.splits) + cur.split) * args.m) * args.n
                             : args.c + batch * args.stride_c;
        write_tile<T, true, Engine::PAIR_M, Engine::PAIR_N, 0, true>(args, e.acc, out, m0, n0, wave_m, wave_n, lane,
                                                                     partial);
        w += stride;
        if (w >= items) break;
    }
}

// The fp32 product with the right operand's column sums over K (Linear's
// weight and bias gradients in one pass).
template <class T, bool A_K>
__global__ __launch_bounds__(T::THREADS)
__attribute__((amdgpu_waves_per_eu(split_waves_per_eu<T>(), split_waves_per_eu<T>())))
void gemm_f32_colsum_kernel(Args args) {
    split_tile<T, A_K, false, kLoadVector, true>(args);
}

// Adds the split partial sums of each output in split order, then applies
// the reference's combine.
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const float* __restrict__ ws, float* c, int64_t m,
                                                            int64_t n, int64_t batches, int splits,
                                                            int64_t stride_c, float scale, int accumulate,
                                                            const float* __restrict__ bias) {
    const int64_t per_matrix = m * n;
    const int64_t total = per_matrix * batches;
    for (int64_t idx = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; idx < total;
         idx += int64_t(gridDim.x) * blockDim.x) {
#pragma clang fp contract(off)
        const int64_t bat = idx / per_matrix;
        const int64_t e = idx % per_matrix;
        const float* src = ws + bat * splits * per_matrix + e;
        float sum = 0.f;
#pragma unroll 8
        for (int s = 0; s < splits; ++s) sum = sum + src[s * per_matrix];
        write_output(c + bat * stride_c + e, sum, scale, accumulate != 0, bias, e % n);
    }
}

// The same for 16-byte-aligned outputs with M*N a multiple of 4: four
// consecutive outputs per thread, 8 splits' 16-byte loads in flight
// (non-temporal: each partial is read once), and the output read (when
// accumulating) and written 16 bytes at a time; each element's combine is
// write_output's, rounded as it rounds.
__global__ __launch_bounds__(256) void splitk_reduce4_kernel(const f32x4* __restrict__ ws, float* c,
                                                             int64_t per_matrix, int64_t n, int64_t batches,
                                                             int splits, int64_t stride_c, float scale,
                                                             int accumulate, const float* __restrict__ bias) {
    const int64_t per_matrix4 = per_matrix / 4;
    const int64_t total = per_matrix4 * batches;
    for (int64_t idx = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; idx < total;
         idx += int64_t(gridDim.x) * blockDim.x) {
#pragma clang fp contract(off)
        const int64_t bat = idx / per_matrix4;
        const int64_t e4 = idx % per_matrix4;
        const f32x4* src = ws + bat * splits * per_matrix4 + e4;
        f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
        for (int s = 0; s < splits; ++s) sum = sum + __builtin_nontemporal_load(src + s * per_matrix4);
        f32x4* dst = reinterpret_cast<f32x4*>(c + bat * stride_c + 4 * e4);
        const f32x4 prior = accumulate ? *dst : f32x4{0.f, 0.f, 0.f, 0.f};
        f32x4 out;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float scaled = scale * sum[j];
            float value = accumulate ? prior[j] + scaled : scaled;
            if (bias != nullptr) value = value + bias[(4 * e4 + j) % n];
            out[j] = value;
        }
        *dst = out;
    }
}

// The split-K model's view of a tile: workgroups per CU, and the rate one CU
// sustains on it.
template <class T>
SplitCost split_cost() {
    SplitCost cost;
    cost.workgroups_per_cu = split_waves_per_eu<T>();
    return cost;
}

template <class T>
Plan f32_plan(const Problem& p, const Env& env) {
    return plan_for<T>(p, env, split_cost<T>());
}

// Products whose 128x128 plan (split K included) has fewer workgroups than
// the device has CUs take 64x64 tiles (four waves of 32x32, four workgroups
// per CU): the 7.1M model's products and the reference's published shapes
// (2048 x 768 x 256: 96 tiles of 128 x 128 on 256 CUs). Measured, 64x64 against
// 128x128: NN 2048 x 768 x 256 12.8 against 17.0 us, 2048 x 1024 x 256 12.7
// against 17.3, 2048 x 256 x 1024 19.0 against 23.6, TN 256 x 1024 x 2048 19.8
// against 23.0; the 42.9M and 111.5M models, whose plans fill the CUs, keep
// 128 x 128.
// Products whose 128x128 plan leaves CU slots empty (under two workgroups
// per CU) with under 24 K-steps per workgroup take 64x64 tiles as well: four
// 64x64 workgroups per CU fill the device without splitting a short K. The line
// was drawn with the fp32 matrix instruction, whose K-steps were 2.7 times as
// long, and holds for some of these only: NN and NT 4096 x 768 x 768 (one GPU's
// share of the 111.5M set over 8) 39.1 and 36.9 us against 43.1 and 42.5, but
// TN 768 x 768 x 4096 50.7 against 39.6 and NN 8192 x 512 x 512 34.4 against
// 30.4, where 128x128 tiles are the better ones now. Longer slices keep
// 128x128 (the 111.5M model's 768 x 768 x 32768 weight gradient, 74 K-steps a
// workgroup: 205 us against 318 on 64x64).
constexpr int64_t kSmallTileMaxK = 768;

// Whether 16-byte loads serve both operands of `p` on tile T.
template <class T>
bool vector_loads(const Problem& p) {
    return buffers_ok<T>(p);
}

// Unaligned operands follow the same rule from kUnalignedSmallMinK inner
// elements on; with fewer, a tile is two K-steps and its edges.
constexpr int64_t kUnalignedSmallMinK = 128;

template <class F>
auto with_f32_tile(const Problem& p, const Env& env, F&& f) {
    if (p.n <= 64) return f(F32Narrow{});
    const Plan square = f32_plan<F32Square>(p, env);
    const int64_t workgroups = int64_t(square.tiles_m) * square.tiles_n * square.splits * p.batch;
    const int64_t cus = std::max(env.cu_count, 1);
    const bool short_slices = workgroups < 2 * cus && square.k_per_split < kSmallTileMaxK;
    const bool small = (workgroups < cus || short_slices) &&
                       (p.k >= kUnalignedSmallMinK || vector_loads<F32Square>(p));
    return small ? f(F32Small{}) : f(F32Square{});
}

// The grid of the persistent kernel for `p` (a multiple of the XCD count, so
// that a workgroup's items stay on its XCD), or 0 when the product takes the
// one-tile kernel: masked products, several launches, tiles with an odd
// number of K-steps, or under two items per workgroup slot.
template <class T>
int64_t persistent_grid(const Problem& p, const Env& env, const Plan& plan, const LaunchShape& shape) {
    if constexpr (T::BM != 128 || T::BN != 128) return 0;
    // Interior tiles that read nothing back: write_tile's one store path.
    if (p.mask != SN_MASK_NONE || shape.batches_per_launch < p.batch || p.k <= kStreamingMaxK ||
        p.m % T::BM != 0 || p.n % T::BN != 0 || (plan.splits == 1 && p.accumulate))
        return 0;
    const int64_t items = int64_t(plan.tiles_m) * plan.tiles_n * plan.splits * p.batch;
    const int64_t slots = int64_t(std::max(env.cu_count, 1)) * split_waves_per_eu<T>() / kXcds * kXcds;
    if (slots < kXcds || items < 2 * slots || items > 0x7FFFFFFF) return 0;
    const int64_t steps = (plan.k_per_split + T::BK - 1) / T::BK;
    const int64_t last_steps = (p.k - int64_t(plan.splits - 1) * plan.k_per_split + T::BK - 1) / T::BK;
    if (steps % 2 != 0 || last_steps % 2 != 0 || last_steps < 2) return 0;
    return slots;
}

template <class T>
hipError_t launch_persistent(const Problem& p, const Env& env, const Plan& plan, int64_t grid, hipStream_t stream) {
    Args args = make_args<T>(p, env, plan);
    args.persistent_items = int32_t(int64_t(plan.tiles_m) * plan.tiles_n * plan.splits * p.batch);
    const dim3 blocks{unsigned(grid)}, threads(T::THREADS);
    if (p.a_k_contiguous && p.b_k_contiguous)
        hipLaunchKernelGGL((gemm_f32_persistent_kernel<T, true, true>), blocks, threads, 0, stream, args);
    else if (p.a_k_contiguous)
        hipLaunchKernelGGL((gemm_f32_persistent_kernel<T, true, false>), blocks, threads, 0, stream, args);
    else if (p.b_k_contiguous)
        hipLaunchKernelGGL((gemm_f32_persistent_kernel<T, false, true>), blocks, threads, 0, stream, args);
    else
        hipLaunchKernelGGL((gemm_f32_persistent_kernel<T, false, false>), blocks, threads, 0, stream, args);
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) return err;
    if (plan.splits > 1) return launch_splitk_reduce(p, env, plan.splits, stream);
    return hipSuccess;
}

// Each K slice also leaves N partial column sums after the product's M x N
// partials: the split count is chosen as if the workspace were M / (M + 1)
// of its size, so that both fit.
template <class T>
Plan column_sums_plan(const Problem& p, const Env& env) {
    Env e = env;
    e.workspace_bytes = env.workspace_bytes / size_t(p.m + 1) * size_t(p.m);
    return f32_plan<T>(p, e);
}

}  // namespace

hipError_t launch_splitk_reduce(const Problem& p, const Env& env, int splits, hipStream_t stream) {
    const int64_t total = p.m * p.n * p.batch;
    if ((p.m * p.n) % 4 == 0 && p.stride_c % 4 == 0 && aligned16(p.c)) {
        const int64_t grid = std::min<int64_t>((total / 4 + 255) / 256, int64_t(env.cu_count) * 16);
        hipLaunchKernelGGL(splitk_reduce4_kernel, dim3(unsigned(grid)), dim3(256), 0, stream,
                           reinterpret_cast<const f32x4*>(env.workspace), p.c, p.m * p.n, p.n, p.batch, splits,
                           p.stride_c, p.scale, p.accumulate ? 1 : 0, p.bias);
        return hipGetLastError();
    }
    const int64_t grid = std::min<int64_t>((total + 255) / 256, int64_t(env.cu_count) * 16);
    hipLaunchKernelGGL(splitk_reduce_kernel, dim3(unsigned(grid)), dim3(256), 0, stream, env.workspace, p.c, p.m,
                       p.n, p.batch, splits, p.stride_c, p.scale, p.accumulate ? 1 : 0, p.bias);
    return hipGetLastError();
}

bool f32_column_sums_applies(const Problem& p, const Env& env) {
    return p.batch == 1 && p.m > 0 && p.k > 0 && p.mask == SN_MASK_NONE && !p.b_k_contiguous && p.bias == nullptr &&
           with_f32_tile(p, env, [&](auto t) { return vector_loads<decltype(t)>(p); });
}

LaunchShape describe_f32_column_sums(const Problem& p, const Env& env) {
    return with_f32_tile(p, env, [&](auto t) {
        using T = decltype(t);
        const Plan plan = column_sums_plan<T>(p, env);
        LaunchShape s = tiled_shape<T>(p, plan, SN_PATH_F32_DIRECT);
        if (plan.splits > 1) s.workspace_bytes += size_t(plan.splits) * size_t(p.n) * sizeof(float);
        return s;
    });
}

hipError_t launch_gemm_f32_column_sums(const Problem& p, const Env& env, hipStream_t stream) {
    return with_f32_tile(p, env, [&](auto t) {
        using T = decltype(t);
        const Plan plan = column_sums_plan<T>(p, env);
        const Args args = make_args<T>(p, env, plan);
        const dim3 grid(unsigned(int64_t(plan.tiles_m) * plan.tiles_n * plan.splits)), block(T::THREADS);
        if (p.a_k_contiguous) hipLaunchKernelGGL((gemm_f32_colsum_kernel<T, true>), grid, block, 0, stream, args);
        else hipLaunchKernelGGL((gemm_f32_colsum_kernel<T, false>), grid, block, 0, stream, args);
        hipError_t err = hipGetLastError();
        if (err != hipSuccess || plan.splits == 1) return err;
        err = launch_splitk_reduce(p, env, plan.splits, stream);
        if (err != hipSuccess) return err;
        return launch_column_sums_finish(env.workspace + int64_t(plan.splits) * p.m * p.n, plan.splits, p.n,
                                         p.column_sums, stream);
    });
}

}  // namespace gemm

LaunchShape describe_gemm_f32(const Problem& p, const Env& env) {
    return gemm::with_f32_tile(p, env, [&](auto t) {
        using T = decltype(t);
        const gemm::Plan plan = gemm::f32_plan<T>(p, env);
        if (!gemm::vector_loads<T>(p)) return gemm::tiled_shape<T>(p, plan, SN_PATH_F32_REGISTER);
        LaunchShape s = gemm::tiled_shape<T>(p, plan, SN_PATH_F32_DIRECT);
        s.persistent_grid = gemm::persistent_grid<T>(p, env, plan, s);
        if (s.persistent_grid > 0) s.path = SN_PATH_F32_PERSISTENT;
        return s;
    });
}

hipError_t launch_gemm_f32(const Problem& p, const Env& env, hipStream_t stream) {
    return gemm::with_f32_tile(p, env, [&](auto t) {
        using T = decltype(t);
        const gemm::Plan plan = gemm::f32_plan<T>(p, env);
        if (!gemm::vector_loads<T>(p)) return gemm::launch_f32_unaligned<T>(p, env, plan, stream);
        const int64_t grid =
            gemm::persistent_grid<T>(p, env, plan, gemm::tiled_shape<T>(p, plan, SN_PATH_F32_DIRECT));
        if constexpr (T::BM == 128 && T::BN == 128)
            if (grid > 0) return gemm::launch_persistent<T>(p, env, plan, grid, stream);
        return gemm::launch_f32_tiles<T, gemm::kLoadVector>(p, env, plan, stream, gemm::streams_output(p, plan));
    });
}

size_t gemm_workspace_bytes(const Problem& p, bool bf16, const Env& env) {
    return bf16 ? describe_gemm_bf16(p, env).workspace_bytes : describe_gemm_f32(p, env).workspace_bytes;
}

}  // namespace sn
