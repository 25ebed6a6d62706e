// Dense softmax cross-entropy (loss + logits gradient) for gfx950.
//
// Semantics: include/ops/cross_entropy.h:25-42; arithmetic of
// src/ops/cpu/backward/cross_entropy_backward_cpu.cpp:122-148:
//   loss = mean_r [ y_r < V ] (log Σ_j e^{z_rj} − z_{r,y_r}),
//   grad_rj = (softmax(z_r)_j − [j = y_r]) · scale / rows   (stored in the logits dtype).
//
// One block per row. Rows of up to 16384 128-bit vectors (131072 16-bit logits, 65536 fp32 ones) are
// loaded once into registers, reduced to (max, Σexp) and turned into the gradient from the registers:
// one read and one write of the logits, wherever a row starts. Longer rows stream: pass 1 keeps an online
// (max, Σexp) pair per thread, pass 2 re-reads the row through the caches. Per-row losses go to
// scratch and one block adds them in a fixed order, where the reference uses a float atomicAdd
// (src/ops/cross_entropy.cu:134-245).
#include "cross_entropy.hpp"

#include <cmath>
#include <limits>

namespace cgptx {
namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / kWave;

struct MaxSum {
    float m, s;
};

__device__ __forceinline__ MaxSum combine(MaxSum a, MaxSum b) {
    const float m = fmaxf(a.m, b.m);
    if (m == -INFINITY) return {m, 0.0f};
    return {m, a.s * __expf(a.m - m) + b.s * __expf(b.m - m)};
}

template <int WAVES = kWaves>
__device__ __forceinline__ MaxSum block_combine(MaxSum v, MaxSum* stage) {
#pragma unroll
    for (int offset = kWave / 2; offset > 0; offset >>= 1) {
        MaxSum other{__shfl_xor(v.m, offset, kWave), __shfl_xor(v.s, offset, kWave)};
        v = combine(v, other);
    }
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    if (lane == 0) stage[wave] = v;
    __syncthreads();
    MaxSum total = stage[0];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) total = combine(total, stage[w]);
    return total;
}

// The mean that the last workgroup of a row launch takes, in place of a launch that begins when all of this one has ended: its first wavefront, which
// looks at the counter behind the gradient's stores. bf16 [16, 900] 7.5 -> 4.6 us a call, [128, 2000] 7.5 -> 5.5. In a graph of calls, where a launch
// takes no host time, 5.5 -> 4.7, at 64 rows 5.6 -> 5.1, at 128 5.5 -> 5.7 (with both of a lane's losses read at once; one after the other, the tree
// of sums on all threads and the counter awaited before the gradient 6.1), [128, 50257] 13.7 -> 12.0. The workgroups meet on one counter, which takes one
// of them every 12 ns: [4096, 1000] would take 52 us for 12, fp32 [512, 50257] 24 for 22.
struct MeanArgs {
    float* loss;
    unsigned int* counter;  // null: no mean
    float inv_rows;
};
constexpr std::size_t kMostMeanRows = kFewMeanRows;

// Streaming kernel for rows that are too long to hold: each row is split into the elements before its first
// 16-byte boundary (a vocabulary that is not a multiple of the vector width moves every row's start), whole 128-bit
// vectors, and the rest. vector_ok: logits and gradient rows have the same alignment phase (or there is no gradient).
// ld_*: row strides; gradient columns past the vocabulary are cleared.
template <typename T, bool WithGradient>
__global__ __launch_bounds__(kThreads) void cross_entropy_row_kernel(float* __restrict__ row_loss,
                                                                    T* gradient,  // may alias logits (in place)
                                                                    const T* logits,
                                                                    const std::uint32_t* __restrict__ targets,
                                                                    unsigned int vocab, std::size_t ld_logits,
                                                                    std::size_t ld_gradient, float factor,
                                                                    bool vector_ok) {
    constexpr int VEC = kVec128<T>;
    __shared__ MaxSum stage[kWaves];
    const T* row = logits + blockIdx.x * ld_logits;
    const unsigned int to_boundary =
        static_cast<unsigned int>(((16u - (reinterpret_cast<std::uintptr_t>(row) & 15u)) & 15u) / sizeof(T));
    const unsigned int head = vector_ok ? (to_boundary < vocab ? to_boundary : vocab) : vocab;
    const unsigned int vectors = (vocab - head) / VEC;
    const unsigned int body_end = head + vectors * VEC;
    const unsigned int edge = head + (vocab - body_end);  // elements handled one by one
    const T* body = row + head;
    const std::uint32_t target = targets[blockIdx.x];
    // Read before the barrier below: in-place use overwrites the row in pass 2.
    const float target_logit = (threadIdx.x == 0 && target < vocab) ? to_f32(row[target]) : 0.0f;

    MaxSum acc{-INFINITY, 0.0f};
    for (unsigned int v = threadIdx.x; v < vectors; v += kThreads) {
        const vec_t<float, VEC> x = vec_to_f32<T, VEC>(load_vec<T, VEC>(body + v * VEC));
        float vmax = x[0];
#pragma unroll
        for (int e = 1; e < VEC; ++e) vmax = fmaxf(vmax, x[e]);
        if (vmax > acc.m) {
            acc.s *= __expf(acc.m - vmax);
            acc.m = vmax;
        }
        if (acc.m != -INFINITY) {
#pragma unroll
            for (int e = 0; e < VEC; ++e) acc.s += __expf(x[e] - acc.m);
        }
    }
    for (unsigned int k = threadIdx.x; k < edge; k += kThreads) {
        const unsigned int i = k < head ? k : body_end + (k - head);
        const float x = to_f32(row[i]);
        if (x > acc.m) {
            acc.s *= __expf(acc.m - x);
            acc.m = x;
        }
        if (acc.m != -INFINITY) acc.s += __expf(x - acc.m);
    }
    const MaxSum total = block_combine(acc, stage);
    if (threadIdx.x == 0) {
        float loss = 0.0f;
        if (target < vocab) loss = __logf(total.s) + total.m - target_logit;
        row_loss[blockIdx.x] = loss;
    }
    if constexpr (WithGradient) {
        const float inv = 1.0f / total.s;
        T* out = gradient + blockIdx.x * ld_gradient;
        for (std::size_t i = vocab + threadIdx.x; i < ld_gradient; i += kThreads) out[i] = from_f32<T>(0.0f);
        for (unsigned int v = threadIdx.x; v < vectors; v += kThreads) {
            const vec_t<float, VEC> x = vec_to_f32<T, VEC>(load_vec<T, VEC>(body + v * VEC));
            vec_t<float, VEC> g;
#pragma unroll
            for (int e = 0; e < VEC; ++e) {
                float value = __expf(x[e] - total.m) * inv;
                if (head + v * VEC + e == target) value -= 1.0f;
                g[e] = value * factor;
            }
            store_vec<T, VEC>(out + head + v * VEC, vec_from_f32<T, VEC>(g));
        }
        for (unsigned int k = threadIdx.x; k < edge; k += kThreads) {
            const unsigned int i = k < head ? k : body_end + (k - head);
            float value = __expf(to_f32(row[i]) - total.m) * inv;
            if (i == target) value -= 1.0f;
            out[i] = from_f32<T>(value * factor);
        }
    }
}

// Rows of up to THREADS * SLOTS 128-bit vectors stay in registers between the two passes: every load of the row is
// in flight at once, and the memory system sees exactly one read and one write of the row (the streaming kernel's
// second pass finds the row in L2 only while the rows in flight on an XCD fit there, which 8 rows of 64 KB per CU do
// not). The vectors start at the row's first element, wherever that lies: an access of 16 bytes per lane that is off
// its boundary touches one cache line more per wavefront, which beats streaming the row twice (fp32 logits
// [512, 50257]: 53 -> 31 us). The up to VEC - 1 elements behind the last vector are held one per thread.
template <typename T>
using anywhere_t __attribute__((aligned(alignof(T)))) = vec_t<T, kVec128<T>>;
template <bool ONCE, typename T>
__device__ __forceinline__ vec_t<T, kVec128<T>> load_anywhere(const T* p) {
    if constexpr (ONCE) return __builtin_nontemporal_load(reinterpret_cast<const anywhere_t<T>*>(p));
    else return *reinterpret_cast<const anywhere_t<T>*>(p);
}
template <bool ONCE, typename T>
__device__ __forceinline__ void store_anywhere(T* p, vec_t<T, kVec128<T>> v) {
    if constexpr (ONCE) __builtin_nontemporal_store(v, reinterpret_cast<anywhere_t<T>*>(p));
    else *reinterpret_cast<anywhere_t<T>*>(p) = v;
}

// ONCE: logits and gradient are accessed as what is used once, see launch_resident.
template <typename T, int THREADS, int SLOTS, bool WithGradient, bool ONCE>
__global__ __launch_bounds__(THREADS) void cross_entropy_row_resident_kernel(
    float* __restrict__ row_loss, T* gradient /* may alias logits */, const T* logits,
    const std::uint32_t* __restrict__ targets, unsigned int vocab, std::size_t ld_logits, std::size_t ld_gradient,
    float factor, MeanArgs mean) {
    constexpr int VEC = kVec128<T>;
    constexpr int WAVES = THREADS / kWave;
    __shared__ MaxSum stage[WAVES];
    const T* row = logits + blockIdx.x * ld_logits;
    const unsigned int vectors = vocab / VEC, tail = vectors * VEC + threadIdx.x;  // tail: this thread's element behind them
    const std::uint32_t target = targets[blockIdx.x];
    // Read before the barrier in block_combine: in-place use overwrites the row after it.
    const float target_logit = (threadIdx.x == 0 && target < vocab) ? to_f32(row[target]) : 0.0f;

    vec_t<T, VEC> held[SLOTS];
#pragma unroll
    for (int s = 0; s < SLOTS; ++s) {
        const unsigned int v = s * THREADS + threadIdx.x;
        if (v < vectors) held[s] = load_anywhere<ONCE, T>(row + v * VEC);
    }
    const float held_tail = tail < vocab ? to_f32(row[tail]) : -INFINITY;
    MaxSum acc{held_tail, 0.0f};
#pragma unroll
    for (int s = 0; s < SLOTS; ++s) {
        if (s * THREADS + threadIdx.x < vectors) {
            const vec_t<float, VEC> x = vec_to_f32<T, VEC>(held[s]);
#pragma unroll
            for (int e = 0; e < VEC; ++e) acc.m = fmaxf(acc.m, x[e]);
        }
    }
    if (acc.m != -INFINITY) {
#pragma unroll
        for (int s = 0; s < SLOTS; ++s) {
            if (s * THREADS + threadIdx.x < vectors) {
                const vec_t<float, VEC> x = vec_to_f32<T, VEC>(held[s]);
#pragma unroll
                for (int e = 0; e < VEC; ++e) acc.s += __expf(x[e] - acc.m);
            }
        }
        if (tail < vocab) acc.s += __expf(held_tail - acc.m);
    }
    const MaxSum total = block_combine<WAVES>(acc, stage);
    unsigned int counted = 0;
    if (threadIdx.x == 0) {
        float loss = 0.0f;
        if (target < vocab) loss = __logf(total.s) + total.m - target_logit;
        if (mean.counter != nullptr)  // before the gradient's stores, which it would wait for
            counted = leave_and_count(row_loss + blockIdx.x, loss, mean.counter, fold_share(static_cast<int>(blockIdx.x), static_cast<int>(gridDim.x)));
        else row_loss[blockIdx.x] = loss;
    }
    if constexpr (WithGradient) {
        const float inv = 1.0f / total.s;
        const unsigned int target_vector = target / VEC;
        T* out = gradient + blockIdx.x * ld_gradient;
#pragma unroll
        for (int s = 0; s < SLOTS; ++s) {
            const unsigned int v = s * THREADS + threadIdx.x;
            if (v < vectors) {
                const vec_t<float, VEC> x = vec_to_f32<T, VEC>(held[s]);
                vec_t<float, VEC> g;
#pragma unroll
                for (int e = 0; e < VEC; ++e) g[e] = __expf(x[e] - total.m) * inv;
                // The target's vector alone looks for its element: compared one by one, the elements' columns cost a
                // quarter of this pass's vector instructions, which a chunk that fits the last-level cache is bound by (bf16
                // [2048, 50257]: 112 -> 101 us).
                if (v == target_vector) {
#pragma unroll
                    for (int e = 0; e < VEC; ++e)
                        if (v * VEC + e == target) g[e] -= 1.0f;
                }
#pragma unroll
                for (int e = 0; e < VEC; ++e) g[e] *= factor;
                store_anywhere<ONCE, T>(out + v * VEC, vec_from_f32<T, VEC>(g));
            }
        }
        if (tail < vocab) {
            float value = __expf(held_tail - total.m) * inv;
            if (tail == target) value -= 1.0f;
            out[tail] = from_f32<T>(value * factor);
        }
        for (std::size_t i = vocab + threadIdx.x; i < ld_gradient; i += THREADS) out[i] = from_f32<T>(0.0f);
    }
    if (mean.counter == nullptr || threadIdx.x >= kWave) return;
    counted = static_cast<unsigned int>(__builtin_amdgcn_readfirstlane(static_cast<int>(counted)));
    if (counted + fold_share(static_cast<int>(blockIdx.x), static_cast<int>(gridDim.x)) != 0u) return;
    mean_of_few_rows(mean.loss, [row_loss](unsigned int i) { return read_left(row_loss + i); }, gridDim.x, mean.inv_rows);
}

template <typename T, int THREADS, int SLOTS>
void launch_resident(float* row_loss, T* gradient, const T* logits, const std::uint32_t* targets, unsigned int rows,
                     unsigned int vocab, std::size_t ld_logits, std::size_t ld_gradient, float factor, const MeanArgs& mean, hipStream_t stream) {
    // More logits and gradients than the memory-side cache holds until somebody reads them again: bf16 [16384, 32000] in place 367 -> 342 us,
    // fp32 [2048, 32000] 107 -> 98, f16 [4096, 20011] (328 MB) 78 -> 72; fp32 [700, 50257] (281 MB), of which a part is still found there, 60 and 64.
    const std::size_t bytes = static_cast<std::size_t>(rows) * vocab * sizeof(T) * (gradient != nullptr && gradient != logits ? 2 : 1);
    const bool once = bytes > kMemoryCacheBytes / 8 * 9;
    auto kernel = gradient == nullptr ? (once ? cross_entropy_row_resident_kernel<T, THREADS, SLOTS, false, true>
                                              : cross_entropy_row_resident_kernel<T, THREADS, SLOTS, false, false>)
                                      : (once ? cross_entropy_row_resident_kernel<T, THREADS, SLOTS, true, true>
                                              : cross_entropy_row_resident_kernel<T, THREADS, SLOTS, true, false>);
    hipLaunchKernelGGL(kernel, dim3(rows), dim3(THREADS), 0, stream, row_loss, gradient, logits, targets, vocab, ld_logits,
                       ld_gradient, factor, mean);
}

}  // namespace

// Shared with the cut-cross-entropy path: loss[0] = (Σ row_loss) / rows, fixed order.
__global__ __launch_bounds__(1024) void mean_reduce_kernel(float* __restrict__ loss,
                                                          const float* __restrict__ row_loss, unsigned int rows,
                                                          float inv_rows) {
    __shared__ double stage[kMeanSums];
    mean_of_rows<1024>(loss, [row_loss](unsigned int i) { return row_loss[i]; }, rows, inv_rows, stage);
}

// Per-row pass: row_loss[r] and (optionally) the gradient, factor = gradient_scale / total_rows.
int cross_entropy_rows(float* row_loss, void* gradient, std::size_t ld_gradient, const void* logits, std::size_t ld_logits,
                       const std::uint32_t* targets, std::size_t rows, std::size_t vocab, float factor, int dtype,
                       hipStream_t stream, float* loss, bool* mean_taken) {
    MeanArgs mean{loss, nullptr, 1.0f / static_cast<float>(rows)};
    if (loss != nullptr && rows <= kMostMeanRows) mean.counter = tickets(stream);
    const auto r = static_cast<unsigned int>(rows), v = static_cast<unsigned int>(vocab);
    return dispatch_dtype(dtype, [&]<typename T>() -> int {
        auto* g = static_cast<T*>(gradient);
        auto* z = static_cast<const T*>(logits);
        // A thread holds up to 16 vectors; 1024 threads where 512 would not reach.
        const unsigned int vectors = v / kVec128<T>;
        if (vectors <= 2u * 512) launch_resident<T, 512, 2>(row_loss, g, z, targets, r, v, ld_logits, ld_gradient, factor, mean, stream);
        else if (vectors <= 8u * 512) launch_resident<T, 512, 8>(row_loss, g, z, targets, r, v, ld_logits, ld_gradient, factor, mean, stream);
        else if (vectors <= 16u * 512) launch_resident<T, 512, 16>(row_loss, g, z, targets, r, v, ld_logits, ld_gradient, factor, mean, stream);
        else if (vectors <= kMostHeldVectors) launch_resident<T, 1024, 16>(row_loss, g, z, targets, r, v, ld_logits, ld_gradient, factor, mean, stream);
        else {
            mean.counter = nullptr;
            // The streaming kernel finds each row's own 16-byte boundary; logits and gradient rows must share it.
            const bool same_phase = g == nullptr || (((reinterpret_cast<std::uintptr_t>(z) ^ reinterpret_cast<std::uintptr_t>(g)) & 15u) == 0 &&
                                                     cross_entropy_in_vectors(vocab, ld_logits, ld_gradient, dtype));
            auto kernel = g != nullptr ? cross_entropy_row_kernel<T, true> : cross_entropy_row_kernel<T, false>;
            hipLaunchKernelGGL(kernel, dim3(r), dim3(kThreads), 0, stream, row_loss, g, z, targets, v, ld_logits, ld_gradient,
                               factor, same_phase);
        }
        CGPTX_LAUNCH_CHECK();
        if (mean_taken != nullptr) *mean_taken = mean.counter != nullptr;
        return CGPTX_OK;
    });
}

std::size_t cross_entropy_gradient_pitch(std::size_t rows, std::size_t hidden, std::size_t vocab, int dtype) {
    const std::size_t pitch = linear_backward_pitch(rows, hidden, vocab, dtype);
    return cross_entropy_in_vectors(vocab, vocab, pitch, dtype) ? pitch : vocab;
}

int mean_reduce(float* loss, const float* row_loss, std::size_t rows, hipStream_t stream) {
    hipLaunchKernelGGL(mean_reduce_kernel, dim3(1), dim3(1024), 0, stream, loss, row_loss,
                       static_cast<unsigned int>(rows), 1.0f / static_cast<float>(rows));
    CGPTX_LAUNCH_CHECK();
    return CGPTX_OK;
}

namespace {

int run(float* loss, void* gradient, const void* logits, const std::uint32_t* targets, std::size_t rows,
        std::size_t vocab, float gradient_scale, int dtype, hipStream_t stream, bool with_gradient,
        const char* name) {
    if (!valid_dtype(dtype)) return fail(CGPTX_INVALID_ARGUMENT, std::string(name) + ": unsupported dtype");
    if (loss == nullptr || logits == nullptr || targets == nullptr || rows == 0 || vocab == 0 ||
        (with_gradient && gradient == nullptr))
        return fail(CGPTX_INVALID_ARGUMENT, std::string(name) + ": invalid tensors or targets");
    if (with_gradient && (!std::isfinite(gradient_scale) || gradient_scale <= 0.0f))
        return fail(CGPTX_INVALID_ARGUMENT, std::string(name) + ": gradient scale must be finite and positive");
    constexpr std::size_t i32max = std::numeric_limits<int>::max();
    if (rows > i32max || vocab > i32max) return fail(CGPTX_OVERFLOW, std::string(name) + ": dimension exceeds int range");
    void* mem = nullptr;
    if (int s = scratch(stream, rows * sizeof(float), &mem)) return s;
    auto* row_loss = static_cast<float*>(mem);
    const float factor = gradient_scale / static_cast<float>(rows);
    bool mean_taken = false;
    if (int s = cross_entropy_rows(row_loss, with_gradient ? gradient : nullptr, vocab, logits, vocab, targets, rows, vocab, factor,
                                   dtype, stream, loss, &mean_taken))
        return s;
    return mean_taken ? CGPTX_OK : mean_reduce(loss, row_loss, rows, stream);
}

}  // namespace
}  // namespace cgptx

extern "C" int cgptx_cross_entropy_forward_backward(float* loss, void* gradient, const void* logits,
                                                    const uint32_t* targets, size_t rows, size_t vocab,
                                                    float gradient_scale, int dtype, cgptx_stream stream) {
    return cgptx::run(loss, gradient, logits, targets, rows, vocab, gradient_scale, dtype,
                      static_cast<hipStream_t>(stream), true, "cross_entropy_forward_backward");
}

extern "C" int cgptx_cross_entropy_forward(float* loss, const void* logits, const uint32_t* targets, size_t rows,
                                           size_t vocab, int dtype, cgptx_stream stream) {
    return cgptx::run(loss, nullptr, logits, targets, rows, vocab, 1.0f, dtype, static_cast<hipStream_t>(stream),
                      false, "cross_entropy_forward");
}
