// linear_forward / linear_backward on top of the MFMA contraction kernels.
//
// Reference interfaces: include/ops/linear.h (Y = X·Wᵀ + b) and
// include/ops/backward/linear_backward.h:36-46 (dX = dY·W, dW = dYᵀ·X,
// db = Σ_rows dY), CPU arithmetic src/ops/cpu/backward/linear_backward_cpu.cpp:131-165.
#include "gemm.hpp"
#include "reduce.hpp"

#include <algorithm>
#include <limits>

namespace cgptx {
namespace {

int validate(const char* name, std::size_t rows, std::size_t in_features, std::size_t out_features, int dtype) {
    if (!valid_dtype(dtype)) return fail(CGPTX_INVALID_ARGUMENT, std::string(name) + ": unsupported dtype");
    if (rows == 0 || in_features == 0 || out_features == 0)
        return fail(CGPTX_INVALID_ARGUMENT, std::string(name) + ": empty shape");
    constexpr std::size_t i32max = std::numeric_limits<int>::max();
    if (rows > i32max || in_features > i32max || out_features > i32max)
        return fail(CGPTX_OVERFLOW, std::string(name) + ": dimension exceeds int range");
    return CGPTX_OK;
}

// An output gradient in rows of whole K tiles.
std::size_t padded(std::size_t out_features) { return (out_features + 31) / 32 * 32; }
// Whether both contractions of a backward pass then stream: whole chunks of input and weight, the streamed kernels' 32-bit offsets.
bool copies_stream(std::size_t rows, std::size_t in_features, std::size_t out_features, std::size_t elem) {
    constexpr std::size_t kSpan = (std::size_t{1} << 31) - (std::size_t{1} << 21);
    return in_features * elem % 16 == 0 && rows * (out_features + 32 + in_features) * elem < kSpan && out_features * in_features * elem < kSpan;
}

// The same with input and weight copied as well.
bool copies_reach(std::size_t rows, std::size_t in_features, std::size_t out_features, std::size_t elem) {
    constexpr std::size_t kSpan = (std::size_t{1} << 31) - (std::size_t{1} << 21);
    return rows * (out_features + in_features + 64) * elem < kSpan && out_features * (in_features + 32) * elem < kSpan;
}

}  // namespace

std::size_t linear_backward_pitch(std::size_t rows, std::size_t in_features, std::size_t out_features, int dtype) {
    const std::size_t elem = dtype_size(dtype);
    return out_features * elem % 16 != 0 && copies_stream(rows, in_features, out_features, elem) ? padded(out_features) : out_features;
}

}  // namespace cgptx

extern "C" int cgptx_linear_forward(void* output, const void* input, const void* weight, const void* bias,
                                    size_t rows, size_t in_features, size_t out_features, int dtype,
                                    cgptx_stream stream) {
    using namespace cgptx;
    if (int s = validate("linear_forward", rows, in_features, out_features, dtype)) return s;
    if (output == nullptr || input == nullptr || weight == nullptr)
        return fail(CGPTX_INVALID_ARGUMENT, "linear_forward: null tensor");
    GemmArgs g;
    g.a = input;
    g.b = weight;
    g.c = output;
    g.bias = bias;
    g.m = rows;
    g.n = out_features;
    g.k = in_features;
    g.lda = in_features;
    g.ldb = in_features;
    g.ldc = out_features;
    g.dtype = dtype;
    return gemm(g, static_cast<hipStream_t>(stream));
}

extern "C" int cgptx_linear_swiglu_forward(void* gate_up, void* activated, const void* input, const void* weight,
                                           size_t rows, size_t in_features, size_t hidden, int dtype,
                                           cgptx_stream stream_) {
    using namespace cgptx;
    if (hidden > std::numeric_limits<std::size_t>::max() / 2)
        return fail(CGPTX_OVERFLOW, "linear_swiglu_forward: dimension exceeds int range");
    if (int s = validate("linear_swiglu_forward", rows, in_features, 2 * hidden, dtype)) return s;
    if (gate_up == nullptr || activated == nullptr || input == nullptr || weight == nullptr)
        return fail(CGPTX_INVALID_ARGUMENT, "linear_swiglu_forward: null tensor");
    auto stream = static_cast<hipStream_t>(stream_);
    GemmArgs g;
    g.a = input;
    g.b = weight;
    g.c = gate_up;
    g.m = rows;
    g.n = 2 * hidden;
    g.k = in_features;
    g.lda = in_features;
    g.ldb = in_features;
    g.ldc = 2 * hidden;
    g.dtype = dtype;
    g.swiglu_out = activated;
    g.ld_swiglu = hidden;
    if (gemm_fuses_swiglu(g)) return gemm(g, stream);
    // Shapes the fused kernel does not take: the two operators one after the other (same bits).
    g.swiglu_out = nullptr;
    if (int s = gemm(g, stream)) return s;
    return cgptx_swiglu_forward_packed(activated, gate_up, rows, hidden, dtype, stream_);
}

extern "C" int cgptx_linear_swiglu_backward(void* grad_gate_up, void* grad_activated, const void* grad_output,
                                            const void* weight, const void* gate_up, size_t rows, size_t hidden,
                                            size_t out_features, int dtype, cgptx_stream stream_) {
    using namespace cgptx;
    if (hidden > std::numeric_limits<std::size_t>::max() / 2)
        return fail(CGPTX_OVERFLOW, "linear_swiglu_backward: dimension exceeds int range");
    if (int s = validate("linear_swiglu_backward", rows, 2 * hidden, out_features, dtype)) return s;
    if (grad_gate_up == nullptr || grad_activated == nullptr || grad_output == nullptr || weight == nullptr || gate_up == nullptr)
        return fail(CGPTX_INVALID_ARGUMENT, "linear_swiglu_backward: null tensor");
    auto stream = static_cast<hipStream_t>(stream_);
    GemmArgs g;  // d(activated)[rows, hidden] = dY[rows, out] · W[out, hidden]
    g.a = grad_output;
    g.b = weight;
    g.c = grad_gate_up;
    g.m = rows;
    g.n = hidden;
    g.k = out_features;
    g.lda = out_features;
    g.ldb = hidden;
    g.ldc = 2 * hidden;
    g.b_k_contiguous = false;
    g.dtype = dtype;
    g.swiglu_saved = gate_up;
    g.ld_swiglu = 2 * hidden;
    if (gemm_fuses_swiglu_gradient(g)) return gemm(g, stream);
    // Shapes the fused kernel does not take: the two operators one after the other (same bits).
    g.swiglu_saved = nullptr;
    g.c = grad_activated;
    g.ldc = hidden;
    if (int s = gemm(g, stream)) return s;
    return cgptx_swiglu_backward_packed(grad_gate_up, grad_activated, gate_up, rows, hidden, 0, dtype, stream_);
}

extern "C" int cgptx_linear_backward_weights_stacked(void* grad_weight, const void* grad_output, const void* input,
                                                     size_t rows, size_t in_features, size_t out_features,
                                                     size_t count, size_t grad_output_stride, size_t input_stride,
                                                     int dtype, cgptx_stream stream_) {
    using namespace cgptx;
    if (int s = validate("linear_backward_weights_stacked", rows, in_features, out_features, dtype)) return s;
    if (grad_weight == nullptr || grad_output == nullptr || input == nullptr)
        return fail(CGPTX_INVALID_ARGUMENT, "linear_backward_weights_stacked: null tensor");
    if (count == 0) return fail(CGPTX_INVALID_ARGUMENT, "linear_backward_weights_stacked: empty stack");
    if (count > static_cast<std::size_t>(std::numeric_limits<int>::max()) / out_features)
        return fail(CGPTX_OVERFLOW, "linear_backward_weights_stacked: dimension exceeds int range");
    auto stream = static_cast<hipStream_t>(stream_);
    GemmArgs g;  // rows j out .. (j + 1) out - 1 of dW = dY_jᵀ[out, rows] · X_j[rows, in]
    g.a = grad_output;
    g.b = input;
    g.c = grad_weight;
    g.m = count * out_features;
    g.n = in_features;
    g.k = rows;
    g.lda = out_features;
    g.ldb = in_features;
    g.ldc = in_features;
    g.a_k_contiguous = false;
    g.b_k_contiguous = false;
    g.dtype = dtype;
    g.batch_rows = out_features;
    g.a_batch_stride = grad_output_stride;
    g.b_batch_stride = input_stride;
    if (count > 1 && gemm_takes_batch(g) && is_aligned16(grad_output) && is_aligned16(input) && is_aligned16(grad_weight))
        return gemm(g, stream);
    // Shapes the stacked launch does not take: one weight gradient after the other.
    const std::size_t elem = dtype_size(dtype);
    for (std::size_t j = 0; j < count; ++j) {
        if (int s = cgptx_linear_backward(nullptr, static_cast<char*>(grad_weight) + j * out_features * in_features * elem,
                                          nullptr, static_cast<const char*>(grad_output) + j * grad_output_stride * elem,
                                          static_cast<const char*>(input) + j * input_stride * elem, nullptr, rows,
                                          in_features, out_features, 0, 0, 0, dtype, stream_))
            return s;
    }
    return CGPTX_OK;
}

extern "C" int cgptx_linear_backward(void* grad_input, void* grad_weight, void* grad_bias, const void* grad_output,
                                     const void* input, const void* weight, size_t rows, size_t in_features,
                                     size_t out_features, int accumulate_input, int accumulate_weight,
                                     int accumulate_bias, int dtype, cgptx_stream stream_) {
    return cgptx::linear_backward(grad_input, grad_weight, grad_bias, grad_output, input, weight, rows, in_features, out_features,
                                  accumulate_input, accumulate_weight, accumulate_bias, dtype, static_cast<hipStream_t>(stream_), nullptr);
}

int cgptx::linear_backward(void* grad_input, void* grad_weight, void* grad_bias, const void* grad_output, const void* input,
                           const void* weight, std::size_t rows, std::size_t in_features, std::size_t out_features,
                           int accumulate_input, int accumulate_weight, int accumulate_bias, int dtype, hipStream_t stream,
                           LinearParts* parts, bool large_pairs, std::size_t grad_output_pitch) {
    if (int s = validate("linear_backward", rows, in_features, out_features, dtype)) return s;
    if (grad_output == nullptr || (grad_input != nullptr && weight == nullptr) ||
        (grad_weight != nullptr && input == nullptr))
        return fail(CGPTX_INVALID_ARGUMENT, "linear_backward: null tensor");
    // An output gradient whose rows are not whole 16-byte chunks feeds both contractions from one padded copy (each would
    // make its own otherwise). So do weight and input of such rows: copied together, they leave the contractions free to share a launch, but for
    // pairs on large tiles whose weight gradient is cut along K: the scratch beside the copies holds no partial tiles for those, and their contractions go one
    // after the other (9000 x 2047 x 200 128 -> 122.6 us). Forward and backward, eager, six to nine launches before: bf16 16 x 1379 x 256 with bias 27 - 33 -> 17.5 us, 1000 x 1021 x 1024 with bias, added
    // to old gradients 48 -> 35, 5005 x 1023 x 2048 118 -> 99, fp32 200 x 1001 x 500 53 -> 35.
    const std::size_t elem = dtype_size(dtype);
    const void *dy = grad_output, *w = weight, *x = input;
    std::size_t in_pitch = in_features;
    std::size_t dy_pitch = grad_output_pitch != 0 ? grad_output_pitch : out_features;
    void* split_room = nullptr;
    std::size_t split_bytes = 0;
    auto input_gradient = [&]() {  // dX[rows, in] = dY[rows, out] · W[out, in]
        GemmArgs g;
        g.a = dy;
        g.b = w;
        g.c = grad_input;
        g.m = rows;
        g.n = in_features;
        g.k = dy_pitch;
        g.b_k = out_features;
        g.b_extent = in_pitch;
        g.lda = dy_pitch;
        g.ldb = in_pitch;
        g.ldc = in_features;
        g.b_k_contiguous = false;
        g.accumulate = accumulate_input != 0;
        g.dtype = dtype;
        g.no_split = split_room != nullptr;
        g.split_workspace = split_room;
        g.split_workspace_bytes = split_bytes;
        return g;
    };
    auto weight_gradient = [&]() {  // dW[out, in] = dYᵀ[out, rows] · X[rows, in]
        GemmArgs g;
        g.a = dy;
        g.b = x;
        g.b_extent = in_pitch;
        g.c = grad_weight;
        g.m = out_features;
        g.a_extent = dy_pitch;
        g.n = in_features;
        g.k = rows;
        g.lda = dy_pitch;
        g.ldb = in_pitch;
        g.ldc = in_features;
        g.a_k_contiguous = false;
        g.b_k_contiguous = false;
        g.accumulate = accumulate_weight != 0;
        g.dtype = dtype;
        g.no_split = split_room != nullptr;
        g.split_workspace = split_room;
        g.split_workspace_bytes = split_bytes;
        return g;
    };
    // Whether no result lies on what one of the contractions reads, nor on another result.
    const std::size_t dy_bytes = rows * std::max(out_features, grad_output_pitch) * elem, x_bytes = rows * in_features * elem, w_bytes = out_features * in_features * elem;
    const std::size_t bias_bytes = out_features * elem;
    auto apart = [](const void* a, std::size_t a_bytes, const void* b, std::size_t b_bytes) {
        const auto at = reinterpret_cast<std::uintptr_t>(a), other = reinterpret_cast<std::uintptr_t>(b);
        return a == nullptr || at >= other + b_bytes || other >= at + a_bytes;
    };
    auto all_apart = [&]() {
        return apart(grad_input, x_bytes, grad_output, dy_bytes) && apart(grad_input, x_bytes, input, x_bytes) &&
               apart(grad_weight, w_bytes, grad_output, dy_bytes) && apart(grad_weight, w_bytes, weight, w_bytes) &&
               apart(grad_bias, bias_bytes, grad_output, dy_bytes) && apart(grad_bias, bias_bytes, weight, w_bytes) &&
               apart(grad_bias, bias_bytes, input, x_bytes) && apart(grad_weight, w_bytes, grad_input, x_bytes) &&
               apart(grad_bias, bias_bytes, grad_input, x_bytes) && apart(grad_bias, bias_bytes, grad_weight, w_bytes);
    };
    const bool both = grad_output_pitch == 0 && grad_input != nullptr && grad_weight != nullptr;
    const bool pad_in = both && in_features * elem % 16 != 0 && copies_reach(rows, in_features, out_features, elem) && all_apart() &&
                        apart(grad_input, x_bytes, weight, w_bytes) && apart(grad_weight, w_bytes, input, x_bytes);
    const bool pad_out = pad_in ? out_features % (64 / elem) != 0 || !is_aligned16(grad_output)
                                : both && (out_features * elem % 16 != 0 || !is_aligned16(grad_output)) && is_aligned16(weight) &&
                                      is_aligned16(input) && copies_stream(rows, in_features, out_features, elem);
    if (pad_in || pad_out) {
        if (pad_out) dy_pitch = padded(out_features);
        if (pad_in) in_pitch = padded(in_features);
        auto bytes_of = [&](std::size_t copy_rows, std::size_t pitch) { return (copy_rows * pitch * elem + 255) & ~std::size_t{255}; };
        const std::size_t dy_copy = pad_out ? bytes_of(rows, dy_pitch) : 0, w_copy = pad_in ? bytes_of(out_features, in_pitch) : 0;
        const std::size_t copy_bytes = dy_copy + w_copy + (pad_in ? bytes_of(rows, in_pitch) : 0);
        split_bytes = std::max(gemm_split_bytes(input_gradient()), gemm_split_bytes(weight_gradient()));
        // fp32 sums in K slices keep them: 2000 x 65 x 67 in one launch, in one sum over 2000 rows, is 4.0e-7 off the sums in 64 bits, in slices 1.4e-7. In 16-bit
        // storage, whose rounding is five hundred times that (f16 2000 x 65 x 67 2.011e-4 off either way), such a sum may be one chain.
        const bool keeps_slices = pad_in && dtype == CGPTX_F32 && split_bytes != 0;
        split_bytes += 256;
        void* mem = nullptr;
        std::size_t held = 0;
        if (!keeps_slices)
            if (int s = scratch_up_to(stream, copy_bytes + split_bytes, &mem, &held)) return s;
        if (!keeps_slices && held >= copy_bytes) {
            char* const base = static_cast<char*>(mem);
            if (pad_out) {
                if (int s = pad_rows(base, grad_output, rows, out_features, out_features, dy_pitch, dtype, stream)) return s;
                dy = base;
            }
            if (pad_in) {
                if (int s = pad_rows_of_two(base + dy_copy, weight, out_features, base + dy_copy + w_copy, input, rows, in_features, in_pitch, dtype, stream))
                    return s;
                w = base + dy_copy;
                x = base + dy_copy + w_copy;
            }
            split_room = base + copy_bytes;
            split_bytes = std::min(split_bytes, held - copy_bytes);
        } else {
            dy_pitch = out_features;  // each contraction goes its own way
            in_pitch = in_features;
        }
    }
    if (grad_input != nullptr && grad_weight != nullptr) {
        // Small calls: both gradients, and the bias's, in one launch, whose parts run in no order. None may write what another
        // one reads, nor what another one writes: overlapping results hold what the last of the separate launches leaves.
        GemmArgs calls[2] = {input_gradient(), weight_gradient()};
        calls[1].a_sums = grad_bias;
        calls[1].a_sums_accumulate = accumulate_bias != 0;
        if (all_apart()) {
            if (const GemmGroup group = gemm_joins(calls, 2, stream, large_pairs); group.joined) {
                if (int s = gemm_joined(calls, 2, group, stream)) return s;
                return parts != nullptr ? parts->done(LinearParts::joined) : CGPTX_OK;
            }
        }
    }
    if (grad_input != nullptr) {
        if (int s = gemm(input_gradient(), stream)) return s;
        if (parts != nullptr)
            if (int s = parts->done(LinearParts::input)) return s;
    }
    if (grad_weight != nullptr) {
        if (int s = gemm(weight_gradient(), stream)) return s;
        if (parts != nullptr)
            if (int s = parts->done(LinearParts::weight)) return s;
    }
    if (grad_bias != nullptr && grad_output_pitch != 0 && grad_output_pitch != out_features)
        return fail(CGPTX_RUNTIME, "linear_backward: no bias gradient of an output gradient in padded rows");
    if (grad_bias != nullptr) {  // db[out] = Σ_rows dY
        const int cols = static_cast<int>(out_features);
        const int slices = rows < 256 ? 1 : (rows < 65536 ? 64 : 256);
        const long rows_per_slice = (static_cast<long>(rows) + slices - 1) / slices;
        void* mem = nullptr;
        if (int s = scratch(stream, static_cast<std::size_t>(slices) * out_features * sizeof(float), &mem)) return s;
        auto* partial = static_cast<float*>(mem);
        const int col_blocks = (cols + kWave - 1) / kWave;
        return dispatch_dtype(dtype, [&]<typename T>() -> int {
            hipLaunchKernelGGL((column_sum_partial_kernel<T>), dim3(col_blocks, slices), dim3(kReduceThreads), 0,
                               stream, partial, static_cast<const T*>(grad_output), static_cast<long>(rows), cols,
                               rows_per_slice);
            CGPTX_LAUNCH_CHECK();
            launch_column_partial_reduce<T>(static_cast<T*>(grad_bias), partial, slices, cols, accumulate_bias != 0 ? 1 : 0, stream);
            CGPTX_LAUNCH_CHECK();
            return CGPTX_OK;
        });
    }
    return CGPTX_OK;
}
