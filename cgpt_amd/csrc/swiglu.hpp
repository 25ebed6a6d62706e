// SwiGLU on whole 16-byte vectors: bodies shared by the operators' kernels (elementwise.hip) and by launches that carry it beside
// other work (rmsnorm.hip).
#pragma once

#include "common.hpp"

namespace cgptx {
namespace {

constexpr int kSwigluThreads = 256;

__device__ __forceinline__ float sigmoid_f32(float x) { return 1.0f / (1.0f + __expf(-x)); }

// Packed input [rows, 2*hidden] = [gate | up] (src/ops/swiglu.cu:152-170): out[r, c] =
// silu(gate_up[r, c]) * gate_up[r, hidden + c]. Workgroup `block` of `blocks`.
template <typename T>
__device__ __forceinline__ void swiglu_forward_packed_vectors(T* __restrict__ out, const T* __restrict__ gate_up, std::size_t rows,
                                                              std::size_t hidden, int block, int blocks) {
    constexpr int VEC = kVec128<T>;
    const std::size_t row_vectors = hidden / VEC;
    const std::size_t vectors = rows * row_vectors;
    for (std::size_t v = static_cast<std::size_t>(block) * kSwigluThreads + threadIdx.x; v < vectors;
         v += static_cast<std::size_t>(blocks) * kSwigluThreads) {
        const std::size_t row = v / row_vectors, col = (v - row * row_vectors) * VEC;
        const T* in = gate_up + row * 2 * hidden + col;
        const vec_t<float, VEC> g = vec_to_f32<T, VEC>(load_vec<T, VEC>(in));
        const vec_t<float, VEC> u = vec_to_f32<T, VEC>(load_vec<T, VEC>(in + hidden));
        vec_t<float, VEC> r;
#pragma unroll
        for (int e = 0; e < VEC; ++e) r[e] = g[e] * sigmoid_f32(g[e]) * u[e];
        store_vec<T, VEC>(out + row * hidden + col, vec_from_f32<T, VEC>(r));
    }
}

// Packed: row-major [rows, 2*hidden] with gate in the first half of each row.
// Separate layout is the special case handled by passing distinct pointers.
// A workgroup takes tiles of kSwigluUnroll x 256 consecutive vectors: a thread requests its kSwigluUnroll
// vectors of all three inputs (and of the old gradients when accumulating) before it computes anything, so that
// twelve 128-bit loads per lane are in flight, and the position inside a packed row comes from 32-bit
// arithmetic (a shift when a row holds a power-of-two number of vectors).
// Below two such tiles per compute unit a tile is 256 vectors: what a small call costs is the serial work of a thread
// (300 x 704 in f16: 7.0 -> 4.2 us, 256 x 2048 in fp32: 6.4 -> 5.1).
template <typename T, bool AccGate, bool AccUp, int kSwigluUnroll>
__device__ __forceinline__ void swiglu_backward_vectors(
    T* grad_gate, T* grad_up, const T* __restrict__ grad_output, const T* __restrict__ gate,
    const T* __restrict__ up, std::size_t vectors, unsigned int row_vectors, int row_shift,
    std::size_t packed_row_stride, int block, int blocks) {
    // packed_row_stride == 0: flat separate tensors. Otherwise gate/up/grad_* are
    // views into [rows, 2*hidden] and index = row * stride + col. row_shift >= 0: row_vectors == 1 << row_shift.
    constexpr int VEC = kVec128<T>;
    constexpr std::size_t kTile = static_cast<std::size_t>(kSwigluThreads) * kSwigluUnroll;
    for (std::size_t base = static_cast<std::size_t>(block) * kTile; base < vectors;
         base += static_cast<std::size_t>(blocks) * kTile) {
        vec_t<T, VEC> dy_raw[kSwigluUnroll], g_raw[kSwigluUnroll], u_raw[kSwigluUnroll], og_raw[kSwigluUnroll],
            ou_raw[kSwigluUnroll];
        std::size_t index[kSwigluUnroll];
        bool live[kSwigluUnroll];
#pragma unroll
        for (int k = 0; k < kSwigluUnroll; ++k) {
            const std::size_t v = base + static_cast<std::size_t>(k) * kSwigluThreads + threadIdx.x;
            live[k] = v < vectors;
            index[k] = v * VEC;
            if (packed_row_stride != 0) {
                std::size_t row;
                if (row_shift >= 0) row = v >> row_shift;
                else if (vectors <= 0xFFFFFFFFull) row = static_cast<unsigned int>(v) / row_vectors;
                else row = v / row_vectors;
                index[k] = row * packed_row_stride + (v - row * row_vectors) * VEC;
            }
            if (live[k]) {
                dy_raw[k] = load_vec<T, VEC>(grad_output + v * VEC);
                g_raw[k] = load_vec<T, VEC>(gate + index[k]);
                u_raw[k] = load_vec<T, VEC>(up + index[k]);
                if constexpr (AccGate) og_raw[k] = load_vec<T, VEC>(grad_gate + index[k]);
                if constexpr (AccUp) ou_raw[k] = load_vec<T, VEC>(grad_up + index[k]);
            }
        }
#pragma unroll
        for (int k = 0; k < kSwigluUnroll; ++k) {
            if (!live[k]) continue;
            const vec_t<float, VEC> dy = vec_to_f32<T, VEC>(dy_raw[k]);
            const vec_t<float, VEC> g = vec_to_f32<T, VEC>(g_raw[k]);
            const vec_t<float, VEC> u = vec_to_f32<T, VEC>(u_raw[k]);
            vec_t<float, VEC> dg, du;
#pragma unroll
            for (int e = 0; e < VEC; ++e) {
                const float s = sigmoid_f32(g[e]);
                dg[e] = dy[e] * u[e] * (s * (1.0f + g[e] * (1.0f - s)));
                du[e] = dy[e] * (g[e] * s);
            }
            if constexpr (AccGate) dg += vec_to_f32<T, VEC>(og_raw[k]);
            if constexpr (AccUp) du += vec_to_f32<T, VEC>(ou_raw[k]);
            store_vec<T, VEC>(grad_gate + index[k], vec_from_f32<T, VEC>(dg));
            store_vec<T, VEC>(grad_up + index[k], vec_from_f32<T, VEC>(du));
        }
    }
}

}  // namespace
}  // namespace cgptx
