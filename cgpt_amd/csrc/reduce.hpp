// Column reductions shared by the norm and linear kernels.
#pragma once

#include "common.hpp"

namespace cgptx {

constexpr int kReduceThreads = 256;
constexpr int kReduceWaves = kReduceThreads / kWave;

// Sums partial[P, H] over P in a fixed order and stores (or adds) in T; `group` = which kColumns columns. The partial sums
// have just been written by the whole chip, so every load is a trip to memory: what counts is how many are in flight. A
// workgroup of 1024 threads takes 32 columns (16 of narrow matrices, so that more workgroups share them), a thread eight
// parts at a time; up to a few thousand parts, what the chip holds of the kernels that leave them, one launch does: 1024 x
// 1024 4.7 us, 1792 x 128 5.7, where two launches (sums over sixteen and more parts, sums of those) took 9.4 and 9.3.
constexpr int kFinishThreads = 1024;
constexpr int finish_columns(int hidden) { return hidden <= 256 ? 16 : 32; }

template <typename T, int COLUMNS>
__device__ __forceinline__ void column_partial_reduce_body(T* __restrict__ out, const float* __restrict__ partial,
                                                           int parts, int hidden, int accumulate, int group) {
    constexpr int kWaves16 = kFinishThreads / kWave, kSlices = kFinishThreads / COLUMNS;
    __shared__ float stage[kWaves16][COLUMNS];
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const int slice = threadIdx.x / COLUMNS;
    const int col = group * COLUMNS + threadIdx.x % COLUMNS;
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = 0.0f;
    if (col < hidden) {
        const float* from = partial + col;
        int p = slice;
        for (; p + 7 * kSlices < parts; p += 8 * kSlices) {
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] += from[static_cast<std::size_t>(p + u * kSlices) * hidden];
        }
#pragma unroll
        for (int u = 0; u < 7; ++u)
            if (p + u * kSlices < parts) v[u] += from[static_cast<std::size_t>(p + u * kSlices) * hidden];
    }
    float total = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
#pragma unroll
    for (int offset = COLUMNS; offset < kWave; offset <<= 1) total += __shfl_xor(total, offset, kWave);
    if (lane < COLUMNS) stage[wave][lane] = total;
    __syncthreads();
    if (threadIdx.x < COLUMNS && col < hidden) {
        float sum = 0.0f;
#pragma unroll
        for (int w = 0; w < kWaves16; ++w) sum += stage[w][threadIdx.x];
        if (accumulate) sum += to_f32(out[col]);
        out[col] = from_f32<T>(sum);
    }
}
template <typename T, int COLUMNS>
__global__ __launch_bounds__(kFinishThreads) void column_partial_reduce_kernel(
    T* __restrict__ out, const float* __restrict__ partial, int parts, int hidden, int accumulate) {
    column_partial_reduce_body<T, COLUMNS>(out, partial, parts, hidden, accumulate, static_cast<int>(blockIdx.x));
}
template <typename T>
void launch_column_partial_reduce(T* out, const float* partial, int parts, int hidden, int accumulate, hipStream_t stream) {
    const int columns = finish_columns(hidden);
    auto kernel = columns == 16 ? column_partial_reduce_kernel<T, 16> : column_partial_reduce_kernel<T, 32>;
    hipLaunchKernelGGL(kernel, dim3((hidden + columns - 1) / columns), dim3(kFinishThreads), 0, stream, out, partial, parts, hidden,
                       accumulate);
}

// The same over a table of reductions (blockIdx.y picks the entry): the same additions in the same order for every entry,
// whatever else is in the table.
template <typename T>
__device__ __forceinline__ void column_partial_reduce_entry(const ColumnReduceEntry& e, int group) {
    if (finish_columns(e.hidden) == 16) column_partial_reduce_body<T, 16>(static_cast<T*>(e.out), e.partial, e.parts, e.hidden, 0, group);
    else column_partial_reduce_body<T, 32>(static_cast<T*>(e.out), e.partial, e.parts, e.hidden, 0, group);
}
static __global__ __launch_bounds__(kFinishThreads) void column_partial_reduce_table_kernel(
    const ColumnReduceEntry* __restrict__ table) {
    const ColumnReduceEntry e = table[blockIdx.y];
    const int group = static_cast<int>(blockIdx.x);
    if (group * finish_columns(e.hidden) >= e.hidden) return;
    switch (e.dtype) {
        case CGPTX_F16: column_partial_reduce_entry<f16_t>(e, group); break;
        case CGPTX_BF16: column_partial_reduce_entry<bf16_t>(e, group); break;
        default: column_partial_reduce_entry<float>(e, group); break;
    }
}

// partial[blockIdx.y, col] = Σ over this block's row slice of in[row, col] (fp32).
template <typename T>
__global__ __launch_bounds__(kReduceThreads) void column_sum_partial_kernel(float* __restrict__ partial,
                                                                           const T* __restrict__ in, long rows,
                                                                           int cols, long rows_per_slice) {
    __shared__ float stage[kReduceWaves][kWave];
    const int lane = threadIdx.x & (kWave - 1);
    const int slice = threadIdx.x / kWave;
    const int col = blockIdx.x * kWave + lane;
    const long row_begin = blockIdx.y * rows_per_slice;
    const long row_end = row_begin + rows_per_slice < rows ? row_begin + rows_per_slice : rows;
    float v = 0.0f;
    if (col < cols) {
        for (long row = row_begin + slice; row < row_end; row += kReduceWaves) v += to_f32(in[row * cols + col]);
    }
    stage[slice][lane] = v;
    __syncthreads();
    if (slice == 0 && col < cols) {
        float total = 0.0f;
#pragma unroll
        for (int s = 0; s < kReduceWaves; ++s) total += stage[s][lane];
        partial[static_cast<long>(blockIdx.y) * cols + col] = total;
    }
}

}  // namespace cgptx
