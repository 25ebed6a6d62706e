// Column reductions shared by the norm and linear kernels.
#pragma once

#include "cross_entropy.hpp"

namespace cgptx {

constexpr int kReduceThreads = 256;
constexpr int kReduceWaves = kReduceThreads / kWave;

// Sums partial[P, H] over P and stores (or adds) in T; `group` = which COLUMNS columns. The order of additions is fixed by P, H and
// the chip, not by how the work is dealt out: P is cut into finish_slices() slices, in a slice every eighth part adds up by
// itself and the eight sums meet as (((0 + 4) + (1 + 5)) + (2 + 6)) + (3 + 7); the slices' sums (with one slice the parts) add up in
// four strands, every fourth each, of four running sums as far as whole groups of sixteen go, and the strands one after the other.
// A norm's weight gradient, and with it a trained step, keeps its bits while that stands.
// The partial sums have just been written by the whole chip, so every load is a trip to memory: what counts is how many are in
// flight. A workgroup of 1024 threads takes 32 columns (16 of narrow matrices, so that more workgroups share them), a wavefront
// a slice at a time (two of 16 columns), a lane eight loads; the slices' sums stay in LDS. The reductions of a step of 32768 tokens
// and two blocks of 768 columns take 9.3 us; two launches, slices and then their sums, took 12.6, one whose threads add every
// 32nd or 64th part, whatever order that is, 8.7.
constexpr int kFinishThreads = 1024;
constexpr int kFolded = 4096;  // slices' sums that a workgroup keeps: at most 256 slices of 16 columns, 128 of 32
constexpr int finish_columns(int hidden) { return hidden <= 256 ? 16 : 32; }
__device__ __host__ __forceinline__ int finish_slices(int parts, int hidden, int units) {
    const int slices = min(min(2 * units / ((hidden + kWave - 1) / kWave), parts / 16), kFolded / finish_columns(hidden));
    return max(slices, 1);
}

template <typename T, int COLUMNS>
__device__ __forceinline__ void column_partial_reduce_body(T* __restrict__ out, const float* __restrict__ partial,
                                                           int parts, int hidden, int accumulate, int group, int units,
                                                           float* folded, float* stage) {
    constexpr int kWaves16 = kFinishThreads / kWave;
    constexpr int kStrands = 4;                          // wavefronts that shared a slice, or the slices, of 64 columns
    constexpr int kOwn = kStrands * COLUMNS / kWave;     // strands of a lane
    constexpr int kAtOnce = 2 / kOwn;                    // slices of a wavefront
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const int column = lane % COLUMNS, sub = lane / COLUMNS;
    const int col = group * COLUMNS + column;
    const int slices = finish_slices(parts, hidden, units);
    if (slices > 1) {
        const float* from = partial + min(col, hidden - 1);
        const int chunk = (parts + slices - 1) / slices;
        for (int i0 = wave; i0 < slices; i0 += kAtOnce * kWaves16) {
            float sum[kAtOnce][kOwn][2];
#pragma unroll
            for (int s = 0; s < kAtOnce; ++s)
#pragma unroll
                for (int j = 0; j < kOwn; ++j) sum[s][j][0] = sum[s][j][1] = 0.0f;
            for (int ahead = 0; ahead < chunk; ahead += 16) {
                float v[kAtOnce][2][kOwn][2];
                bool live[kAtOnce][2][kOwn][2];
#pragma unroll
                for (int s = 0; s < kAtOnce; ++s)
#pragma unroll
                    for (int t = 0; t < 2; ++t)
#pragma unroll
                        for (int j = 0; j < kOwn; ++j)
#pragma unroll
                            for (int u = 0; u < 2; ++u) {
                                const int within = ahead + 8 * t + sub * kOwn + j + 4 * u;
                                const int p = (i0 + s * kWaves16) * chunk + within;
                                live[s][t][j][u] = within < chunk && p < parts;
                                v[s][t][j][u] = from[static_cast<std::size_t>(live[s][t][j][u] ? p : 0) * hidden];
                            }
#pragma unroll
                for (int s = 0; s < kAtOnce; ++s)
#pragma unroll
                    for (int t = 0; t < 2; ++t)
#pragma unroll
                        for (int j = 0; j < kOwn; ++j)
#pragma unroll
                            for (int u = 0; u < 2; ++u) sum[s][j][u] += live[s][t][j][u] ? v[s][t][j][u] : 0.0f;
            }
#pragma unroll
            for (int s = 0; s < kAtOnce; ++s) {
                float total = 0.0f;
#pragma unroll
                for (int w = 0; w < kStrands; ++w)
                    total += __shfl(sum[s][w % kOwn][0] + sum[s][w % kOwn][1], (w / kOwn) * COLUMNS + column, kWave);
                if (sub == 0 && i0 + s * kWaves16 < slices) folded[(i0 + s * kWaves16) * COLUMNS + column] = total;
            }
        }
        __syncthreads();
    }
    const int strand = threadIdx.x / COLUMNS;
    if (strand < kStrands && group * COLUMNS + static_cast<int>(threadIdx.x) % COLUMNS < hidden) {
        const int c = threadIdx.x % COLUMNS;
        auto add = [&](const float* from, std::size_t pitch, int count) __attribute__((always_inline)) {
            float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
            int p = strand;
            for (; p + 3 * kStrands < count; p += 4 * kStrands) {
#pragma unroll
                for (int u = 0; u < 4; ++u) v[u] += from[(p + u * kStrands) * pitch];
            }
            for (; p < count; p += kStrands) v[0] += from[p * pitch];
            return (v[0] + v[1]) + (v[2] + v[3]);
        };
        if (slices > 1) stage[strand * COLUMNS + c] = add(folded + c, COLUMNS, slices);
        else stage[strand * COLUMNS + c] = add(partial + group * COLUMNS + c, hidden, parts);
    }
    __syncthreads();
    if (threadIdx.x < COLUMNS && col < hidden) {
        float sum = 0.0f;
#pragma unroll
        for (int w = 0; w < kStrands; ++w) sum += stage[w * COLUMNS + threadIdx.x];
        if (accumulate) sum += to_f32(out[col]);
        out[col] = from_f32<T>(sum);
    }
}
template <typename T, int COLUMNS>
__global__ __launch_bounds__(kFinishThreads) void column_partial_reduce_kernel(
    T* __restrict__ out, const float* __restrict__ partial, int parts, int hidden, int accumulate, int units) {
    __shared__ float folded[kFolded], stage[4 * COLUMNS];
    column_partial_reduce_body<T, COLUMNS>(out, partial, parts, hidden, accumulate, static_cast<int>(blockIdx.x), units, folded, stage);
}
template <typename T>
void launch_column_partial_reduce(T* out, const float* partial, int parts, int hidden, int accumulate, hipStream_t stream) {
    const int columns = finish_columns(hidden);
    auto kernel = columns == 16 ? column_partial_reduce_kernel<T, 16> : column_partial_reduce_kernel<T, 32>;
    hipLaunchKernelGGL(kernel, dim3((hidden + columns - 1) / columns), dim3(kFinishThreads), 0, stream, out, partial, parts, hidden,
                       accumulate, compute_units());
}

// The same over a table of reductions (blockIdx.y picks the entry): the same additions in the same order for every entry,
// whatever else is in the table.
template <typename T>
__device__ __forceinline__ void column_partial_reduce_entry(const ColumnReduceEntry& e, int group, int units, float* folded, float* stage) {
    if (finish_columns(e.hidden) == 16) column_partial_reduce_body<T, 16>(static_cast<T*>(e.out), e.partial, e.parts, e.hidden, 0, group, units, folded, stage);
    else column_partial_reduce_body<T, 32>(static_cast<T*>(e.out), e.partial, e.parts, e.hidden, 0, group, units, folded, stage);
}
static __global__ __launch_bounds__(kFinishThreads) void column_partial_reduce_table_kernel(
    const ColumnReduceEntry* __restrict__ table, int entries, int units, MeanEntry mean) {
    __shared__ __align__(8) float folded[kFolded];
    __shared__ float stage[4 * 32];
    static_assert(sizeof(folded) >= kMeanSums * sizeof(double), "the mean's sums fit");
    if (static_cast<int>(blockIdx.y) == entries) {  // a launch of its own would take a step of 300 tokens 4 us
        if (blockIdx.x == 0)
            mean_of_rows<kFinishThreads>(mean.loss, [&](unsigned int i) { return mean.row_losses[i]; }, mean.rows,
                                         1.0f / static_cast<float>(mean.rows), reinterpret_cast<double*>(folded));
        return;
    }
    const ColumnReduceEntry e = table[blockIdx.y];
    const int group = static_cast<int>(blockIdx.x);
    if (group * finish_columns(e.hidden) >= e.hidden) return;
    switch (e.dtype) {
        case CGPTX_F16: column_partial_reduce_entry<f16_t>(e, group, units, folded, stage); break;
        case CGPTX_BF16: column_partial_reduce_entry<bf16_t>(e, group, units, folded, stage); break;
        default: column_partial_reduce_entry<float>(e, group, units, folded, stage); break;
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
