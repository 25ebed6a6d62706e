// Internal interface of the softmax cross-entropy row kernels (used by the dense and the cut path).
#pragma once

#include "common.hpp"

namespace cgptx {

// row_loss[r] = [y_r < V](logsumexp z_r − z_{r,y_r}); gradient (may be null, may be the logits' own memory) =
// (softmax − onehot)·factor. Rows are ld_logits and ld_gradient elements apart; gradient columns from vocab to
// ld_gradient are cleared. loss (may be null): where the mean over these rows goes if they are few (*mean_taken; see mean_reduce).
int cross_entropy_rows(float* row_loss, void* gradient, std::size_t ld_gradient, const void* logits, std::size_t ld_logits,
                       const std::uint32_t* targets, std::size_t rows, std::size_t vocab, float factor, int dtype,
                       hipStream_t stream, float* loss = nullptr, bool* mean_taken = nullptr);

// Rows of up to this many 16-byte vectors stay in registers between the row pass's two passes; longer ones are streamed twice.
constexpr std::size_t kMostHeldVectors = 16 * 1024;
// Whether the row pass accesses logits and gradient, both on 16 bytes and in rows of these lengths, by whole vectors: streamed rows only where
// a logits' row and its gradient's lie alike within their vectors (else by elements).
inline bool cross_entropy_in_vectors(std::size_t vocab, std::size_t ld_logits, std::size_t ld_gradient, int dtype) {
    const std::size_t vec = 16 / dtype_size(dtype);
    return vocab / vec <= kMostHeldVectors || (ld_logits - ld_gradient) % vec == 0;
}
// The row length of the gradient that a dense loss over logits in rows of `vocab` leaves for linear_backward: what that reads as it lies, but
// where rows are streamed that of the logits (linear_backward then copies it).
std::size_t cross_entropy_gradient_pitch(std::size_t rows, std::size_t hidden, std::size_t vocab, int dtype);

// loss[0] = (Σ row_loss) / rows, summed in a fixed order.
int mean_reduce(float* loss, const float* row_loss, std::size_t rows, hipStream_t stream);

// cgptx_cut_cross_entropy_forward_backward whose rows' losses are left in row_losses; the mean is the caller's to take.
int cut_cross_entropy(float* row_losses, void* input_gradient, void* classifier_gradient, const void* input, const void* classifier,
                      const std::uint32_t* targets, std::size_t rows, std::size_t hidden, std::size_t vocab, float gradient_scale,
                      int dtype, hipStream_t stream);

// (Σ row_loss) / rows by a workgroup of THREADS. 1024 partial sums of four running ones each: the order of additions is fixed by
// the rows alone, so the result is reproducible. read: how a row's loss is read.
constexpr int kMeanSums = 1024;  // what tree_sum_1024 adds up
template <int THREADS, typename Read>
__device__ __forceinline__ void mean_of_rows(float* __restrict__ loss, Read&& read, unsigned int rows, float inv_rows, double* stage) {
    for (unsigned int t = threadIdx.x; t < kMeanSums; t += THREADS) {
        double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
        unsigned int i = t;
        for (; i + 3 * kMeanSums < rows; i += 4 * kMeanSums) {
            s0 += static_cast<double>(read(i));
            s1 += static_cast<double>(read(i + kMeanSums));
            s2 += static_cast<double>(read(i + 2 * kMeanSums));
            s3 += static_cast<double>(read(i + 3 * kMeanSums));
        }
        for (; i < rows; i += kMeanSums) s0 += static_cast<double>(read(i));
        stage[t] = (s0 + s1) + (s2 + s3);
    }
    __syncthreads();
    if (threadIdx.x >= kWave) return;
    const double sum = tree_sum_1024(stage);
    if (threadIdx.x == 0) loss[0] = static_cast<float>(sum) * inv_rows;
}
// The same sum of at most 128 rows, by the first wavefront: the other partial sums, and so the first levels of their tree, are zeros.
constexpr unsigned int kFewMeanRows = 2 * kWave;
template <typename Read>
__device__ __forceinline__ void mean_of_few_rows(float* __restrict__ loss, Read&& read, unsigned int rows, float inv_rows) {
    const unsigned int lane = threadIdx.x, last = rows - 1;
    const float first = read(lane < last ? lane : last), second = read(lane + kWave < last ? lane + kWave : last);  // both on their way at once
    const double sum = tree_sum_64((lane < rows ? 0.0 + static_cast<double>(first) : 0.0) + (lane + kWave < rows ? 0.0 + static_cast<double>(second) : 0.0));
    if (threadIdx.x == 0) loss[0] = static_cast<float>(sum) * inv_rows;
}

}  // namespace cgptx
