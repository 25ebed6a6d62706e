// Internal interface of the softmax cross-entropy row kernels (used by the dense and the cut path).
#pragma once

#include "common.hpp"

namespace cgptx {

// row_loss[r] = [y_r < V](logsumexp z_r − z_{r,y_r}); gradient (may be null, may be the logits' own memory) =
// (softmax − onehot)·factor. Rows are ld_logits and ld_gradient elements apart; gradient columns from vocab to
// ld_gradient are cleared. loss (may be null): where the mean over these rows goes, see mean_reduce.
int cross_entropy_rows(float* row_loss, void* gradient, std::size_t ld_gradient, const void* logits, std::size_t ld_logits,
                       const std::uint32_t* targets, std::size_t rows, std::size_t vocab, float factor, int dtype,
                       hipStream_t stream, float* loss = nullptr);

// loss[0] = (Σ row_loss) / rows, summed in a fixed order.
int mean_reduce(float* loss, const float* row_loss, std::size_t rows, hipStream_t stream);

}  // namespace cgptx
