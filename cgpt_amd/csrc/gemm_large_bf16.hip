// Persistent contraction kernels, bf16 storage.
#include "gemm_large_kernel.hpp"

namespace cgptx {
int gemm_large_bf16(const LargeCall& call, hipStream_t stream) { return launch_large<bf16_t>(call, stream); }
int gemm_pair_bf16(const PairArgs& pair, hipStream_t stream) { return launch_pair<bf16_t>(pair, stream); }
}  // namespace cgptx
