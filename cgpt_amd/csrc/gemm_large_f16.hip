// Persistent contraction kernels, f16 storage.
#include "gemm_large_kernel.hpp"

namespace cgptx {
int gemm_large_f16(const LargeCall& call, hipStream_t stream) { return launch_large<f16_t>(call, stream); }
int gemm_pair_f16(const PairArgs& pair, hipStream_t stream) { return launch_pair<f16_t>(pair, stream); }
}  // namespace cgptx
