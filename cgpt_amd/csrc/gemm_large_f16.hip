// Persistent contraction kernels, f16 storage.
#include "gemm_large_kernel.hpp"

namespace cgptx {
int gemm_large_f16(const LargeCall& call, hipStream_t stream) { return launch_large<f16_t>(call, stream); }
}  // namespace cgptx
