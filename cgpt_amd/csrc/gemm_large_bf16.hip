// Persistent contraction kernels, bf16 storage.
#include "gemm_large_kernel.hpp"

namespace cgptx {
int gemm_large_bf16(const LargeCall& call, hipStream_t stream) { return launch_large<bf16_t>(call, stream); }
}  // namespace cgptx
