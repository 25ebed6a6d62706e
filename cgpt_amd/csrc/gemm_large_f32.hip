// Persistent contraction kernels, fp32 storage.
#include "gemm_large_kernel.hpp"

namespace cgptx {
int gemm_large_f32(const LargeCall& call, hipStream_t stream) { return launch_large<float>(call, stream); }
}  // namespace cgptx
