// Oblong tiles, bf16 storage.
#include "gemm_large_kernel.hpp"

namespace cgptx {
int gemm_oblong_bf16(const LargeCall& call, hipStream_t stream) { return launch_oblong<bf16_t>(call, stream); }
}  // namespace cgptx
