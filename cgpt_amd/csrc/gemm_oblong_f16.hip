// Oblong tiles, f16 storage.
#include "gemm_large_kernel.hpp"

namespace cgptx {
int gemm_oblong_f16(const LargeCall& call, hipStream_t stream) { return launch_oblong<f16_t>(call, stream); }
}  // namespace cgptx
