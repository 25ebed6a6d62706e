// Small contractions, f16 storage.
#include "gemm_small_kernel.hpp"

namespace cgptx {
int gemm_small_f16(const SmallCall& call, hipStream_t stream) { return launch_small<f16_t>(call, stream); }
}  // namespace cgptx
