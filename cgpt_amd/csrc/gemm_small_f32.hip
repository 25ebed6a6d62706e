// Small contractions, f32 storage.
#include "gemm_small_kernel.hpp"

namespace cgptx {
int gemm_small_f32(const SmallCall& call, hipStream_t stream) { return launch_small<float>(call, stream); }
}  // namespace cgptx
