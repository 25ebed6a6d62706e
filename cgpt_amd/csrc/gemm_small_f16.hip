// Small contractions, f16 storage.
#include "gemm_small_kernel.hpp"

namespace cgptx {
int gemm_small_f16(const SmallCall& call, hipStream_t stream) { return launch_small<f16_t>(call, stream); }
int gemm_small_f16(const SmallGroup<kGroupCalls>& group, int blocks, bool deep, hipStream_t stream) { return launch_small_group<f16_t>(group, blocks, deep, stream); }
}  // namespace cgptx
