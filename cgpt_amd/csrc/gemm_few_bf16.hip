// Groups of up to kFewCalls small contractions, bf16 storage.
#include "gemm_small_kernel.hpp"

namespace cgptx {
int gemm_small_bf16(const SmallGroup<kFewCalls>& group, int blocks, bool deep, hipStream_t stream) { return launch_small_group<bf16_t>(group, blocks, deep, stream); }
}  // namespace cgptx
