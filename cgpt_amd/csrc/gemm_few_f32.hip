// Groups of up to kFewCalls small contractions, f32 storage.
#include "gemm_small_kernel.hpp"

namespace cgptx {
int gemm_small_f32(const SmallGroup<kFewCalls>& group, int blocks, bool deep, hipStream_t stream) { return launch_small_group<float>(group, blocks, deep, stream); }
}  // namespace cgptx
