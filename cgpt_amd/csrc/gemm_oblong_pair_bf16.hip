// Pairs of gradients on oblong tiles, bf16 storage.
#include "gemm_large_kernel.hpp"

namespace cgptx {
int gemm_oblong_pair_bf16(const PairArgs& pair, hipStream_t stream) { return launch_oblong_pair<bf16_t>(pair, stream); }
}  // namespace cgptx
