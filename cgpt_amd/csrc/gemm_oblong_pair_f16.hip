// Pairs of gradients on oblong tiles, f16 storage.
#include "gemm_large_kernel.hpp"

namespace cgptx {
int gemm_oblong_pair_f16(const PairArgs& pair, hipStream_t stream) { return launch_oblong_pair<f16_t>(pair, stream); }
}  // namespace cgptx
