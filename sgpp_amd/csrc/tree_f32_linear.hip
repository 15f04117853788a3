// Subspace-tree kernels: FP32, Linear.
#include "tree_kernels.hpp"

namespace sgpp_hip {
template TreeLaunch tree_launch<float, false>(int, int, bool);
}  // namespace sgpp_hip
