// Subspace-tree kernels: FP32, ModLinear.
#include "tree_kernels.hpp"

namespace sgpp_hip {
template TreeLaunch tree_launch<float, true>(int, int, bool);
}  // namespace sgpp_hip
