// Subspace-tree kernels: FP64, ModLinear.
#include "tree_kernels.hpp"

namespace sgpp_hip {
template TreeLaunch tree_launch<double, true>(int, int, bool);
}  // namespace sgpp_hip
