// Subspace-tree kernels: FP64, Linear.
#include "tree_kernels.hpp"

namespace sgpp_hip {
template TreeLaunch tree_launch<double, false>(int, int, bool);
}  // namespace sgpp_hip
