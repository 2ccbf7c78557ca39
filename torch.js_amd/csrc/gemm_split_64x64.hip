// The split-product GEMM kernels of the 64 x 64 tile.
#include "gemm_split.h"

namespace tjh {
template void launch_split<3>(const GemmArgs&, dim3, int, int, bool);
}  // namespace tjh
