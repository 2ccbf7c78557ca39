// The split-product GEMM kernels of the 256 x 128 tile.
#include "gemm_split.h"

namespace tjh {
template void launch_split<0>(const GemmArgs&, dim3, int, int, bool);
}  // namespace tjh
