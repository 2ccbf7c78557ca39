// The split-product GEMM kernels of the 128 x 64 tile.
#include "gemm_split.h"

namespace tjh {
template void launch_split<2>(const GemmArgs&, dim3, int, int, bool);
}  // namespace tjh
