// float64 GEMM kernels on 64 x 64 block tiles.
#include "gemm_tiles.h"

namespace dtmi {

template void launch_layout<double, 64, 64>(const GemmArgs&, dim3, int, int, bool, bool, bool);

}  // namespace dtmi
