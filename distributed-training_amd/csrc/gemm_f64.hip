// float64 GEMM kernels on 128 x 128 block tiles.
#include "gemm_tiles.h"

namespace dtmi {

template void launch_layout<double, 128, 128>(const GemmArgs&, dim3, int, int, bool, bool, bool);

}  // namespace dtmi
