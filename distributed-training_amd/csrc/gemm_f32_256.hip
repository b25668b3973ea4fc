// float32 GEMM kernels on 256 x 128 block tiles.
#include "gemm_tiles.h"

namespace dtmi {

template void launch_layout<float, 256, 128>(const GemmArgs&, dim3, int, int, bool, bool, bool);

}  // namespace dtmi
