// The launches between two fused kernels with 32-bit population storage.
#include "front_launch.hpp"

namespace lbdem {
template void launch_front<float>(const FsArgs<float>&, const HydroArgs&, const Consts&, const NbrArgs&, const ForceArgs&, int,
                               hipStream_t);
}
