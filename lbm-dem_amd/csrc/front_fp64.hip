// The launches between two fused kernels with 64-bit population storage.
#include "front_launch.hpp"

namespace lbdem {
template void launch_front<double>(const FsArgs<double>&, const HydroArgs&, const Consts&, const NbrArgs&, const ForceArgs&, int,
                               hipStream_t);
}
