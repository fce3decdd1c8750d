// The launches between two fused kernels with 16-bit population storage.
#include "front_launch.hpp"

namespace lbdem {
template void launch_front<__half>(const FsArgs<__half>&, const HydroArgs&, const Consts&, const NbrArgs&, const ForceArgs&, int,
                               hipStream_t);
}
