// The fused kernel with 64-bit population storage.
#include "fused.hpp"

namespace lbdem {
template void launch_fused<double>(Box&, const Consts&, const PartLB*, const ObjLB*, DevScalars*, bool, hipStream_t,
                               hipEvent_t, hipEvent_t);
}
