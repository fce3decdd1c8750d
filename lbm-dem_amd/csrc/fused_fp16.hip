// The fused kernel with 16-bit population storage.
#include "fused.hpp"

namespace lbdem {
template void launch_fused<__half>(Box&, const Consts&, const PartLB*, const ObjLB*, DevScalars*, bool, hipStream_t,
                               hipEvent_t, hipEvent_t);
}
