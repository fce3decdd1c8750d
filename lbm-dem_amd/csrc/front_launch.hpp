// launch_front (front.hpp), instantiated once per storage type.
#pragma once
#include "front.hpp"

namespace lbdem {

template <typename S>
void launch_front(const FsArgs<S>& a, const HydroArgs& h, const Consts& k, const NbrArgs& n, const ForceArgs& f, int L,
                  hipStream_t s) {
    const int bs = FS_THREADS;
    if (const int g = h.blocks + a.blocks + n.pBlocks; g > 0) {
        if (L == 1) launch<&k_front1<S, 1>, FS_THREADS, 1>(g, bs, s, a, h, k, n);
        else launch<&k_front1<S, 0>, FS_THREADS, 1>(g, bs, s, a, h, k, n);
    }
    if (const int g = n.scanBlocks + a.blocks; g > 0) launch<&k_front2<S>, FS_THREADS, 1>(g, bs, s, a, n);
    if (const int g = a.blocks + n.pBlocks; g > 0) launch<&k_front3<S>, FS_THREADS, 1>(g, bs, s, a, n);
    if (const int g = a.blocks + n.buildBlocks; g > 0) {
        if (L == 1) launch<&k_front4<S, 1>, FS_THREADS, 1>(g, bs, s, a, k, n);
        else launch<&k_front4<S, 0>, FS_THREADS, 1>(g, bs, s, a, k, n);
    }
    if (const int g = a.blocks + n.slotBlocks; g > 0) launch<&k_front5<S>, FS_THREADS, 1>(g, bs, s, a, n);
    const RedistArgs r{a.type, a.list2, a.filled, a.newIf, a.count2, a.marker, a.changed, a.cap, a.changedCap, a.blocks, a.sc};
    if (r.blocks + f.blocks > 0) launch_front6(r, a.mass, f, s);
}

}  // namespace lbdem
