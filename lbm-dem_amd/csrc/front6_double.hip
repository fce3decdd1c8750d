// Redistribution and forces (front.hpp) with double node masses.
#include "front.hpp"

namespace lbdem {

template <>
void launch_front6<double>(const RedistArgs& r, double* mass, const ForceArgs& f, hipStream_t s) {
    const int g = r.blocks + f.blocks, bs = FS_THREADS;
    const bool few = f.lanes == DEM_LANES_FEW;
    if (f.p.stress) {
        if (few) launch<&k_front6<double, true, DEM_LANES_FEW>, FS_THREADS, 1>(g, bs, s, r, mass, f);
        else launch<&k_front6<double, true, DEM_LANES_MANY>, FS_THREADS, 1>(g, bs, s, r, mass, f);
    } else {
        if (few) launch<&k_front6<double, false, DEM_LANES_FEW>, FS_THREADS, 1>(g, bs, s, r, mass, f);
        else launch<&k_front6<double, false, DEM_LANES_MANY>, FS_THREADS, 1>(g, bs, s, r, mass, f);
    }
}

}  // namespace lbdem
