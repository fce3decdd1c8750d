// DEM integration, object and wall totals and record packing (compiled without contraction so the
// arithmetic rounds like the reference's scalar code): integration and periodic wrap
// (DEM.cpp:2676-2836). The neighbour list and the forces are in dem.hpp, launched with the free
// surface's passes (front.hpp).
#include "dem.hpp"
#pragma clang fp contract(off)

namespace lbdem {

int dem_force_lanes(int nPart, bool inBatch) { return !inBatch && nPart <= DEM_FEW ? DEM_LANES_FEW : DEM_LANES_MANY; }
int dem_force_blocks(int nPart, bool inBatch) {
    return int((int64_t(nPart) * dem_force_lanes(nPart, inBatch) + 255) / 256);
}

// One block (the last block of the integration launch, which runs beside the particles' blocks:
// neither reads what the other writes): the sums of the impactor and wall columns over the force
// pass's blocks (in block order within four interleaved shares), then, on thread 0, objects:
// totals and integration (DEM.cpp:786-790, 2742-2758) and walls: totals (DEM.cpp:773-775).
constexpr int OBJ_THREADS = 256;
// the numbers of the blocks that wrote sums, in order, in LDS (RED_LIST of them at most: the callers' rounds)
__device__ inline int flagged_blocks(const int* flag, int n, int* list, int* sWave) {
    int base = 0;
    for (int b0 = 0; b0 < n; b0 += OBJ_THREADS) {
        const int b = b0 + int(threadIdx.x);
        const bool f = b < n && flag[b] != 0;
        const unsigned long long m = __ballot(f);
        const int wave = threadIdx.x / 64;
        if (__lane_id() == 0) sWave[wave] = __popcll(m);
        __syncthreads();
        int off = base, tot = 0;
        for (int w = 0; w < OBJ_THREADS / 64; ++w) {
            if (w < wave) off += sWave[w];
            tot += sWave[w];
        }
        if (f) list[off + __popcll(m & ((1ull << __lane_id()) - 1ull))] = b;
        base += tot;
        __syncthreads();
    }
    return base;
}
static_assert(DEM_RED_COLS <= 64 && OBJ_THREADS == 4 * 64, "four threads per column");
constexpr int RED_LIST = 2048;  // block numbers per round
__device__ inline void dem_objects(DemParams P, DemState d, int redBlocks, int demTimeStep) {
#pragma clang fp contract(off)
    __shared__ double sObj[12 * MAX_OBJECTS], sWall[6 * MAX_WALLS];
    __shared__ double sShare[4][64];
    __shared__ int list[RED_LIST], sWave[OBJ_THREADS / 64];
    const int t = threadIdx.x;
    const int nco = 12 * P.nObj, ncw = 6 * P.nWall;
    const int col = t % 64, share = t / 64;
    double acc = 0.0;
    for (int b0 = 0; b0 < redBlocks; b0 += RED_LIST) {
        const int n = flagged_blocks(d.redFlag + b0, min(RED_LIST, redBlocks - b0), list, sWave);
        if (col < nco + ncw) {
            const double* part = d.redPart + int64_t(b0) * DEM_RED_COLS + col;
            int k = share;
            for (; k + 28 < n; k += 32) {  // eight loads in flight
                double v[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) v[u] = part[int64_t(list[k + 4 * u]) * DEM_RED_COLS];
#pragma unroll
                for (int u = 0; u < 8; ++u) acc += v[u];
            }
            for (; k < n; k += 4) acc += part[int64_t(list[k]) * DEM_RED_COLS];
        }
        __syncthreads();
    }
    sShare[share][col] = acc;
    __syncthreads();
    if (t < 12 * MAX_OBJECTS) sObj[t] = 0.0;
    if (t < 6 * MAX_WALLS) sWall[t] = 0.0;
    __syncthreads();
    if (t < nco + ncw) {
        const double s = ((sShare[0][t] + sShare[1][t]) + sShare[2][t]) + sShare[3][t];
        if (t < nco) sObj[t] = s;
        else sWall[t - nco] = s;
    }
    const double* objSum;
    const double* wallSum;
    __syncthreads();
    if (t != 0) return;
    objSum = sObj;
    wallSum = sWall;
    // body-spring forces (DEM.cpp:798-869), on the positions before this step's integration
    double spring[MAX_OBJECTS];  // y component of each object's FSpring
    for (int o = 0; o < MAX_OBJECTS; ++o) spring[o] = 0.0;
    const bool waited = demTimeStep >= P.objWaitTime;
    for (int b = 0; b < P.nBody; ++b) {
        double* B = d.body + b * LBDEM_B_REC;
        double fsB = 0.0;
        if (waited) {
            for (int o = 0; o < P.nObj; ++o) {
                const double L = B[LBDEM_B_X0 + 1] - d.ox0[3 * o + 1];
                B[LBDEM_B_L] = L;
                const double rx = B[LBDEM_B_X0] - d.ox0[3 * o], ry = L, rz = B[LBDEM_B_X0 + 2] - d.ox0[3 * o + 2];
                const double rn = sqrt(rx * rx + ry * ry + rz * rz);
                const double ny = ry / rn;
                const double k = B[LBDEM_B_K], del = B[LBDEM_B_L0] - L, sigma = B[LBDEM_B_R];
                const double bodyDamp = 2.0 * sqrt(B[LBDEM_B_M] * k) * P.springDamp;
                const double objDamp = 2.0 * sqrt(d.om[o] * k) * P.springDamp;
                double fs, fdo = -d.ox1[3 * o + 1] * objDamp, fdb = -B[LBDEM_B_X1 + 1] * bodyDamp;
                if (P.nonLinType == 0) {
                    fs = k * del * ny;
                    fdo = 0.0;
                    fdb = 0.0;
                } else if (P.nonLinType == 1) {
                    fs = (k * del) * ny;
                } else if (P.nonLinType == 2) {
                    fs = (k * del + P.k13 * k * (del * del * del)) * ny;
                } else if (P.nonLinType == 3) {
                    fs = (k * del + (24.0 * P.epsilon / rn) * 2.0 * (pow((sigma / rn), 12.0))) * ny;
                } else {  // 4: WCA repulsion inside 2^(1/6) sigma
                    if (rn <= pow(2.0, 1.0 / 6.0) * sigma)
                        fs = (k * del + (24.0 * P.epsilon / rn) * ((2.0 * pow(sigma / rn, 12.0)) - (pow(sigma / rn, 6.0)))) * ny;
                    else
                        fs = (k * del) * ny;
                }
                spring[o] -= fs;
                fsB += fs;
                spring[o] += fdo;
                fsB += fdb;
            }
        }
        // totals (DEM.cpp:792-794): FTotal = FGrav + FSpring; integration (DEM.cpp:2730-2740)
        const double FT[3] = {B[LBDEM_B_FGRAV] + 0.0, B[LBDEM_B_FGRAV + 1] + fsB, B[LBDEM_B_FGRAV + 2] + 0.0};
        B[LBDEM_B_FSPRING] = 0.0; B[LBDEM_B_FSPRING + 1] = fsB; B[LBDEM_B_FSPRING + 2] = 0.0;
        for (int c = 0; c < 3; ++c) B[LBDEM_B_FTOTAL + c] = FT[c];
        if (waited) {
            const double dt = P.deltat, im = 1.0 / B[LBDEM_B_M];
            for (int c = 0; c < 3; ++c) B[LBDEM_B_X0 + c] += dt * B[LBDEM_B_X1 + c] + dt * dt * FT[c] * im;
            for (int c = 0; c < 3; ++c) B[LBDEM_B_X1 + c] += dt * FT[c] * im;
        }
    }
    for (int o = 0; o < P.nObj; ++o) {
        const double* s = objSum + 12 * o;
        const V Fc{s[0], s[1], s[2]}, Mc{s[3], s[4], s[5]}, Fl{s[6], s[7], s[8]}, Ml{s[9], s[10], s[11]};
        st3(d.oFContact, o, Fc); st3(d.oMContact, o, Mc); st3(d.oFLub, o, Fl); st3(d.oMLub, o, Ml);
        const V FH = ld3(d.oFHydro, o), MH = ld3(d.oMHydro, o), FG = ld3(d.oFGrav, o);
        const V FT = add(add(add(add(FH, Fc), Fl), FG), V{0, spring[o], 0});
        const V MT = add(add(MH, Mc), Ml);
        st3(d.oFTotal, o, FT); st3(d.oMTotal, o, MT);
        if (demTimeStep >= P.objWaitTime) {
            const double dt = P.deltat, im = d.oim[o], iI = d.oiI[o];
            double* x0 = d.ox0 + 3 * o; double* x1 = d.ox1 + 3 * o; double* w1 = d.ow1 + 3 * o;
            const double F[3] = {FT.x, FT.y, FT.z}, M[3] = {MT.x, MT.y, MT.z};
            for (int c = 0; c < 3; ++c) x0[c] += dt * x1[c] + dt * dt * F[c] * im;
            for (int c = 0; c < 3; ++c) x1[c] += dt * F[c] * im;
            for (int c = 0; c < 3; ++c) w1[c] += dt * M[c] * iI;
        }
        ObjLB ol;
        for (int c = 0; c < 3; ++c) { ol.c[c] = d.ox0[3 * o + c] / P.unitLength; ol.u[c] = d.ox1[3 * o + c] / P.unitSpeed; }
        ol.r = d.or_[o] / P.unitLength;
        ol.pad = 0.0;
        d.olb[o] = ol;
    }
    for (int w = 0; w < P.nWall; ++w) {
        const double* s = wallSum + 6 * w;
        const V Fc{s[0], s[1], s[2]}, Fl{s[3], s[4], s[5]};
        st3(d.wFContact, w, Fc); st3(d.wFLub, w, Fl);
        st3(d.wFTotal, w, add(add(add(ld3(d.wFHydro, w), Fc), Fl), V{0, 0, 0}));
    }
}

// particle p: totals, gravity switch-off, integration, periodic wrap, lattice view; returns |v|^2
__device__ inline double integrate_particle(const DemParams& P, const DemState& d, int demTimeStep, int p) {
#pragma clang fp contract(off)
    const V FT = add(add(add(add(ld3(d.FHydro, p), ld3(d.FContact, p)), ld3(d.FLub, p)), ld3(d.FGrav, p)), ld3(d.FRep, p));
    const V MT = add(add(ld3(d.MHydro, p), ld3(d.MContact, p)), ld3(d.MLub, p));
    st3(d.FTotal, p, FT); st3(d.MTotal, p, MT);
    if (demTimeStep <= P.objWaitTime) st3(d.FGrav, p, V{0, 0, 0});
    const double dt = P.deltat, im = d.im[p], iI = d.iI[p];
    double* x0 = d.x0 + 3 * p; double* x1 = d.x1 + 3 * p; double* w1 = d.w1 + 3 * p;
    const double F[3] = {FT.x, FT.y, FT.z}, M[3] = {MT.x, MT.y, MT.z};
    for (int c = 0; c < 3; ++c) x0[c] += dt * x1[c] + dt * dt * F[c] * im;
    for (int c = 0; c < 3; ++c) x1[c] += dt * F[c] * im;
    for (int c = 0; c < 3; ++c) w1[c] += dt * M[c] * iI;
    if (P.stress) {  // DEM.cpp:2705, 2721-2725 (before the periodic wrap, which follows the integration)
        for (int c = 0; c < 3; ++c) d.disp[3 * p + c] = d.xi0[3 * p + c] - x0[c];
        if (demTimeStep == P.objWaitTime)
            for (int c = 0; c < 3; ++c) d.xi0[3 * p + c] = x0[c];
    }
    for (int c = 0; c < 3; ++c)
        if (P.periodic[c]) {
            if (x0[c] > P.demSize[c]) x0[c] -= P.demSize[c];
            if (x0[c] < 0.0) x0[c] += P.demSize[c];
        }
    PartLB v;
    for (int c = 0; c < 3; ++c) {
        v.c[c] = x0[c] / P.unitLength;
        v.v[c] = x1[c] / P.unitSpeed;
        v.w[c] = w1[c] / P.unitAngVel;
    }
    v.r = d.r[p] / P.unitLength;
    d.plb[p] = v;
    return x1[0] * x1[0] + x1[1] * x1[1] + x1[2] * x1[2];
}
// Blocks [0, nb) integrate the particles (OBJ_THREADS per block), block nb does the objects and
// walls (dem_objects); later blocks (a batch launch sized for a larger box) return.
__device__ inline void k_dem_integrate(DemParams P, DemState d, int redBlocks, int demTimeStep, int nb) {
#pragma clang fp contract(off)
    if (int(blockIdx.x) >= nb) {
        if (int(blockIdx.x) == nb) dem_objects(P, d, redBlocks, demTimeStep);
        return;
    }
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    double v2 = 0.0;  // |v|^2 after the update, for the next step's neighbour-list trigger
    if (p < P.nPart) v2 = integrate_particle(P, d, demTimeStep, p);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const double o = __shfl_xor(v2, off, 64);
        v2 = o > v2 ? o : v2;
    }
    if (__lane_id() == 0 && v2 > 0.0)
        atomicMax(d.blockMax + blockIdx.x % VEL_SLOTS, (unsigned long long)__double_as_longlong(v2));
}

__device__ inline void k_dem_views(DemParams P, DemState d) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p < P.nPart) {
        PartLB v;
        for (int c = 0; c < 3; ++c) {
            v.c[c] = d.x0[3 * p + c] / P.unitLength;
            v.v[c] = d.x1[3 * p + c] / P.unitSpeed;
            v.w[c] = d.w1[3 * p + c] / P.unitAngVel;
        }
        v.r = d.r[p] / P.unitLength;
        d.plb[p] = v;
    }
    if (p < P.nObj) {
        ObjLB ol;
        for (int c = 0; c < 3; ++c) { ol.c[c] = d.ox0[3 * p + c] / P.unitLength; ol.u[c] = d.ox1[3 * p + c] / P.unitSpeed; }
        ol.r = d.or_[p] / P.unitLength;
        ol.pad = 0.0;
        d.olb[p] = ol;
    }
}


void dem_refresh_views(const DemParams& p, DemState& d, hipStream_t s) {
    const int n = p.nPart > p.nObj ? p.nPart : p.nObj;
    if (n > 0) launch<&k_dem_views, 1024, 1>((n + 255) / 256, 256, s, p, d);
}

// the records of a download in one pass: thread e writes value e of the record table, so the stores
// are contiguous and the loads of a column are strided by its array's width. One launch and one copy
// replace a copy, a wait and a host loop per array: particle records of the 256x320x256 box
// (31 000 x 48 values) 18 copies before; a step and its records on a 14x20x14 box 627 us with them.
__device__ inline void k_pack_records(RecordMap m, int n, double* out) {
    const int64_t e = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (e >= int64_t(n) * m.cols) return;
    const int i = int(e / m.cols), q = int(e - int64_t(i) * m.cols);
    out[e] = m.src[q][int64_t(i) * m.width[q] + m.comp[q]];
}
void dem_pack_records(const RecordMap& m, int n, double* out, hipStream_t s) {
    const int64_t total = int64_t(n) * m.cols;
    if (total > 0) launch<&k_pack_records, 256, 1>(int((total + 255) / 256), 256, s, m, n, out);
}

NbrArgs nbr_args(const DemParams& p, DemState& d, DevScalars* sc, bool force) {
    NbrArgs a{};
    a.p = p; a.x0 = d.x0; a.r = d.r;
    a.cellCount = d.cellCount; a.cellStart = d.cellStart; a.cellFill = d.cellFill; a.cellItems = d.cellItems;
    a.cellKey = d.cellKey; a.nbrCount = d.nbrCount; a.nbrList = d.nbrList; a.nbrSlot = d.nbrSlot;
    a.xi = d.xiCur; a.oldCount = d.nbrCountOld; a.oldList = d.nbrListOld; a.velMax = d.blockMax;
    a.force = force ? 1 : 0;
    a.scanBlocks = 1;
    const bool cells = p.nlx > 0 && p.nlz > 0;
    a.pBlocks = cells ? (p.nPart + 255) / 256 : 0;
    a.buildBlocks = (p.nPart + NBR_GROUPS - 1) / NBR_GROUPS;
    a.slotBlocks = int((int64_t(p.nPart) * SLOT_LANES + 255) / 256);  // SLOT_LANES threads per particle
    a.sc = sc;
    return a;
}
ForceArgs force_args(const DemParams& p, DemState& d, int demTimeStep) {
    ForceArgs f{};
    f.p = p; f.x0 = d.x0; f.x1 = d.x1; f.w1 = d.w1; f.r = d.r;
    f.FContact = d.FContact; f.MContact = d.MContact; f.FLub = d.FLub; f.MLub = d.MLub; f.FRep = d.FRep;
    f.xiw = d.xiw; f.xio = d.xio; f.nbrCount = d.nbrCount; f.nbrList = d.nbrList; f.nbrSlot = d.nbrSlot;
    f.xiOld = d.xiCur; f.xiNew = d.xiNext;
    f.ox0 = d.ox0; f.ox1 = d.ox1; f.ow1 = d.ow1; f.or_ = d.or_;
    f.redPart = d.redPart; f.redFlag = d.redFlag; f.lanes = dem_force_lanes(p.nPart, d.inBatch); f.blocks = dem_force_blocks(p.nPart, d.inBatch);
    f.demTimeStep = demTimeStep;
    f.stressPart = d.stressPart; f.shydro = d.shydro;
    return f;
}

void dem_integrate(const DemParams& p, DemState& d, int demTimeStep, hipStream_t s) {
    const int nb = (p.nPart + OBJ_THREADS - 1) / OBJ_THREADS;
    launch<&k_dem_integrate, OBJ_THREADS, 1>(nb + 1, OBJ_THREADS, s, p, d, dem_force_blocks(p.nPart, d.inBatch), demTimeStep, nb);
}

}  // namespace lbdem
