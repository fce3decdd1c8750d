// The fused collide-stream kernel (reconstruct, particle interior forcing, BGK/Guo collision, AA
// streaming with the boundary conditions resolved by the storing node; LB.cpp:1261-1544, 1901-1978,
// node.cpp:75-207) and the slip pass that follows it. fused_fp64.hip, fused_fp32.hip and
// fused_fp16.hip instantiate it, one storage type each, so that the variants compile in parallel.
#pragma once
#include "lattice.hpp"

namespace lbdem {

template <typename S>
struct FusedArgs {
    Geom g;
    S* f;
    S* fq[Q];  // population planes (f + q N): uniform bases of the fused kernel's accesses
    uint8_t* type;
    const int32_t* solid;
    typename Types<S>::M* mass;
    typename Types<S>::C* aux;
    typename Types<S>::C* visc;  // node viscosities (the NN variant of the kernel only)
    int32_t* ifList;
    int ifCap;
    const PartLB* plb;
    const ObjLB* olb;
    double* hacc;
    double* blockPart;
    const uint64_t* bcm;
    DevScalars* sc;
    int nseg, nby, nbz;  // 64-node segments per row (tiles per row with 2-byte storage), row groups, z-slabs
    int gridBlocks;  // the box's grid (a batch launch covers the largest box; the rest return)
    int sumMask;     // nodes of a tile, which share one sum in 32 bits before the block's FP64 table, less 1
    int storeVel;    // every active node's density and velocity into aux (else interface nodes only)
    Consts k;
};

// moving-object link (LB.cpp:1427-1453): bounce-back with the velocity of the object whose sphere
// holds the neighbour (the last one, as the reference scans objects in order), momentum exchange
// into the partials of the object named by the neighbour's solid index oi
template <typename S>
__device__ inline typename Types<S>::C object_value(const FusedArgs<S>& a, int j, int32_t yj, int oi,
                                                   typename Types<S>::C gj, typename Types<S>::C n, double mi,
                                                   double* sPart, const ObjLB* sObj) {
    using C = typename Types<S>::C;
    const int nObj = a.k.nObj;
    int yx, yy, yz;
    cell_xyz(a.g, yj, yx, yy, yz);
    // the impactor node's velocity (LB.cpp:1440): updateObjectBoundaries (LB.cpp:822-837) gives
    // every impactor node a fresh node each step and the velocity of the last impactor whose
    // sphere holds it, or none (zero) when no sphere holds it (a node a restart file typed as
    // impactor away from where the impactor now is)
    int ov = -1;
    for (int oo = 0; oo < nObj; ++oo)
        if (inside_sphere(yx, yy, yz, sObj[oo].c[0], sObj[oo].c[1], sObj[oo].c[2], sObj[oo].r)) ov = oo;
    const double cuo =
        ov < 0 ? 0.0 : sObj[ov].u[0] * cx_rt(j) + sObj[ov].u[1] * cy_rt(j) + sObj[ov].u[2] * cz_rt(j);
    const C BBi = C(6.0) * n * C(w_rt(j)) * C(cuo);
    if (oi >= 0 && oi < nObj && oi < MAX_OBJ_PART) {
        const double fm = 2.0 * double(gj) - double(BBi);
        const double Fb[3] = {fm * cx_rt(j), fm * cy_rt(j), fm * cz_rt(j)};
        const double rr[3] = {yx - sObj[oi].c[0], yy - sObj[oi].c[1], yz - sObj[oi].c[2]};
        const double M[3] = {rr[1] * Fb[2] - rr[2] * Fb[1], rr[2] * Fb[0] - rr[0] * Fb[2], rr[0] * Fb[1] - rr[1] * Fb[0]};
        double* sp = &sPart[7 * oi];
#pragma unroll
        for (int c = 0; c < 3; ++c) { atomicAdd(sp + c, Fb[c]); atomicAdd(sp + 3 + c, M[c]); }
    }
    atomicAdd(&sPart[PART_BB], double(BBi) * mi);
    return gj - BBi;
}

// boundary link of the storing cell (LB.cpp:1390-1453): value reflected into the slot the cell
// itself loads next step; momentum exchange into the block partials
template <typename S>
__device__ inline typename Types<S>::C boundary_value(const FusedArgs<S>& a, int j, int32_t yj, uint8_t ty,
                                                     typename Types<S>::C gj, typename Types<S>::C n,
                                                     typename Types<S>::C sx, typename Types<S>::C sy,
                                                     typename Types<S>::C sz, typename Types<S>::C usq, double mi,
                                                     double* sPart, const ObjLB* sObj) {
    using C = typename Types<S>::C;
    const Consts& k = a.k;
    if (ty == T_GAS) {
        const C cu = C(cx_rt(j)) * sx + C(cy_rt(j)) * sy + C(cz_rt(j)) * sz;
        return -gj + C(w_rt(j)) * (C(9) * (cu * cu) - C(3) * usq);
    }
    if (ty == T_WALL) {
        if (k.nWall > 0 && !k.slip) {
            int wi = a.solid[yj];
            wi = (wi >= 0 && wi < k.nWall) ? wi : 0;
            const double v2 = 2.0 * double(gj);
            if (cx_rt(j)) atomicAdd(&sPart[PART_WALL + 3 * wi + 0], v2 * cx_rt(j));
            if (cy_rt(j)) atomicAdd(&sPart[PART_WALL + 3 * wi + 1], v2 * cy_rt(j));
            if (cz_rt(j)) atomicAdd(&sPart[PART_WALL + 3 * wi + 2], v2 * cz_rt(j));
        }
        return gj;
    }
    if (ty == T_OBJ) return object_value<S>(a, j, yj, a.solid[yj], gj, n, mi, sPart, sObj);
    atomicOr(&a.sc->typeError, 1);
    return gj;
}

// Population addresses in the fused kernel: a uniform part in scalar registers (plane, row and
// the wrapped y/z steps: a wavefront is one x-row segment, so y and z are the same on all its
// lanes) plus a 32-bit per-lane byte offset (x, or x -+ 1 wrapped through periodic x faces) that
// stays fixed along the z-walk. Loads and stores take the scalar-base form: no 64-bit address
// arithmetic per access, no per-lane wrap registers.
struct LaneX {
    uint32_t m, o, p;  // byte offsets of x - 1, x, x + 1 within a row (wrapped, LB.cpp:632-678)
    __device__ LaneX(const Geom& g, int x, uint32_t elt) {
        const int xm = (x == 1 && g.per[0]) ? g.X - 2 : x - 1;
        const int xp = (x == g.X - 2 && g.per[1]) ? 1 : x + 1;
        m = uint32_t(xm) * elt;
        o = uint32_t(x) * elt;
        p = uint32_t(xp) * elt;
    }
    __device__ uint32_t sel(int cx) const { return cx < 0 ? m : (cx > 0 ? p : o); }
};
struct RowYZ {  // uniform across a wavefront
    int32_t row;             // index of node (0, y, z)
    int32_t ym, yp, zm, zp;  // index steps to the wrapped rows y -+ 1 and z -+ 1
    __device__ RowYZ(const Geom& g, int y, int z) {
        const int32_t sy = g.X, sz = g.X * g.Y;
        row = sy * y + sz * z;
        ym = (y == 1 && g.per[2]) ? (g.Y - 3) * sy : -sy;
        yp = (y == g.Y - 2 && g.per[3]) ? -(g.Y - 3) * sy : sy;
        zm = (z == 1 && g.per[4]) ? (g.Z - 3) * sz : -sz;
        zp = (z == g.Z - 2 && g.per[5]) ? -(g.Z - 3) * sz : sz;
    }
    // index of (0, y, z) of the row holding the wrapped neighbour in direction q
    __device__ int32_t nb(int q) const {
        return row + (cyq(q) < 0 ? ym : (cyq(q) > 0 ? yp : 0)) + (czq(q) < 0 ? zm : (czq(q) > 0 ? zp : 0));
    }
};
// element of a plane (uniform base) at a uniform row index plus a per-lane byte offset; a node's
// byte offset within a plane fits 32 bits (19 N < 2^31 nodes, at most 8 bytes each)
template <typename T>
__device__ inline T* at(T* plane, int32_t rowIdx, uint32_t laneBytes) {
    return reinterpret_cast<T*>(reinterpret_cast<char*>(plane) + (uint32_t(rowIdx) * uint32_t(sizeof(T)) + laneBytes));
}

// populations of a node before collision (its post-streaming values). PAR 0: the node's own
// slots; PAR 1: the slots its neighbours wrote (the neighbour in direction opp(q) holds slot
// opp(q)), wrapped through periodic faces
template <typename S, int PAR>
__device__ inline void load_pop(const FusedArgs<S>& a, const RowYZ& r, const LaneX& lx, bool act,
                                typename StoreT<S>::Raw* gq) {
    if (!act) return;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        if (PAR == 0) gq[q] = StoreT<S>::raw(at(a.fq[q], r.row, lx.o));
        else gq[q] = StoreT<S>::raw(at(a.fq[oppq(q)], r.nb(oppq(q)), lx.sel(cxq(oppq(q)))));
    }
}

// streaming of the post-collision values (LB.cpp:1375-1389): PAR 0 into the node's own slots
// (opposite direction), PAR 1 into the neighbours' slots (wrapped as in load_pop)
template <typename S, int PAR>
__device__ inline void store_pop(const FusedArgs<S>& a, const RowYZ& r, const LaneX& lx, bool act,
                                 const typename Types<S>::C* gq) {
    if (!act) return;
    StoreT<S>::st(at(a.fq[0], r.row, lx.o), gq[0]);
#pragma unroll
    for (int j = 1; j < Q; ++j) {
        if (PAR == 0) StoreT<S>::st(at(a.fq[oppq(j)], r.row, lx.o), gq[j]);
        else StoreT<S>::st(at(a.fq[j], r.nb(j), lx.sel(cxq(j))), gq[j]);
    }
}

// c_q . (x, y, z) without the products by zero, which the compiler has to keep (a NaN times zero)
// (419 -> 348 vector instructions a node; a step of the 256x320x256 impact box FP16 0.626 -> 0.619 ms,
// FP32 0.792 -> 0.788, of 128^3 FP32 0.156 -> 0.152; the larger boxes mostly wait for memory)
template <typename C>
__device__ inline C dir_dot(int q, C x, C y, C z) {
    C r = 0;
    bool any = false;
    if (cxq(q)) { r = cxq(q) > 0 ? x : -x; any = true; }
    if (cyq(q)) { const C v = cyq(q) > 0 ? y : -y; r = any ? r + v : v; any = true; }
    if (czq(q)) { const C v = czq(q) > 0 ? z : -z; r = any ? r + v : v; }
    return r;
}

// one node's collision (node.cpp:75-207): reconstruct, interior forcing of particle nodes
// (LB.cpp:1919-1962), BGK with Guo forcing. gc holds the post-streaming populations on entry
// and the post-collision ones on return.
template <typename S>
struct CellOut {
    typename Types<S>::C n, sx, sy, sz, usq, hx, hy, hz;
    typename Types<S>::C d[7];  // particle contribution: F(3), M(3), fluid volume
    typename Types<S>::C visc;  // the node's viscosity after the collision (NN variant)
    int key;                    // particle index or -1
};

// apparent viscosity (node.cpp:113-168): the shear-rate tensor from the non-equilibrium part of the
// post-streaming populations, relaxed with the node's previous viscosity nu, its magnitude
// (tinyMatrix::magnitude, myvector.cpp:546-550), the rheology model's viscosity plus the
// Smagorinsky term, clamped as std::max(minVisc, std::min(maxVisc, .)) clamps it (a NaN from 0 / 0
// becomes maxVisc). Second moments see a pair of opposite directions only through its sum, so the
// pair's even equilibrium part is subtracted once per pair: a third of the operations of the sum
// over the directions, whose products with zero components the compiler has to keep (50 steps and
// their records on a 150x110x100 box with BINGHAM and the Smagorinsky term, FP32: 13.1 -> 9.4 ms,
// about 1 ms of it from the record reads; the error against 64 bits stays what it was).
template <typename C>
__device__ inline C apparent_viscosity(const Consts& k, const C* gc, C n, C sx, C sy, C sz, C usq, C nu) {
    const C even = (n - C(1)) - C(1.5) * n * usq, n45 = C(4.5) * n;
    auto pair = [&](int q, C cu) { return (gc[q] + gc[q + 1]) - C(2 * wq(q)) * (even + n45 * (cu * cu)); };
    const C p7 = pair(7, sx + sy), p9 = pair(9, sy - sx), p11 = pair(11, sy + sz), p13 = pair(13, sz - sy);
    const C p15 = pair(15, sx + sz), p17 = pair(17, sx - sz);
    C xx = pair(1, sx) + ((p7 + p9) + (p15 + p17));
    C yy = pair(3, sy) + ((p7 + p9) + (p11 + p13));
    C zz = pair(5, sz) + ((p11 + p13) + (p15 + p17));
    C xy = p7 - p9, xz = p15 - p17, yz = p11 - p13;
    const C tau = C(0.5) + C(3) * nu;
    const C sc = C(1.5) / (tau * n);
    xx *= sc; yy *= sc; zz *= sc; xy *= sc; xz *= sc; yz *= sc;
    const C shear = C(2) * sqrt(C(0.5) * (xx * xx + yy * yy + zz * zz + C(2) * (xy * xy + xz * xz + yz * yz)));
    C app;
    if (k.rheo == LBDEM_RHEO_BINGHAM) {
        app = C(k.plasticVisc) + C(k.yieldStress) / shear;
    } else if (k.rheo == LBDEM_RHEO_FRICTIONAL || k.rheo == LBDEM_RHEO_VOELLMY) {
        const C pr = C(0.33333333) * (n - C(1));
        const C pressure = C(0) < pr ? pr : C(0);  // std::max(0.0, .)
        app = k.rheo == LBDEM_RHEO_FRICTIONAL ? C(k.visc) + C(k.frictionCoef) * pressure / shear
                                              : (C(k.frictionCoef) * pressure + usq / C(k.voellmyCoef)) / shear;
    } else {
        app = C(k.visc);
    }
    if (k.turb) app += C(k.turbConst) * shear;
    const C lo = C(k.minVisc), hi = C(k.maxVisc);
    const C m = app < hi ? app : hi;  // std::min(maxVisc, app)
    return lo < m ? m : lo;           // std::max(minVisc, .)
}
template <typename S, bool NN>
__device__ inline void collide_cell(const FusedArgs<S>& a, int32_t sp, uint8_t t, int x, int y, int z, double mi,
                                    typename Types<S>::C* gc, typename Types<S>::C nuIn, CellOut<S>& r) {
    using C = typename Types<S>::C;
    const Consts& k = a.k;
    C sum = 0, jx = 0, jy = 0, jz = 0;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        sum += gc[q];
        if (cxq(q)) jx += C(cxq(q)) * gc[q];
        if (cyq(q)) jy += C(cyq(q)) * gc[q];
        if (czq(q)) jz += C(czq(q)) * gc[q];
    }
    const C n = C(1) + sum;
    const C inv = C(1) / n;  // one division per node: the quotients below differ by rounding only
    const C ux = jx * inv, uy = jy * inv, uz = jz * inv;
    C hx = 0, hy = 0, hz = 0;
    if (t & T_PMASK) {
        const PartLB P = a.plb[sp];
        const C rx = C(double(x) - P.c[0]), ry = C(double(y) - P.c[1]), rz = C(double(z) - P.c[2]);
        const C wx = C(P.w[0]), wy = C(P.w[1]), wz = C(P.w[2]);
        const C lvx = C(P.v[0]) + (wy * rz - wz * ry);
        const C lvy = C(P.v[1]) + (wz * rx - wx * rz);
        const C lvz = C(P.v[2]) + (wx * ry - wy * rx);
        const C lf = C(mi) * inv;
        const C dfx = lf * (ux - lvx), dfy = lf * (uy - lvy), dfz = lf * (uz - lvz);
        hx = -dfx; hy = -dfy; hz = -dfz;
        r.d[0] = dfx; r.d[1] = dfy; r.d[2] = dfz;
        r.d[3] = ry * dfz - rz * dfy; r.d[4] = rz * dfx - rx * dfz; r.d[5] = rx * dfy - ry * dfx;
        r.d[6] = C(mi);
        r.key = sp;
    }
    const C Fx = C(k.lbF[0]) + hx, Fy = C(k.lbF[1]) + hy, Fz = C(k.lbF[2]) + hz;
    const C sx = ux + C(0.5) * Fx * inv, sy = uy + C(0.5) * Fy * inv, sz = uz + C(0.5) * Fz * inv;
    // The order of the fused products is written out where the results hang on their rounding (free-surface
    // and particle flags; 2-byte storage most): which one the compiler fuses depends on the code around.
    C usq, uF;
    if constexpr (NN) {
        usq = sx * sx + sy * sy + sz * sz;
        uF = sx * Fx + sy * Fy + sz * Fz;
    } else {
        usq = sizeof(S) == 2 ? fma(sz, sz, fma(sx, sx, sy * sy)) : fma(sz, sz, fma(sy, sy, sx * sx));
        uF = fma(sz, Fz, fma(sy, Fy, sx * Fx));
    }
    C om = C(k.omega), omf = C(k.omegaf);
    if constexpr (NN) {  // the node's own viscosity, updated first when the model asks for it
        const C nu = k.viscUpdate ? apparent_viscosity<C>(k, gc, n, sx, sy, sz, usq, nuIn) : nuIn;
        om = C(1) / (C(0.5) + C(3) * nu);
        omf = C(1) - C(1) / (C(1) + C(6) * nu);
        r.visc = nu;
    }
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const C cu = dir_dot(q, sx, sy, sz);
        const C cF = dir_dot(q, Fx, Fy, Fz);
        const C e = fma(C(-1.5), usq, fma(C(3), cu, C(4.5) * cu * cu));
        const C fq = fma(cF, C(9) * cu, C(3) * (cF - uF));
        // gc + om (geq - gc) + omf w fq with geq = w (n - 1 + n e)
        gc[q] = fma(omf * C(wq(q)), fq, fma(om, fma(fma(n, e, n - C(1)), C(wq(q)), -gc[q]), gc[q]));
    }
    r.n = n; r.sx = sx; r.sy = sy; r.sz = sz; r.usq = usq; r.hx = hx; r.hy = hy; r.hz = hz;
}

// one thread's running sums of particle key into the block's table (LDS hash; global atomics
// when the table is full)
template <typename C>
__device__ inline void add_particle(int key, const C* s, int* hkey, double (*hval)[7], double* hacc) {
    int slot = key & (HS - 1);
    int probes = 0;
    for (; probes < HS; ++probes) {
        const int old = atomicCAS(&hkey[slot], -1, key);
        if (old == -1 || old == key) break;
        slot = (slot + 1) & (HS - 1);
    }
    if (probes < HS) {
#pragma unroll
        for (int c = 0; c < 7; ++c) atomicAdd(&hval[slot][c], double(s[c]));
    } else {
        double* hp = hacc + int64_t(key) * 8;
#pragma unroll
        for (int c = 0; c < 7; ++c) atomicAdd(hp + c, double(s[c]));
    }
}

__device__ inline void flush_particles(int tid, int nthreads, const int* hkey, double (*hval)[7], double* hacc) {
    for (int s = tid; s < HS; s += nthreads) {
        const int key = hkey[s];
        if (key >= 0) {
            double* hp = hacc + int64_t(key) * 8;
            for (int c = 0; c < 7; ++c) atomicAdd(hp + c, hval[s][c]);
        }
    }
}

// Fused collide-stream over the box. Block = FX x FY columns; each thread walks FZ nodes along z.
// Per node the loads of the next node (populations, mass, solid index, boundary-link classes)
// and the type byte of the node after it go out before this node's stores (in either AA parity a
// node loads and stores only its own slot set, so no store of node z aliases a load of node
// z+1). Edge nodes are handled by the same waves as their row neighbours, so every population
// access stays coalesced; their boundary links run in a rolled loop over the precomputed link
// classes, without further loads for gas and wall links.
// Launch bounds of the fused kernel, in blocks (one wavefront per SIMD each) per CU: four for
// 4- and 2-byte storage (128 VGPRs: two words of the prologue's are spilled across the walk, none
// inside it; LDS is at most 13 KB per block), two for
// FP64 (its populations alone take 38 VGPRs per node, and two nodes are live).
template <typename S> struct FusedOcc { static constexpr int value = sizeof(S) == 8 ? 2 : 4; };
// Block-to-node mapping. Row order (see k_fused) for 4- and 8-byte storage; measured on the
// 256x320x256 impact box in the impact phase: FP32 0.726 -> 0.631 ms per launch, FP64
// 1.310 -> 1.198 ms against 64 x 4 tiles spread over the XCDs (a probe of the bare AA accesses:
// 5.2 TB/s in either parity in row order, 3.8 TB/s odd / 4.6 TB/s even with the tiles). 2-byte
// storage keeps the tiles (0.521 ms there against 0.656 ms in row order).
template <typename S> struct FusedRowOrder { static constexpr bool value = sizeof(S) >= 4; };
// nodes whose bundle is loaded ahead of the one being collided. Measured as above: none 0.71 ms,
// one 0.69 ms, two 0.78 ms (more loads in flight per CU slow the memory system down).
template <typename S> struct FusedAhead { static constexpr int value = 1; };

// Gas and wall links of edge nodes from the registers of the collision, one unrolled direction after
// the other, instead of reading each value back from where it was stored, link by link: every link of
// the rolled loop waits for a store and a load. For one-node walks (the boxes too small to fill the
// GPU with longer ones, where one node's chain of waits is the launch) and FP64, which have the
// registers; with 4- and 2-byte storage and a walk the next node's populations are live as well, the
// kernel spills, and edge rows are few (256x320x256 FP32: 0.80 -> 0.83 ms a step with it). Whole
// passes: 128^3 FP32 18.6 -> 18.0 ms, 91^3 FP64 closed box 8.6 -> 8.2 ms, 256x320x256 FP64 67.9 -> 67.3 ms.
template <typename S, int FZ> struct FusedRegLinks { static constexpr bool value = FZ == 1 || sizeof(S) == 8; };

// per-node bundle: type byte, populations, mass (particle or edge node), solid index (particle
// node); the boundary-link classes of edge nodes (rare) are loaded where they are used. The
// populations stay as loaded until the node collides: converted here, 2-byte values would make the
// wavefront wait for the next node's loads before this node's arithmetic instead of behind it
// (256x320x256 impact box, FP16 storage, four-node walk: 0.70 -> 0.62 ms a step)
template <typename S>
struct Bundle {
    typename StoreT<S>::Raw g[Q];
    typename Types<S>::M m;
    int32_t s;
    uint8_t t;
    bool act;
};
template <typename S, int PAR>
__device__ inline void load_bundle(const FusedArgs<S>& a, const RowYZ& r, const LaneX& lx, int32_t i, uint8_t t,
                                   Bundle<S>& n) {
    using M = typename Types<S>::M;
    n.t = t;
    n.act = is_active(t);
    load_pop<S, PAR>(a, r, lx, n.act, n.g);
    n.m = (n.act && (t & (T_PMASK | T_EDGE))) ? a.mass[i] : M(0);
    n.s = (n.act && (t & T_PMASK)) ? a.solid[i] : 0;
}

template <typename S, int PAR, bool FSURF, int FZ, bool NN>
__device__ inline void k_fused(FusedArgs<S> a) {
    using C = typename Types<S>::C;
    using M = typename Types<S>::M;
    constexpr int NT = FX * FY;
    constexpr bool REGLINKS = FusedRegLinks<S, FZ>::value;
    constexpr bool SUBTILES = sizeof(S) == 2 && FZ > 2;
    if (int(blockIdx.x) >= a.gridBlocks) return;
    __shared__ int hkey[HS];
    __shared__ double hval[HS][7];
    __shared__ double sPart[PART_STRIDE]; // object / wall partials of the block (FP64 LDS atomics)
    __shared__ int32_t sIf[NT * FZ];      // interface nodes of the block
    __shared__ int sIfCount, sIfBase;
    __shared__ ObjLB sObj[MAX_OBJ_PART];  // the impactors' centres, radii and velocities
    const int tid = threadIdx.x + FX * threadIdx.y;
    if (tid < MAX_OBJ_PART * 8 && tid / 8 < a.k.nObj)
        reinterpret_cast<double*>(sObj)[tid] = reinterpret_cast<const double*>(a.olb)[tid];
    for (int s = tid; s < HS; s += NT) {
        hkey[s] = -1;
        for (int c = 0; c < 7; ++c) hval[s][c] = 0.0;
    }
    if (tid < PART_STRIDE) sPart[tid] = 0.0;
    if (tid == 0) sIfCount = 0;
    __syncthreads();

    static_assert(FX == 64, "a wavefront is one x-row segment: y and z are uniform across it");
    const Geom& g = a.g;
    const int b0 = blockIdx.x;
    int x, y, bz;
    bool col_ok;
    if constexpr (FusedRowOrder<S>::value) {
        // Row order: wavefront threadIdx.y of block b takes row segment s = FY b + threadIdx.y, i.e.
        // segment seg (64 nodes along x) of row y of z-slab bz, s = (bz Y + y) nseg + seg, and walks
        // the slab's FZ nodes in z. The blocks resident at a time then cover a few consecutive
        // z-planes, and the x -+ 1 accesses of a segment's edge lanes meet the neighbouring
        // segment's in the same or the next block while both are in flight.
        const int sid = b0 * FY + int(threadIdx.y);
        const int seg = sid % a.nseg, rest = sid / a.nseg;
        y = rest % g.Y;
        bz = rest / g.Y;
        x = seg * FX + threadIdx.x;
        col_ok = bz < a.nbz && x < g.X;
    } else {
        // 64 x 4 tiles, consecutive tiles on one XCD (tile = (b % 8) per + b / 8)
        const int nblk = a.nseg * a.nby * a.nbz;
        const int per = (nblk + 7) / 8;
        const int tile = (b0 % 8) * per + b0 / 8;
        const int bx = tile % a.nseg, by = (tile / a.nseg) % a.nby;
        bz = tile / (a.nseg * a.nby);
        x = bx * FX + threadIdx.x;
        y = by * FY + threadIdx.y;
        col_ok = tile < nblk && x < g.X && y < g.Y;
    }
    const int yw = __builtin_amdgcn_readfirstlane(y);
    const int32_t N = int32_t(g.N), SZ = g.X * g.Y;
    const int lane = __lane_id();
    const int z0 = __builtin_amdgcn_readfirstlane(bz) * FZ;
    auto type_at = [&](int zz) -> uint8_t {
        return (col_ok && zz < FZ && z0 + zz < g.Z) ? a.type[int32_t(cidx(g, x, yw, z0 + zz))] : uint8_t(T_WALL);
    };

    // Bundles of the current node and of the AH nodes after it are in registers; per node the
    // thread loads the bundle AH nodes ahead and the type byte one further before it collides and
    // stores the current node. In either AA parity a node loads and stores only its own slot set,
    // so no load of a node ahead reads a slot that a store of the current node writes.
    constexpr int AH = FusedAhead<S>::value;
    Bundle<S> nb[AH + 1];  // nb[0]: current node, nb[k]: k nodes ahead
    int32_t ic = col_ok ? int32_t(cidx(g, x, yw, z0)) : 0;
    const LaneX lx(g, x, uint32_t(sizeof(S)));
#pragma unroll
    for (int k = 0; k < AH; ++k) load_bundle<S, PAR>(a, RowYZ(g, yw, z0 + k), lx, ic + k * SZ, type_at(k), nb[k]);
    uint8_t tAhead = type_at(AH);  // type byte of the node AH ahead
    int accKey = -1;  // particle whose contributions acc holds
    C acc[7];
#pragma unroll
    for (int c = 0; c < 7; ++c) acc[c] = 0;
    for (int zz = 0; zz < FZ; ++zz) {
        const int z = z0 + zz;
        const uint8_t tFar = type_at(zz + AH + 1);
        // The wavefront issues its memory operations at raised priority, so that with three
        // wavefronts per SIMD the next node's loads (and the current node's stores) leave ahead of
        // the other wavefronts' arithmetic: measured 1 % faster (0.688 -> 0.679 ms per launch on
        // the 256x320x256 impact box, FP32) than at the default priority throughout.
        __builtin_amdgcn_s_setprio(2);
        load_bundle<S, PAR>(a, RowYZ(g, yw, z + AH), lx, ic + AH * SZ, tAhead, nb[AH]);
        __builtin_amdgcn_s_setprio(0);
        C gc[Q];
#pragma unroll
        for (int q = 0; q < Q; ++q) gc[q] = StoreT<S>::value(nb[0].g[q]);
        const bool actc = nb[0].act;
        const uint8_t tc = nb[0].t;
        const double mc = double(nb[0].m);
        const int32_t sc_ = nb[0].s;

        CellOut<S> r;
        r.key = -1;
#pragma unroll
        for (int c = 0; c < 7; ++c) r.d[c] = 0;
        r.n = 1; r.sx = 0; r.sy = 0; r.sz = 0; r.usq = 0;
        uint64_t bcEarly = 0;  // the link classes of edge nodes, on their way while the node collides
        if constexpr (REGLINKS) {
            if (actc && (tc & T_EDGE)) bcEarly = a.bcm[ic];
        }
        C nu = 0;
        if constexpr (NN) {
            if (actc) nu = a.visc[ic];
        }
        if (actc) collide_cell<S, NN>(a, sc_, tc, x, yw, z, mc, gc, nu, r);
        if constexpr (NN) {
            if (actc && a.k.viscUpdate) a.visc[ic] = r.visc;
        }
        __builtin_amdgcn_s_setprio(1);
        store_pop<S, PAR>(a, RowYZ(g, yw, z), lx, actc, gc);
        __builtin_amdgcn_s_setprio(0);

        // boundary links of edge nodes (LB.cpp:1390-1528): the value reflected into the slot
        // this node loads next step (FusedRegLinks: gas and wall links from registers)
        const bool edge = actc && (tc & T_EDGE);
        // In the rolled loop the post-collision value of link j is read back from where store_pop just
        // put it (PAR 0: the node's own slot opp(j); PAR 1: slot j of the neighbour), which the same
        // lane wrote, so it needs no staging; the reflected value then goes to the slot the node loads
        // next step.
        if (__ballot(edge)) {
            const uint64_t bc_ = REGLINKS ? bcEarly : (edge ? a.bcm[ic] : 0);
            uint32_t lm = 0;
            if constexpr (REGLINKS) {
                double wf[3] = {0.0, 0.0, 0.0};
                const RowYZ rw(g, yw, z);
#pragma unroll
                for (int j = 1; j < Q; ++j) {
                    const int cls = int(bc_ >> (BC_BITS * (j - 1))) & 7;
                    if (cls == BC_NONE) continue;
                    if (cls != BC_GAS && cls != BC_WALL) {
                        lm |= 1u << j;
                        continue;
                    }
                    const C gj = StoreT<S>::stored(gc[j]);
                    C bcv = gj;
                    if (cls == BC_GAS) {
                        const C cu = C(cxq(j)) * r.sx + C(cyq(j)) * r.sy + C(czq(j)) * r.sz;
                        bcv = -gj + C(wq(j)) * (C(9) * (cu * cu) - C(3) * r.usq);
                    } else {
                        const double v2 = 2.0 * double(gj);
                        if (cxq(j)) wf[0] += cxq(j) > 0 ? v2 : -v2;
                        if (cyq(j)) wf[1] += cyq(j) > 0 ? v2 : -v2;
                        if (czq(j)) wf[2] += czq(j) > 0 ? v2 : -v2;
                    }
                    if (PAR == 0) StoreT<S>::st(at(a.fq[j], rw.nb(j), lx.sel(cxq(j))), bcv);
                    else StoreT<S>::st(at(a.fq[oppq(j)], rw.row, lx.o), bcv);
                }
                // wall force of the node's links into the block's partials; the lanes of a wavefront
                // nearly always face one wall, and add up before the one atomic per component
                if (a.k.nWall > 0 && !a.k.slip) {  // slip walls take no force (LB.cpp:1454-1482)
                    const int wp = int(bc_ >> BC_WALL_SHIFT) & 7;
                    const bool hit = wf[0] != 0.0 || wf[1] != 0.0 || wf[2] != 0.0;
                    const unsigned long long hm = __ballot(hit);
                    if (hm) {
                        const int w0 = __shfl(wp, __ffsll(hm) - 1, 64);
                        if (__ballot(hit && wp != w0) == 0) {
#pragma unroll
                            for (int c = 0; c < 3; ++c) {
#pragma unroll
                                for (int off = 32; off > 0; off >>= 1) wf[c] += __shfl_xor(wf[c], off, 64);
                                if (lane == 0 && wf[c] != 0.0) atomicAdd(&sPart[PART_WALL + 3 * w0 + c], wf[c]);
                            }
                        } else if (hit) {
#pragma unroll
                            for (int c = 0; c < 3; ++c)
                                if (wf[c] != 0.0) atomicAdd(&sPart[PART_WALL + 3 * wp + c], wf[c]);
                        }
                    }
                }
            } else if (edge) {
#pragma unroll
                for (int j = 1; j < Q; ++j)
                    if ((bc_ >> (BC_BITS * (j - 1))) & 7u) lm |= 1u << j;
            }
            const Offs o(g, x, yw, z);
            const int wprim = int(bc_ >> BC_WALL_SHIFT) & 7;
            while (lm) {
                const int j = __ffs(lm) - 1;
                lm &= lm - 1u;
                const int cls = int(bc_ >> (BC_BITS * (j - 1))) & 7;
                const int32_t yj = ic + offs_rt(o, j);
                S* const own = a.f + int64_t(opp_rt(j)) * N + ic;  // slot opp(j) of this node
                S* const nbs = a.f + int64_t(j) * N + yj;          // slot j of the neighbour
                const C gj = StoreT<S>::ld(PAR == 0 ? own : nbs);
                C bcv;
                if (!REGLINKS && cls == BC_GAS) {
                    const C cu = C(cx_rt(j)) * r.sx + C(cy_rt(j)) * r.sy + C(cz_rt(j)) * r.sz;
                    bcv = -gj + C(w_rt(j)) * (C(9) * (cu * cu) - C(3) * r.usq);
                } else if (!REGLINKS && cls == BC_WALL) {
                    if (a.k.nWall > 0 && !a.k.slip) {  // slip walls take no force (LB.cpp:1454-1482)
                        const double v2 = 2.0 * double(gj);
                        double* wp = &sPart[PART_WALL + 3 * wprim];
                        if (cx_rt(j)) atomicAdd(wp + 0, v2 * cx_rt(j));
                        if (cy_rt(j)) atomicAdd(wp + 1, v2 * cy_rt(j));
                        if (cz_rt(j)) atomicAdd(wp + 2, v2 * cz_rt(j));
                    }
                    bcv = gj;
                } else if (cls == BC_OBJ0 || cls == BC_OBJ1) {
                    bcv = object_value<S>(a, j, yj, cls - BC_OBJ0, gj, r.n, mc, sPart, sObj);
                } else {
                    const uint8_t ty = a.type[yj] & T_BASE;
                    if (ty == T_FLUID || ty == T_IF) continue;  // an object node uncovered since marking
                    bcv = boundary_value<S>(a, j, yj, ty, gj, r.n, r.sx, r.sy, r.sz, r.usq, mc, sPart, sObj);
                }
                StoreT<S>::st(PAR == 0 ? nbs : own, bcv);
            }
        }
        if (FSURF) {
            const bool isIf = actc && (tc & T_BASE) == T_IF;
            if (actc && !isIf) a.mass[ic] = M(r.n);
            if (isIf || (actc && a.storeVel)) {
                a.aux[ic] = r.n;
                a.aux[N + ic] = r.sx; a.aux[2 * N + ic] = r.sy; a.aux[3 * N + ic] = r.sz;
                a.aux[4 * N + ic] = r.hx; a.aux[5 * N + ic] = r.hy; a.aux[6 * N + ic] = r.hz;
            }
            // interface list: one LDS reservation per wave
            const unsigned long long m = __ballot(isIf);
            if (m) {
                const int leader = __ffsll((unsigned long long)m) - 1;
                int base = 0;
                if (lane == leader) base = atomicAdd(&sIfCount, __popcll(m));
                base = __shfl(base, leader, 64);
                if (isIf) sIf[base + __popcll(m & ((1ull << lane) - 1ull))] = ic;
            }
        } else if (actc && a.storeVel) {
            a.aux[ic] = r.n;
            a.aux[N + ic] = r.sx; a.aux[2 * N + ic] = r.sy; a.aux[3 * N + ic] = r.sz;
            a.aux[4 * N + ic] = r.hx; a.aux[5 * N + ic] = r.hy; a.aux[6 * N + ic] = r.hz;
        }
        // particle sums: the thread's z-walk usually stays in one sphere for several nodes, so the
        // contributions are summed in registers while the particle index is unchanged and added
        // to the block's table when it changes (and after the walk)
        if (r.key != accKey || (SUBTILES && (zz & a.sumMask) == 0)) {
            if (accKey >= 0) add_particle<C>(accKey, acc, hkey, hval, a.hacc);
            accKey = r.key;
#pragma unroll
            for (int c = 0; c < 7; ++c) acc[c] = r.d[c];
        } else if (r.key >= 0) {
#pragma unroll
            for (int c = 0; c < 7; ++c) acc[c] += r.d[c];
        }
        // advance the column
        ic += SZ;
        tAhead = tFar;
#pragma unroll
        for (int k = 0; k < AH; ++k) nb[k] = nb[k + 1];
    }
    if (accKey >= 0) add_particle<C>(accKey, acc, hkey, hval, a.hacc);
    __syncthreads();
    int tx = threadIdx.x + FX * threadIdx.y;
    asm volatile("" : "+v"(tx));
    flush_particles(tx, NT, hkey, hval, a.hacc);
    if (FSURF) {
        // interface list: one global reservation per block
        const int n = sIfCount;
        if (n > 0) {
            if (tx == 0) sIfBase = atomicAdd(&a.sc->nIf, n);
            __syncthreads();
            const int base = sIfBase;
            for (int k = tx; k < n; k += NT) {
                if (base + k < a.ifCap) a.ifList[base + k] = sIf[k];
                else atomicOr(&a.sc->listOverflow, 1);
            }
        }
    }
    // object / wall partials: a block that has any appends them, column by column, to the records
    // the finalisation sums (the sums above are complete since the block's synchronisation before
    // flush_particles; one wavefront holds them all). The impactor's records, a few hundred, have a
    // list of their own: the free surface needs their extra mass first.
    static_assert(PART_STRIDE <= FX, "one wavefront appends the block's partials");
    if (threadIdx.y == 0) {
        const bool used = tx < PART_STRIDE && sPart[tx] != 0.0;
        const uint32_t m = uint32_t(__ballot(used));
        constexpr uint32_t objBits = (1u << PART_WALL) - 1u;
        int pos = 0;
        if (tx == 0 && (m & objBits)) pos = atomicAdd(&a.sc->nPartObj, 1);
        if (tx == PART_WALL && (m & ~objBits)) pos = atomicAdd(&a.sc->nPartWall, 1);
        const int po = __shfl(pos, 0, 64), pw = __shfl(pos, PART_WALL, 64);
        const int64_t col = int64_t(tx) * part_stride(g);
        if ((m & objBits) && tx < PART_WALL) a.blockPart[col + po] = sPart[tx];
        if ((m & ~objBits) && tx >= PART_WALL && tx < PART_STRIDE)
            a.blockPart[col + pw] = sPart[tx];
    }
}

// Slip walls (LB.cpp:1454-1482, slip static walls): a diagonal link j (j > 6) of an active node A
// into a wall, with exactly one of its two check nodes A + c(slip1Check[j]), A + c(slip2Check[j])
// active, receives S1 times that active check node B's post-collision population k = slip1[j]
// (or slip2[j]) plus S2 = 1 - S1 times A's own post-collision population j; every other wall link
// bounces back, as the fused kernel has already written. Runs right after the fused kernel of
// parity PAR, over the nodes next to a wall: it reads post-collision values where that kernel
// stored them (PAR 0: slot opp(k) of the node itself; PAR 1: slot k of the node's neighbour in
// direction k, here always the inactive check node or the wall) and overwrites the slot A loads
// next step (PAR 0: slot j of the wall node; PAR 1: A's own slot opp(j)), none of which is read here.
template <typename S, int PAR>
__device__ inline void k_slip(Geom g, S* f, const uint8_t* type, const int32_t* list, int n, double s1) {
    using C = typename StoreT<S>::C;
    const int i = int(blockIdx.x * blockDim.x + threadIdx.x);
    if (i >= n) return;
    const int32_t a = list[i];
    if (!is_active(type[a])) return;
    int x, y, z;
    cell_xyz(g, a, x, y, z);
    const Offs oa(g, x, y, z);
    const int64_t N = g.N;
#pragma unroll
    for (int j = 7; j < Q; ++j) {
        const int32_t w = a + oa.d(j);
        if ((type[w] & T_BASE) != T_WALL) continue;
        const bool act1 = is_active(type[a + oa.d(slip1Check(j))]);
        const bool act2 = is_active(type[a + oa.d(slip2Check(j))]);
        if (act1 == act2) continue;  // bounce-back, written by the fused kernel
        const int32_t b = a + oa.d(act1 ? slip1Check(j) : slip2Check(j));
        const int kk = act1 ? slip1Dir(j) : slip2Dir(j);
        C fb, fa;
        if (PAR == 0) {
            fb = StoreT<S>::ld(f + int64_t(oppq(kk)) * N + b);
            fa = StoreT<S>::ld(f + int64_t(oppq(j)) * N + a);
        } else {
            int bx, by, bz;
            cell_xyz(g, b, bx, by, bz);
            const Offs ob(g, bx, by, bz);
            fb = StoreT<S>::ld(f + int64_t(kk) * N + b + ob.d(kk));
            fa = StoreT<S>::ld(f + int64_t(j) * N + w);
        }
        // offset storage: S1 (fb + w) + S2 (fa + w) - w = S1 fb + S2 fa (the weights of j and kk agree)
        const C v = C(s1) * fb + (C(1) - C(s1)) * fa;
        if (PAR == 0) StoreT<S>::st(f + int64_t(j) * N + w, v);
        else StoreT<S>::st(f + int64_t(oppq(j)) * N + a, v);
    }
}

template <typename S>
static void launch_slip(const Box& b, double s1, hipStream_t s) {
    const int bs = 256, nb = (b.nSlip + bs - 1) / bs;
    if (b.parity == 0) launch<&k_slip<S, 0>, 256, 1>(nb, bs, s, b.g, (S*)b.f, b.type, b.slipList, b.nSlip, s1);
    else launch<&k_slip<S, 1>, 256, 1>(nb, bs, s, b.g, (S*)b.f, b.type, b.slipList, b.nSlip, s1);
}

template <typename S>
void launch_fused(Box& b, const Consts& k, const PartLB* plb, const ObjLB* olb, DevScalars* sc,
                         bool storeVel, hipStream_t s, hipEvent_t ev0, hipEvent_t ev1) {
    FusedArgs<S> a;
    a.g = b.g; a.f = (S*)b.f; a.type = b.type; a.solid = b.solid;
    for (int q = 0; q < Q; ++q) a.fq[q] = a.f + int64_t(q) * b.g.N;
    a.mass = (typename Types<S>::M*)b.mass; a.aux = (typename Types<S>::C*)b.aux;
    a.visc = (typename Types<S>::C*)b.visc;
    a.ifList = b.ifList; a.ifCap = b.ifCap;
    a.plb = plb; a.olb = olb; a.hacc = b.hacc; a.blockPart = b.blockPart; a.bcm = b.bcm; a.sc = sc;
    a.k = k;
    const int fz = b.fz;
    a.nseg = (b.g.X + FX - 1) / FX; a.nby = (b.g.Y + FY - 1) / FY; a.nbz = (b.g.Z + fz - 1) / fz;
    const int grid = fused_grid_blocks(b.g, fz, b.prec);
    a.gridBlocks = grid;
    a.sumMask = b.tz - 1;
    a.storeVel = storeVel ? 1 : 0;
    const bool fs = k.freeSurface != 0;
    if (ev0) (void)hipEventRecord(ev0, s);
    const bool nn = b.visc != nullptr;
#define LBDEM_FUSED(P, F, Z, V) \
    launch<&k_fused<S, P, F, Z, V>, FX * FY, FusedOcc<S>::value>(dim3(grid), dim3(FX, FY, 1), s, a)
#define LBDEM_FUSED_Z(P, F, V)                 \
    switch (fz) {                             \
        case 1: LBDEM_FUSED(P, F, 1, V); break; \
        case 2: LBDEM_FUSED(P, F, 2, V); break; \
        case 4: LBDEM_FUSED(P, F, 4, V); break; \
        default: LBDEM_FUSED(P, F, 8, V); break; \
    }
#define LBDEM_FUSED_FS(P, V) \
    if (fs) { LBDEM_FUSED_Z(P, true, V); } else { LBDEM_FUSED_Z(P, false, V); }
    if (nn) {
        if (b.parity == 0) { LBDEM_FUSED_FS(0, true) } else { LBDEM_FUSED_FS(1, true) }
    } else {
        if (b.parity == 0) { LBDEM_FUSED_FS(0, false) } else { LBDEM_FUSED_FS(1, false) }
    }
#undef LBDEM_FUSED_FS
#undef LBDEM_FUSED_Z
#undef LBDEM_FUSED
    if (ev1) (void)hipEventRecord(ev1, s);
    if (b.slipList && b.nSlip > 0) launch_slip<S>(b, k.slipCoef, s);
    b.parity ^= 1;
}

}  // namespace lbdem
