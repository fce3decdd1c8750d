// The launches between two fused kernels up to the particles' integration: the finalisation of the
// fused kernel's sums, the free surface (LB.cpp:1548-1852) and the next step's neighbour list and
// forces (dem.hpp).
//
// The free surface reads and writes the lattice (populations, types, mass, interface lists), the DEM
// step the particles, so the two commute; each is a chain of six short passes, every one of which
// needs all of the previous one. One launch holds the blocks of the n-th pass of either chain: six
// launches in a row instead of two chains on two streams. A graph with two branches is issued kernel
// by kernel by the host (about 4 us each, 88-124 us a step of 30 tiny kernels), a graph without
// branches is handed to the device as a whole (1.6-1.8 us a kernel, 48-52 us a step).
#pragma once
#include "dem.hpp"
#include "lattice.hpp"

namespace lbdem {

// sum of v[0 .. n) over a block of 256 threads, the same on every thread and for every block that
// sums the same values: strided sums per thread (four loads in flight), a wavefront butterfly, then
// the wavefronts in order
constexpr int HF_THREADS = 256;
__device__ inline double block_sum(const double* v, int n, double* red) {
    const int tid = threadIdx.x;
    double acc = 0.0;
    int b = tid;
    for (; b + 3 * HF_THREADS < n; b += 4 * HF_THREADS) {
        const double v0 = v[b], v1 = v[b + HF_THREADS], v2 = v[b + 2 * HF_THREADS], v3 = v[b + 3 * HF_THREADS];
        acc += v0; acc += v1; acc += v2; acc += v3;
    }
    for (; b < n; b += HF_THREADS) acc += v[b];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
    if ((tid & 63) == 0) red[tid / 64] = acc;
    __syncthreads();
    double s = 0.0;
    for (int w = 0; w < HF_THREADS / 64; ++w) s += red[w];
    __syncthreads();
    return s;
}

// the fused kernel's sums: impactors and walls from the blocks' records, one block per column, the
// particles' accumulators, one thread each; unit conversion (LB.cpp:1966-1977, 1536-1543)
struct HydroArgs {
    const double* part;
    int stride;      // of the columns of part
    double* hacc;
    double *FHydro, *MHydro, *fluidVol, *objFH, *objMH, *wallFH;
    int blocks;      // of the finalisation (0: none)
};
__device__ inline void hydro_finalize(const HydroArgs& a, const Consts& k, DevScalars* sc, int blk, double* red) {
    const int tid = threadIdx.x;
    if (blk == 0 && tid == 0) sc->nChanged = sc->fullMark = 0;  // taken by the marking before the fused kernel
    if (blk < PART_STRIDE) {
        const int c = blk;
        const bool obj = c < PART_WALL;
        if (obj && c / 7 >= k.nObj && c != PART_BB) return;            // no such object
        if (!obj && (c - PART_WALL) / 3 >= k.nWall) return;  // no such wall
        const double v = block_sum(a.part + int64_t(c) * a.stride, obj ? sc->nPartObj : sc->nPartWall, red);
        if (tid != 0) return;
        if (obj) {
            const int o = c / 7, comp = c % 7;
            if (o < k.nObj) {
                if (comp < 3) a.objFH[3 * o + comp] = v * k.unitForce;
                else if (comp < 6) a.objMH[3 * o + comp - 3] = v * k.unitTorque;
            }
            if (c == PART_BB) { sc->extraMass = v; sc->lastExtraMass = v; }
        } else {
            const int w = (c - PART_WALL) / 3, comp = (c - PART_WALL) % 3;
            if (w < k.nWall) a.wallFH[3 * w + comp] = v * k.unitForce;
        }
    } else {
        const int p = (blk - PART_STRIDE) * HF_THREADS + tid;
        if (p < k.nPart) {
            double* h = a.hacc + int64_t(p) * 8;
            for (int c = 0; c < 3; ++c) {
                a.FHydro[3 * p + c] = h[c] * k.unitForce;
                a.MHydro[3 * p + c] = h[3 + c] * k.unitTorque;
            }
            a.fluidVol[p] = h[6] * k.unitVolume;
            for (int c = 0; c < 8; ++c) h[c] = 0.0;  // zero for the next LB step's sums
        }
    }
}

// ------------------------------------------------------------------------------------------
// free surface (LB.cpp:1548-1852)
// ------------------------------------------------------------------------------------------
constexpr int FS_THREADS = 256;
static_assert(FS_THREADS == HF_THREADS, "one launch holds the blocks of all passes");

// Entries of a list whose counter went past its capacity (reported as an overflow at the next
// synchronisation) that are there to read.
__device__ inline int list_len(int count, int cap) { return min(count, cap); }

template <typename S>
struct FsArgs {
    Geom g;
    S* f;
    uint8_t* type;
    typename Types<S>::M* mass;
    typename Types<S>::C* aux;
    typename Types<S>::C* visc;
    const int32_t* ifList;
    typename Types<S>::M* newMass;
    int32_t *list2, *filled, *emptied, *newIf, *marker, *changed;
    int* count2;
    DevScalars* sc;
    int cap, changedCap;
    int slipDyn;
    double s1;
    int blocks;  // of each pass (0: no free surface in this launch)
};

// Mass exchange (LB.cpp:1548-1666). Of the fused kernel's sums it needs only the impactors' extra
// mass, which every block adds up for itself from the few hundred records of blocks with impactor
// links (the same value in every block); so it runs beside the finalisation. Its first block also
// resets the counters of the passes that follow (LB.cpp:422-430).
template <typename S, int L>
__device__ inline void fs_mass(const FsArgs<S>& a, const HydroArgs& h, int blk, double* red) {
    using C = typename Types<S>::C;
    using M = typename Types<S>::M;
    const Geom& g = a.g;
    const S* const f = a.f;
    const uint8_t* const type = a.type;
    const M* const mass = a.mass;
    const int32_t* const ifList = a.ifList;
    M* const newMass = a.newMass;
    DevScalars* const sc = a.sc;
    const int nblk = a.blocks, slipDyn = a.slipDyn;
    const double s1 = a.s1;
    if (blk == 0 && threadIdx.x == 0) {
        sc->surplus = 0.0;
        sc->nFilled = sc->nEmptied = sc->nNewIf = 0;
        sc->nIfFinal = 0;
        *a.count2 = 0;
    }
    const int nIf = sc->nIf;
    if (blk * HF_THREADS >= nIf) return;
    const double extra = block_sum(h.part + int64_t(PART_BB) * h.stride, sc->nPartObj, red);
    const double addE = extra / double(nIf);
    const int listed = list_len(nIf, a.cap);
    for (int k = blk * HF_THREADS + threadIdx.x; k < listed; k += nblk * HF_THREADS) {
        const int64_t i = ifList[k];
        int x, y, z;
        cell_xyz(g, i, x, y, z);
        const Offs o(g, x, y, z);
        const C mi = C(double(mass[i]) + addE);
        // every neighbour's type, populations and mass are loaded up front (all addresses are
        // nodes of the box), so the loads overlap; the sum then runs in direction order
        uint8_t ty[Q];
        C a1[Q], a2[Q], mj[Q];
#pragma unroll
        for (int j = 1; j < Q; ++j) {
            const int64_t yj = i + o.d(j);
            ty[j] = type[yj] & T_BASE;
            a1[j] = StoreT<S>::ld(f + int64_t(j) * g.N + yj);
            a2[j] = StoreT<S>::ld(f + int64_t(oppq(j)) * g.N + i);
            mj[j] = C(mass[yj]);
        }
        C dm = 0;
#pragma unroll
        for (int j = 1; j < Q; ++j) {
            const bool slipLink = slipDyn && ty[j] == T_WALL;
            if (ty[j] != T_IF && ty[j] != T_FLUID && ty[j] != T_OBJ && !slipLink) continue;
            const C ms = L == 1 ? (a1[j] - a2[j]) : (a2[j] - a1[j]);  // incoming(opp j) - outgoing(j), offsets
            if (ty[j] == T_IF) dm += C(0.5) * (C(double(mj[j]) + addE) + mi) * ms;
            else if (ty[j] == T_FLUID) dm += ms;
            else if (slipLink) {  // moving slip wall (LB.cpp:1595-1625): (1 - S) of the mass on a slip link
                bool slipped = false;
                if (j > 6) {
                    const uint8_t t1 = ty[slip1Check(j)], t2 = ty[slip2Check(j)];
                    slipped = (t1 == T_FLUID || t1 == T_IF) != (t2 == T_FLUID || t2 == T_IF);
                }
                dm += (slipped ? C(1.0 - s1) * mi : mi) * ms;
            } else {
                dm += mi * ms;
            }
        }
        newMass[k] = M(mi + dm);
    }
}

// assign new mass, classify filled / emptied (findInterfaceMutants, LB.cpp:1669-1698)
template <typename S>
__device__ inline void fs_mutants(const FsArgs<S>& a, int blk) {
    uint8_t* const type = a.type;
    DevScalars* const sc = a.sc;
    const int nIf = list_len(sc->nIf, a.cap);
    for (int k = blk * FS_THREADS + threadIdx.x; k < nIf; k += a.blocks * FS_THREADS) {
        const int64_t i = a.ifList[k];
        const auto m = a.newMass[k];
        a.mass[i] = m;
        const auto n = a.aux[i];
        if (m > n) {
            type[i] = (type[i] & (T_PMASK | T_EDGE)) | T_FLUID;  // active to active: edge bit stays
            a.marker[i] = -3;
            list_push(a.filled, &sc->nFilled, a.cap, int32_t(i), &sc->listOverflow);
        } else if (m < 0) {
            type[i] = (type[i] & T_PMASK) | T_GAS;
            list_push(a.emptied, &sc->nEmptied, a.cap, int32_t(i), &sc->listOverflow);
            push_changed(a.changed, a.changedCap, sc, int32_t(i));
        }
    }
}

// Neighbours of the converted nodes, two independent passes in one launch: a filled node offers itself
// as donor to its gas neighbours, each of which takes the highest-index one and joins the new
// interface nodes (LB.cpp:1704-1728); a fluid neighbour of an emptied node becomes an interface node
// with 99% of its density (LB.cpp:1730-1748). The first reads gas types, which the second does not
// change, and the second fluid types, which the first does not change. Both append to newIf; a node
// from a donor has donor[] >= 0, one from an emptied node a marker below -1.
template <typename S>
__device__ inline void fs_neighbours(const FsArgs<S>& a, int blk) {
    const Geom& g = a.g;
    uint8_t* const type = a.type;
    typename Types<S>::M* const mass = a.mass;
    typename Types<S>::C* const aux = a.aux;
    const int32_t* const filled = a.filled;
    const int32_t* const emptied = a.emptied;
    int32_t* const marker = a.marker;
    int32_t* const newIf = a.newIf;
    DevScalars* const sc = a.sc;
    const int cap = a.cap;
    using C = typename Types<S>::C;
    using M = typename Types<S>::M;
    const int nF = list_len(sc->nFilled, cap), nE = list_len(sc->nEmptied, cap);
    if (blk * FS_THREADS >= nF + nE) return;
    double gained = 0.0;
    for (int k = blk * FS_THREADS + threadIdx.x; k < nF + nE; k += a.blocks * FS_THREADS) {
        const bool isF = k < nF;
        const int64_t i = isF ? filled[k] : emptied[k - nF];
        int x, y, z;
        cell_xyz(g, i, x, y, z);
        const Offs o(g, x, y, z);
        // neighbour types loaded up front so the loads overlap; the marker CAS below decides which
        // thread converts a node, so a type read early changes nothing
        const uint8_t want = isF ? T_GAS : T_FLUID;
        uint32_t mask = 0;
#pragma unroll
        for (int j = 1; j < Q; ++j) mask |= uint32_t((type[i + o.d(j)] & T_BASE) == want) << j;
        for (uint32_t m = mask; m; m &= m - 1u) {  // in direction order
            const int j = __ffs(m) - 1;
            const int64_t l = i + o.d(j);
            if (isF) {
                if (!stencil_in_arrays(g, l)) {  // gas that an impactor left on a z face of the box
                    atomicOr(&sc->typeError, 1);
                    continue;
                }
                const int old = atomicMax(&marker[l], int32_t(i));
                if (old < 0) list_push(newIf, &sc->nNewIf, cap, int32_t(l), &sc->listOverflow);
                continue;
            }
            double nl;
            const int old = atomicCAS(&marker[l], -1, -2);
            if (old == -1) {
                nl = double(mass[l]);               // ordinary fluid node: mass holds its density
            } else if (old == -3 && atomicCAS(&marker[l], -3, -4) == -3) {
                nl = double(aux[l]);                // filled this step: density kept in aux
            } else {
                continue;
            }
            type[l] = (type[l] & (T_PMASK | T_EDGE)) | T_IF;  // active to active: edge bit stays
            mass[l] = M(0.99 * nl);
            aux[l] = C(nl);
            gained += 0.01 * nl;
            list_push(newIf, &sc->nNewIf, cap, int32_t(l), &sc->listOverflow);
        }
    }
    wave_add(&sc->surplus, gained);
}

// The new interface nodes from their donor (node::initialize with the donor's u, visc and
// hydroForce + lbF, mass 0.01 rho0), and updateMutants (LB.cpp:1751-1790) over the filled and
// emptied nodes, which tells by the marker what the type will be: a filled node is still fluid while
// its marker is -3, an emptied node still gas while it has no donor.
template <typename S, int L>
__device__ inline void fs_settle(const FsArgs<S>& a, const Consts& k, int blk) {
    const Geom& g = a.g;
    S* const f = a.f;
    uint8_t* const type = a.type;
    typename Types<S>::M* const mass = a.mass;
    typename Types<S>::C* const aux = a.aux;
    typename Types<S>::C* const visc = a.visc;
    const int32_t* const filled = a.filled;
    const int32_t* const emptied = a.emptied;
    const int32_t* const newIf = a.newIf;
    const int32_t* const marker = a.marker;
    DevScalars* const sc = a.sc;
    int32_t* const changed = a.changed;
    const int changedCap = a.changedCap;
    using C = typename Types<S>::C;
    using M = typename Types<S>::M;
    const int nN = list_len(sc->nNewIf, a.cap), nF = list_len(sc->nFilled, a.cap), nE = list_len(sc->nEmptied, a.cap);
    const int tot = nN + nF + nE;
    if (blk * FS_THREADS >= tot) return;
    const int64_t N = g.N;
    double acc = 0.0;
    for (int kk = blk * FS_THREADS + threadIdx.x; kk < tot; kk += a.blocks * FS_THREADS) {
        if (kk >= nN + nF) {
            const int64_t i = emptied[kk - nN - nF];
            if (marker[i] < 0) acc += double(mass[i]);
            continue;
        }
        if (kk >= nN) {
            const int64_t i = filled[kk - nN];
            if (marker[i] == -3) {
                acc += double(mass[i]) - double(aux[i]);
                mass[i] = M(aux[i]);
            }
            continue;
        }
        const int64_t gi = newIf[kk];
        const int64_t d = marker[gi];
        if (d < 0) continue;  // from an emptied neighbour: complete
        type[gi] = (type[gi] & T_PMASK) | T_IF;
        push_changed(changed, changedCap, sc, int32_t(gi));
        const double n = k.rho0;
        const double ux = (double(aux[4 * N + d]) + k.lbF[0]) / 2.0 / n + double(aux[N + d]);
        const double uy = (double(aux[5 * N + d]) + k.lbF[1]) / 2.0 / n + double(aux[2 * N + d]);
        const double uz = (double(aux[6 * N + d]) + k.lbF[2]) / 2.0 / n + double(aux[3 * N + d]);
        int x, y, z;
        cell_xyz(g, gi, x, y, z);
        const Offs o(g, x, y, z);
        const double usq = ux * ux + uy * uy + uz * uz;
        for (int q = 0; q < Q; ++q) {
            const double vu = ux * cxq(q) + uy * cyq(q) + uz * czq(q);
            const double feq = wq(q) * n * (1.0 + 3.0 * vu + 4.5 * vu * vu - 1.5 * usq);
            StoreT<S>::st(f + load_slot(g, gi, o, q, L), C(feq - wq(q)));
        }
        mass[gi] = M(0.01 * k.rho0);
        acc -= 0.01 * k.rho0;
        aux[gi] = C(n);
        aux[N + gi] = C(ux); aux[2 * N + gi] = C(uy); aux[3 * N + gi] = C(uz);
        aux[4 * N + gi] = C(0); aux[5 * N + gi] = C(0); aux[6 * N + gi] = C(0);
        if (visc) visc[gi] = visc[d];  // the donor's viscosity (LB.cpp:1719)
    }
    wave_add(&sc->surplus, acc);
}

// removeIsolated (LB.cpp:1796-1841): interface nodes without gas neighbours become fluid, then those
// without fluid neighbours become gas. Both in one pass over the interface list after the
// conversions (the old interface nodes left untouched, then the new ones), compacted into list2 for
// the redistribution. A node's first test reads gas types and its second fluid types:
//   * nodes turned to gas are entered in list2 as ~i and change type in the redistribution, so no
//     first test sees them;
//   * a fluid neighbour seen is one before or one from the first test, either of which counts;
//   * a node that sees neither (rare) looks at its interface neighbours for one that the first test
//     turns to fluid, that is one without gas neighbours, which is the same before and after.
// Two passes with a launch between them took 9 and 8 us on the 256x320x256 box.
template <typename S>
__device__ inline void fs_isolated(const FsArgs<S>& a, int blk) {
    const Geom& g = a.g;
    uint8_t* const type = a.type;
    typename Types<S>::M* const mass = a.mass;
    const typename Types<S>::C* const aux = a.aux;
    const int32_t* const ifList = a.ifList;
    const int32_t* const newIf = a.newIf;
    const int32_t* const marker = a.marker;
    int32_t* const list2 = a.list2;
    int* const count2 = a.count2;
    DevScalars* const sc = a.sc;
    const int cap = a.cap;
    const int nIf = list_len(sc->nIf, cap), nN = list_len(sc->nNewIf, cap);
    if (blk * FS_THREADS >= nIf + nN) return;
    __shared__ int sPos[8];
    __shared__ double sSum[8];
    __shared__ int sCnt[8];
    double acc = 0.0;
    int keep = 0;
    // the loop runs the same number of times on every thread of a block (block_reserve)
    for (int k0 = blk * FS_THREADS; k0 < nIf + nN; k0 += a.blocks * FS_THREADS) {
        const int k = k0 + int(threadIdx.x);
        int64_t i = -1;
        if (k < nIf) {
            i = ifList[k];
            if ((type[i] & T_BASE) != T_IF || marker[i] != -1) i = -1;
        } else if (k < nIf + nN) {
            i = newIf[k - nIf];
        }
        bool stay = false, toGas = false;
        if (i >= 0) {
            int x, y, z;
            cell_xyz(g, i, x, y, z);
            const Offs o(g, x, y, z);
            bool gasNb = false, fluidNb = false;
            uint32_t ifNb = 0;
#pragma unroll
            for (int j = 1; j < Q; ++j) {  // the 18 loads overlap
                const uint8_t t = type[i + o.d(j)] & T_BASE;
                gasNb |= t == T_GAS;
                fluidNb |= t == T_FLUID;
                ifNb |= uint32_t(t == T_IF) << j;
            }
            if (!gasNb) {
                acc += double(mass[i]) - double(aux[i]);
                mass[i] = typename Types<S>::M(aux[i]);
                type[i] = (type[i] & (T_PMASK | T_EDGE)) | T_FLUID;  // active to active: edge bit stays
            } else {
                for (uint32_t m = ifNb; m && !fluidNb; m &= m - 1u) {
                    const int64_t l = i + o.d(__ffs(m) - 1);
                    cell_xyz(g, l, x, y, z);
                    const Offs ol(g, x, y, z);
                    bool gas = false;
#pragma unroll
                    for (int j = 1; j < Q; ++j) gas |= (type[l + ol.d(j)] & T_BASE) == T_GAS;
                    fluidNb = !gas;
                }
                stay = fluidNb;
                toGas = !fluidNb;
                if (toGas) acc += double(mass[i]);
                else keep++;
            }
        }
        const int pos = block_reserve(count2, stay || toGas, sPos);
        if (stay || toGas) {
            if (pos < cap) list2[pos] = stay ? int32_t(i) : ~int32_t(i);
            else atomicOr(&sc->listOverflow, 1);
        }
    }
    block_add(&sc->surplus, acc, sSum);
    block_add(&sc->nIfFinal, keep, sCnt);
}

// redistributeMass (LB.cpp:1844-1852), the isolated nodes' change to gas, and the marker reset
struct RedistArgs {  // of FsArgs, for the pass that does not depend on the storage type
    uint8_t* type;
    const int32_t *list2, *filled, *newIf;
    const int* count2;
    int32_t *marker, *changed;
    int cap, changedCap, blocks;
    DevScalars* sc;
};
template <typename M>
__device__ inline void fs_redistribute(const RedistArgs& a, M* mass, int blk) {
    uint8_t* const type = a.type;
    const int32_t* const list2 = a.list2;
    const int32_t* const filled = a.filled;
    const int32_t* const newIf = a.newIf;
    int32_t* const marker = a.marker;
    int32_t* const changed = a.changed;
    const int* const count2 = a.count2;
    const int changedCap = a.changedCap;
    DevScalars* const sc = a.sc;
    const int n2 = list_len(*count2, a.cap);
    const double add = sc->surplus / double(sc->nIfFinal);
    for (int k = blk * FS_THREADS + threadIdx.x; k < n2; k += a.blocks * FS_THREADS) {
        const int32_t v = list2[k];
        if (v >= 0) {
            mass[v] = M(double(mass[v]) + add);
        } else {
            type[~v] = (type[~v] & T_PMASK) | T_GAS;
            push_changed(changed, changedCap, sc, ~v);
        }
    }
    const int nF = list_len(sc->nFilled, a.cap), nN = list_len(sc->nNewIf, a.cap);
    for (int k = blk * FS_THREADS + threadIdx.x; k < nF + nN; k += a.blocks * FS_THREADS)
        marker[k < nF ? filled[k] : newIf[k - nF]] = -1;
    if (blk == 0 && threadIdx.x == 0) sc->lastSurplus = sc->surplus;
}

// ------------------------------------------------------------------------------------------
// the launches
// ------------------------------------------------------------------------------------------
template <typename S, int L>
__device__ inline void k_front1(FsArgs<S> a, HydroArgs h, Consts k, NbrArgs n) {
    __shared__ double red[HF_THREADS / 64];
    int blk = int(blockIdx.x);
    if (blk < h.blocks) return hydro_finalize(h, k, a.sc, blk, red);
    blk -= h.blocks;
    if (blk < a.blocks) return fs_mass<S, L>(a, h, blk, red);
    blk -= a.blocks;
    if (blk < n.pBlocks) nbr_assign(n, blk);
}
template <typename S>
__device__ inline void k_front2(FsArgs<S> a, NbrArgs n) {
    // the one block of the list scan goes first: its loop over the cells is the longest
    int blk = int(blockIdx.x);
    if (blk < n.scanBlocks) return nbr_scan(n);
    blk -= n.scanBlocks;
    if (blk < a.blocks) fs_mutants<S>(a, blk);
}
template <typename S>
__device__ inline void k_front3(FsArgs<S> a, NbrArgs n) {
    int blk = int(blockIdx.x);
    if (blk < a.blocks) return fs_neighbours<S>(a, blk);
    blk -= a.blocks;
    if (blk < n.pBlocks) nbr_fill(n, blk);
}
template <typename S, int L>
__device__ inline void k_front4(FsArgs<S> a, Consts k, NbrArgs n) {
    int blk = int(blockIdx.x);
    if (blk < a.blocks) return fs_settle<S, L>(a, k, blk);
    blk -= a.blocks;
    if (blk < n.buildBlocks) nbr_build(n, blk);
}
template <typename S>
__device__ inline void k_front5(FsArgs<S> a, NbrArgs n) {
    int blk = int(blockIdx.x);
    if (blk < a.blocks) return fs_isolated<S>(a, blk);
    blk -= a.blocks;
    if (blk < n.slotBlocks) nbr_slots(n, blk, n.slotBlocks);
}
template <typename M, bool STRESS, int LANES>
__device__ inline void k_front6(RedistArgs a, M* mass, const ForceArgs& f) {  // (walls indexed by a variable)
    int blk = int(blockIdx.x);
    if (blk < f.blocks) return dem_forces<STRESS, LANES>(f, blk);  // the longer pass first
    blk -= f.blocks;
    if (blk < a.blocks) fs_redistribute<M>(a, mass, blk);
}

// launches of the passes; fs.blocks, h.blocks and the DEM block counts say which are there
template <typename S>
void launch_front(const FsArgs<S>& a, const HydroArgs& h, const Consts& k, const NbrArgs& n, const ForceArgs& f, int L,
                  hipStream_t s);
template <typename M>
void launch_front6(const RedistArgs& r, M* mass, const ForceArgs& f, hipStream_t s);

}  // namespace lbdem
