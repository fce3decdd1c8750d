// Lattice kernels of the coupled step on gfx950:
//   * the fused collide-stream kernel is in fused.hpp; here its boundary-link classes and the
//     finalisation of its sums
//   * free-surface mass exchange and interface conversion (LB.cpp:1548-1852)
//   * particle flags and the moving-object (impactor) node update (LB.cpp:683-711, 797-943,
//     1875-1899, 1980-2029; findNewSolid, LB.cpp:2032-2100, changes no flag)
#include "front.hpp"

#include <utility>

namespace lbdem {

// ------------------------------------------------------------------------------------------
// initial populations (node::initialize, node.cpp:26-73) for fluid and interface nodes
// ------------------------------------------------------------------------------------------
template <typename S>
__device__ inline void k_init_fields(Geom g, S* f, const uint8_t* type, typename Types<S>::M* mass,
                              typename Types<S>::C* aux, typename Types<S>::C* visc, Consts k) {
    using C = typename Types<S>::C;
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= g.N) return;
    const uint8_t t = type[i] & T_BASE;
    if (t != T_FLUID && t != T_IF) return;
    const double n = k.rho0;
    const double ux = k.lbF[0] / 2.0 / n + k.initVel[0];
    const double uy = k.lbF[1] / 2.0 / n + k.initVel[1];
    const double uz = k.lbF[2] / 2.0 / n + k.initVel[2];
    const double usq = ux * ux + uy * uy + uz * uz;
    for (int q = 0; q < Q; ++q) {
        const double vu = ux * cxq(q) + uy * cyq(q) + uz * czq(q);
        const double feq = wq(q) * n * (1.0 + 3.0 * vu + 4.5 * vu * vu - 1.5 * usq);
        StoreT<S>::st(f + int64_t(q) * g.N + i, C(feq - wq(q)));
    }
    mass[i] = typename Types<S>::M(t == T_FLUID ? k.rho0 : 0.5 * k.rho0);
    // density and velocity of every active node (the interface nodes' for the free surface, all
    // of them for a velocity read-back before the first LB step)
    aux[i] = C(n);
    aux[g.N + i] = C(ux); aux[2 * g.N + i] = C(uy); aux[3 * g.N + i] = C(uz);
    aux[4 * g.N + i] = C(0); aux[5 * g.N + i] = C(0); aux[6 * g.N + i] = C(0);
    if (visc) visc[i] = C(k.visc);  // initDynVisc (LB.cpp:1083-1090)
}

// restartVariables (LB.cpp:1098-1138) for record r of the restart file, at active node node[r]:
// populations f = restF, mass = restMass + 1, density n = restN + 1 and velocity u (node::restart,
// node.cpp:38-51, with initDensity 1); hydrodynamic force zero (a fresh node)
template <typename S>
__device__ inline void k_restart_fields(Geom g, S* f, typename Types<S>::M* mass, typename Types<S>::C* aux,
                                        typename Types<S>::C* visc, const double* rec, const int32_t* node, int nrec) {
    using C = typename Types<S>::C;
    const int r = int(blockIdx.x * blockDim.x + threadIdx.x);
    if (r >= nrec) return;
    const int64_t i = node[r];
    const double* v = rec + int64_t(r) * LBDEM_RESTART_REC;
    for (int q = 0; q < Q; ++q) StoreT<S>::st(f + int64_t(q) * g.N + i, C(v[6 + q] - wq(q)));
    mass[i] = typename Types<S>::M(v[4] + 1.0);
    aux[i] = C(v[0] + 1.0);
    aux[g.N + i] = C(v[1]); aux[2 * g.N + i] = C(v[2]); aux[3 * g.N + i] = C(v[3]);
    aux[4 * g.N + i] = C(0); aux[5 * g.N + i] = C(0); aux[6 * g.N + i] = C(0);
    if (visc) visc[i] = C(v[5]);
}
void lb_restart_fields(const Box& b, const double* rec, const int32_t* node, int nrec, hipStream_t s) {
    const int bs = 256, nb = (nrec + bs - 1) / bs;
    if (b.prec == LBDEM_PREC_FP64)
        launch<&k_restart_fields<double>, 1024, 1>(nb, bs, s, b.g, (double*)b.f, (double*)b.mass, (double*)b.aux,
                                                   (double*)b.visc, rec, node, nrec);
    else if (b.prec == LBDEM_PREC_FP32)
        launch<&k_restart_fields<float>, 1024, 1>(nb, bs, s, b.g, (float*)b.f, (float*)b.mass, (float*)b.aux,
                                                  (float*)b.visc, rec, node, nrec);
    else
        launch<&k_restart_fields<__half>, 1024, 1>(nb, bs, s, b.g, (__half*)b.f, (float*)b.mass, (float*)b.aux,
                                                   (float*)b.visc, rec, node, nrec);
}

// node viscosities (the per-node plane), zero at nodes that are not active
template <typename C>
__device__ inline void k_download_visc(int64_t N, const uint8_t* type, const C* visc, double* out) {
    for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < N; i += int64_t(gridDim.x) * blockDim.x)
        out[i] = is_active(type[i]) ? double(visc[i]) : 0.0;
}
void lb_download_visc(const Box& b, double* out, hipStream_t s) {
    if (b.prec == LBDEM_PREC_FP64) launch<&k_download_visc<double>, 1024, 1>(4096, 256, s, b.g.N, b.type, (const double*)b.visc, out);
    else launch<&k_download_visc<float>, 1024, 1>(4096, 256, s, b.g.N, b.type, (const float*)b.visc, out);
}

// velocity of every active node (aux planes 1-3), x y z per node, zero elsewhere
template <typename C>
__device__ inline void k_download_vel(int64_t N, const uint8_t* type, const C* aux, double* out) {
    for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < N; i += int64_t(gridDim.x) * blockDim.x) {
        const bool act = is_active(type[i]);
        for (int a = 0; a < 3; ++a) out[3 * i + a] = act ? double(aux[(1 + a) * N + i]) : 0.0;
    }
}
void lb_download_velocity(const Box& b, double* out, hipStream_t s) {
    if (b.prec == LBDEM_PREC_FP64) launch<&k_download_vel<double>, 1024, 1>(4096, 256, s, b.g.N, b.type, (const double*)b.aux, out);
    else launch<&k_download_vel<float>, 1024, 1>(4096, 256, s, b.g.N, b.type, (const float*)b.aux, out);
}

// SHydro of every particle (LB.cpp:1951-1959): the sum over the active nodes inside it of
// radius (x) diffVel in physical units, with diffVel = -(the node's hydrodynamic force), which the
// LB step just stored in aux planes 4-6 (it runs with every active node's values stored). One
// thread per (x, y) column and run of HS_ZRUN nodes in z walks its run and sums in registers while
// the particle is unchanged; the sums go to the block's LDS table (global atomics when it is
// full), which adds them to the particles once per block.
__device__ inline void k_zero_doubles(double* p, int64_t n) {
    for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += int64_t(gridDim.x) * blockDim.x)
        p[i] = 0.0;
}
constexpr int HS_ZRUN = 16, HS_SLOTS = 128;
__device__ inline void hydro_stress_add(int key, const double* acc, int* hk, double (*hv)[9], double* shydro) {
    int slot = key & (HS_SLOTS - 1), probes = 0;
    for (; probes < HS_SLOTS; ++probes) {
        const int old = atomicCAS(&hk[slot], -1, key);
        if (old == -1 || old == key) break;
        slot = (slot + 1) & (HS_SLOTS - 1);
    }
    if (probes < HS_SLOTS)
        for (int e = 0; e < 9; ++e) atomicAdd(&hv[slot][e], acc[e]);
    else
        for (int e = 0; e < 9; ++e) atomicAdd(shydro + 9 * int64_t(key) + e, acc[e]);
}
template <typename M>
__device__ inline void k_hydro_stress(Geom g, const uint8_t* type, const int32_t* solid, const M* aux,
                                      const PartLB* plb, double L, double F, double* shydro) {
#pragma clang fp contract(off)
    __shared__ int hk[HS_SLOTS];
    __shared__ double hv[HS_SLOTS][9];
    for (int s = threadIdx.x; s < HS_SLOTS; s += blockDim.x) {
        hk[s] = -1;
        for (int e = 0; e < 9; ++e) hv[s][e] = 0.0;
    }
    __syncthreads();
    const int64_t SZ = int64_t(g.X) * g.Y, N = g.N;
    const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    const int64_t col = t % SZ, run = t / SZ;
    const int x = int(col % g.X), y = int(col / g.X);
    const int z0 = int(run) * HS_ZRUN, z1 = min(g.Z, z0 + HS_ZRUN);  // empty past the last run
    int key = -1;
    double acc[9];
    for (int e = 0; e < 9; ++e) acc[e] = 0.0;
    for (int z = z0; z < z1; ++z) {
        const int64_t i = col + SZ * z;
        const uint8_t ty = type[i];
        const int k = (is_active(ty) && (ty & T_PMASK)) ? solid[i] : -1;
        if (k != key) {
            if (key >= 0) hydro_stress_add(key, acc, hk, hv, shydro);
            key = k;
            for (int e = 0; e < 9; ++e) acc[e] = 0.0;
        }
        if (k < 0) continue;
        const PartLB P = plb[k];
        const double r[3] = {double(x) - P.c[0], double(y) - P.c[1], double(z) - P.c[2]};
        const double d[3] = {-double(aux[4 * N + i]), -double(aux[5 * N + i]), -double(aux[6 * N + i])};
        for (int a = 0; a < 3; ++a)
            for (int c = 0; c < 3; ++c) acc[3 * a + c] += r[a] * L * d[c] * F;
    }
    if (key >= 0) hydro_stress_add(key, acc, hk, hv, shydro);
    __syncthreads();
    for (int s = threadIdx.x; s < HS_SLOTS; s += blockDim.x)
        if (hk[s] >= 0)
            for (int e = 0; e < 9; ++e) atomicAdd(shydro + 9 * int64_t(hk[s]) + e, hv[s][e]);
}
void lb_hydro_stress(const Box& b, const PartLB* plb, int nPart, double L, double F, double* shydro, hipStream_t s) {
    const int64_t n9 = 9 * int64_t(nPart > 0 ? nPart : 1);
    launch<&k_zero_doubles, 1024, 1>(int((n9 + 255) / 256), 256, s, shydro, n9);
    if (nPart <= 0) return;
    const int64_t threads = int64_t(b.g.X) * b.g.Y * ((b.g.Z + HS_ZRUN - 1) / HS_ZRUN);
    const int nb = int((threads + 255) / 256);
    if (b.prec == LBDEM_PREC_FP64)
        launch<&k_hydro_stress<double>, 1024, 1>(nb, 256, s, b.g, b.type, b.solid, (const double*)b.aux, plb, L, F, shydro);
    else
        launch<&k_hydro_stress<float>, 1024, 1>(nb, 256, s, b.g, b.type, b.solid, (const float*)b.aux, plb, L, F, shydro);
}

void lb_init_fields(const Box& b, const Consts& k, hipStream_t s) {
    const int bs = 256;
    const int nb = int((b.g.N + bs - 1) / bs);
    if (b.prec == LBDEM_PREC_FP64)
        launch<&k_init_fields<double>, 1024, 1>(nb, bs, s, b.g, (double*)b.f, b.type, (double*)b.mass, (double*)b.aux,
                                                (double*)b.visc, k);
    else if (b.prec == LBDEM_PREC_FP32)
        launch<&k_init_fields<float>, 1024, 1>(nb, bs, s, b.g, (float*)b.f, b.type, (float*)b.mass, (float*)b.aux,
                                               (float*)b.visc, k);
    else
        launch<&k_init_fields<__half>, 1024, 1>(nb, bs, s, b.g, (__half*)b.f, b.type, (float*)b.mass, (float*)b.aux,
                                                (float*)b.visc, k);
}

// ------------------------------------------------------------------------------------------
// edge bits and link classes for the fused kernel, its launch and its sums
// ------------------------------------------------------------------------------------------
// boundary-link classes of the active node i at (x, y, z), over its wrapped neighbours
__device__ inline uint64_t link_classes(const Geom& g, const uint8_t* type, const int32_t* solid, int32_t i, int x,
                                        int y, int z) {
    const Offs o(g, x, y, z);
    uint64_t m = 0;
    int wprim = -1;
    // every neighbour's type and solid index loaded up front, so that the loads overlap: an index
    // loaded only for impactor neighbours is one dependent load after the other (k_mark 8.2 us on a
    // 64^3 box, 15 us on 256x320x256, most of it that)
    uint8_t tfs[Q];
    int32_t sis[Q];
#pragma unroll
    for (int j = 1; j < Q; ++j) {
        tfs[j] = type[i + o.d(j)];
        sis[j] = solid[i + o.d(j)];
    }
#pragma unroll
    for (int j = 1; j < Q; ++j) {
        const uint8_t tf = tfs[j];
        const uint8_t ty = tf & T_BASE;
        uint64_t cls = BC_OTHER;
        if (ty == T_FLUID || ty == T_IF) {
            cls = BC_NONE;
        } else if (ty == T_GAS) {
            cls = BC_GAS;
        } else if (ty == T_WALL) {
            const int w = (tf >> T_WSHIFT) & 7;
            if (wprim < 0) wprim = w;
            cls = w == wprim ? BC_WALL : BC_OTHER;
        } else if (ty == T_OBJ) {
            const int32_t si = sis[j];
            cls = si == 0 ? BC_OBJ0 : (si == 1 ? BC_OBJ1 : BC_OTHER);
        }
        m |= cls << (BC_BITS * (j - 1));
    }
    if (wprim > 0) m |= uint64_t(wprim) << BC_WALL_SHIFT;
    return m;
}

// Edge bits (T_EDGE) and boundary-link classes. An active node is an edge node when some wrapped
// neighbour (D3Q19 stencil) is not active. The full pass runs at initialisation, after a particle
// flag rebuild that cleared wall indices, and when the change list overflowed; otherwise only the
// stencil neighbourhoods of the nodes on the change list are re-marked (only transitions between
// active and non-active types, or among non-active types, change edge bits or classes).
//
// Full pass, rows of a multiple of four bytes: one thread per four nodes of a row (one 32-bit
// word of type bytes). Neighbour rows (wrapped through periodic faces) are read as words; the test
// uses three masks of non-active bytes: the node's own row (x - 1, x + 1), the four rows sharing
// one axis with it (x - 1 .. x + 1) and the four diagonal rows (same x).
__device__ inline uint32_t inactive_bytes(uint32_t w) {
    // a byte is active when its type is 0 (fluid) or 3 (interface); types fit in 4 bits, so the
    // per-byte additions below cannot carry into the next byte
    const uint32_t base = w & 0x0F0F0F0Fu;
    const uint32_t nz0 = (base + 0x7F7F7F7Fu) & 0x80808080u;               // type != 0
    const uint32_t nz3 = ((base ^ 0x03030303u) + 0x7F7F7F7Fu) & 0x80808080u;  // type != 3
    uint32_t m = (nz0 & nz3) >> 7;
    m |= m >> 7;
    m |= m >> 14;
    return m & 0xFu;
}
constexpr int MARK_GRID = 512;  // blocks of k_mark (grid-stride; the full pass is rare)
__device__ __attribute__((always_inline)) inline void mark_full_w(Geom g, uint8_t* type, const int32_t* solid, uint64_t* bcm) {
    const int W = g.X / 4;
    const uint32_t* t32 = reinterpret_cast<const uint32_t*>(type);
    const int64_t total = int64_t(g.Y) * g.Z * W;
    for (int64_t gid = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; gid < total;
         gid += int64_t(gridDim.x) * blockDim.x) {
        const int w = int(gid % W);
        const int64_t row = gid / W;
        const int y = int(row % g.Y), z = int(row / g.Y);
        if (y == 0 || y == g.Y - 1 || z == 0 || z == g.Z - 1) continue;
        const int64_t c0 = row * W + w;
        const uint32_t cw = t32[c0];
        if (inactive_bytes(cw) == 0xFu) continue;  // no active node in this word
        const int ym = (y == 1 && g.per[2]) ? g.Y - 2 : y - 1, yp = (y == g.Y - 2 && g.per[3]) ? 1 : y + 1;
        const int zm = (z == 1 && g.per[4]) ? g.Z - 2 : z - 1, zp = (z == g.Z - 2 && g.per[5]) ? 1 : z + 1;
        auto rowWord = [&](int yy, int zz) { return (int64_t(zz) * g.Y + yy) * W; };
        // 6-bit window of a row: bit 0 = byte x-1, bits 1-4 = the word, bit 5 = byte x+4; bytes of
        // the boundary layer of a periodic x face are replaced by their wrapped partners
        auto window = [&](int64_t rw) {
            uint32_t mid = inactive_bytes(t32[rw + w]);
            if (w == 0 && g.per[0]) {
                const uint32_t b = (t32[rw + W - 1] >> 16) & 0xFFu;  // x = X - 2
                mid = (mid & ~1u) | (is_active(uint8_t(b)) ? 0u : 1u);
            }
            if (w == W - 1 && g.per[1]) {
                const uint32_t b = (t32[rw] >> 8) & 0xFFu;  // x = 1
                mid = (mid & ~8u) | (is_active(uint8_t(b)) ? 0u : 8u);
            }
            const uint32_t lo = w > 0 ? uint32_t(!is_active(uint8_t(t32[rw + w - 1] >> 24))) : 1u;
            const uint32_t hi = w < W - 1 ? uint32_t(!is_active(uint8_t(t32[rw + w + 1]))) : 1u;
            return lo | (mid << 1) | (hi << 5);
        };
        const uint32_t own = window(rowWord(y, z));
        const uint32_t side = window(rowWord(ym, z)) | window(rowWord(yp, z)) | window(rowWord(y, zm)) |
                              window(rowWord(y, zp));
        const uint32_t diag = inactive_bytes(t32[rowWord(ym, zm) + w]) | inactive_bytes(t32[rowWord(ym, zp) + w]) |
                              inactive_bytes(t32[rowWord(yp, zm) + w]) | inactive_bytes(t32[rowWord(yp, zp) + w]);
        uint32_t nw = cw;
        // rolled: one inlined copy of the link-class code keeps the kernel free of calls and scratch
#pragma unroll 1
        for (int k = 0; k < 4; ++k) {
            const uint8_t t = uint8_t(cw >> (8 * k));
            if (!is_active(t)) continue;
            const bool edge = ((own >> k) & 5u) || ((side >> k) & 7u) || ((diag >> k) & 1u);
            const uint8_t nt = edge ? uint8_t(t | T_EDGE) : uint8_t(t & ~T_EDGE);
            nw = (nw & ~(0xFFu << (8 * k))) | (uint32_t(nt) << (8 * k));
            if (edge) bcm[c0 * 4 + k] = link_classes(g, type, solid, int32_t(c0 * 4 + k), 4 * w + k, y, z);
        }
        // other threads read this word concurrently; they only test the type bits, which do not change
        if (nw != cw) reinterpret_cast<uint32_t*>(type)[c0] = nw;
    }
}
// one active node: edge bit and classes from its wrapped neighbours
__device__ inline void mark_node(const Geom& g, uint8_t* type, const int32_t* solid, uint64_t* bcm, int32_t i) {
    const uint8_t t = type[i];
    if (!is_active(t)) return;
    int x, y, z;
    cell_xyz(g, i, x, y, z);
    const uint64_t m = link_classes(g, type, solid, i, x, y, z);
    const bool edge = m != 0;
    if (edge) bcm[i] = m;
    const uint8_t nt = edge ? uint8_t(t | T_EDGE) : uint8_t(t & ~T_EDGE);
    if (nt != t) type[i] = nt;
}
// full pass for rows whose length is not a multiple of four: one thread per node
__device__ inline void mark_full_b(Geom g, uint8_t* type, const int32_t* solid, uint64_t* bcm) {
    for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < g.N; i += int64_t(gridDim.x) * blockDim.x)
        mark_node(g, type, solid, bcm, int32_t(i));
}
// end of the coupling step's flag pass (flags_compute set kminP to INT_MAX) or of its search for the
// lowest flagged node: in the marking of the LB step that was enqueued with the coupling, or in a launch of
// its own. (An LB step without a coupling leaves a list rebuild to the next coupling.)
__device__ inline void couple_end(DevScalars* sc) {
    if (sc->newNeighborList) {
        if (sc->kminP == INT_MAX) sc->kminP = -1;
        sc->newNeighborList = 0;
    } else if (sc->fnaDue) {
        sc->kminP = sc->fnaBest ? INT_MAX - sc->fnaBest : -1;
        sc->fnaDue = sc->fnaBest = 0;
    }
}
__device__ inline void k_couple_end(DevScalars* sc) { couple_end(sc); }

// One launch: the full pass when the full-pass flag is set (initialisation, a flag rebuild that
// clears wall indices, change-list overflow), else the incremental pass: the stencil
// neighbourhood (wrapped) of every node on the change list. A node reached from several changed
// nodes is marked several times with the same result.
__device__ inline void k_mark(Geom g, uint8_t* type, const int32_t* solid, uint64_t* bcm, const int32_t* changed, int cap,
                              int endCoupling, DevScalars* sc) {
    // the fused kernel comes next: its counters start at zero
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        if (endCoupling) couple_end(sc);
        sc->nIf = 0;
        sc->nPartObj = sc->nPartWall = 0;
    }
    if (sc->fullMark) {
        if (g.X % 4 == 0) mark_full_w(g, type, solid, bcm);
        else mark_full_b(g, type, solid, bcm);
        return;
    }
    const int n = min(sc->nChanged, cap);
    for (int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; t < int64_t(n) * Q;
         t += int64_t(gridDim.x) * blockDim.x) {
        const int32_t c = changed[t / Q];
        const int j = int(t % Q);
        int x, y, z;
        cell_xyz(g, c, x, y, z);
        const Offs o(g, x, y, z);
        const int64_t p = int64_t(c) + offs_rt(o, j);
        if (p >= 0 && p < g.N) mark_node(g, type, solid, bcm, int32_t(p));  // (changed boundary-layer nodes)
    }
}

void lb_mark_edges(const Box& b, DevScalars* sc, bool endCoupling, hipStream_t s) {
    launch_gs<&k_mark, 256, 1>(MARK_GRID, 256, s, b.g, b.type, b.solid, b.bcm, b.changed, b.changedCap, endCoupling ? 1 : 0, sc);
    // the list and the full-pass flag are reset by the finalisation of the fused kernel's sums
}

int fused_grid_blocks(const Geom& g, int fz, int prec) {
    const int nseg = (g.X + FX - 1) / FX, nby = (g.Y + FY - 1) / FY, nbz = (g.Z + fz - 1) / fz;
    if (prec != LBDEM_PREC_FP16) return (nseg * g.Y * nbz + FY - 1) / FY;  // row order
    return ((nseg * nby * nbz + 7) / 8) * 8;                              // XCD-spread tiles
}

void lb_fused_step(Box& b, const Consts& k, const PartLB* plb, const ObjLB* olb, DevScalars* sc,
                   bool storeVel, hipStream_t s, hipEvent_t ev0, hipEvent_t ev1) {
    if (b.prec == LBDEM_PREC_FP64) launch_fused<double>(b, k, plb, olb, sc, storeVel, s, ev0, ev1);
    else if (b.prec == LBDEM_PREC_FP32) launch_fused<float>(b, k, plb, olb, sc, storeVel, s, ev0, ev1);
    else launch_fused<__half>(b, k, plb, olb, sc, storeVel, s, ev0, ev1);
}

__device__ inline void k_hydro_finalize(HydroArgs a, Consts k, DevScalars* sc) {
    __shared__ double red[HF_THREADS / 64];
    if (int(blockIdx.x) < a.blocks) hydro_finalize(a, k, sc, int(blockIdx.x), red);
}
static HydroArgs hydro_args(const Box& b, const Consts& k, double* FHydro, double* MHydro, double* fluidVol, double* objFH,
                            double* objMH, double* wallFH) {
    HydroArgs a;
    a.part = b.blockPart; a.stride = part_stride(b.g); a.hacc = b.hacc;
    a.FHydro = FHydro; a.MHydro = MHydro; a.fluidVol = fluidVol; a.objFH = objFH; a.objMH = objMH; a.wallFH = wallFH;
    a.blocks = PART_STRIDE + (k.nPart + HF_THREADS - 1) / HF_THREADS;
    return a;
}

void lb_hydro_finalize(const Box& b, const Consts& k, double* FHydro, double* MHydro, double* fluidVol,
                       DevScalars* sc, double* objFH, double* objMH, double* wallFH, hipStream_t s) {
    const HydroArgs a = hydro_args(b, k, FHydro, MHydro, fluidVol, objFH, objMH, wallFH);
    launch<&k_hydro_finalize, HF_THREADS, 1>(a.blocks, HF_THREADS, s, a, k, sc);
}

// blocks of the free surface's passes over the interface list, which holds about one node per column
// of the box (the passes stride over longer lists)
static int fs_blocks(const Geom& g) {
    const int64_t n = (int64_t(g.X) * g.Z * 5 / 4 + FS_THREADS - 1) / FS_THREADS;
    return int(n < 8 ? 8 : (n > 256 ? 256 : n));
}
template <typename S>
static void front(Box& b, const Consts& k, DevScalars* sc, const HydroArgs& h, bool fs, const NbrArgs& n,
                  const ForceArgs& f, hipStream_t s) {
    FsArgs<S> a;
    a.g = b.g; a.f = (S*)b.f; a.type = b.type;
    a.mass = (typename Types<S>::M*)b.mass; a.aux = (typename Types<S>::C*)b.aux; a.visc = (typename Types<S>::C*)b.visc;
    a.ifList = b.ifList; a.newMass = (typename Types<S>::M*)b.ifNewMass; a.list2 = b.ifList2;
    a.filled = b.filled; a.emptied = b.emptied; a.newIf = b.newIf; a.marker = b.donor; a.changed = b.changed;
    a.count2 = (int*)(b.ifList2 + b.ifCap);  // counter stored after the list
    a.sc = sc; a.cap = b.ifCap; a.changedCap = b.changedCap;
    a.slipDyn = k.slip == 2 ? 1 : 0; a.s1 = k.slipCoef;
    a.blocks = fs ? fs_blocks(b.g) : 0;
    launch_front<S>(a, h, k, n, f, b.parity, s);
}
void lb_front(Box& b, const Consts& k, DevScalars* sc, bool hydro, bool fs, double* FHydro, double* MHydro,
              double* fluidVol, double* objFH, double* objMH, double* wallFH, const DemParams* dp, DemState* ds,
              int demTimeStep, bool forceList, hipStream_t s) {
    HydroArgs h = hydro_args(b, k, FHydro, MHydro, fluidVol, objFH, objMH, wallFH);
    if (!hydro) h.blocks = 0;
    NbrArgs n{};
    ForceArgs f{};
    if (ds && (dp->nPart > 0 || forceList)) {
        n = nbr_args(*dp, *ds, sc, forceList);
        if (!forceList) f = force_args(*dp, *ds, demTimeStep);
    }
    if (b.prec == LBDEM_PREC_FP64) front<double>(b, k, sc, h, fs, n, f, s);
    else if (b.prec == LBDEM_PREC_FP32) front<float>(b, k, sc, h, fs, n, f, s);
    else front<__half>(b, k, sc, h, fs, n, f, s);
    if (f.blocks > 0) std::swap(ds->xiCur, ds->xiNext);
}

// ------------------------------------------------------------------------------------------
// particle flags (LB.cpp:683-711 via 1875-1899; findNewActive LB.cpp:1980-2029)
// ------------------------------------------------------------------------------------------
// One wavefront per particle, over the particle's bounding box: active nodes inside the sphere,
// highest index wins. A node inside particle p and inside a higher-index particle q has
// |c_p - c_q| < r_p + r_q, so q is on p's Verlet list, which this rebuild step built from positions
// one step earlier with a skin of two length units (DEM.cpp:585-627). So p first gathers the
// higher-index partners whose spheres overlap its own (one list entry per lane), then writes every
// node inside its sphere and inside none of them with a plain store: each node gets exactly one
// writer, the highest index (the atomic maximum the list-free path uses gives the same). Without a
// list (no link cell along z, where the reference builds none) the atomic maximum is used.
// Particles are taken in link-cell order when the rebuild sorted them (neighbouring particles
// then share the type lines they read), in one contiguous share of that order per XCD (blocks
// b, b + 8, ... run on one XCD, whose L2 then holds one region). A wavefront walks its box 64 nodes
// per lane step, FLAGS_UNROLL steps at a time so that their type loads are in flight together; the
// sphere test keeps the reference's operations (LB.cpp:705, myvector.cpp:171-175).
constexpr int FLAGS_GRID = 2048, FLAGS_APPLY_GRID = 1024;  // blocks of the flag passes (grid-stride; most steps return early)
constexpr int FLAGS_WAVES = 4;     // wavefronts (particles at a time) per block
constexpr int FLAGS_UNROLL = 6;
__device__ inline void flags_compute(int blk, int nblk, Geom g, const uint8_t* type, const PartLB* plb, int nPart, int32_t* flagNew,
                                DevScalars* sc, const int* nbrCount, const int* nbrList, int useList,
                                const int* order) {
    if (blk == 0 && threadIdx.x == 0) sc->kminP = INT_MAX;  // lowest flagged index, from flags_apply
    __shared__ double sq[FLAGS_WAVES][NBR_CAP][4];  // centre and radius of overlapping higher-index partners
    const int wv = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6), lane = int(threadIdx.x) & 63;
    double(*hq)[4] = sq[wv];
    const int dims[3] = {g.X, g.Y, g.Z};
    // this wavefront's particles: positions k0, k0 + step, ... below k1 of the (sorted) order
    int k0 = blk * FLAGS_WAVES + wv, k1 = nPart, step = nblk * FLAGS_WAVES;
    if (nblk % 8 == 0) {
        const int share = (nPart + 7) / 8, xcd = blk % 8;
        k0 = xcd * share + (blk / 8) * FLAGS_WAVES + wv;
        k1 = min(nPart, (xcd + 1) * share);
        step = (nblk / 8) * FLAGS_WAVES;
    }
    for (int k = k0; k < k1; k += step) {
        const int p = order ? order[k] : k;
        const PartLB P = plb[p];
        int nHigher = 0;
        if (useList) {
            const int cnt = nbrCount[p];  // at most NBR_CAP - 1 entries: one lane each
            bool keep = false;
            double qc[4] = {0.0, 0.0, 0.0, 0.0};
            if (lane < cnt) {
                const int q = nbrList[p * NBR_CAP + lane];
                if (q > p) {
                    const PartLB Qp = plb[q];
                    const double dx = Qp.c[0] - P.c[0], dy = Qp.c[1] - P.c[1], dz = Qp.c[2] - P.c[2];
                    const double rs = P.r + Qp.r + 1e-9;  // a margin: a spare candidate only costs a test
                    keep = dx * dx + dy * dy + dz * dz < rs * rs;
                    qc[0] = Qp.c[0]; qc[1] = Qp.c[1]; qc[2] = Qp.c[2]; qc[3] = Qp.r;
                }
            }
            const uint64_t m = __ballot(keep);
            // the previous particle's reads of hq are done (LDS requests of a wavefront complete in order)
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            if (keep) {
                const int slot = __popcll(m & ((uint64_t(1) << lane) - 1));
                hq[slot][0] = qc[0]; hq[slot][1] = qc[1]; hq[slot][2] = qc[2]; hq[slot][3] = qc[3];
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            nHigher = __popcll(m);
        }
        int lo[3], hi[3];
        for (int ax = 0; ax < 3; ++ax) {
            lo[ax] = int(floor(P.c[ax] - P.r)) - 1;
            hi[ax] = int(ceil(P.c[ax] + P.r)) + 1;
            lo[ax] = lo[ax] < 0 ? 0 : lo[ax];
            hi[ax] = hi[ax] > dims[ax] - 1 ? dims[ax] - 1 : hi[ax];
        }
        if (lo[0] > hi[0] || lo[1] > hi[1] || lo[2] > hi[2]) continue;
        const int nx = hi[0] - lo[0] + 1, ny = hi[1] - lo[1] + 1, nxy = nx * ny, tot = nxy * (hi[2] - lo[2] + 1);
        // node c = lane + 64 j of the box, as (x, y, z) offsets advanced by 64 nodes per step
        const int sx = 64 % nx, sy = (64 / nx) % ny, sz = 64 / nxy;
        int ox = lane % nx, oy = (lane / nx) % ny, oz = lane / nxy;
        for (int c0 = 0; c0 < tot; c0 += 64 * FLAGS_UNROLL) {
            int64_t idx[FLAGS_UNROLL];
            bool in[FLAGS_UNROLL];
            uint8_t t[FLAGS_UNROLL];
#pragma unroll
            for (int u = 0; u < FLAGS_UNROLL; ++u) {
                const int x = lo[0] + ox, y = lo[1] + oy, z = lo[2] + oz;
                const bool ok = c0 + 64 * u + lane < tot;
                idx[u] = cidx(g, ok ? x : lo[0], ok ? y : lo[1], ok ? z : lo[2]);
                t[u] = type[idx[u]];
                in[u] = ok && inside_sphere(x, y, z, P.c[0], P.c[1], P.c[2], P.r);
                if (in[u] && useList)
                    for (int j = 0; j < nHigher && in[u]; ++j)
                        in[u] = !inside_sphere(x, y, z, hq[j][0], hq[j][1], hq[j][2], hq[j][3]);
                ox += sx;
                const int cy = ox >= nx ? 1 : 0;
                ox -= cy * nx;
                oy += sy + cy;
                const int cz = oy >= ny ? 1 : 0;
                oy -= cz * ny;
                oz += sz + cz;
            }
#pragma unroll
            for (int u = 0; u < FLAGS_UNROLL; ++u) {
                if (!in[u] || !is_active(t[u])) continue;
                if (useList) flagNew[idx[u]] = p;
                else atomicMax(&flagNew[idx[u]], p);
            }
        }
    }
}

// clear every flag and solid index, apply the new flags (initializeParticleBoundaries)
__device__ inline void flags_apply(int blk, int nblk, int64_t N, uint8_t* type, int32_t* solid, int32_t* flagNew,
                                   DevScalars* sc, int32_t* changed, int changedCap) {
    __shared__ int bmin;
    if (threadIdx.x == 0) bmin = INT_MAX;
    __syncthreads();
    int mymin = INT_MAX;
    bool remark = false;  // a cleared wall index: link classes need a full pass
    for (int64_t i = int64_t(blk) * 256 + threadIdx.x; i < N; i += int64_t(nblk) * 256) {
        const int32_t s = flagNew[i];
        const uint8_t t = type[i];
        // an object node's index is part of its neighbours' link classes: re-mark around it
        // (a node covered by an impactor after the flags were computed takes a particle index)
        const bool obj = (t & T_BASE) == T_OBJ;
        if (s >= 0) {
            if (obj && solid[i] != s) push_changed(changed, changedCap, sc, int32_t(i));
            type[i] = uint8_t(t | T_PMASK);  // flagged nodes were active: the edge bit stays
            solid[i] = s;
            flagNew[i] = -1;
            mymin = min(mymin, int(i));
        } else {
            // active nodes keep their edge bit; other nodes lose the flag and a wall index
            const uint8_t nt = is_active(t) ? uint8_t(t & ~T_PMASK) : uint8_t(t & T_BASE);
            if (!is_active(t) && (t & 0x70)) remark = true;
            if (obj && solid[i] != 0) push_changed(changed, changedCap, sc, int32_t(i));
            if (nt != t) type[i] = nt;
            solid[i] = 0;
        }
    }
    if (__syncthreads_or(remark) && threadIdx.x == 0) atomicOr(&sc->fullMark, 1);
    if (mymin != INT_MAX) atomicMin(&bmin, mymin);
    __syncthreads();
    // blocks run roughly in index order: only a smaller minimum needs the global atomic
    if (threadIdx.x == 0 && bmin != INT_MAX &&
        bmin < __hip_atomic_load(&sc->kminP, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
        atomicMin(&sc->kminP, bmin);
}

// findNewActive (LB.cpp:1980-2029): when the lowest flagged node has left its particle, the flagged nodes
// below the first one still inside its own lose their flag, and that one is the lowest from then on. No
// node below the lowest is flagged. The search (in the coupling's first launch) takes stripes of 16 384
// nodes upwards from it, one per block and round; a block stops once a lower stripe has a hit, so that
// a search that ends a few thousand nodes on, in the same sphere or the next, costs one round, and one
// that runs through the whole box, as when the only spheres low in the box leave it through a periodic
// face, runs on every compute unit: a step with such a search of a 256x320x256 box takes 0.69 ms, as the
// steps beside it, and 3.2 ms with one block. The flags go in the coupling's last launch (fna_unflag). In
// between only the cover pass changes what the search reads, the index of the nodes an impactor covers,
// which the search takes as they will be. A step that rebuilt the flags has nothing to do: every flag was
// set from this step's positions.
constexpr int FNA_WORDS = 16;       // words of four type bytes per thread and round
constexpr int FNA_MAX_BLOCKS = 256; // one per compute unit
constexpr int FNA_STRIPE = 256 * FNA_WORDS * 4;  // nodes of a block's round
__device__ inline int inside_which(int x, int y, int z, const ObjLB* olb, int nObj) {
    int which = -1;
    for (int o = 0; o < nObj; ++o)
        if (inside_sphere(x, y, z, olb[o].c[0], olb[o].c[1], olb[o].c[2], olb[o].r)) which = o;
    return which;
}
// word w of the type bytes, the last N % 4 of them as one short word
__device__ inline uint32_t type_word(const uint8_t* type, int64_t N, int64_t w) {
    const int64_t nw = N / 4;
    if (w < nw) return reinterpret_cast<const uint32_t*>(type)[w];
    uint32_t t = 0;
    if (w == nw)
        for (int64_t i = 4 * nw; i < N; ++i) t |= uint32_t(type[i]) << (8 * int(i - 4 * nw));
    return t;
}
__device__ inline void fna_scan(int blk, int nblk, const Geom& g, const uint8_t* type, const int32_t* solid, const PartLB* plb,
                                int nPart, const ObjLB* olb, int nObj, DevScalars* sc) {
    __shared__ int sBest, sStop;
    const int kp = sc->kminP;
    if (kp < 0) return;
    auto inside = [&](int64_t i) {
        int x, y, z;
        cell_xyz(g, i, x, y, z);
        int sp = inside_which(x, y, z, olb, nObj);  // (the cover pass stores the impactor's index)
        if (sp < 0) sp = solid[i];
        if (sp < 0 || sp >= nPart) return false;
        const PartLB P = plb[sp];
        return inside_sphere(x, y, z, P.c[0], P.c[1], P.c[2], P.r);
    };
    if (inside(kp)) return;
    if (blk == 0 && threadIdx.x == 0) sc->fnaDue = 1;
    for (int64_t w0 = kp / 4 + int64_t(blk) * (FNA_STRIPE / 4); 4 * w0 < g.N; w0 += int64_t(nblk) * (FNA_STRIPE / 4)) {
        if (threadIdx.x == 0) {
            const int best = __hip_atomic_load(&sc->fnaBest, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            sStop = best > 0 && INT_MAX - best < 4 * w0;
            sBest = 0;
        }
        __syncthreads();
        if (sStop) break;
        uint32_t t[FNA_WORDS];
#pragma unroll
        for (int u = 0; u < FNA_WORDS; ++u) t[u] = type_word(type, g.N, w0 + int64_t(u) * 256 + threadIdx.x);
        int mymin = INT_MAX;
        for (int u = 0; u < FNA_WORDS && mymin == INT_MAX; ++u)
            for (uint32_t m = t[u] & 0x80808080u; m && mymin == INT_MAX; m &= m - 1u) {
                const int64_t i = 4 * (w0 + int64_t(u) * 256 + threadIdx.x) + (__ffs(m) - 1) / 8;
                if (inside(i)) mymin = int(i);
            }
        if (mymin != INT_MAX) atomicMax(&sBest, INT_MAX - mymin);
        __syncthreads();
        const int best = sBest;
        if (best == 0) continue;
        if (threadIdx.x == 0) atomicMax(&sc->fnaBest, best);
        break;
    }
}
__device__ inline void fna_unflag(int blk, int nblk, int64_t N, uint8_t* type, int32_t* solid, const DevScalars* sc) {
    if (!sc->fnaDue) return;
    const int64_t end = sc->fnaBest ? int64_t(INT_MAX - sc->fnaBest) : N;
    for (int64_t w = sc->kminP / 4 + int64_t(blk) * 256 + threadIdx.x; 4 * w < end; w += int64_t(nblk) * 256)
        for (uint32_t m = type_word(type, N, w) & 0x80808080u; m; m &= m - 1u) {
            const int64_t i = 4 * w + (__ffs(m) - 1) / 8;
            if (i < end) { type[i] &= uint8_t(~T_PMASK); solid[i] = 0; }
        }
}

// ------------------------------------------------------------------------------------------
// impactor nodes (updateObjectBoundaries + findNewActiveObject, LB.cpp:797-943)
// ------------------------------------------------------------------------------------------
// uncovered object nodes (LB.cpp:846-943). The previous object nodes (ascending list) that the
// moved sphere no longer covers become fluid, interface or gas nodes. Pass 1 (obj_uncover_find,
// many blocks) compacts them in ascending order, each block over its slice of the list. Each
// conversion reads the node types its predecessors in that order wrote, so pass 2
// (k_obj_uncover, one block) takes the candidates in chunks of UNC_CHUNK: it stages their neighbour types in LDS, finds
// neighbours that are candidates of the chunk through a hash table, decides the new types (see
// below) and writes a chunk's results back before the next chunk stages its neighbourhood.
constexpr int UNCOVER_THREADS = 1024, UNC_CHUNK = 1024;
constexpr int UNC_MAX_BLOCKS = UNCOVER_BLOCKS_MAX, UNC_NODES_PER_BLOCK = 1024, FIND_THREADS = 256;
constexpr int UNC_HASH = 2048;  // open-addressing table of a chunk's candidates (at most half full)
__device__ inline uint32_t unc_hash(int32_t key) { return (uint32_t(key) * 2654435761u) >> (32 - 11); }
__device__ inline uint8_t uncover_type(bool anyFluid, bool anyGas) {
    return !anyFluid ? uint8_t(T_GAS) : (anyGas ? uint8_t(T_IF) : uint8_t(T_FLUID));
}
__device__ inline int block_exclusive_scan(int v, int* sWave, int& total) {
    const int lane = __lane_id(), wave = threadIdx.x / 64, nw = blockDim.x / 64;
    int incl = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int o = __shfl_up(incl, d, 64);
        if (lane >= d) incl += o;
    }
    if (lane == 63) sWave[wave] = incl;
    __syncthreads();
    if (threadIdx.x == 0) {
        int acc = 0;
        for (int w = 0; w < nw; ++w) { const int c = sWave[w]; sWave[w] = acc; acc += c; }
        sWave[nw] = acc;
    }
    __syncthreads();
    const int r = sWave[wave] + incl - v;
    total = sWave[nw];
    __syncthreads();
    return r;
}

// pass 1: ordered compaction of the nodes of each block's slice of the list that left the sphere,
// into the same slice of cand
__device__ inline void obj_uncover_find(int blk, Geom g, const int32_t* objList, int32_t* cand, int* blockCount, int G,
                                        const DevScalars* sc, const ObjLB* olb) {
    __shared__ int sWave[FIND_THREADS / 64 + 1];
    const int tid = threadIdx.x;
    const int n = sc->nObjList;
    const int per = (n + G - 1) / G;
    const ObjLB O = olb[0];
    const int beg = min(n, blk * per), end = min(n, beg + per);
    int m = 0;
    for (int base = beg; base < end; base += FIND_THREADS) {
        const int kk = base + tid;
        int32_t i = 0;
        int flag = 0;
        if (kk < end) {
            i = objList[kk];
            int x, y, z;
            cell_xyz(g, i, x, y, z);
            flag = !inside_sphere(x, y, z, O.c[0], O.c[1], O.c[2], O.r);
        }
        int tot;
        const int pos = block_exclusive_scan(flag, sWave, tot);
        if (flag) cand[beg + m + pos] = i;
        m += tot;
    }
    if (tid == 0) blockCount[blk] = m;
}

// pass 2 (one block): the candidates of the G slices in order
template <typename S, int L>
__device__ inline void k_obj_uncover(Geom g, S* f, uint8_t* type,
                                                                 typename Types<S>::M* mass,
                                                                 typename Types<S>::C* aux, typename Types<S>::C* visc,
                                                                 const int32_t* cand, const int* blockCount, int G,
                                                                 DevScalars* sc, Consts k, int32_t* changed, int changedCap) {
    using C = typename Types<S>::C;
    __shared__ int sWave[UNCOVER_THREADS / 64 + 1];
    __shared__ uint8_t nbT[Q - 1][UNC_CHUNK];   // neighbour base types (values before this pass)
    __shared__ uint8_t newT[UNC_CHUNK];
    __shared__ int32_t sCand[UNC_CHUNK];
    __shared__ int32_t hKey[UNC_HASH];          // chunk candidates: node index -> position
    __shared__ int16_t hPos[UNC_HASH];
    __shared__ int sPre[UNC_MAX_BLOCKS + 1];   // exclusive prefix of the slices' candidate counts
    __shared__ uint8_t ownT[UNC_CHUNK];        // the candidates' own types (staged with the neighbours')
    __shared__ int sChBase;                    // the chunk's first slot on the change list
    const int tid = threadIdx.x;
    const int n = sc->nObjList;
    const int per = (n + G - 1) / G;
    {
        const int c = tid < G ? blockCount[tid] : 0;
        int tot;
        const int ex = block_exclusive_scan(c, sWave, tot);
        if (tid < G) sPre[tid] = ex;
        if (tid == 0) sPre[G] = tot;
    }
    __syncthreads();
    const int m = sPre[G];
    // pass 2: candidates in ascending node order, in chunks; a candidate's new type depends on
    // the new types of earlier candidates among its neighbours (the reference's sequential order)
    for (int c0 = 0; c0 < m; c0 += UNC_CHUNK) {
        const int cnt = min(UNC_CHUNK, m - c0);
        if (tid < cnt) {
            const int q = c0 + tid;
            int lo = 0, hi = G - 1;  // block b with sPre[b] <= q < sPre[b + 1]
            while (lo < hi) {
                const int mid = (lo + hi + 1) >> 1;
                if (sPre[mid] <= q) lo = mid; else hi = mid - 1;
            }
            sCand[tid] = cand[min(n, lo * per) + (q - sPre[lo])];
        }
        for (int h = tid; h < UNC_HASH; h += UNCOVER_THREADS) hKey[h] = -1;
        __syncthreads();
        if (tid < cnt) {  // position of every candidate, by node index
            const int32_t key = sCand[tid];
            for (uint32_t h = unc_hash(key);; h = (h + 1) & (UNC_HASH - 1))
                if (atomicCAS(&hKey[h], -1, key) == -1) { hPos[h] = int16_t(tid); break; }
        }
        if (tid == 0) sChBase = atomicAdd(&sc->nChanged, cnt);  // every candidate goes on the change list
        if (tid < cnt) {
            const int32_t i = sCand[tid];
            int x, y, z;
            cell_xyz(g, i, x, y, z);
            uint8_t nt[Q];  // the 19 loads are issued together, then written to LDS
            nt[0] = type[i];
#pragma unroll
            for (int j = 1; j < Q; ++j) nt[j] = type[nbr_plain(g, x, y, z, j)] & T_BASE;
            ownT[tid] = nt[0];
#pragma unroll
            for (int j = 1; j < Q; ++j) nbT[j - 1][tid] = nt[j];
        }
        __syncthreads();
        // The new type of candidate t: gas without a fluid neighbour, interface with fluid and gas
        // neighbours, fluid otherwise, over the types its neighbours have when the reference
        // reaches t (earlier candidates converted, later ones still object nodes). One wavefront
        // takes 64 candidates at a time: types of earlier groups are final; dependencies inside
        // the group are resolved by repeating the decision with the group's current types until
        // none changes. On the dependency order (a candidate depends on earlier ones only) the
        // only fixed point is the sequential result, reached after at most depth + 1 rounds.
        if (tid < 64) {
            const int lane = tid;
            for (int s0 = 0; s0 < cnt; s0 += 64) {
                const int t = s0 + lane;
                const bool valid = t < cnt;
                bool baseF = false, baseG = false;
                uint64_t dep = 0;
                if (valid) {
                    int x, y, z;
                    cell_xyz(g, sCand[t], x, y, z);
                    for (int j = 1; j < Q; ++j) {
                        const int32_t nb = int32_t(nbr_plain(g, x, y, z, j));
                        int pos = -1;
                        for (uint32_t h = unc_hash(nb);; h = (h + 1) & (UNC_HASH - 1)) {
                            const int32_t kk = hKey[h];
                            if (kk == nb) { pos = hPos[h]; break; }
                            if (kk == -1) break;
                        }
                        uint8_t ty = nbT[j - 1][t];
                        if (pos >= 0 && pos < t) {
                            if (pos < s0) ty = newT[pos];
                            else { dep |= 1ull << (pos - s0); continue; }
                        }
                        baseF |= ty == T_FLUID;
                        baseG |= ty == T_GAS;
                    }
                }
                uint8_t myT = uncover_type(baseF, baseG);
                for (int round = 0; round <= 64; ++round) {
                    const uint64_t fm = __ballot(valid && myT == T_FLUID);
                    const uint64_t gm = __ballot(valid && myT == T_GAS);
                    const uint8_t nt = uncover_type(baseF || (dep & fm), baseG || (dep & gm));
                    const uint64_t ch = __ballot(valid && nt != myT);
                    myT = nt;
                    if (!ch) break;
                }
                if (valid) newT[t] = myT;
                __threadfence_block();  // the next group of this wavefront reads these
            }
        }
        __syncthreads();
        if (tid < cnt) {
            const int32_t i = sCand[tid];
            uint8_t nt = newT[tid];
            if (nt != T_GAS && !stencil_in_arrays(g, i)) {  // left behind on a z face of the box
                nt = T_GAS;
                atomicOr(&sc->typeError, 1);
            }
            type[i] = uint8_t((ownT[tid] & T_PMASK) | nt);  // no other thread writes a candidate's type
            const int pos = sChBase + tid;
            if (pos < changedCap) changed[pos] = i;
            else atomicOr(&sc->fullMark, 1);
            if (nt != T_GAS) {
                const bool isIf = nt == T_IF;
                int x, y, z;
                cell_xyz(g, i, x, y, z);
                const double nn = k.rho0;
                const double ux = k.lbF[0] / 2.0 / nn + (isIf ? 0.0 : k.initVel[0]);
                const double uy = k.lbF[1] / 2.0 / nn + (isIf ? 0.0 : k.initVel[1]);
                const double uz = k.lbF[2] / 2.0 / nn + (isIf ? 0.0 : k.initVel[2]);
                const double usq = ux * ux + uy * uy + uz * uz;
                const Offs o(g, x, y, z);
                for (int q = 0; q < Q; ++q) {
                    const double vu = ux * cxq(q) + uy * cyq(q) + uz * czq(q);
                    const double feq = wq(q) * nn * (1.0 + 3.0 * vu + 4.5 * vu * vu - 1.5 * usq);
                    StoreT<S>::st(f + load_slot(g, i, o, q, L), C(feq - wq(q)));
                }
                mass[i] = typename Types<S>::M(isIf ? 0.5 * k.rho0 : k.rho0);
                aux[i] = C(nn);
                aux[g.N + i] = C(ux); aux[2 * g.N + i] = C(uy); aux[3 * g.N + i] = C(uz);
                aux[4 * g.N + i] = C(0); aux[5 * g.N + i] = C(0); aux[6 * g.N + i] = C(0);
                if (visc) visc[i] = C(k.visc);  // initDynVisc (LB.cpp:928-934)
            }
        }
        __threadfence_block();
        __syncthreads();
    }
}

// cover: every node inside an object sphere becomes an object node; ascending object node list.
// Pass a covers the union box of the spheres and counts per block (blocks own consecutive
// ranges of the box); pass b writes the list at the blocks' exclusive prefix offsets.
constexpr int COVER_BS = 256;
struct CoverBox {
    int lo[3], n[3], tot;
};
__device__ inline CoverBox cover_box(const Geom& g, const ObjLB* olb, int nObj) {
    int lo[3] = {INT_MAX, INT_MAX, INT_MAX}, hi[3] = {INT_MIN, INT_MIN, INT_MIN};
    const int dims[3] = {g.X, g.Y, g.Z};
    for (int o = 0; o < nObj; ++o)
        for (int a = 0; a < 3; ++a) {
            const int l = int(floor(olb[o].c[a] - olb[o].r)) - 1, h = int(ceil(olb[o].c[a] + olb[o].r)) + 1;
            lo[a] = min(lo[a], max(l, 0));
            hi[a] = max(hi[a], min(h, dims[a] - 1));
        }
    CoverBox b;
    for (int a = 0; a < 3; ++a) { b.lo[a] = lo[a]; b.n[a] = max(hi[a] - lo[a] + 1, 0); }
    b.tot = b.n[0] * b.n[1] * b.n[2];
    return b;
}
__device__ inline void k_obj_cover_a(int G, Geom g, uint8_t* type, int32_t* solid, const ObjLB* olb,
                                                          int nObj, int* blockCount, int32_t* seg, int segCap,
                                                          int32_t* changed, int changedCap, DevScalars* sc) {
    if (int(blockIdx.x) >= G) return;  // G: the box's grid
    __shared__ int sWave[COVER_BS / 64 + 1];
    const CoverBox cb = cover_box(g, olb, nObj);
    const int per = (cb.tot + G - 1) / G;
    const int beg = min(cb.tot, int(blockIdx.x) * per), end = min(cb.tot, beg + per);
    const bool segmented = cb.tot <= segCap;  // the block's nodes go to seg[beg ...] in order
    int cnt = 0;
    for (int c0 = beg; c0 < end; c0 += COVER_BS) {
        const int c = c0 + threadIdx.x;
        int in = 0;
        int64_t i = 0;
        if (c < end) {
            const int x = cb.lo[0] + c % cb.n[0], y = cb.lo[1] + (c / cb.n[0]) % cb.n[1], z = cb.lo[2] + c / (cb.n[0] * cb.n[1]);
            const int which = inside_which(x, y, z, olb, nObj);
            if (which >= 0) {
                i = cidx(g, x, y, z);
                const uint8_t t = type[i];
                // the link classes of neighbouring edge nodes hold the type and the object index
                if ((t & T_BASE) != T_OBJ || solid[i] != which) push_changed(changed, changedCap, sc, int32_t(i));
                type[i] = uint8_t((t & T_PMASK) | T_OBJ);
                solid[i] = which;
                in = 1;
            }
        }
        if (segmented) {
            int tot;
            const int pos = block_exclusive_scan(in, sWave, tot);
            if (in) seg[beg + cnt + pos] = int32_t(i);
            cnt += tot;
        } else {
            cnt += __syncthreads_count(in);
        }
    }
    if (threadIdx.x == 0) blockCount[blockIdx.x] = cnt;
}
// the object node list: every block's nodes at the exclusive prefix of the block counts
__device__ inline void obj_cover_b(int blk, int G, Geom g, const uint8_t* type, const ObjLB* olb, int nObj,
                                                          const int* blockCount, const int32_t* seg, int segCap,
                                                          int32_t* objList, int cap, DevScalars* sc) {
    __shared__ int sWave[COVER_BS / 64 + 1];
    __shared__ int sOff, sTot;
    const CoverBox cb = cover_box(g, olb, nObj);
    {
        int before = 0, all = 0;
        for (int b = threadIdx.x; b < G; b += COVER_BS) {
            const int v = blockCount[b];
            all += v;
            if (b < blk) before += v;
        }
        int t1, t2;
        (void)block_exclusive_scan(before, sWave, t1);
        (void)block_exclusive_scan(all, sWave, t2);
        if (threadIdx.x == 0) { sOff = t1; sTot = t2; }
        __syncthreads();
    }
    if (blk == 0 && threadIdx.x == 0) {
        sc->nObjList = sTot < cap ? sTot : cap;
        if (sTot > cap) sc->listOverflow |= 1;
    }
    int off = sOff;
    const int per = (cb.tot + G - 1) / G;
    const int beg = min(cb.tot, blk * per), end = min(cb.tot, beg + per);
    if (cb.tot <= segCap) {
        const int cnt = blockCount[blk];
        for (int k = threadIdx.x; k < cnt; k += COVER_BS)
            if (off + k < cap) objList[off + k] = seg[beg + k];
        return;
    }
    // union box larger than the staging buffer (impactors far apart): scan the box again
    for (int c0 = beg; c0 < end; c0 += COVER_BS) {
        const int c = c0 + threadIdx.x;
        int in = 0;
        int64_t i = 0;
        if (c < end) {
            const int x = cb.lo[0] + c % cb.n[0], y = cb.lo[1] + (c / cb.n[0]) % cb.n[1], z = cb.lo[2] + c / (cb.n[0] * cb.n[1]);
            i = cidx(g, x, y, z);
            in = (type[i] & T_BASE) == T_OBJ && inside_which(x, y, z, olb, nObj) >= 0;
        }
        int tot;
        const int pos = block_exclusive_scan(in, sWave, tot);
        if (in && off + pos < cap) objList[off + pos] = int32_t(i);
        off += tot;
    }
}

// First launch of the coupling: the particle flags of a list rebuild, or findNewActive's search, and the
// nodes the impactor left (none reads what another writes; all read the types before the impactor's nodes
// change).
struct CoupleArgs {
    Geom g;
    uint8_t* type;
    int32_t *solid, *flagNew, *objList, *objCand, *changed;
    int *coverCount, *uncCount;
    const PartLB* plb;
    const ObjLB* olb;
    DevScalars* sc;
    const int *nbrCount, *nbrList, *order;
    int nPart, nObj, useList, objCap, changedCap;
    int flagBlocks, scanBlocks, findBlocks, coverBlocks, applyBlocks;
};
__device__ inline void k_couple_first(CoupleArgs a) {
    int blk = int(blockIdx.x);
    const int flags = max(a.flagBlocks, a.scanBlocks);
    if (blk < flags) {
        if (a.sc->newNeighborList) {
            if (blk < a.flagBlocks)
                flags_compute(blk, a.flagBlocks, a.g, a.type, a.plb, a.nPart, a.flagNew, a.sc, a.nbrCount, a.nbrList, a.useList,
                              a.order);
        } else if (blk < a.scanBlocks) {
            fna_scan(blk, a.scanBlocks, a.g, a.type, a.solid, a.plb, a.nPart, a.olb, a.nObj, a.sc);
        }
        return;
    }
    blk -= flags;
    if (blk < a.findBlocks) obj_uncover_find(blk, a.g, a.objList, a.objCand, a.uncCount, a.findBlocks, a.sc, a.olb);
}
// Last launch: the impactor's node list and the new flags, or the flags that findNewActive takes away. The
// list is made from the cover pass's counts and reads base types at most, so the two do not meet.
__device__ inline void k_couple_last(CoupleArgs a) {
    int blk = int(blockIdx.x);
    if (blk < a.coverBlocks)
        return obj_cover_b(blk, a.coverBlocks, a.g, a.type, a.olb, a.nObj, a.coverCount, a.objCand, a.objCap, a.objList,
                           a.objCap, a.sc);
    blk -= a.coverBlocks;
    if (blk < a.applyBlocks) {
        if (a.sc->newNeighborList)
            flags_apply(blk, a.applyBlocks, a.g.N, a.type, a.solid, a.flagNew, a.sc, a.changed, a.changedCap);
        else
            fna_unflag(blk, a.applyBlocks, a.g.N, a.type, a.solid, a.sc);
    }
}

template <typename S>
static void obj_uncover(Box& b, const Consts& k, const CoupleArgs& a, hipStream_t s) {
    using M = typename Types<S>::M;
    using C = typename Types<S>::C;
    if (b.parity == 0)
        launch<&k_obj_uncover<S, 0>, UNCOVER_THREADS, 1>(1, UNCOVER_THREADS, s, b.g, (S*)b.f, b.type, (M*)b.mass, (C*)b.aux,
                                                         (C*)b.visc, b.objCand, a.uncCount, a.findBlocks, a.sc, k, b.changed, b.changedCap);
    else
        launch<&k_obj_uncover<S, 1>, UNCOVER_THREADS, 1>(1, UNCOVER_THREADS, s, b.g, (S*)b.f, b.type, (M*)b.mass, (C*)b.aux,
                                                         (C*)b.visc, b.objCand, a.uncCount, a.findBlocks, a.sc, k, b.changed, b.changedCap);
}

// The coupling step (LB.cpp:432-467): flags, impactor nodes, findNewActive, in four launches (two
// without an impactor). order: the particles sorted by link cell (the rebuild's cell list), or null.
// markFollows: lb_mark_edges is enqueued next and ends the coupling (endCoupling); else a launch of its own does.
void lb_coupling(Box& b, const Consts& k, const PartLB* plb, const ObjLB* olb, DevScalars* sc, const int* nbrCount,
                 const int* nbrList, bool useList, const int* order, bool markFollows, hipStream_t s) {
    CoupleArgs a;
    a.g = b.g; a.type = b.type; a.solid = b.solid; a.flagNew = b.flagNew; a.objList = b.objList; a.objCand = b.objCand;
    a.changed = b.changed; a.coverCount = b.coverCount; a.uncCount = b.coverCount + COVER_BLOCKS;
    a.plb = plb; a.olb = olb; a.sc = sc; a.nbrCount = nbrCount; a.nbrList = nbrList; a.order = order;
    a.nPart = k.nPart; a.nObj = k.nObj; a.useList = useList ? 1 : 0; a.objCap = b.objCap; a.changedCap = b.changedCap;
    // the flag passes stride (two particles a wavefront, sixteen nodes a thread or more): most steps only
    // test a flag and return
    a.flagBlocks = k.nPart > 0 ? std::min((k.nPart + 2 * FLAGS_WAVES - 1) / (2 * FLAGS_WAVES), FLAGS_GRID) : 0;
    if (a.flagBlocks > 8) a.flagBlocks = (a.flagBlocks + 7) / 8 * 8;  // one share of the cell order per XCD
    a.scanBlocks = k.nPart > 0 ? int(std::min<int64_t>((b.g.N + FNA_STRIPE - 1) / FNA_STRIPE, FNA_MAX_BLOCKS)) : 0;
    a.applyBlocks = int(std::min<int64_t>((b.g.N + 4095) / 4096, FLAGS_APPLY_GRID));
    a.findBlocks = a.coverBlocks = 0;
    if (k.nObj > 0) {
        // the impactors' node list and the union of their boxes hold about objCap nodes
        a.findBlocks = std::max(1, std::min(UNC_MAX_BLOCKS, (b.objCap + UNC_NODES_PER_BLOCK - 1) / UNC_NODES_PER_BLOCK));
        a.coverBlocks = std::max(16, std::min(COVER_BLOCKS, (b.objCap + 255) / 256));
    }
    const int first = std::max(a.flagBlocks, a.scanBlocks) + a.findBlocks;
    if (first > 0) launch<&k_couple_first, 256, 8>(first, 256, s, a);
    if (k.nObj > 0) {
        if (b.prec == LBDEM_PREC_FP64) obj_uncover<double>(b, k, a, s);
        else if (b.prec == LBDEM_PREC_FP32) obj_uncover<float>(b, k, a, s);
        else obj_uncover<__half>(b, k, a, s);
        // the candidate buffer of the uncover pass stages the cover pass's per-block node lists
        launch<&k_obj_cover_a, COVER_BS, 1>(a.coverBlocks, COVER_BS, s, a.coverBlocks, b.g, b.type, b.solid, olb, k.nObj,
                                            b.coverCount, b.objCand, b.objCap, b.changed, b.changedCap, sc);
    }
    launch<&k_couple_last, 256, 1>(a.coverBlocks + a.applyBlocks, 256, s, a);
    if (!markFollows) launch<&k_couple_end, 64, 1>(1, 1, s, sc);
}

// ------------------------------------------------------------------------------------------
// downloads
// ------------------------------------------------------------------------------------------
// post-streaming populations q0 <= q < q1 of every node in FP64 (plane q at out + (q - q0) N),
// zero where the node is not active
template <typename S>
__device__ inline void k_download_f(Geom g, const S* f, const uint8_t* type, int L, int q0, int q1, double* out) {
    for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < g.N; i += int64_t(gridDim.x) * blockDim.x) {
        const bool act = is_active(type[i]);
        int x, y, z;
        cell_xyz(g, i, x, y, z);
        if (!act) { for (int q = q0; q < q1; ++q) out[int64_t(q - q0) * g.N + i] = 0.0; continue; }
        const Offs o(g, x, y, z);
        for (int q = q0; q < q1; ++q)
            out[int64_t(q - q0) * g.N + i] = wq(q) + double(StoreT<S>::ld(f + load_slot(g, i, o, q, L)));
    }
}
void lb_download_f(const Box& b, double* out, hipStream_t s, int q0, int q1) {
    const int grid = 4096;
    if (b.prec == LBDEM_PREC_FP64) launch<&k_download_f<double>, 1024, 1>(grid, 256, s, b.g, (const double*)b.f, b.type, b.parity, q0, q1, out);
    else if (b.prec == LBDEM_PREC_FP32) launch<&k_download_f<float>, 1024, 1>(grid, 256, s, b.g, (const float*)b.f, b.type, b.parity, q0, q1, out);
    else launch<&k_download_f<__half>, 1024, 1>(grid, 256, s, b.g, (const __half*)b.f, b.type, b.parity, q0, q1, out);
}

// mass field in FP64, zero where the node is not active
template <typename M>
__device__ inline void k_download_mass(int64_t N, const uint8_t* type, const M* mass, double* out) {
    for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < N; i += int64_t(gridDim.x) * blockDim.x)
        out[i] = is_active(type[i]) ? double(mass[i]) : 0.0;
}
void lb_download_mass(const Box& b, double* out, hipStream_t s) {
    if (b.prec == LBDEM_PREC_FP64) launch<&k_download_mass<double>, 1024, 1>(4096, 256, s, b.g.N, b.type, (const double*)b.mass, out);
    else launch<&k_download_mass<float>, 1024, 1>(4096, 256, s, b.g.N, b.type, (const float*)b.mass, out);
}

template <typename S>
__device__ inline void k_download_n(Geom g, const uint8_t* type, const typename Types<S>::M* mass,
                             const typename Types<S>::C* aux, double* out) {
    for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < g.N; i += int64_t(gridDim.x) * blockDim.x) {
        const uint8_t t = type[i] & T_BASE;
        out[i] = t == T_FLUID ? double(mass[i]) : (t == T_IF ? double(aux[i]) : 0.0);
    }
}
void lb_download_n(const Box& b, const Consts& k, double* out, hipStream_t s) {
    (void)k;
    if (b.prec == LBDEM_PREC_FP64) launch<&k_download_n<double>, 1024, 1>(4096, 256, s, b.g, b.type, (const double*)b.mass, (const double*)b.aux, out);
    else launch<&k_download_n<float>, 1024, 1>(4096, 256, s, b.g, b.type, (const float*)b.mass, (const float*)b.aux, out);
}

// total fluid mass: active nodes outside particles (LB.cpp:388-395)
template <typename M>
__device__ inline void k_total_mass(int64_t N, const uint8_t* type, const M* mass, double* out) {
    __shared__ double red[256];
    double acc = 0.0;
    for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < N; i += int64_t(gridDim.x) * blockDim.x) {
        const uint8_t t = type[i];
        if (!(t & T_PMASK) && ((t & T_BASE) == T_FLUID || (t & T_BASE) == T_IF)) acc += double(mass[i]);
    }
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[blockIdx.x] = red[0];
}
void lb_total_mass(const Box& b, double* out, hipStream_t s) {
    // out: 1024 per-block partials, summed on the host in block order
    if (b.prec == LBDEM_PREC_FP64) launch<&k_total_mass<double>, 1024, 1>(1024, 256, s, b.g.N, b.type, (const double*)b.mass, out);
    else launch<&k_total_mass<float>, 1024, 1>(1024, 256, s, b.g.N, b.type, (const float*)b.mass, out);
}

// node counts by kind, read as words of four type bytes (N type bytes are padded to 256 by the
// allocator, the tail is taken byte by byte). Each thread keeps its counts in registers and a block
// adds them once per kind: with one atomic per thread the five counters took 177 us on the
// 256x320x256 box and 78 us on a 64^3 box (a quarter of a million atomics on one cache line).
constexpr int CNT_BLOCKS = 512, CNT_KINDS = 5;
__device__ inline void k_count_types(int64_t N, const uint8_t* type, int* counts) {
    __shared__ int red[CNT_KINDS];
    if (threadIdx.x < CNT_KINDS) red[threadIdx.x] = 0;
    __syncthreads();
    int c[CNT_KINDS] = {0, 0, 0, 0, 0};
    auto one = [&](uint32_t t) {
        const uint32_t b = t & T_BASE;
        c[0] += b == T_FLUID; c[1] += b == T_IF; c[2] += b == T_OBJ; c[3] += (t & T_PMASK) != 0;
        c[4] += b == T_GAS;
    };
    const uint32_t* t32 = reinterpret_cast<const uint32_t*>(type);
    const int64_t nw = N / 4, step = int64_t(gridDim.x) * blockDim.x, t0 = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    for (int64_t i = t0; i < nw; i += step) {
        const uint32_t w = t32[i];
#pragma unroll
        for (int k = 0; k < 4; ++k) one((w >> (8 * k)) & 0xFFu);
    }
    for (int64_t i = 4 * nw + t0; i < N; i += step) one(type[i]);
#pragma unroll
    for (int j = 0; j < CNT_KINDS; ++j) {
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) c[j] += __shfl_xor(c[j], off, 64);
        if (__lane_id() == 0 && c[j]) atomicAdd(&red[j], c[j]);
    }
    __syncthreads();
    if (threadIdx.x < CNT_KINDS && red[threadIdx.x]) atomicAdd(&counts[threadIdx.x], red[threadIdx.x]);
}
void lb_count_types(const Box& b, int* counts, hipStream_t s) {
    launch<&k_count_types, 256, 1>(CNT_BLOCKS, 256, s, b.g.N, b.type, counts);
}

}  // namespace lbdem
