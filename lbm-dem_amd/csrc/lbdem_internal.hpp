// Internal declarations of the MI355X lbdem library: device data layout, lattice constants,
// neighbour rules and the launcher interface shared by lb.hip, dem.hip and api.hip.
//
// Data layout in HBM (one box, N = X*Y*Z cells, index i = x + X*(y + Y*z)):
//   f      : 19 SoA planes of the population offset g_q = f_q - w_q (FP64 / FP32 / scaled FP16),
//            updated in place with the AA pattern (even steps read/write the cell's own slots,
//            odd steps read/write the neighbours' slots); boundary conditions are resolved by
//            the cell that stores, which writes the reflected value into the slot its own load
//            will read next step.
//   type   : uint8 node type (0 fluid, 2 gas, 3 interface, 4 periodic, 7 wall, 12 object),
//            bit 7 = inside-particle flag
//   solid  : int32 solid index (particle / wall / object index, as the reference's solidIndex)
//   mass   : free-surface mass (fluid cells carry their density)
//   aux    : density, shifted velocity and hydrodynamic force of interface cells (donor data)
// Particles, objects and walls are FP64 (positions, velocities, forces, reductions).
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <cstdint>

#include "../../include/lbdem.h"

namespace lbdem {

constexpr int Q = 19;
constexpr int NBR_CAP = 64;        // Verlet partners per particle
constexpr int MAX_OBJECTS = 8;
constexpr int MAX_WALLS = 6;
constexpr float FP16_SCALE = 4096.0f;   // FP16 storage holds g * 2^12

// D3Q19 (reference lattice.h:33-57, 134, 147-150)
__host__ __device__ constexpr int cxq(int q) {
    constexpr int c[Q] = {0, 1, -1, 0, 0, 0, 0, 1, -1, -1, 1, 0, 0, 0, 0, 1, -1, 1, -1};
    return c[q];
}
__host__ __device__ constexpr int cyq(int q) {
    constexpr int c[Q] = {0, 0, 0, 1, -1, 0, 0, 1, -1, 1, -1, 1, -1, -1, 1, 0, 0, 0, 0};
    return c[q];
}
__host__ __device__ constexpr int czq(int q) {
    constexpr int c[Q] = {0, 0, 0, 0, 0, 1, -1, 0, 0, 0, 0, 1, -1, 1, -1, 1, -1, -1, 1};
    return c[q];
}
__host__ __device__ constexpr int oppq(int q) {
    constexpr int o[Q] = {0, 2, 1, 4, 3, 6, 5, 8, 7, 10, 9, 12, 11, 14, 13, 16, 15, 18, 17};
    return o[q];
}
__host__ __device__ constexpr double wq(int q) { return q == 0 ? 12.0 / 36.0 : (q < 7 ? 2.0 / 36.0 : 1.0 / 36.0); }

// type byte: bits 0-3 node type; active nodes: bit 6 'edge' (some wrapped neighbour is not active;
// kept up to date before every lattice step), bit 7 inside-particle flag; wall nodes: bits 4-6 the wall that receives the node's link forces
// (its solid index when that is a wall index, else 0; cleared with the solid index when the
// particle flags are rebuilt)
enum : uint8_t { T_FLUID = 0, T_GAS = 2, T_IF = 3, T_PER = 4, T_WALL = 7, T_OBJ = 12, T_EDGE = 0x40, T_PMASK = 0x80,
                 T_BASE = 0x0F, T_WSHIFT = 4 };
// Boundary-link classes of an edge node, 2 bits per direction j = 1..18 at bit 2(j-1):
// 0 active neighbour (no boundary), 1 gas, 2 wall receiving the node's primary wall index
// (bits 36-38), 3 anything else (object node, another wall, unexpected type: resolved from the
// neighbour's type and solid index).
// boundary-link classes of an edge node: 3 bits per direction 1..18, then the primary wall index.
// OBJ0/OBJ1: object node whose solid index is 0/1; OTHER: anything else (type reloaded in the
// fused kernel)
enum : int { BC_NONE = 0, BC_GAS = 1, BC_WALL = 2, BC_OBJ0 = 3, BC_OBJ1 = 4, BC_OTHER = 7, BC_BITS = 3,
             BC_WALL_SHIFT = 54 };

// Geometry of one box: sizes and which faces wrap (reference LB.cpp:85-126, 632-678:
// an active node wraps along an axis when its face neighbour on that side is periodic).
struct Geom {
    int X, Y, Z;
    int64_t N;
    int per[6];      // boundary[k] == 4
};

__host__ __device__ inline int64_t cidx(const Geom& g, int x, int y, int z) {
    return int64_t(x) + int64_t(g.X) * (int64_t(y) + int64_t(g.Y) * int64_t(z));
}
// neighbour of an active (or gas) node in direction q: wrapped rule
__host__ __device__ inline int64_t nbr_wrapped(const Geom& g, int x, int y, int z, int q) {
    int nx = x + cxq(q), ny = y + cyq(q), nz = z + czq(q);
    if (nx == 0 && g.per[0]) nx = g.X - 2; else if (nx == g.X - 1 && g.per[1]) nx = 1;
    if (ny == 0 && g.per[2]) ny = g.Y - 2; else if (ny == g.Y - 1 && g.per[3]) ny = 1;
    if (nz == 0 && g.per[4]) nz = g.Z - 2; else if (nz == g.Z - 1 && g.per[5]) nz = 1;
    return cidx(g, nx, ny, nz);
}
// neighbour of a node that is neither wall nor active (object nodes): plain index offset
// (reference LB.cpp:570-572), clamped into the box
__host__ __device__ inline int64_t nbr_plain(const Geom& g, int x, int y, int z, int q) {
    int nx = x + cxq(q), ny = y + cyq(q), nz = z + czq(q);
    nx = nx < 0 ? 0 : (nx >= g.X ? g.X - 1 : nx);
    ny = ny < 0 ? 0 : (ny >= g.Y ? g.Y - 1 : ny);
    nz = nz < 0 ? 0 : (nz >= g.Z ? g.Z - 1 : nz);
    return cidx(g, nx, ny, nz);
}

// Particle view used by the lattice kernels (lattice units), refreshed after each DEM step.
struct PartLB {
    double c[3];     // x0 / unit.Length
    double r;        // r / unit.Length
    double v[3];     // x1 / unit.Speed
    double w[3];     // w1 / unit.AngVel
};
struct ObjLB {
    double c[3];     // x0 / unit.Length
    double r;        // r / unit.Length
    double u[3];     // x1 / unit.Speed (object node velocity)
    double pad;
};
static_assert(sizeof(ObjLB) == 8 * sizeof(double), "ObjLB is staged as 8 doubles");

// Scalars shared between kernels (device memory). Doubles first.
struct DevScalars {
    double extraMass;          // streaming extra mass (LB.cpp:1453)
    double surplus;            // free-surface mass surplus (LB.cpp:1644)
    double maxDisp;            // DEM neighbour-list trigger accumulator (DEM.cpp:460-470)
    double obj_F[MAX_OBJECTS][6];   // hydrodynamic F, M per object (lattice units) of the last LB step
    double wall_F[MAX_WALLS][3];    // hydrodynamic F per wall (lattice units, diagnostics)
    double lastExtraMass, lastSurplus;
    int rebuild;               // DEM rebuilt its list this step
    int newNeighborList;       // DEM::newNeighborList
    int builds;                // neighbour list builds
    int nbrOverflow;
    int typeError;             // streaming met an unsupported neighbour type
    int listOverflow;          // a compaction list overflowed
    int nIf;                   // interface list length (LB step)
    int nFilled, nEmptied, nNewIf;
    int nIfFinal;              // interface cells after removeIsolated
    int nObjList;              // object node list length
    int nChanged;              // nodes whose type changed between active and non-active (or among
                               // non-active types) since the last LB step
    int fullMark;              // edge bits and link classes must be recomputed for the whole box
    int kminP;                 // lowest index of a particle-flagged node (-1: none)
    int nPartObj, nPartWall;   // block partials of the fused kernel with impactor / wall links
    int fnaDue, fnaBest;       // findNewActive (fna_scan): due this step; INT_MAX less the new lowest node (0: none)
    int pad[1];
};

template <typename Tst> struct StoreT;
template <> struct StoreT<double> {
    using C = double;
    using Raw = double;  // what a load in flight holds
    __device__ static Raw raw(const double* p) { return *p; }
    __device__ static double value(Raw r) { return r; }
    __device__ static double ld(const double* p) { return *p; }
    __device__ static void st(double* p, double v) { *p = v; }
    __device__ static double stored(double v) { return v; }  // the value a store and a load give back
};
template <> struct StoreT<float> {
    using C = float;
    using Raw = float;
    __device__ static Raw raw(const float* p) { return *p; }
    __device__ static float value(Raw r) { return r; }
    __device__ static float ld(const float* p) { return *p; }
    __device__ static void st(float* p, float v) { *p = v; }
    __device__ static float stored(float v) { return v; }
};
template <> struct StoreT<__half> {
    using C = float;
    using Raw = __half_raw;
    __device__ static Raw raw(const __half* p) { return *reinterpret_cast<const __half_raw*>(p); }
    __device__ static float value(Raw r) {
#pragma clang fp contract(off)  // the product is exact; fused into a sum it would keep that sum's other product from being fused
        return __half2float(__half(r)) * (1.0f / FP16_SCALE);
    }
    __device__ static float ld(const __half* p) { return __half2float(*p) * (1.0f / FP16_SCALE); }
    __device__ static void st(__half* p, float v) { *p = __float2half_rn(v * FP16_SCALE); }
    __device__ static float stored(float v) { return __half2float(__float2half_rn(v * FP16_SCALE)) * (1.0f / FP16_SCALE); }
};

// The device state of one box.
struct Box {
    Geom g;
    int prec;
    int tz = 8;                // nodes along z of a tile, whose particle sums a thread adds together (1, 2, 4 or 8)
    int fz = 8;                // nodes a thread of the fused kernel walks along z: tz, or with 2-byte storage
                               // several tiles of two
    void use_tile(int tile, int walk) { tz = tile; fz = walk; }
    void* f;                   // 19*N storage elements
    uint8_t* type;
    int32_t* solid;
    void* mass;                // N (double for FP64, float otherwise)
    void* aux;                 // 7*N compute-type values: rho, u(3), h(3) for interface cells
    int32_t* ifList;           // interface list (LB step)
    void* ifNewMass;           // per-list new mass
    int32_t* ifList2;          // interface list after conversions
    int32_t* filled;
    int32_t* emptied;
    int32_t* newIf;
    int32_t* donor;            // N, -1 = none
    int32_t* flagNew;          // N, -1 = none (particle flags computed at a rebuild)
    int32_t* objList;          // object nodes, ascending
    int32_t* objCand;          // uncovered object nodes of the current step, ascending
    int* coverCount;           // per-block counts of the object cover and uncover passes
    int32_t* changed;          // nodes to re-mark (see DevScalars::nChanged)
    int changedCap;
    int ifCap, objCap;
    double* blockPart;         // per-block partials of the fused kernel (object F/M, extra mass, walls)
    uint64_t* bcm;             // N, boundary-link classes of edge nodes (valid where T_EDGE is set)
    int32_t* slipList;         // nodes with a diagonal link into a wall, when the walls slip (else null)
    int nSlip;
    void* visc;                // N compute-type node viscosities (lattice units), or null: every node
                               // has the run's viscosity (Newtonian, no turbulence, no restart values)
    int blockPartCap;
    double* hacc;              // per-particle hydro accumulators: F3 M3 vol (lattice units)
    int parity;                // 0: populations in natural layout, 1: swapped
};

struct Consts {
    // lattice-unit parameters
    double lbF[3];              // force in lattice units (zero once collision() ran without forceField)
    double initVel[3];
    double visc;                // lattice kinematic viscosity (initDynVisc)
    double rho0;
    double omega, omegaf;       // 1/(0.5+3 nu), 1 - 1/(1+6 nu)
    // apparent viscosity (node.cpp:113-168; with per-node viscosities only): rheology model
    // (LBDEM_RHEO_*), its parameters in lattice units, the Smagorinsky constant, the clamp range
    int rheo, turb, viscUpdate;
    int slip;                   // walls slip (1: boundary0 = 5, 2: boundary0 = 6, moving with zero velocity):
                                // no wall forces; the slip pass follows the fused kernel; 2 also
                                // enters the free-surface mass exchange
    double slipCoef;            // slipCoefficient (LB.cpp:313, 1344-1345)
    double plasticVisc, yieldStress, frictionCoef, voellmyCoef, turbConst, minVisc, maxVisc;
    int freeSurface;
    int nPart, nObj, nWall;
    double unitLength, unitSpeed, unitAngVel, unitForce, unitTorque, unitVolume;
};

struct DemParams;
struct DemState;

// ---------------- launchers (lb.hip) ----------------
void lb_init_fields(const Box& b, const Consts& k, hipStream_t s);
// rec: LBDEM_RESTART_REC values per record, written at active node node[r]
void lb_restart_fields(const Box& b, const double* rec, const int32_t* node, int nrec, hipStream_t s);
// 3 N values: the velocity held in aux for every active node, zero elsewhere
void lb_download_velocity(const Box& b, double* out, hipStream_t s);
// N values: the node viscosity plane (b.visc must be set) at active nodes, zero elsewhere
void lb_download_visc(const Box& b, double* out, hipStream_t s);
// SHydro of every particle (9 per particle, physical units: L, F = unit.Length, unit.Force) from
// the aux planes an LB step with storeVel left
void lb_hydro_stress(const Box& b, const PartLB* plb, int nPart, double L, double F, double* shydro, hipStream_t s);
void lb_mark_edges(const Box& b, DevScalars* sc, bool endCoupling, hipStream_t s);  // endCoupling: of lb_coupling
// storeVel: every active node's density and velocity into aux (else the interface nodes' only)
void lb_fused_step(Box& b, const Consts& k, const PartLB* plb, const ObjLB* olb, DevScalars* sc,
                   bool storeVel, hipStream_t s, hipEvent_t ev0 = nullptr, hipEvent_t ev1 = nullptr);
void lb_hydro_finalize(const Box& b, const Consts& k, double* FHydro, double* MHydro, double* fluidVol,
                       DevScalars* sc, double* objFH, double* objMH, double* wallFH, hipStream_t s);
// The launches between two fused kernels (front.hpp): hydro: the finalisation of the fused kernel's
// sums; fs: the free surface; dp, ds (may be null): the neighbour list (forceList: built without asking
// the trigger, and no forces) and the forces of DEM step demTimeStep
void lb_front(Box& b, const Consts& k, DevScalars* sc, bool hydro, bool fs, double* FHydro, double* MHydro,
              double* fluidVol, double* objFH, double* objMH, double* wallFH, const DemParams* dp, DemState* ds,
              int demTimeStep, bool forceList, hipStream_t s);
// the coupling step; useList: the Verlet lists of a rebuild resolve overlapping spheres (highest index
// wins) without atomics; order: the particles sorted by link cell, or null; markFollows:
// lb_mark_edges is enqueued next
void lb_coupling(Box& b, const Consts& k, const PartLB* plb, const ObjLB* olb, DevScalars* sc, const int* nbrCount,
                 const int* nbrList, bool useList, const int* order, bool markFollows, hipStream_t s);
constexpr int PART_STRIDE_ = 32;
int fused_grid_blocks(const Geom& g, int fz, int prec);  // blocks of the fused kernel for z-walk length fz
// With 2-byte storage a rounding of the particle sums in 32 bits decides a particle flag within some
// hundred steps, so the results depend on how many nodes share one. Walks of 4 and 8 nodes are therefore
// walks over tiles of two there whenever it is the library that chooses the walk, by timing or by the size
// of the box: walks of 2, 4 and 8 then give the same sums, and the tile says which (two: the fastest walk
// of large boxes while it waited for each load). The caller may still fix a tile of 4 or 8.
inline int tile_of_walk(int prec, int walk) { return prec == LBDEM_PREC_FP16 && walk > 2 ? 2 : walk; }
// The walk that a fixed tile takes; blocks4: blocks of the four-node walk over all boxes of a launch.
// Event-timed launches with 2-byte storage, walks of four and two nodes: 9216 blocks 234 and 233 us, 7488
// blocks 194 and 194, 4800 blocks 122 and 111, 256 blocks 44 and 29; 10 000 blocks 228 and 234, 12 544 blocks
// 290 and 300, 20 480 blocks 458 and 485.
constexpr int64_t WALK4_BLOCKS = 9600;
inline int walk_of_tile(int prec, int tile, int64_t blocks4) {
    return prec == LBDEM_PREC_FP16 && tile == 2 && blocks4 >= WALK4_BLOCKS ? 4 : tile;
}
constexpr int FUSED_TILE_X = 64, FUSED_TILE_Y = 4;  // threads of a fused-kernel tile (x, y)
// largest grid of the fused kernel over its walks and mappings: columns of the partials are this far apart
__host__ __device__ inline int part_stride(const Geom& g) {
    const int nseg = (g.X + FUSED_TILE_X - 1) / FUSED_TILE_X, nby = (g.Y + FUSED_TILE_Y - 1) / FUSED_TILE_Y;
    return nseg * nby * g.Z + 8;
}
constexpr int COVER_BLOCKS = 512, UNCOVER_BLOCKS_MAX = 1024;  // grids of the impactor node passes
void lb_download_f(const Box& b, double* out, hipStream_t s, int q0 = 0, int q1 = Q);
void lb_download_mass(const Box& b, double* out, hipStream_t s);
void lb_download_n(const Box& b, const Consts& k, double* out, hipStream_t s);
void lb_total_mass(const Box& b, double* out, hipStream_t s);
void lb_count_types(const Box& b, int* counts, hipStream_t s);

// ---------------- DEM (dem.hip) ----------------
struct DemParams {
    double demSize[3];
    double deltat;
    double linearStiff, dampCoeff, frictionCoefPart, kinVisc;
    double lubNormal, lubTangential, lubRotation, lubCutoff;
    double electroForce, debyeLength;
    double rmax;
    int objWaitTime;
    int periodic[3];           // both faces periodic along axis
    int nlx, nly, nlz;         // cell grid: all 0 for the direct sum; else nlx, nly >= 3, nlz >= 0
    int nPart, nObj, nWall;
    int nBody, nonLinType;     // body-spring impactor (DEM.cpp:63-73, 798-869)
    double springDamp, epsilon, k13;
    double wallP[MAX_WALLS][3], wallN[MAX_WALLS][3];
    double unitLength, unitSpeed, unitAngVel;
    int stress;                // accumulate the stress diagnostics (DemState::stressPart, disp)
};
// per-particle stress record of the last DEM step (doubles): the stresslet SHydro the force kernel
// copied from DemState::shydro, SLub, the contact stress of the particle pairs (each pair adds the
// same tensor to both of its spheres), the contact stress of walls and impactors, SRep, the
// elastic and viscous parts of the contact stress (SElas, SVisc before SVisc_h is added), FElas,
// the contact and normal-lubrication counts; tensors m00 m01 m02 m10 ... m22
enum { SP_HYDRO = 0, SP_LUB = 9, SP_CPAIR = 18, SP_CWALL = 27, SP_REP = 36, SP_ELAS = 45, SP_VISC = 54,
       SP_FELAS = 63, SP_COORD = 66, SP_LUBC = 67, SP_REC = 68 };
constexpr int VEL_SLOTS = 64;  // slots of the particle speed maximum (DemState::blockMax)
struct DemState {
    bool inBatch = false;  // stepped by a batch, whose launches hold many boxes (dem_force_lanes)
    // particles (FP64, vectors stored as 3 consecutive doubles)
    double *x0, *x1, *w1, *r, *m, *I, *im, *iI;
    double *FHydro, *MHydro, *FContact, *MContact, *FLub, *MLub, *FRep, *FTotal, *MTotal, *FGrav, *fluidVol;
    double *xiw, *xio;
    int* nbrCount;             // partners per particle
    int* nbrList;              // NBR_CAP per particle, ascending
    int* nbrSlot;              // history slot of each entry (in the list of the higher index)
    int* nbrCountOld;
    int* nbrListOld;
    double* xiCur;             // tangential history per slot (3 per slot), read by the force kernel
    double* xiNext;            // written by the force kernel (buffers swap every step); between steps free
                               // to use (lbdem_get_particles packs its records there)
    int* cellCount;
    int* cellStart;
    int* cellFill;
    int* cellItems;
    int* cellKey;
    double* redPart;           // per block of the force pass: impactor and wall sums (DEM_RED_COLS columns)
    int* redFlag;              // per block: the sums are written
    unsigned long long* blockMax;  // [VEL_SLOTS]: largest particle |v|^2 of the last integration, per slot (bit patterns)
    // objects
    double *ox0, *ox1, *ow1, *or_, *om, *oI, *oim, *oiI;
    double *oFHydro, *oMHydro, *oFContact, *oMContact, *oFLub, *oMLub, *oFTotal, *oMTotal, *oFGrav;
    // bodies: LBDEM_B_REC doubles each (include/lbdem.h layout)
    double* body;
    // stress diagnostics (null unless DemParams::stress)
    double* stressPart;        // SP_REC per particle
    double* shydro;            // 9 per particle: SHydro of the last LB step (physical units)
    double* xi0;               // 3 per particle: x_i, the position at the start or at objWaitTime
    double* disp;              // 3 per particle: x_i - x0 after the last integration
    // walls
    double *wFHydro, *wFContact, *wFLub, *wFTotal;
    PartLB* plb;
    ObjLB* olb;
};
int dem_force_lanes(int nPart, bool inBatch);   // lanes per particle of the force pass
int dem_force_blocks(int nPart, bool inBatch);  // its blocks
constexpr int DEM_RED_COLS = 12 * 2 + 6 * MAX_WALLS;  // columns of redPart: at most two impactors (lbdem_set_objects)
// totals, integration, objects and walls (after the forces and the hydrodynamic sums)
void dem_integrate(const DemParams& p, DemState& d, int demTimeStep, hipStream_t s);
void dem_refresh_views(const DemParams& p, DemState& d, hipStream_t s);

// records of a download (particles, impactors, walls): column q of a record is component comp[q]
// of an array with width[q] values per item
constexpr int REC_COLS = 48;
struct RecordMap {
    const double* src[REC_COLS];
    uint8_t width[REC_COLS], comp[REC_COLS];
    int cols;
    void add(int col, const double* p, int w) {
        for (int a = 0; a < w; ++a) { src[col + a] = p; width[col + a] = uint8_t(w); comp[col + a] = uint8_t(a); }
    }
};
void dem_pack_records(const RecordMap& m, int n, double* out, hipStream_t s);

// run pool hooks: a context carves its buffers from [base, base+bytes) instead of allocating
// them (set before lbdem_init); the stream a context enqueues on
int ctx_use_region(lbdem_ctx* c, void* base, size_t bytes);
hipStream_t ctx_stream(const lbdem_ctx* c);
// a batch's argument tables in [base, base+bytes) (set before its first cycle); its stream
int batch_use_region(lbdem_batch* b, void* base, size_t bytes);
hipStream_t batch_stream(const lbdem_batch* b);
// start-up over (a batch may take the context); AA/history phase; storage precision
bool ctx_steady(const lbdem_ctx* c);
int ctx_phase(const lbdem_ctx* c);
int ctx_precision(const lbdem_ctx* c);

}  // namespace lbdem
