// Device helpers shared by the lattice kernels (lb.hip and the fused kernel's translation units).
#pragma once
#include "lbdem_internal.hpp"
#include "launch.hpp"

#include <climits>

namespace lbdem {

template <typename S> struct Types;
template <> struct Types<double> { using C = double; using M = double; };
template <> struct Types<float> { using C = float; using M = float; };
template <> struct Types<__half> { using C = float; using M = float; };

__device__ inline bool is_active(uint8_t t) { t &= T_BASE; return t == T_FLUID || t == T_IF; }

// insideSphere with the reference's rounding (myvector.cpp:171-176): no contraction
__device__ inline bool inside_sphere(double px, double py, double pz, double cx, double cy, double cz, double r) {
#pragma clang fp contract(off)
    const double dx = px - cx, dy = py - cy, dz = pz - cz;
    const double s = dx * dx + dy * dy + dz * dz;
    return s < r * r;
}

__device__ inline void cell_xyz(const Geom& g, int64_t i, int& x, int& y, int& z) {
    if ((uint64_t(i) | uint64_t(g.X) * uint64_t(g.Y)) <= 0xffffffffull) {  // 32-bit quotients
        const uint32_t u = uint32_t(i), sxy = uint32_t(g.X) * uint32_t(g.Y);
        const uint32_t zz = u / sxy, rem = u - zz * sxy, yy = rem / uint32_t(g.X);
        z = int(zz);
        y = int(yy);
        x = int(rem - yy * uint32_t(g.X));
        return;
    }
    z = int(i / (int64_t(g.X) * g.Y));
    const int64_t rem = i - int64_t(z) * g.X * g.Y;
    y = int(rem / g.X);
    x = int(rem - int64_t(y) * g.X);
}

// lattice vectors for a direction index known only at run time: 2-bit fields of packed words
constexpr uint64_t pack_dir(int axis) {
    uint64_t k = 0;
    for (int q = 0; q < Q; ++q) k |= uint64_t((axis == 0 ? cxq(q) : axis == 1 ? cyq(q) : czq(q)) + 1) << (2 * q);
    return k;
}
constexpr uint64_t PACK_CX = pack_dir(0), PACK_CY = pack_dir(1), PACK_CZ = pack_dir(2);
constexpr bool opp_rule_ok() {
    for (int q = 1; q < Q; ++q)
        if (oppq(q) != ((q - 1) ^ 1) + 1) return false;
    return true;
}
static_assert(opp_rule_ok(), "opposite-direction rule");
__device__ inline int cx_rt(int q) { return int((PACK_CX >> (2 * q)) & 3u) - 1; }
__device__ inline int cy_rt(int q) { return int((PACK_CY >> (2 * q)) & 3u) - 1; }
__device__ inline int cz_rt(int q) { return int((PACK_CZ >> (2 * q)) & 3u) - 1; }
__device__ inline int opp_rt(int q) { return q == 0 ? 0 : ((q - 1) ^ 1) + 1; }
__device__ inline double w_rt(int q) { return q == 0 ? 12.0 / 36.0 : (q < 7 ? 2.0 / 36.0 : 1.0 / 36.0); }
// Per-axis index offsets of the wrapped neighbour rule: nb(q) = i + ox[cx+1] + oy[cy+1] + oz[cz+1]
// (offsets fit 32 bits: initialisation rejects boxes with 19*N >= 2^31)
struct Offs {
    int32_t ox[3], oy[3], oz[3];
    __device__ Offs(const Geom& g, int x, int y, int z) {
        const int32_t sy = g.X, sz = g.X * g.Y;
        ox[1] = 0; oy[1] = 0; oz[1] = 0;
        ox[0] = (x - 1 == 0 && g.per[0]) ? g.X - 3 : -1;
        ox[2] = (x + 1 == g.X - 1 && g.per[1]) ? -(g.X - 3) : 1;
        oy[0] = (y - 1 == 0 && g.per[2]) ? (g.Y - 3) * sy : -sy;
        oy[2] = (y + 1 == g.Y - 1 && g.per[3]) ? -(g.Y - 3) * sy : sy;
        oz[0] = (z - 1 == 0 && g.per[4]) ? (g.Z - 3) * sz : -sz;
        oz[2] = (z + 1 == g.Z - 1 && g.per[5]) ? -(g.Z - 3) * sz : sz;
    }
    // selects and packed direction words, not indexed arrays: a direction known only at run
    // time must not put tables or offsets in scratch memory
    __device__ int32_t d(int q) const {
        const int cx = cx_rt(q), cy = cy_rt(q), cz = cz_rt(q);
        return (cx < 0 ? ox[0] : (cx > 0 ? ox[2] : 0)) + (cy < 0 ? oy[0] : (cy > 0 ? oy[2] : 0)) +
               (cz < 0 ? oz[0] : (cz > 0 ? oz[2] : 0));
    }
};

__device__ inline int32_t offs_rt(const Offs& o, int q) { return o.d(q); }

// Whether all neighbours of node i lie within the lattice arrays, wrapped or not: so it is for every node
// inside the outer layer, and of the layer for all but its z faces and the two rows next to them (indices
// below XY + X or not below N - XY - X). Only such nodes may become active: an impactor that passes a z face
// leaves nodes behind on it whose populations would stream out of the arrays (in the fused kernel by 4 GiB,
// its offsets being unsigned). A node that may not is reported as a type error, as the step that streams
// into a periodic layer is.
__device__ inline bool stencil_in_arrays(const Geom& g, int64_t i) {
    const int64_t reach = int64_t(g.X) * g.Y + g.X;
    return i >= reach && i < g.N - reach;
}

// slot holding the post-streaming population q of cell i in layout L (0 natural, 1 swapped)
__device__ inline int64_t load_slot(const Geom& g, int64_t i, const Offs& o, int q, int L) {
    return L == 0 ? int64_t(q) * g.N + i : int64_t(opp_rt(q)) * g.N + i + o.d(opp_rt(q));
}

constexpr int FX = FUSED_TILE_X, FY = FUSED_TILE_Y;  // 64x4 threads: 4 row segments, each lane walks FZ cells
                                                     // along z (FZ 1, 2, 4 or 8, chosen per box)
constexpr int HS = 64;                  // per-block particle hash slots
constexpr int PART_STRIDE = PART_STRIDE_;  // per-block partials: obj (7*MAX_OBJ_PART) + walls 18
constexpr int MAX_OBJ_PART = 2;
// block partials of the fused kernel (sPart, doubles): object o's force and torque at 7 o, the
// bounce-back mass term of all object links at 6, wall w's force at 7 MAX_OBJ_PART + 3 w
constexpr int PART_BB = 6, PART_WALL = 7 * MAX_OBJ_PART;

// Position in a list for each lane of the wavefront that calls this now (any subset of its
// lanes, in divergent code too): one atomic reservation per wavefront, lanes in lane order.
__device__ inline int wave_reserve(int* count) {
    const unsigned long long m = __ballot(1);
    const int lane = __lane_id();
    const int leader = __ffsll(m) - 1;
    int base = 0;
    if (lane == leader) base = atomicAdd(count, __popcll(m));
    base = __shfl(base, leader, 64);
    return base + __popcll(m & ((1ull << lane) - 1ull));
}

// a node changed between active and non-active (or among non-active types): its neighbourhood is
// re-marked before the next LB step; an overflowing list asks for a full re-mark instead
__device__ inline void push_changed(int32_t* changed, int cap, DevScalars* sc, int32_t i) {
    const int pos = wave_reserve(&sc->nChanged);
    if (pos < cap) changed[pos] = i;
    else atomicOr(&sc->fullMark, 1);
}

__device__ inline void list_push(int32_t* list, int* count, int cap, int32_t v, int* overflow) {
    const int pos = wave_reserve(count);
    if (pos < cap) list[pos] = v;
    else atomicOr(overflow, 1);
}

// Block-wide forms of the two above for the passes over the whole interface list, where one
// atomic per wavefront on one counter serialises (every thread of the block must call them, the
// same number of times; sTmp: blockDim.x / 64 + 1 ints or doubles of LDS, reused by the next call):
// positions in a list for the threads with `want`, one reservation per block, block-major then
// wave then lane order; and a sum into one global total, one atomic per block.
__device__ inline int block_reserve(int* count, bool want, int* sTmp) {
    const unsigned long long m = __ballot(want);
    const int lane = __lane_id(), wave = threadIdx.x / 64, nw = blockDim.x / 64;
    if (lane == 0) sTmp[wave] = __popcll(m);
    __syncthreads();
    if (threadIdx.x == 0) {
        int acc = 0;
        for (int w = 0; w < nw; ++w) {
            const int c = sTmp[w];
            sTmp[w] = acc;
            acc += c;
        }
        sTmp[nw] = acc ? atomicAdd(count, acc) : 0;
    }
    __syncthreads();
    const int r = sTmp[nw] + sTmp[wave] + __popcll(m & ((1ull << lane) - 1ull));
    __syncthreads();
    return r;
}
template <typename T>
__device__ inline void block_add(T* dst, T v, T* sTmp) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    const int wave = threadIdx.x / 64, nw = blockDim.x / 64;
    if (__lane_id() == 0) sTmp[wave] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        T t = 0;
        for (int w = 0; w < nw; ++w) t += sTmp[w];
        if (t != T(0)) atomicAdd(dst, t);
    }
    __syncthreads();
}

// per-thread partial sums into one global total: summed over the wavefront first (every lane of
// the wavefront must call this), one atomic per wavefront that has a nonzero sum
__device__ inline void wave_add(double* dst, double v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    if (__lane_id() == 0 && v != 0.0) atomicAdd(dst, v);
}

// check nodes and source directions of the slip reflection (LB.cpp:1454-1482; see k_slip)
__host__ __device__ constexpr int slip1Check(int j) {
    constexpr int c[Q] = {0, 0, 0, 0, 0, 0, 0, 1, 2, 3, 4, 3, 4, 5, 6, 1, 2, 6, 5};
    return c[j];
}
__host__ __device__ constexpr int slip1Dir(int j) {
    constexpr int c[Q] = {0, 0, 0, 0, 0, 0, 0, 9, 10, 8, 7, 13, 14, 12, 11, 18, 17, 15, 16};
    return c[j];
}
__host__ __device__ constexpr int slip2Check(int j) {
    constexpr int c[Q] = {0, 0, 0, 0, 0, 0, 0, 3, 4, 2, 1, 5, 6, 4, 3, 5, 6, 1, 2};
    return c[j];
}
__host__ __device__ constexpr int slip2Dir(int j) {
    constexpr int c[Q] = {0, 0, 0, 0, 0, 0, 0, 10, 9, 7, 8, 14, 13, 11, 12, 17, 18, 16, 15};
    return c[j];
}

// the fused step in storage type S (fused.hpp, instantiated once per storage type)
template <typename S>
void launch_fused(Box& b, const Consts& k, const PartLB* plb, const ObjLB* olb, DevScalars* sc,
                  bool storeVel, hipStream_t s, hipEvent_t ev0, hipEvent_t ev1);

}  // namespace lbdem
