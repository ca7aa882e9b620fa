// Device definitions shared by the two forms of the detour-DAG routing kernels
// (src/Lshape_route_detour.hpp); the pattern kernels take the wire segments'.
#pragma once
#include "igr_dev.h"

namespace igr_dev {

constexpr uint64_t INIT_KEY = 7208259049189261824ULL;  // :106
constexpr uint32_t ID_MUL = 1000;

// DP keys pack the FP32 cost (as an order-preserving int) above a 32-bit id,
// node * 1000 + choice with the node's index inside its own net, so the
// 64-bit minimum picks the smallest cost and, among equal costs, the smallest
// (node, choice) pair exactly as the reference's global ids do.
__device__ __forceinline__ uint64_t pack_key(float cost, uint32_t id) {
    int32_t i = __float_as_int(cost);
    int32_t o = i >= 0 ? i : i ^ 0x7FFFFFFF;
    return ((uint64_t)(int64_t)o << 32) | (uint64_t)id;
}
__device__ __forceinline__ float unpack_costf(uint64_t k) {
    int32_t o = (int32_t)(k >> 32);
    return __int_as_float(o >= 0 ? o : o ^ 0x7FFFFFFF);
}
__device__ __forceinline__ double unpack_cost(uint64_t k) { return (double)unpack_costf(k); }

__device__ __forceinline__ double wseg(const GridDev& g, int l, int xmin, int xmax, int ymin, int ymax) {
    return g.presum[gidx(g, l, xmax, ymax)] - g.presum[gidx(g, l, xmin, ymin)];
}

// Difference-array form of one wire segment (src/graph.hpp:105-117).
__device__ __forceinline__ void add_segment(const GridDev& g, int l, int minx, int maxx, int miny, int maxy,
                                            int stamp) {
    atomicAdd(&g.pre[gidx(g, l, minx, miny)], 1);
    if (g.dirty) g.dirty[track_id(g, l, minx, miny)] = 1;
    if (minx == maxx) {
        atomicAdd(&g.pre[gidx(g, l, minx, maxy)], -1);
        g.ts[gidx(g, l, minx, maxy)] = stamp;
    }
    if (miny == maxy) {
        atomicAdd(&g.pre[gidx(g, l, maxx, miny)], -1);
        g.ts[gidx(g, l, maxx, miny)] = stamp;
    }
}

// Rip-up footprint of one routed net, by RIP_LANES consecutive lanes, a route
// pair each (a thread per net waits for its pairs one after another): +1/-1
// wire differences at the two ends of each wire, +1/-1 covered-cell
// differences at its first cell and one past its last, one count per via cut,
// and the dirty flag of every track touched.  Wires that do not run along
// their layer's direction set *bad.  A launch over the 2600 nets of an average
// 800x800 batch took 132 us with a thread per net, 21 us with 16 lanes.
constexpr int RIP_LANES = 16;
__device__ __forceinline__ void rip_route(const GridDev& g, const int* r, int* bad) {
    const int XY = g.X * g.Y;
    const int end = r[0];
    for (int i = 1 + 2 * (threadIdx.x & (RIP_LANES - 1)); i < end; i += 2 * RIP_LANES) {
        const int a = r[i], b = r[i + 1];
        const int la = a / XY, lb = b / XY;
        const int x0 = a / g.Y % g.X, y0 = a % g.Y, x1 = b / g.Y % g.X, y1 = b % g.Y;
        if (la == lb) {
            const int d = layer_dir(la, g.DIR);
            if ((d == 0 && y0 != y1) || (d == 1 && x0 != x1)) { atomicOr(bad, 1); continue; }
            const int lo = d ? min(y0, y1) : min(x0, x1), hi = d ? max(y0, y1) : max(x0, x1);
            const int len = d ? g.Y : g.X;
            const int64_t c0 = d ? gidx(g, la, x0, lo) : gidx(g, la, lo, y0);
            const int64_t c1 = d ? gidx(g, la, x0, hi) : gidx(g, la, hi, y0);
            if (lo < hi) {
                atomicAdd(&g.rpre[c0], 1);
                atomicAdd(&g.rpre[c1], -1);
            }
            atomicAdd(&g.rcov[c0], 1);
            if (hi + 1 < len) atomicAdd(&g.rcov[c1 + 1], -1);
            g.dirty[track_id(g, la, x0, y0)] = 1;
        } else {
            const int lo = min(la, lb), hi = max(la, lb);
            for (int l = lo; l < hi; l++) {
                atomicAdd(&g.rvc[gidx(g, l, x0, y0)], 1);
                g.dirty[track_id(g, l, x0, y0)] = 1;
            }
        }
    }
}

} // namespace igr_dev
