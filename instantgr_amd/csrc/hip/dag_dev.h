// Device definitions shared by the two forms of the detour-DAG routing
// kernels (src/Lshape_route_detour.hpp).
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

} // namespace igr_dev
