// Device layout of one rip-up-and-reroute pass's DAGs (batched form).
//
// The host uploads the DAGs as the builder produced them (net list order,
// local parent indices); once the scheduler has fixed the routing order,
// device kernels compute the per-net bases of that order.  One 64-lane workgroup per routed net then
// writes the net's node records grouped by depth level, its parent-edge records
// grouped by child in the same order (a child's edges keep their own order),
// the level boundaries and the node positions (the order inside a level is
// free: the DAG kernels combine a level's nodes with minima over keys that
// carry the node id, and emit routes in node order), and checks the DAG's
// structure (node range, slot counts, a single source, parents before children
// and at a smaller depth, valid slots), raising *err on a violation.
#include "igr_ctx.hpp"

namespace igr_dev {

namespace {

constexpr int WG = 64;

__device__ __forceinline__ int wave_incl_scan(int v) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int t = __shfl_up(v, d, 64);
        if (lane >= d) v += t;
    }
    return v;
}

__global__ void __launch_bounds__(WG) k_dag_layout(DagLayoutArgs a) {
    const int64_t r = blockIdx.x;
    const int lane = threadIdx.x;
    const int64_t i = a.rorder[r];
    const int64_t b0 = a.node_off[i];
    const int nn = (int)(a.node_off[i + 1] - b0);
    const int64_t g0 = a.nbase[r], ge0 = a.ebase[r];
    const int nl = (int)(a.lbase[r + 1] - a.lbase[r]);
    const int64_t lo = a.lbase[r] + r;   // nl + 1 level boundaries per net
    const int XY = a.X * a.Y;
    for (int d = lane; d <= nl; d += WG) a.lcur[lo + d] = 0;
    __syncthreads();
    bool bad = false;
    int carry = 0;
    for (int base = 0; base < nn; base += WG) {
        const int k = base + lane;
        const int cn = k < nn ? a.child_num[b0 + k] : 0;
        const int incl = wave_incl_scan(cn);
        if (k < nn) {
            const int v = a.nodes[b0 + k];
            bad |= v < 0 || v >= a.node_limit || cn < 0 || cn > 10;
            const int l = v / XY, x = v / a.Y % a.X, y = v % a.Y;
            a.npos[g0 + k] = (uint32_t)l << (2 * DAG_POS_BITS) | (uint32_t)x << DAG_POS_BITS | (uint32_t)y;
            a.lslot[g0 + k] = carry + incl - cn;
            bad |= (k == 0) != (a.par_off[b0 + k + 1] == a.par_off[b0 + k]);
            const int d = a.depth[b0 + k];
            if (d < 0 || d >= nl) bad = true;
            else atomicAdd(&a.lcur[lo + d], 1);
        }
        carry += __shfl(incl, 63, 64);
    }
    if (__any(bad)) {
        if (lane == 0) atomicOr(a.err, 1);
        return;
    }
    __syncthreads();
    // level boundaries (exclusive prefix of the counts); the counters become
    // the fill cursors
    int lcarry = 0;
    for (int base = 0; base <= nl; base += WG) {
        const int d = base + lane;
        const int cn = d < nl ? a.lcur[lo + d] : 0;
        const int incl = wave_incl_scan(cn);
        if (d <= nl) {
            a.lvl[lo + d] = lcarry + incl - cn;
            a.lcur[lo + d] = lcarry + incl - cn;
        }
        lcarry += __shfl(incl, 63, 64);
    }
    __syncthreads();
    // records by level, with the edge counts where the edge bases go
    for (int k = lane; k < nn; k += WG) {
        const int pos = atomicAdd(&a.lcur[lo + a.depth[b0 + k]], 1);
        a.nrec[g0 + pos] = DagNode{a.npos[g0 + k], (uint32_t)k,
                                   (uint32_t)a.lslot[g0 + k] | (uint32_t)a.child_num[b0 + k] << 28,
                                   (uint32_t)(a.par_off[b0 + k + 1] - a.par_off[b0 + k])};
        a.lpos[g0 + k] = pos;
    }
    __syncthreads();
    carry = 0;
    for (int base = 0; base < nn; base += WG) {
        const int q = base + lane;
        const int cn = q < nn ? (int)a.nrec[g0 + q].ebeg : 0;
        const int incl = wave_incl_scan(cn);
        if (q < nn) a.nrec[g0 + q].ebeg = (uint32_t)(carry + incl - cn);
        carry += __shfl(incl, 63, 64);
    }
    __syncthreads();
    for (int k = lane; k < nn; k += WG) {
        const int pos = a.lpos[g0 + k];
        const int64_t pb = a.par_off[b0 + k], pe = a.par_off[b0 + k + 1];
        DagEdge* o = a.edge + ge0 + a.nrec[g0 + pos].ebeg;
        for (int64_t q = pb; q < pe; q++) {
            const int p = a.par[q], sl = a.slot[q];
            if (p < 0 || p >= k || sl < 0 || sl >= a.child_num[b0 + p] || a.depth[b0 + p] >= a.depth[b0 + k]) {
                bad = true;
                continue;
            }
            o[q - pb] = DagEdge{a.npos[g0 + k], a.npos[g0 + p], (uint32_t)(a.lslot[g0 + p] + sl), (uint32_t)pos};
        }
    }
    if (bad) atomicOr(a.err, 1);
}

} // namespace

void launch_dag_layout(igr_ctx* c, const DagLayoutArgs& a, int64_t n) {
    if (n == 0) return;
    k_dag_layout<<<(unsigned)n, WG, 0, c->stream>>>(a);
    HIP_OK(hipGetLastError());
}

} // namespace igr_dev
