// Detour-DAG routing, batched form (src/Lshape_route_detour.hpp:75-694): per
// batch one launch prices every parent edge of its DAGs (k_dag_edge_costs),
// then one launch routes the nets, a workgroup each (k_dag_net).  Both read
// the level-ordered records the layout kernel writes once per pass
// (dag_layout.hip).  Costs, keys and tie rules are those of the plain form's
// kernels (dag_kernels.hip), so both forms' routes are identical.
#include "dag_dev.h"
#include "igr_ctx.hpp"
#include "row.h"

#include <algorithm>

namespace igr_dev {

namespace {

constexpr int TPB = 256;
constexpr int64_t EDGE_WAVES = 8192;  // waves an edge launch fills first

// Direction-layer count of either direction is at most (L + 1) / 2; an edge's
// costs over (parent layer, child layer) pairs of its direction are one row
// block of stride ND * ND, parent-major.
__host__ __device__ constexpr int dir_layers(int L) { return (L + 1) / 2; }

__device__ __forceinline__ int pos_x(uint32_t p) { return (int)(p >> DAG_POS_BITS) & ((1 << DAG_POS_BITS) - 1); }
__device__ __forceinline__ int pos_y(uint32_t p) { return (int)p & ((1 << DAG_POS_BITS) - 1); }

struct EdgeGeom {
    int fx, fy, tx, ty, dist;
    bool vert, straight;
};
__device__ __forceinline__ EdgeGeom edge_geom(uint32_t from, uint32_t to) {
    EdgeGeom e;
    e.fx = pos_x(from); e.fy = pos_y(from); e.tx = pos_x(to); e.ty = pos_y(to);
    e.dist = abs(e.tx - e.fx) + abs(e.ty - e.fy);
    e.vert = e.fx == e.tx;
    e.straight = e.vert || e.fy == e.ty;
    return e;
}
// First routing layer of direction d, and how many there are.
__device__ __forceinline__ int dir_first(const GridDev& g, int d) { return d ^ g.DIR; }
__device__ __forceinline__ int dir_count(int L, int first) { return (L - first + 1) / 2; }

// ---------------------------------------------------------------------------
// Edge costs.  For a straight edge and every pair (parent layer tl, child
// layer fl) of its direction: the wire cost along the layer where tl == fl;
// where they differ and the edge is longer than 4 gcells, the smallest cost of
// one layer change at a sampled position (precompute_cost_edge, :123-195).
//
// A wave takes CH consecutive edges.  Lane i first prices edge i's same-layer
// wires; then the wave takes the long edges one after another: every lane
// stages via and prefix-sum values of the edge's samples in LDS (at most 39
// samples: dd = dist / min(dist, 20)), then owns one unordered layer pair and
// every S-th sample (S = 64 / pairs), forms the via stack once for both
// directions of the change, and the S lanes of a pair combine their minima by
// (cost, sample).  The via cuts are summed from the lower layer up and the two
// wire pieces added after, as the reference does; the first smallest sample
// wins.
// ---------------------------------------------------------------------------
constexpr int EW_SAMPLES = 40;
constexpr int EW_WAVES = TPB / 64;

struct EdgeArgs {
    GridDev g;
    const DagEdge* edge;      // the batch's edges
    int64_t n;
    double* cost;             // n blocks of ND * ND
    uint16_t* change;         // the sample of each entry's layer change
    int chunk;                // edges per wave
    unsigned edge_blocks;     // workgroups from here on rip up
    const int* rip_nets;      // the next batch's nets
    int64_t rip_n;
    int* const* rptr;
    int* bad;
};

template <int L>
__global__ void __launch_bounds__(TPB) k_dag_edge_costs(EdgeArgs a) {
    constexpr int ND = dir_layers(L), LV = L > 1 ? L - 1 : 1;
    __shared__ float s_v[EW_WAVES][EW_SAMPLES * LV];       // via cut cost at (sample, layer)
    __shared__ double s_ps[EW_WAVES][EW_SAMPLES * ND];     // prefix sum at (sample, direction layer)
    __shared__ double s_pe[EW_WAVES][2 * ND];              // prefix sum at the child / parent end
    const GridDev& g = a.g;
    if (blockIdx.x >= a.edge_blocks) {
        // The rip-up scatter of the next batch: it reads other nets' old
        // routes and writes only the rip-up difference arrays, so it shares
        // the launch with the edges of this batch.
        const int64_t t = ((int64_t)(blockIdx.x - a.edge_blocks) * TPB + threadIdx.x) / RIP_LANES;
        if (t < a.rip_n) rip_route(g, a.rptr[a.rip_nets[t]], a.bad);
        return;
    }
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int64_t w0 = ((int64_t)blockIdx.x * EW_WAVES + wv) * a.chunk;
    if (w0 >= a.n) return;                                 // whole waves; no workgroup barrier below
    const int cnt = (int)(a.n - w0 < a.chunk ? a.n - w0 : a.chunk);
    uint32_t from = 0, to = 0;
    bool lng = false;
    if (lane < cnt) {
        const DagEdge e = a.edge[w0 + lane];
        from = e.from;
        to = e.to;
        const EdgeGeom q = edge_geom(from, to);
        if (q.straight && q.dist > 0) {
            const int dir = q.vert ? 1 : 0, first = dir_first(g, dir), nd = dir_count(L, first);
            const int x0 = min(q.fx, q.tx), x1 = max(q.fx, q.tx), y0 = min(q.fy, q.ty), y1 = max(q.fy, q.ty);
            double* c = a.cost + (w0 + lane) * (ND * ND);
#pragma unroll
            for (int b = 0; b < ND; b++)
                if (b < nd) c[b * ND + b] = wseg(g, first + 2 * b, x0, x1, y0, y1);
            lng = q.dist > 4 && nd > 1;
        }
    }
    uint64_t todo = __ballot(lng);
    float* sv = s_v[wv];
    double *sps = s_ps[wv], *spe = s_pe[wv];
    while (todo) {
        const int i = __builtin_ctzll(todo);
        todo &= todo - 1;
        const EdgeGeom q = edge_geom((uint32_t)__builtin_amdgcn_readlane((int)from, i),
                                     (uint32_t)__builtin_amdgcn_readlane((int)to, i));
        const int dir = q.vert ? 1 : 0, first = dir_first(g, dir), nd = dir_count(L, first);
        const int dd = q.dist / min(q.dist, 20);
        const int fpos = q.vert ? q.fy : q.fx, tpos = q.vert ? q.ty : q.tx;
        const int s0 = min(fpos, tpos), s1 = max(fpos, tpos);
        const int ns = (s1 - 1 - s0) / dd;                 // samples s0 + dd, ..., < s1
        for (int t = lane; t < ns * LV; t += 64) {
            const int k = t / LV, l = t - k * LV;
            const int sp = s0 + (k + 1) * dd;
            sv[t] = g.vcost[q.vert ? gidx(g, l, q.fx, sp) : gidx(g, l, sp, q.fy)];
        }
        for (int t = lane; t < ns * nd; t += 64) {
            const int k = t / nd, b = t - k * nd;
            const int sp = s0 + (k + 1) * dd;
            sps[k * ND + b] = g.presum[q.vert ? gidx(g, first + 2 * b, q.fx, sp) : gidx(g, first + 2 * b, sp, q.fy)];
        }
        if (lane < 2 * nd) {
            const int end = lane >= nd, b = lane - end * nd;
            spe[end * ND + b] = g.presum[gidx(g, first + 2 * b, end ? q.tx : q.fx, end ? q.ty : q.fy)];
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
        __builtin_amdgcn_wave_barrier();
        const int np = nd * (nd - 1) / 2, S = 64 / np;
        const int sub = lane / np, pr = lane - sub * np;
        // pair pr: direction layers lo < hi
        int lo = 0, r = pr;
        while (r >= nd - 1 - lo) r -= nd - 1 - lo++;
        const int hi = lo + 1 + r;
        // up: child on the lower layer, parent on the higher; dn: the reverse
        double mu = INF, md = INF;
        int ku = EW_SAMPLES, kd = EW_SAMPLES;
        if (sub < S) {
            const int l0 = first + 2 * lo, l1 = first + 2 * hi;
            const double fl = spe[lo], fh = spe[hi], tl = spe[ND + lo], th = spe[ND + hi];
            for (int k = sub; k < ns; k += S) {
                const int sp = s0 + (k + 1) * dd;
                double via = 0;
                for (int l = l0; l < l1; l++) via += (double)sv[k * LV + l];
                const double pl = sps[k * ND + lo], ph = sps[k * ND + hi];
                const bool f = sp >= fpos, t = sp >= tpos;
                // presum[max] - presum[min] of each piece
                const double up = via + ((f ? pl - fl : fl - pl) + (t ? ph - th : th - ph));
                const double dn = via + ((f ? ph - fh : fh - ph) + (t ? pl - tl : tl - pl));
                if (up < mu) { mu = up; ku = k; }
                if (dn < md) { md = dn; kd = k; }
            }
        }
        // lanes pr, pr + np, ... hold the pair's samples in stripes
        for (int d = 1; d < S; d <<= 1) {
            const int src = lane + d * np;
            const double ou = __shfl(mu, src & 63), od = __shfl(md, src & 63);
            const int qu = __shfl(ku, src & 63), qd = __shfl(kd, src & 63);
            if (src < S * np) {
                if (ou < mu || (ou == mu && qu < ku)) { mu = ou; ku = qu; }
                if (od < md || (od == md && qd < kd)) { md = od; kd = qd; }
            }
        }
        if (lane < np) {
            double* c = a.cost + (w0 + i) * (ND * ND);
            uint16_t* ch = a.change + (w0 + i) * (ND * ND);
            c[hi * ND + lo] = mu;
            ch[hi * ND + lo] = (uint16_t)(s0 + (ku + 1) * dd);
            c[lo * ND + hi] = md;
            ch[lo * ND + hi] = (uint16_t)(s0 + (kd + 1) * dd);
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
        __builtin_amdgcn_wave_barrier();
    }
}

// ---------------------------------------------------------------------------
// Net routing: NW waves per net, nodes sixteen lanes each, level by level
// from the deepest, then the extraction from the source down and the route.
//
// A net is a chain of levels, so its time is the latency of a level: the
// records and via costs of the next step are loaded during the current one,
// the edge costs before the node costs they are added to, and the keys, layer
// ranges and decisions live in LDS, where the minima over a slot's candidates
// are LDS atomics.  The batch's edge costs come from the launch before, so no
// grid gather but the nodes' via costs is left in the chain.  A node's child
// choices are not stored per layer: the range behind each layer's cost (one
// byte) lets the extraction find the one it needs.  Four waves a net: two lose
// 7% of a 20k-net run (180 against 168 ms) and win 1% of a 438k-net pass.
// Average launch, 9 layers, against a wave per net with tables in global
// memory and four shuffled prefix steps per child and lowest layer: 200x200, 20k
// nets 65 us (477), 800x800, 438k nets 153 us (727), 600x600 with heavy
// nets 106 us (840), a 40-net request 38 us (250).
// ---------------------------------------------------------------------------
struct NetArgs {
    GridDev g;
    const DagNode* node;          // per net by level
    const DagEdge* edge;          // per net by child in level order
    const uint32_t* npos;         // per net in node order: position and layer
    const int* lvl;               // per net: nlev + 1 level boundaries
    const int64_t *nbase, *ebase, *sbase, *lbase;   // by routed net
    const int* rorder;            // by routed net: its list entry
    const int64_t* list_node;     // by list entry: the nodes before it
    const double* cost;           // the batch's edge costs and layer-change samples
    const uint16_t* change;
    const int* nets;
    int64_t net0, n, edge0;       // the batch's nets
    int* queue;
    int* routes;
    int** rptr;
    int stamp;
    int lds_bytes;                // dynamic LDS of the launch
    // tables of the nets that exceed it, indexed from the batch's first slot,
    // node (null when none does)
    uint64_t* big_key;
    uint8_t* big_range;
    uint2* big_dec;
    int64_t node0, slot0;
};

// Key table access: LDS, or global memory for the nets whose tables exceed it
// (their keys are updated by atomics that complete in L2, so they are read
// with device-scope loads).
template <bool LDS>
__device__ __forceinline__ uint64_t key_load(const uint64_t* p) {
    if constexpr (LDS) return *p;
    else return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <bool LDS>
__device__ __forceinline__ void key_store(uint64_t* p, uint64_t v) {
    if constexpr (LDS) *p = v;
    else __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

constexpr uint64_t NO_CHILD = ~0ull;   // entry 0 of a slot: no child chosen
constexpr float INF_BELOW = 9.999999778196308e21f;   // the largest float below INF

// Cost of every layer s (this lane's) of a node and the layer range behind it
// (Lshape_route_node_layer_change_cuda, :281-353): the smallest, over ranges
// low <= s <= hi that hold the node's pin, of the via stack of the range plus
// every child slot's smallest key cost within it; ties go to the smaller low,
// then the smaller hi, which is the order the reference's loops keep.  Lane hi
// of the row forms the costs of its ranges for every low: the via sums in
// layer order, and per child the running minimum over the layers from hi
// down, in FP32 where the keys live, so every sum is the reference's.
template <int L, bool LDS>
__device__ __forceinline__ double node_cost(const uint64_t* keys, int nc, int ncw, int fixed, float vl, bool valid,
                                            int& range) {
    constexpr int ML = L + 1;
    const int s = threadIdx.x & 15;
    const double PINF = __longlong_as_double(0x7ff0000000000000LL);
    const int low_top = fixed == ML ? L : fixed;       // a pin's range starts at or below it
    const bool as_hi = valid && s >= 1 && s <= L && (fixed == ML || s >= fixed);
    double cost[L];                                    // by low - 1
    double vm[L];                                      // via cut t - 2, zero above s
    unrolled<L - 1>([&](auto I) {
        constexpr int t = I + 2;
        const float v = row_bcast<I>(vl);
        vm[I] = t <= s ? (double)v : 0.0;
    });
    unrolled<L>([&](auto I) {
        constexpr int low = I + 1;
        double acc = 0.0;
#pragma unroll
        for (int t = low + 1; t <= L; t++) acc += vm[t - 2];
        cost[I] = acc;
    });
    for (int k = 0; k < ncw; k++) {
        float c = 0.0f;
        if (k < nc && s >= 1 && s <= L) {
            c = unpack_costf(key_load<LDS>(keys + k * ML + s));
            c = c <= INF_BELOW ? c : __int_as_float(0x7f800000);
        }
        float m = c;
        unrolled<L>([&](auto I) {
            constexpr int low = L - I;
            const float below = row_bcast<low>(c);        // outside the selects: every lane takes part
            m = __builtin_amdgcn_fmed3f(m, below, -__builtin_inff());   // their minimum
            m = low >= s ? c : m;
            cost[low - 1] += (double)m;
        });
    }
    double best = INF;
    int code = 0;
    uint64_t at = 0;
    unrolled<L>([&](auto I) {
        constexpr int low = I + 1;
        const bool ok = as_hi & (s >= low) & (low <= low_top) & (cost[I] < INF);
        const double own = ok ? cost[I] : PINF;
        double c = own;
        auto lower = [&](double o) { c = o < c ? o : c; };
        lower(row_above<1>(c));
        lower(row_above<2>(c));
        if constexpr (L > 4) lower(row_above<4>(c));
        if constexpr (L > 8) lower(row_above<8>(c));
        const uint64_t mine = __ballot(own == c);      // where the minimum from here up is the lane's own
        const bool better = (s >= low) & (c < best);
        best = better ? c : best;
        code = better ? low : code;
        at = better ? mine : at;
    });
    const int lane = threadIdx.x & 63;
    if (code) code |= (s + __builtin_ctzll(at >> lane)) << 4;
    range = code;
    return best;
}

template <int L, int NW, bool LDS>
__device__ void route_net(const NetArgs& a, int64_t r, uint64_t* K, uint8_t* R, uint2* dec, int* slvl,
                          double (*s_cst)[16], int* s_loc, int* s_out, int* s_scan) {
    constexpr int ML = L + 1, LL = L * L, SENT = LL + 1, T = NW * 64, CH = NW * 4, ND = dir_layers(L);
    const GridDev& g = a.g;
    const int tid = threadIdx.x, lane = tid & 63, s = tid & 15, gi = tid >> 4;
    const int64_t n0 = a.nbase[r], e0 = a.ebase[r], l0 = a.lbase[r] + r;
    const int nn = (int)(a.nbase[r + 1] - n0), ne = (int)(a.ebase[r + 1] - e0);
    const int ns = (int)(a.sbase[r + 1] - a.sbase[r]), nlev = (int)(a.lbase[r + 1] - a.lbase[r]);
    const DagNode* node = a.node + n0;
    const DagEdge* edge = a.edge + e0;
    const double* ecost = a.cost + (e0 - a.edge0) * (ND * ND);
    if constexpr (LDS)
        for (int k = tid; k <= nlev; k += T) slvl[k] = a.lvl[l0 + k];
    for (int k = tid; k < ns * ML; k += T) key_store<LDS>(&K[k], INIT_KEY);
    for (int k = tid; k < nn; k += T) dec[k] = make_uint2(0, 0);
    __syncthreads();
    for (int k = tid; k < ns; k += T) key_store<LDS>(&K[k * ML], NO_CHILD);

    // Bottom-up, CH nodes of a level at a time.  The records and via costs of
    // the next CH nodes are loaded while the current ones are worked on.
    int d = nlev - 1, c0 = 0;
    while (d >= 0 && slvl[d] == slvl[d + 1]) d--;
    c0 = d >= 0 ? slvl[d] : 0;
    DagNode rec{0, 0, 0, 0};
    float vl = 0.0f;
    int eb = 0, ee = 0;
    auto fetch = [&](int dd, int cc, DagNode& o, int& b, int& e) {
        const int hi = slvl[dd + 1];
        o = DagNode{0, 0, 0, 0};
        if (cc + gi < hi) o = node[cc + gi];
        const int c1 = min(cc + CH, hi);
        b = (int)node[cc].ebeg;
        e = c1 < nn ? (int)node[c1].ebeg : ne;
    };
    auto via_at = [&](int dd, int cc, const DagNode& o) {
        return cc + gi < slvl[dd + 1] && s < L - 1 ? g.vcost[gidx(g, s, pos_x(o.pos), pos_y(o.pos))] : 0.0f;
    };
    if (d >= 0) {
        fetch(d, c0, rec, eb, ee);
        vl = via_at(d, c0, rec);
    }
    while (d >= 0) {
        const int hi = slvl[d + 1];
        // the next step
        int dn = d, cn = c0 + CH;
        if (cn >= hi) {
            dn--;
            while (dn >= 0 && slvl[dn] == slvl[dn + 1]) dn--;
            cn = dn >= 0 ? slvl[dn] : 0;
        }
        DagNode nrec{0, 0, 0, 0};
        int neb = 0, nee = 0;
        if (dn >= 0) fetch(dn, cn, nrec, neb, nee);
        // this step's first edge of the lane's eight-lane group, before it is needed
        const int eg = tid >> 3, b = tid & 7;
        int e = eb + eg;
        DagEdge er{0, 0, 0, 0};
        double ec[ND];
        auto fetch_edge = [&]() {
            er = edge[e];
#pragma unroll
            for (int q = 0; q < ND; q++) ec[q] = b < ND ? ecost[(int64_t)e * (ND * ND) + b * ND + q] : 0.0;
        };
        if (e < ee) fetch_edge();
        const bool valid = c0 + gi < hi;
        const int nc = valid ? (int)(rec.slots >> 28) : 0;
        const int cs = (int)(rec.slots & 0xfffffff);
        const uint64_t act = __ballot(valid);
        if (act) {
            int ncw = nc;
            ncw = max(ncw, __shfl_xor(ncw, 16, 64));
            ncw = max(ncw, __shfl_xor(ncw, 32, 64));
            int range = 0;
            const int fixed = 1 + (int)(rec.pos >> (2 * DAG_POS_BITS));
            const double c = node_cost<L, LDS>(K + (int64_t)cs * ML, nc, ncw, fixed, vl, valid, range);
            if (valid) {
                s_cst[gi][s] = c;
                if (s <= L) R[(c0 + gi) * 16 + s] = (uint8_t)range;
                if (s == 0) s_loc[gi] = (int)rec.loc;
                if (rec.loc == 0) {
                    // the source's layer: the first smallest cost
                    double m = s >= 1 && s <= L ? c : __longlong_as_double(0x7ff0000000000000LL);
                    int ml = s;
#pragma unroll
                    for (int o = 1; o < 16; o <<= 1) {
                        const double om = __shfl_xor(m, o, 16);
                        const int ol = __shfl_xor(ml, o, 16);
                        if (om < m || (om == m && ol < ml)) { m = om; ml = ol; }
                    }
                    if (s == 0) *s_out = m < INF ? ml : 0;
                }
            }
        }
        const float nvl = dn >= 0 ? via_at(dn, cn, nrec) : 0.0f;
        __syncthreads();
        // Parent edges of these nodes (:355-406): eight lanes an edge, a lane
        // per parent layer of the edge's direction, which takes the smallest
        // key over the child's layers to the parent's slot.
        for (; e < ee;) {
            const int ci = (int)er.child - c0;
            const EdgeGeom q = edge_geom(er.from, er.to);
            const uint32_t id = (uint32_t)s_loc[ci] * ID_MUL;
            uint64_t* ks = K + (int64_t)er.slot * ML;
            if (q.dist == 0) {
                // same gcell: every layer continues at no cost
                for (int l = b; l < L; l += 8)
                    atomicMin((unsigned long long*)&ks[l + 1],
                              (unsigned long long)pack_key((float)s_cst[ci][l + 1], id + SENT));
            } else if (q.straight) {
                const int first = dir_first(g, q.vert ? 1 : 0), nd = dir_count(L, first);
                if (b < nd) {
                    uint64_t key = ~0ull;
#pragma unroll
                    for (int f = 0; f < ND; f++) {
                        if (f >= nd || (f != b && q.dist <= 4)) continue;
                        if (f != b && !(ec[f] < INF)) continue;
                        const double cost = s_cst[ci][first + 2 * f + 1] + ec[f];
                        const uint32_t ch = f == b ? SENT : (uint32_t)((first + 2 * f) * L + first + 2 * b);
                        const uint64_t kk = pack_key((float)cost, id + ch);
                        key = kk < key ? kk : key;
                    }
                    atomicMin((unsigned long long*)&ks[first + 2 * b + 1], (unsigned long long)key);
                }
            }
            e += T / 8;
            if (e < ee) fetch_edge();
        }
        __syncthreads();
        d = dn;
        c0 = cn;
        rec = nrec;
        vl = nvl;
        eb = neb;
        ee = nee;
    }

    // Top-down (get_routing_tree_layer_change_cuda, :520-694): a node takes
    // the first of its parent edges whose slot its parent gave to it, and
    // gives each of its own slots to the child behind the smallest key within
    // its layer range (entry 0 of the slot: layer above the key's id).
    for (int dd = 0; dd < nlev; dd++) {
        for (int k = slvl[dd] + tid; k < slvl[dd + 1]; k += T) {
            const DagNode o = node[k];
            int out = -1, ein = 0;
            if (o.loc == 0) {
                out = *s_out;
            } else {
                const int e1 = k + 1 < nn ? (int)node[k + 1].ebeg : ne;
                for (int e = (int)o.ebeg; e < e1; e++) {
                    const uint64_t ch = key_load<LDS>(&K[(int64_t)edge[e].slot * ML]);
                    if (ch == NO_CHILD || (uint32_t)ch / ID_MUL != o.loc) continue;
                    const int choice = (int)((uint32_t)ch % ID_MUL);
                    out = choice == SENT ? (int)(ch >> 32) : choice / L + 1;
                    ein = e;
                    break;
                }
            }
            if (out < 1) continue;
            const int l = (int)(o.pos >> (2 * DAG_POS_BITS));
            int minl = l + 1, maxl = l + 1 == ML ? 1 : minl;
            minl = min(minl, out);
            maxl = max(maxl, out);
            const int code = R[k * 16 + out];
            if (code) {
                const int lo = code & 15, hi = code >> 4, nc = (int)(o.slots >> 28);
                uint64_t* ks = K + (int64_t)(o.slots & 0xfffffff) * ML;
                for (int c = 0; c < nc; c++, ks += ML) {
                    double m = INF;
                    uint64_t pick = NO_CHILD;
                    for (int li = lo; li <= hi; li++) {
                        const uint64_t key = key_load<LDS>(&ks[li]);
                        const double v = unpack_cost(key);
                        if (v < m) {
                            m = v;
                            pick = ((uint64_t)li << 32) | (uint32_t)key;
                        }
                    }
                    key_store<LDS>(ks, pick);
                    if (pick != NO_CHILD) {
                        minl = min(minl, (int)(pick >> 32));
                        maxl = max(maxl, (int)(pick >> 32));
                    }
                }
            }
            dec[o.loc] = make_uint2((uint32_t)ein, (uint32_t)(out | minl << 8 | maxl << 16));
        }
        __syncthreads();
    }

    // Routes in node order: each node's piece of its parent edge, then its
    // via stack; wires and vias are scattered for the fused track update.
    const int XY = g.X * g.Y;
    const int64_t entry = a.rorder[r];
    int* rt = a.routes + dag_route_slot(a.list_node[entry], entry);
    int base = 1;
    for (int k0 = 0; k0 < nn; k0 += T) {
        const int k = k0 + tid;
        const uint2 dc = k < nn ? dec[k] : make_uint2(0, 0);
        const int out = (int)(dc.y & 255), minl = (int)(dc.y >> 8 & 255), maxl = (int)(dc.y >> 16);
        EdgeGeom q{0, 0, 0, 0, 0, false, false};
        int choice = SENT, cx = 0, cy = 0;
        int cnt = 0;
        if (out) {
            const uint32_t p = a.npos[n0 + k];
            cx = pos_x(p);
            cy = pos_y(p);
            if (k > 0) {
                const DagEdge er = edge[dc.x];
                q = edge_geom(er.from, er.to);
                choice = (int)((uint32_t)key_load<LDS>(&K[(int64_t)er.slot * ML]) % ID_MUL);
                if (q.straight && q.dist > 0) cnt = choice == SENT ? 1 : 3;
            }
            if (minl < maxl) cnt++;
        }
        int incl = cnt;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int v = __shfl_up(incl, o, 64);
            if (lane >= o) incl += v;
        }
        int before = 0, total = 0;
        if (NW > 1) {
            if (lane == 63) s_scan[tid >> 6] = incl;
            __syncthreads();
#pragma unroll
            for (int w = 0; w < NW; w++) {
                if (w < tid >> 6) before += s_scan[w];
                total += s_scan[w];
            }
            __syncthreads();
        } else {
            total = __shfl(incl, 63, 64);
        }
        if (cnt) {
            int* o = rt + base + 2 * (before + incl - cnt);
            auto push = [&](int u, int v) {
                o[0] = u;
                o[1] = v;
                o += 2;
            };
            auto cell = [&](int l, int x, int y) { return l * XY + x * g.Y + y; };
            if (k > 0 && q.straight && q.dist > 0) {
                const int px = q.tx, py = q.ty;
                if (choice == SENT) {
                    const int x0 = min(px, cx), x1 = max(px, cx), y0 = min(py, cy), y1 = max(py, cy);
                    add_segment(g, out - 1, x0, x1, y0, y1, a.stamp);
                    push(cell(out - 1, x0, y0), cell(out - 1, x1, y1));
                } else {
                    const int fl = choice / L, tl = choice % L, first = fl & 1;
                    const int ch = a.change[(e0 - a.edge0 + dc.x) * (ND * ND) + (tl - first) / 2 * ND + (fl - first) / 2];
                    const int hx = q.vert ? cx : ch, hy = q.vert ? ch : cy;   // the layer change
                    add_segment(g, fl, min(cx, hx), max(cx, hx), min(cy, hy), max(cy, hy), a.stamp);
                    add_segment(g, tl, min(px, hx), max(px, hx), min(py, hy), max(py, hy), a.stamp);
                    push(cell(fl, min(cx, hx), min(cy, hy)), cell(fl, max(cx, hx), max(cy, hy)));
                    push(cell(min(fl, tl), hx, hy), cell(max(fl, tl), hx, hy));
                    emit_via(g, fl, tl, hx, hy);
                    push(cell(tl, min(px, hx), min(py, hy)), cell(tl, max(px, hx), max(py, hy)));
                }
            }
            if (minl < maxl) {
                push(cell(minl - 1, cx, cy), cell(maxl - 1, cx, cy));
                emit_via(g, minl - 1, maxl - 1, cx, cy);
            }
        }
        base += 2 * total;
    }
    if (tid == 0) {
        rt[0] = base;
        a.rptr[a.nets[r]] = rt;
    }
}

// Workgroups pull the batch's nets from its queue (one counter per batch,
// zero at the pass start) in launch order (dag_order), and exit when the
// counter passes n.
template <int L, int NW>
__global__ void __launch_bounds__(64 * NW) k_dag_net(NetArgs a) {
    extern __shared__ __align__(16) unsigned char s_dyn[];
    __shared__ double s_cst[NW * 4][16];
    __shared__ int s_loc[NW * 4], s_scan[NW], s_out, s_next;
    constexpr int ML = L + 1;
    for (;;) {
        if (threadIdx.x == 0) s_next = atomicAdd(a.queue, 1);
        __syncthreads();
        const int qi = s_next;
        if (qi >= a.n) return;
        const int64_t r = a.net0 + qi;
        const int64_t nn = a.nbase[r + 1] - a.nbase[r], ns = a.sbase[r + 1] - a.sbase[r];
        const int64_t nl = a.lbase[r + 1] - a.lbase[r];
        if (dag_net_lds_bytes(nn, ns, nl, ML) <= a.lds_bytes) {
            uint64_t* K = reinterpret_cast<uint64_t*>(s_dyn);
            uint2* dec = reinterpret_cast<uint2*>(K + ns * ML);
            uint8_t* R = reinterpret_cast<uint8_t*>(dec + nn);
            int* lv = reinterpret_cast<int*>(R + 16 * nn);
            route_net<L, NW, true>(a, r, K, R, dec, lv, s_cst, s_loc, &s_out, s_scan);
        } else {
            const int64_t no = a.nbase[r] - a.node0, so = a.sbase[r] - a.slot0;
            route_net<L, NW, false>(a, r, a.big_key + so * ML, a.big_range + no * 16, a.big_dec + no,
                                    const_cast<int*>(a.lvl) + a.lbase[r] + r, s_cst, s_loc, &s_out, s_scan);
        }
        __syncthreads();   // the tables, s_next and s_out are free again
    }
}

inline unsigned blocks(int64_t n) { return (unsigned)((n + TPB - 1) / TPB); }

__global__ void k_queue_zero(int* p, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * TPB + threadIdx.x;
    if (i < n) p[i] = 0;
}

} // namespace

template <int L>
static void dag_batch(igr_ctx* c, const DagBatch& b, const DagBatch* rip, int stamp) {
    DagDev& D = c->dag;
    const int64_t n = b.net1 - b.net0, ne = b.edge1 - b.edge0;
    hipStream_t st = c->stream;
    const int64_t nr = rip ? rip->net1 - rip->net0 : 0;
    if (ne > 0 || nr > 0) {
        KScope ks(c, K_DAG_EDGES, b.bytes_edges);
        // edges per wave: enough waves to fill the GPU first, then up to a
        // record per lane
        const int64_t per = ne / EDGE_WAVES;
        const int chunk = per >= 64 ? 64 : per >= 32 ? 32 : per >= 16 ? 16 : per >= 8 ? 8 : 4;
        const unsigned eb = (unsigned)((ne + (int64_t)chunk * EW_WAVES - 1) / (chunk * EW_WAVES));
        EdgeArgs a{c->g, D.edge.p + b.edge0, ne, D.cost_edges.p, D.change.p, chunk, eb,
                   rip ? D.nets.p + rip->net0 : nullptr, nr, c->nets.rptr.p, c->bad.p};
        k_dag_edge_costs<L><<<eb + blocks(nr * RIP_LANES), TPB, 0, st>>>(a);
        HIP_OK(hipGetLastError());
    }
    if (n == 0) return;
    KScope ks(c, K_DAG_DP, b.bytes_dp);
    const unsigned grid = (unsigned)std::min<int64_t>(n, c->tune.dag_grid ? c->tune.dag_grid : DEF_DAG_GRID);
    NetArgs a{c->g, D.nrec.p, D.edge.p, D.npos.p, D.lvl.p, D.node_off.p, D.ebase.p, D.sbase.p, D.lbase.p,
              D.rorder.p, D.r_node_off.p, D.cost_edges.p, D.change.p, D.nets.p, b.net0, n, b.edge0,
              D.queue.p + b.index, c->nets.dag_routes.back()->p, c->nets.rptr.p, stamp, b.lds, D.packed.p,
              D.big_range.p, D.big_dec.p, b.node0, b.slot0};
    if (c->tune.dag_waves == 2) k_dag_net<L, 2><<<grid, 128, b.lds, st>>>(a);
    else k_dag_net<L, 4><<<grid, 256, b.lds, st>>>(a);
    HIP_OK(hipGetLastError());
}

void launch_dag_batch_wave(igr_ctx* c, const DagBatch& b, const DagBatch* rip, int stamp) {
    switch (c->g.L) {
#define CASE(LV) case LV: dag_batch<LV>(c, b, rip, stamp); break;
        CASE(1) CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(7) CASE(8) CASE(9) CASE(10) CASE(11) CASE(12)
#undef CASE
    default: throw std::runtime_error("unsupported routing layer count");
    }
}

void launch_dag_queue_reset(igr_ctx* c, int64_t batches) {
    const int64_t n = std::max<int64_t>(1, batches);
    c->dag.queue.alloc(n);
    k_queue_zero<<<blocks(n), TPB, 0, c->stream>>>(c->dag.queue.p, n);
    HIP_OK(hipGetLastError());
}

} // namespace igr_dev
