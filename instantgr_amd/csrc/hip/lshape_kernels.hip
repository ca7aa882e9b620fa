// L-shape pattern routing with 3-D layer assignment (src/Lshape_route.hpp:9-153).
//
// Plain form: one thread per net, the reference's launch structure.  The
// per-node DP tables (dist over layer ranges, back-pointers) live in a
// per-batch global scratch slab; each thread walks its tree bottom-up, then
// traces the chosen layer ranges top-down, writes the route and adds its wire
// segments to the demand difference array.  The arithmetic follows the
// reference exactly: FP64 accumulation in the same order (sequential via
// sums, children added in decreasing node order), strict '<' keeping the
// first minimum and '<=' in the layer-range prefix minimum.
#include "dag_dev.h"
#include "igr_ctx.hpp"
#include "row.h"

namespace igr_dev {

namespace {

constexpr int TPB = 256;

template <int L>
__global__ void __launch_bounds__(TPB) k_lshape_plain(GridDev g, const int* nets, const int64_t* scr_off, int64_t n,
                                                      const int64_t* node_off, const int* node, const int* parent,
                                                      const int64_t* route_off, int* routes, double* dist, int* from,
                                                      int* lrbuf, int stamp) {
    int64_t t = (int64_t)blockIdx.x * TPB + threadIdx.x;
    if (t >= n) return;
    constexpr int LL = L * L;
    const int net = nets[t];
    const int64_t nb = node_off[net];
    const int nn = (int)(node_off[net + 1] - nb);
    const int* nd_pos = node + nb;
    const int* par = parent + nb;
    double* D = dist + scr_off[t] * LL;
    int* F = from + scr_off[t] * LL;
    int* lr = lrbuf + scr_off[t];
    int* r = routes + route_off[net];
    const int X = g.X, Y = g.Y, XY = X * Y;

    for (int i = 0; i < nn; i++) {
        int l = nd_pos[i] / XY, x = nd_pos[i] / Y % X, y = nd_pos[i] % Y;
        double* nd = D + i * LL;
        for (int minl = 0; minl < L; minl++) {
            nd[minl * L + minl] = 0;
            for (int maxl = minl + 1; maxl < L; maxl++)
                nd[minl * L + maxl] = nd[minl * L + maxl - 1] + (double)g.vcost[gidx(g, maxl - 1, x, y)];
            for (int maxl = minl; maxl < L; maxl++)
                if (l < L && (minl > l || maxl < l)) nd[minl * L + maxl] = INF;
        }
    }
    double mcc[L], mcp[LL];
    int cur_from[L];
    for (int i = nn - 1; i >= 1; i--) {
        int x = nd_pos[i] / Y % X, y = nd_pos[i] % Y;
        int p = par[i];
        int px = nd_pos[p] / Y % X, py = nd_pos[p] % Y;
        int minx = min(x, px), maxx = max(x, px), miny = min(y, py), maxy = max(y, py);
        const double* nd = D + i * LL;
        double* pd = D + p * LL;
        int* prev = F + i * LL;
        for (int l = 0; l < L; l++) {
            mcc[l] = mcp[l * L + l] = INF;
            cur_from[l] = 0;
            for (int minl = 0; minl <= l; minl++)
                for (int maxl = l; maxl < L; maxl++)
                    if (nd[minl * L + maxl] < mcc[l]) { mcc[l] = nd[minl * L + maxl]; cur_from[l] = minl * L + maxl; }
        }
        if (x == px || y == py) {
            for (int l = 0; l < L; l++) {
                if (layer_dir(l, g.DIR) == 0 && y != py) continue;
                if (layer_dir(l, g.DIR) == 1 && x != px) continue;
                mcp[l * L + l] = mcc[l] + wseg(g, l, minx, maxx, miny, maxy);
                prev[l * L + l] = cur_from[l] * LL + l * L + l;
            }
        } else {
            for (int curl = 0; curl < L; curl++) {
                double cost = mcc[curl];
                const int cd = layer_dir(curl, g.DIR);
                if (cd == 1) cost += wseg(g, curl, x, x, miny, maxy);
                else cost += wseg(g, curl, minx, maxx, y, y);
                for (int parl = (curl & 1) ^ 1; parl < L; parl += 2) {
                    double cost2 = 0;
                    for (int l = min(curl, parl) + 1; l < max(curl, parl); l++)
                        cost2 += (double)(cd == 1 ? g.vcost[gidx(g, l, x, py)] : g.vcost[gidx(g, l, px, y)]);
                    if (layer_dir(parl, g.DIR) == 1) cost2 += wseg(g, parl, px, px, miny, maxy);
                    else cost2 += wseg(g, parl, minx, maxx, py, py);
                    if (cost + cost2 < mcp[parl * L + parl]) {
                        mcp[parl * L + parl] = cost + cost2;
                        prev[parl * L + parl] = cur_from[curl] * LL + curl * L + parl;
                    }
                }
            }
        }
        for (int minl = 0; minl < L; minl++) {
            for (int maxl = minl + 1; maxl < L; maxl++) {
                if (mcp[minl * L + maxl - 1] <= mcp[maxl * L + maxl]) {
                    mcp[minl * L + maxl] = mcp[minl * L + maxl - 1];
                    prev[minl * L + maxl] = prev[minl * L + maxl - 1];
                } else {
                    mcp[minl * L + maxl] = mcp[maxl * L + maxl];
                    prev[minl * L + maxl] = prev[maxl * L + maxl];
                }
            }
            for (int maxl = minl; maxl < L; maxl++) pd[minl * L + maxl] += mcp[minl * L + maxl];
        }
    }

    int cnt = 1;
    lr[0] = 0;
    for (int minl = 0; minl < L; minl++)
        for (int maxl = minl; maxl < L; maxl++)
            if (D[minl * L + maxl] < D[lr[0]]) lr[0] = minl * L + maxl;
    auto push = [&](int a, int b) { r[cnt] = a; r[cnt + 1] = b; cnt += 2; };
    for (int i = 0; i < nn; i++) {
        const int* prev = F + i * LL;
        if (i > 0) lr[i] = prev[lr[par[i]]] / LL;
        int minl = lr[i] / L, maxl = lr[i] % L;
        int x = nd_pos[i] / Y % X, y = nd_pos[i] % Y;
        if (minl < maxl) {
            push(minl * XY + x * Y + y, maxl * XY + x * Y + y);
            if (g.vc) emit_via(g, minl, maxl, x, y);
        }
        if (i == 0) continue;
        int p = par[i];
        int px = nd_pos[p] / Y % X, py = nd_pos[p] % Y;
        int minx = min(x, px), maxx = max(x, px), miny = min(y, py), maxy = max(y, py);
        int code = prev[lr[p]];
        int curl = code / L % L, parl = code % L;
        if (px == x || py == y) {
            push(curl * XY + minx * Y + miny, curl * XY + maxx * Y + maxy);
            add_segment(g, curl, minx, maxx, miny, maxy, stamp);
        } else if (layer_dir(curl, g.DIR) == 1) {
            push(curl * XY + x * Y + y, curl * XY + x * Y + py);
            add_segment(g, curl, x, x, miny, maxy, stamp);
            push(curl * XY + x * Y + py, parl * XY + x * Y + py);
            if (g.vc) emit_via(g, curl, parl, x, py);
            push(parl * XY + x * Y + py, parl * XY + px * Y + py);
            add_segment(g, parl, minx, maxx, py, py, stamp);
        } else {
            push(curl * XY + x * Y + y, curl * XY + px * Y + y);
            add_segment(g, curl, minx, maxx, y, y, stamp);
            push(curl * XY + px * Y + y, parl * XY + px * Y + y);
            if (g.vc) emit_via(g, curl, parl, px, y);
            push(parl * XY + px * Y + y, parl * XY + px * Y + py);
            add_segment(g, parl, px, px, miny, maxy, stamp);
        }
    }
    r[0] = cnt;
}


// ---------------------------------------------------------------------------
// Batched form: a row of 16 lanes per net, four nets per wave, lane s for
// layer s - 1.  A node's cost over its layer ranges is never stored: with its
// children's edge costs per layer in LDS (L doubles a node), lane hi forms the
// cost of every range [low, hi] (via stack, then the children in decreasing
// node order, each the running minimum of its edge costs over the range), and
// the row keeps per layer the smallest range that holds it and its two ends,
// ties to the smaller low, then the smaller hi.  The same FP64 operations in
// the same order as the thread-per-net kernel above, so routes and costs are
// bit-identical.  Which child layers a range used is found again on the way
// down, for the ranges chosen.
//
// Nets are short chains of nodes, so a net's time is the latency of a node
// (some 1350 instructions): the prefix sums and via costs of the next node and
// its parent edge are loaded while the current one is worked on.  One launch
// takes a batch: nets of one wave have similar node counts (the device sorts
// them), and at most 3.4 KB of LDS a net (24 nodes, 12 layers; 2.8 with 9)
// leave the waves to the registers.  With
// the layer-range tables in LDS (450 bytes a node), the grid read inside the
// chain and a launch per node-count class, a batch took 295 us on 200x200 (20k
// nets, 40 batches), 252 us on 800x800 (500k nets, 58 batches) and 315 us on
// 1237x989 with 11 layers; this kernel takes 43, 71 and 80 us.
// ---------------------------------------------------------------------------
// What a node's step reads from the grid, by lane.
struct NodeIn {
    float vl;                     // via cut of layer lane (lanes 0 .. L - 2) at the node
    double wc, wp;                // the edge's wire on the lane's layer at the node's side, at the parent's
    float va, vb;                 // via cut of the lane's layer at the L corners (x, py) and (px, y)
};

// Batches of at most this many nets leave most of the chip's 1024 SIMDs idle
// with four nets a wave, and a batch then takes as long as its longest net: a
// wave takes one net, its four rows up to four nodes of a depth level.  Larger
// batches are bound by the instructions issued, which one net a wave does not
// reduce.  Four nets a wave against one, us a launch inside pattern passes with
// 9 layers, by the batch's nets: up to 512 43 / 32, 513..1024 70 / 49, 1025..2048
// 76 / 50, 3073..4096 78 / 64, 4097..5120 83 / 76, 5121..6144 86 / 89, 8193..9216
// 94 / 107; with 11 layers the two meet near 11000.
constexpr int64_t LSWAVE_WIDE_NETS = 5120;
__host__ __device__ constexpr int lswave_net_lds(int L, int cap) { return (cap * (8 * L + 12 + 34) + 15) / 16 * 16; }

template <int L, bool WIDE>
__global__ void __launch_bounds__(64) k_lshape_wave(GridDev g, const int* __restrict__ nets, int64_t n, int cap,
                                                    const int64_t* __restrict__ node_off,
                                                    const int* __restrict__ node, const int* __restrict__ parent,
                                                    const int64_t* __restrict__ route_off, int* routes, int stamp) {
    constexpr int LL = L * L;
    extern __shared__ __align__(16) double s_dyn[];
    // per net, cap nodes of: edge cost by parent layer; position, parent, the
    // choice made on the way down; by layer, the edge's child layer and the
    // best range's ends; last child and next lower sibling (0: none)
    const int gi = threadIdx.x >> 4, lane = threadIdx.x & 15, s = lane;
    unsigned char* base = reinterpret_cast<unsigned char*>(s_dyn) + (WIDE ? 0 : gi * lswave_net_lds(L, cap));
    double* mcp = reinterpret_cast<double*>(base);
    int* pos = reinterpret_cast<int*>(mcp + cap * L);
    int* par = pos + cap;
    int* pick = par + cap;
    uint8_t* curl_of = reinterpret_cast<uint8_t*>(pick + cap);
    uint8_t* range_of = curl_of + 16 * cap;
    uint8_t* child_of = range_of + 16 * cap;
    uint8_t* sib_of = child_of + cap;
    // WIDE: the nodes by falling depth, and the ends of each one's level there
    uint8_t* ord = reinterpret_cast<uint8_t*>(s_dyn) + lswave_net_lds(L, cap);
    uint8_t* lvl_beg = ord + cap;
    uint8_t* lvl_end = lvl_beg + cap;
    const int64_t t = WIDE ? blockIdx.x : (int64_t)blockIdx.x * 4 + gi;
    int nn = 0, net = 0;
    int64_t nb = 0;
    if (t < n) {
        net = nets[t];
        nb = node_off[net];
        nn = (int)(node_off[net + 1] - nb);
    }
    const int X = g.X, Y = g.Y, XY = X * Y;
    for (int k = lane; k < nn; k += 16) {
        pos[k] = node[nb + k];
        par[k] = parent[nb + k];
    }
    int nmax = nn;
    nmax = max(nmax, __shfl_xor(nmax, 16, 64));
    nmax = max(nmax, __shfl_xor(nmax, 32, 64));
    __syncthreads();
    for (int k = lane; k < nn; k += 16) {
        const int p = par[k];
        int c = 0, b = 0;
        for (int q = 1; q < nn; q++) {
            const int pq = par[q];
            if (pq == k) c = q;
            if (q < k && pq == p) b = q;
        }
        child_of[k] = (uint8_t)c;
        sib_of[k] = (uint8_t)b;
        if (WIDE) {
            int d = 0;
            for (int q = k; q > 0; q = par[q]) d++;
            pick[k] = d;
        }
    }
    __syncthreads();
    if (WIDE) {
        for (int k = lane; k < nn; k += 16) {
            const int d = pick[k];
            int deeper = 0, same = 0, before = 0;
            for (int q = 0; q < nn; q++) {
                const int dq = pick[q];
                deeper += dq > d;
                same += dq == d;
                before += dq == d && q > k;
            }
            ord[deeper + before] = (uint8_t)k;
            lvl_beg[deeper + before] = (uint8_t)deeper;
            lvl_end[deeper + before] = (uint8_t)(deeper + same);
        }
        __syncthreads();
    }
    // The row's node in the step that starts at 'at' (WIDE: up to four nodes of
    // a level from there; else node 'at' of the row's own net), -1 for none.
    auto node_at = [&](int at) {
        if (!WIDE) return at < nn ? at : -1;
        return at >= 0 && at < nn && at + gi < lvl_end[at] ? (int)ord[at + gi] : -1;
    };
    const int l = s - 1;                               // the lane's layer
    const bool on = s >= 1 && s <= L;
    const int dl = layer_dir(l & 15, g.DIR);
    auto fetch = [&](int i) {
        NodeIn in{0, 0, 0, 0, 0};
        if (i < 0) return in;
        const int v = pos[i] % XY, x = v / Y, y = v - x * Y;
        if (lane < L - 1) in.vl = g.vcost[gidx(g, lane, x, y)];
        if (i > 0 && on) {
            const int u = pos[par[i]] % XY, px = u / Y, py = u - px * Y;
            const int minx = min(x, px), maxx = max(x, px), miny = min(y, py), maxy = max(y, py);
            if (x == px || y == py) {
                if ((dl == 0 && y == py) || (dl == 1 && x == px)) in.wc = wseg(g, l, minx, maxx, miny, maxy);
            } else {
                in.wc = dl == 1 ? wseg(g, l, x, x, miny, maxy) : wseg(g, l, minx, maxx, y, y);
                in.wp = dl == 1 ? wseg(g, l, px, px, miny, maxy) : wseg(g, l, minx, maxx, py, py);
                in.va = g.vcost[gidx(g, l, x, py)];
                in.vb = g.vcost[gidx(g, l, px, y)];
            }
        }
        return in;
    };
    const double PINF = __longlong_as_double(0x7ff0000000000000LL);
    int step = WIDE ? 0 : nmax - 1;
    NodeIn in = fetch(node_at(step));
    while (WIDE ? step < nn : step >= 0) {
        const int after = WIDE ? min(step + 4, (int)lvl_end[step]) : step - 1;
        const NodeIn next = (WIDE ? after < nn : after >= 0) ? fetch(node_at(after)) : NodeIn{0, 0, 0, 0, 0};
        const int own_node = node_at(step), i = max(own_node, 0);
        const bool act = own_node >= 0;
        const bool root = WIDE ? step == nn - 1 : step == 0;
        const int v = act ? pos[i] : 0;
        const int pl = v / XY;                         // the pin's layer, L for none
        // cost[low - 1] of the range [low, s]
        double cost[L], vm[L];
        unrolled<L - 1>([&](auto I) {
            const float via = row_bcast<I>(in.vl);
            vm[I] = I + 2 <= s ? (double)via : 0.0;    // zero above the range's top
        });
        unrolled<L>([&](auto I) {
            double acc = 0.0;
#pragma unroll
            for (int k = I; k < L - 1; k++) acc += vm[k];
            cost[I] = acc;
        });
        // children, in decreasing node order
        for (int c = act ? child_of[i] : 0; __ballot(c != 0); c = c ? sib_of[c] : 0) {
            const double e = c && on ? mcp[c * L + l] : 0.0;
            double m = e;
            unrolled<L>([&](auto I) {
                constexpr int low = L - I;
                const double below = row_bcast<low>(e);
                m = below < m ? below : m;
                m = low >= s ? e : m;
                cost[low - 1] += m;
            });
        }
        // per layer, the smallest range through it
        double best = INF;
        int code = 0;
        uint64_t at = 0;
        unrolled<L>([&](auto I) {
            constexpr int low = I + 1;
            const bool ok = act & on & (s >= low) & ((pl >= L) | ((low - 1 <= pl) & (pl < s))) & (cost[I] < INF);
            const double own = ok ? cost[I] : PINF;
            double c = own;
            auto lower = [&](double o) { c = o < c ? o : c; };
            lower(row_above<1>(c));
            lower(row_above<2>(c));
            if constexpr (L > 4) lower(row_above<4>(c));
            if constexpr (L > 8) lower(row_above<8>(c));
            const uint64_t mine = __ballot(own == c);
            const bool better = (s >= low) & (c < best);
            best = better ? c : best;
            code = better ? low : code;
            at = better ? mine : at;
        });
        if (code) code |= (s + __builtin_ctzll(at >> (threadIdx.x & 63))) << 4;
        if (act && on) range_of[i * 16 + l] = (uint8_t)code;
        if (root) {
            // the root's range: the smallest cost, ties to the smaller low,
            // then the smaller hi (every range through the best layer is one
            // of the candidates, so the row's smallest (cost, range) is it)
            double m = on ? best : PINF;
            int cd = on && code ? (code & 15) << 4 | code >> 4 : 0x11;
#pragma unroll
            for (int o = 1; o < 16; o <<= 1) {
                const double om = __shfl_xor(m, o, 16);
                const int oc = __shfl_xor(cd, o, 16);
                if (om < m || (om == m && oc < cd)) { m = om; cd = oc; }
            }
            if (lane == 0 && act) pick[0] = (cd >> 4) | (cd & 15) << 4;
            break;
        }
        // edge to the parent: cost by parent layer and the child layer it uses
        double up = INF;
        int uc = 0;
        int u = 0;
        if (act) u = pos[par[i]] % XY;
        const int w = v % XY;
        const bool straight = w / Y == u / Y || w % Y == u % Y;
        if (__ballot(act && straight)) {
            const bool along = dl == 0 ? w % Y == u % Y : w / Y == u / Y;
            if (act && straight && on && along) {
                up = best + in.wc;
                uc = l;
            }
        }
        if (__ballot(act && !straight)) {
            const double from = best + in.wc;
            double cu = INF;
            int cc = 0;
            unrolled<L>([&](auto I) {
                // child layer I; the corner's vias lie on the layers between,
                // where the child's direction meets the parent's
                constexpr int cl = I;
                const bool vert = layer_dir(cl, g.DIR) == 1;
                const double cost1 = row_bcast<cl + 1>(from);
                double cost2 = 0.0;
                unrolled<L>([&](auto K) {
                    constexpr int k = K;
                    if constexpr (k != cl && k != 0) {
                        const float cut = row_bcast<k + 1>(vert ? in.va : in.vb);
                        const bool between = k > cl ? k < l : k > l;
                        cost2 += between ? (double)cut : 0.0;
                    }
                });
                cost2 += in.wp;
                const double sum = cost1 + cost2;
                const bool take = (((cl ^ l) & 1) != 0) & (sum < cu);
                cu = take ? sum : cu;
                cc = take ? cl : cc;
            });
            if (!straight) { up = cu; uc = cc; }
        }
        if (act && on) {
            mcp[i * L + l] = up;
            curl_of[i * 16 + l] = (uint8_t)uc;
        }
        __syncthreads();
        in = next;
        step = after;
    }
    __syncthreads();
    // Top-down (parents first): within the parent's range the lowest of the
    // cheapest layers, the child layer its edge uses, and that layer's range.
    for (int at2 = WIDE ? nn - 2 : 1; WIDE ? at2 >= 0 : at2 < nmax;) {
        const int first = WIDE ? max((int)lvl_beg[at2], at2 - 3) : at2;
        const int node2 = WIDE ? (first + gi <= at2 ? (int)ord[first + gi] : -1) : at2 < nn ? at2 : -1;
        const int i = max(node2, 0);
        const bool act = node2 >= 0;
        at2 = WIDE ? first - 1 : at2 + 1;
        const int up = act ? pick[par[i]] : 0;
        const int low = up & 15, hi = up >> 4 & 15;
        double c = act && s >= low && s <= hi ? mcp[i * L + l] : PINF;
        const double own = c;
#pragma unroll
        for (int o = 1; o < 16; o <<= 1) {
            const double oc = __shfl_xor(c, o, 16);
            c = oc < c ? oc : c;
        }
        const uint64_t mine = __ballot(act && own == c) >> (threadIdx.x & 48);
        if (act) {
            const int parl = __builtin_ctzll(mine | 1ull << 16) - 1;
            const int curl = parl < L ? curl_of[i * 16 + parl] : 0;
            const int code = range_of[i * 16 + curl];
            if (lane == 0) pick[i] = (code ? code : 0x11) | curl << 8 | (parl & 15) << 12;
        }
        __syncthreads();
    }
    if (t >= n || (WIDE && gi != 0)) return;
    // Route pairs in node order: the node's via stack, then the edge to its
    // parent (one piece, or wire-via-wire for an L).
    int* r = routes + route_off[net];
    int done = 0;
    for (int c0 = 0; c0 < nn; c0 += 16) {
        const int i = c0 + lane;
        int cnt = 0;
        int minl = 0, maxl = 0, x = 0, y = 0, px = 0, py = 0, curl = 0, parl = 0;
        if (i < nn) {
            const int pk = pick[i], v = pos[i] % XY;
            minl = (pk & 15) - 1;
            maxl = (pk >> 4 & 15) - 1;
            x = v / Y;
            y = v - x * Y;
            cnt = minl < maxl;
            if (i > 0) {
                const int u = pos[par[i]] % XY;
                px = u / Y;
                py = u - px * Y;
                curl = pk >> 8 & 15;
                parl = pk >> 12;
                cnt += (px == x || py == y) ? 1 : 3;
            }
        }
        int incl = cnt;
        for (int off = 1; off < 16; off <<= 1) {
            const int v = __shfl_up(incl, off, 16);
            if (lane >= off) incl += v;
        }
        const int total = __shfl(incl, 15, 16);
        if (i < nn) {
            int* o = r + 1 + 2 * (done + incl - cnt);
            auto push = [&](int a, int b) {
                o[0] = a;
                o[1] = b;
                o += 2;
            };
            if (minl < maxl) {
                push(minl * XY + x * Y + y, maxl * XY + x * Y + y);
                if (g.vc) emit_via(g, minl, maxl, x, y);
            }
            if (i > 0) {
                const int minx = min(x, px), maxx = max(x, px), miny = min(y, py), maxy = max(y, py);
                if (px == x || py == y) {
                    push(curl * XY + minx * Y + miny, curl * XY + maxx * Y + maxy);
                    add_segment(g, curl, minx, maxx, miny, maxy, stamp);
                } else {
                    // the corner (x, py) when the child's layer runs along y, else (px, y)
                    const bool vert = layer_dir(curl, g.DIR) == 1;
                    const int hx = vert ? x : px, hy = vert ? py : y;
                    push(curl * XY + x * Y + y, curl * XY + hx * Y + hy);
                    add_segment(g, curl, min(x, hx), max(x, hx), min(y, hy), max(y, hy), stamp);
                    push(curl * XY + hx * Y + hy, parl * XY + hx * Y + hy);
                    if (g.vc) emit_via(g, curl, parl, hx, hy);
                    push(parl * XY + hx * Y + hy, parl * XY + px * Y + py);
                    add_segment(g, parl, min(px, hx), max(px, hx), min(py, hy), max(py, hy), stamp);
                }
            }
        }
        done += total;
    }
    if (lane == 0) r[0] = 1 + 2 * done;
}

} // namespace

void launch_lshape_wave(igr_ctx* c, const int* d_nets, int64_t n, int nodes, int stamp, double bytes) {
    if (n == 0) return;
    if (nodes < 1 || nodes > LSWAVE_MAX_NODES) throw std::runtime_error("L-shape node count out of range");
    KScope ks(c, K_LSHAPE, bytes);
    NetsDev& N = c->nets;
    const bool wide = n <= LSWAVE_WIDE_NETS;
    const unsigned grid = (unsigned)(wide ? n : (n + 3) / 4);
#define ARGS c->g, d_nets, n, nodes, N.node_off.p, N.node.p, N.parent.p, N.route_off.p, N.routes.p, stamp
#define CASE(LV)                                                                                                    \
    case LV:                                                                                                        \
        if (wide) k_lshape_wave<LV, true><<<grid, 64, lswave_net_lds(LV, nodes) + 3 * nodes, c->stream>>>(ARGS);     \
        else k_lshape_wave<LV, false><<<grid, 64, 4 * lswave_net_lds(LV, nodes), c->stream>>>(ARGS);                \
        break;
    switch (c->g.L) {
        CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(7) CASE(8) CASE(9) CASE(10) CASE(11) CASE(12)
    default: throw std::runtime_error("unsupported routing layer count");
    }
#undef CASE
#undef ARGS
    HIP_OK(hipGetLastError());
}

void launch_lshape_plain(igr_ctx* c, const int* d_nets, const int64_t* d_scr_off, int64_t n, int stamp,
                         double bytes) {
    if (n == 0) return;
    KScope ks(c, K_LSHAPE, bytes);
    const unsigned grid = (unsigned)((n + TPB - 1) / TPB);
    NetsDev& N = c->nets;
#define CASE(LV)                                                                                               \
    case LV:                                                                                                   \
        k_lshape_plain<LV><<<grid, TPB, 0, c->stream>>>(c->g, d_nets, d_scr_off, n, N.node_off.p, N.node.p,    \
                                                        N.parent.p, N.route_off.p, N.routes.p,                 \
                                                        c->scratch.dist.p, c->scratch.from.p, c->scratch.lr.p, \
                                                        stamp);                                                \
        break;
    switch (c->g.L) {
        CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(7) CASE(8) CASE(9) CASE(10) CASE(11) CASE(12)
    default: throw std::runtime_error("unsupported routing layer count");
    }
#undef CASE
    HIP_OK(hipGetLastError());
}

} // namespace igr_dev
