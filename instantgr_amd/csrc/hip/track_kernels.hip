// Batched form of the grid updates: one fused pass per dirty track.
//
// Between two routed batches the reference runs, over the whole grid, the
// wire-demand scan and commit (src/graph.hpp:104-137), the via commit
// (:496-543), for rip-up batches the wire and via rip-up (:468-543 with
// K = -1), then the logistic cost update (:40-71) and the FP64 prefix sums
// (:405-430).  Each of these only touches cells of one track (a via cut at
// (l, x, y) adds demand to the two edges of that cell's track on layer l), so
// one workgroup per track does them all in registers, in the reference's
// order, and streams each array once:
//   1. wire commit: inclusive scan of the difference array, demand += count,
//      timestamp = commit stamp on covered edges;
//   2. via commit: cuts whose cell timestamp is older than the commit stamp
//      add half a track to each adjacent edge (a whole one at track ends);
//   3. rip-up of the next batch: demand -= covering wire count, timestamp =
//      rip stamp on covered cells, then the gated via cuts subtract;
//   4. wcost / vcost from the new demand, FP64 prefix sums of wcost.
// Demand changes by integers and halves, so from demand on the half grid, which
// every pass leaves, the result equals the sequential one; from any other float
// demand the FP32 sums round in the order above, a batch's count at a time.  A
// track no scatter touched keeps its demand and so its costs: the routing
// kernels and the rip-up scatter flag every track they write into.
#include "dag_dev.h"
#include "igr_ctx.hpp"
#include "scan.h"

namespace igr_dev {

namespace {

constexpr int SB = 256;   // block size of the scatter and fill kernels

// Inclusive sums of a wave's lanes (integers: any order).
__device__ __forceinline__ int wave_sum(int v) {
    v += dpp_move<0x111, 0xf, 0xf>(0, v);
    v += dpp_move<0x112, 0xf, 0xf>(0, v);
    v += dpp_move<0x114, 0xf, 0xf>(0, v);
    v += dpp_move<0x118, 0xf, 0xf>(0, v);
    v += dpp_move<0x142, 0xa, 0xf>(0, v);
    v += dpp_move<0x143, 0xc, 0xf>(0, v);
    return v;
}
__device__ __forceinline__ int row_sum(int v) {
    v += dpp_move<0x111, 0xf, 0xf>(0, v);
    v += dpp_move<0x112, 0xf, 0xf>(0, v);
    v += dpp_move<0x114, 0xf, 0xf>(0, v);
    v += dpp_move<0x118, 0xf, 0xf>(0, v);
    return v;
}

// Inclusive prefix sums of three integer arrays over the workgroup, with one
// barrier (tot: the waves' totals).
template <int K>
__device__ __forceinline__ void block_sums(int (&a)[K], int (&b)[K], int (&c)[K], int4* tot, int nw) {
#pragma unroll
    for (int j = 1; j < K; j++) {
        a[j] += a[j - 1];
        b[j] += b[j - 1];
        c[j] += c[j - 1];
    }
    const int ta = a[K - 1], tb = b[K - 1], tc = c[K - 1];
    int pa = wave_sum(ta), pb = wave_sum(tb), pc = wave_sum(tc);
    if (nw > 1) {
        const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        if (lane == 63) tot[wave] = make_int4(pa, pb, pc, 0);
        __syncthreads();
        const int4 t = (lane & 15) < nw ? tot[lane & 15] : make_int4(0, 0, 0, 0);
        const int sa = row_sum(t.x), sb = row_sum(t.y), sc = row_sum(t.z);
        if (wave > 0) {
            pa += lane_read(sa, wave - 1);
            pb += lane_read(sb, wave - 1);
            pc += lane_read(sc, wave - 1);
        }
    }
#pragma unroll
    for (int j = 0; j < K; j++) {
        a[j] += pa - ta;
        b[j] += pb - tb;
        c[j] += pc - tc;
    }
}

// K consecutive elements of a track per thread.  With K a multiple of 4 and
// 16-byte aligned tracks (v4), four elements move in one 16-byte access, so a
// wave reads or writes one contiguous span.
template <int K, typename T, typename V4>
__device__ __forceinline__ void load_k(const T* __restrict__ src, int64_t base, int p0, int len, bool v4,
                                       T (&dst)[K]) {
    if constexpr (K % 4 == 0) {
        if (v4) {
#pragma unroll
            for (int j = 0; j < K; j += 4) {
                if (p0 + j < len) {
                    const V4 q = *reinterpret_cast<const V4*>(src + base + p0 + j);
                    dst[j] = q.x; dst[j + 1] = q.y; dst[j + 2] = q.z; dst[j + 3] = q.w;
                } else {
                    dst[j] = dst[j + 1] = dst[j + 2] = dst[j + 3] = T(0);
                }
            }
            return;
        }
    }
#pragma unroll
    for (int j = 0; j < K; j++) dst[j] = p0 + j < len ? src[base + p0 + j] : T(0);
}

template <int K>
__device__ __forceinline__ void store_k(float* __restrict__ dst, int64_t base, int p0, int len, bool v4,
                                        const float (&v)[K]) {
    if constexpr (K % 4 == 0) {
        if (v4) {
#pragma unroll
            for (int j = 0; j < K; j += 4)
                if (p0 + j < len)
                    *reinterpret_cast<float4*>(dst + base + p0 + j) = make_float4(v[j], v[j + 1], v[j + 2], v[j + 3]);
            return;
        }
    }
#pragma unroll
    for (int j = 0; j < K; j++)
        if (p0 + j < len) dst[base + p0 + j] = v[j];
}

template <int K>
__device__ __forceinline__ void store_k(double* __restrict__ dst, int64_t base, int p0, int len, bool v4,
                                        const double (&v)[K]) {
    if constexpr (K % 4 == 0) {
        if (v4) {
#pragma unroll
            for (int j = 0; j < K; j += 2)
                if (p0 + j < len) *reinterpret_cast<double2*>(dst + base + p0 + j) = make_double2(v[j], v[j + 1]);
            return;
        }
    }
#pragma unroll
    for (int j = 0; j < K; j++)
        if (p0 + j < len) dst[base + p0 + j] = v[j];
}

// Via cuts gv at the cells apply sign * (1 or 1/2) to the adjacent edges.
template <int K>
__device__ __forceinline__ void apply_vias(float (&dem)[K], const int (&gv)[K], int gnext, int len, float sign) {
#pragma unroll
    for (int j = 0; j < K; j++) {
        const int e = threadIdx.x * K + j;
        if (e > len - 2) continue;
        const int g0 = gv[j];
        const int g1 = j + 1 < K ? gv[j + 1] : gnext;
        if (g0) dem[j] += sign * (e == 0 ? (float)g0 : 0.5f * (float)g0);
        if (g1) dem[j] += sign * (e + 1 == len - 1 ? (float)g1 : 0.5f * (float)g1);
    }
}

// Wire costs, via costs and the exclusive prefix inputs (the predecessor's
// wire cost) of a thread's K cells from their demand and capacity.  The
// increments are formed once per cell; those of the cell before the thread's
// first come from the thread before (sh: one entry per wave, one barrier).
struct CellCost {
    double a1, ah;                // increments of one and of half a track
    float wc;
};
template <int K, bool TAB>
__device__ __forceinline__ void own_costs(const GridDev& g, int l, int len, int p0, const float (&dem)[K],
                                          const float (&cap)[K], const int (&el)[K], const float* tab,
                                          double (&a1)[K], double (&ah)[K], float (&wc)[K]) {
    const double w = g.w[l];
#pragma unroll
    for (int j = 0; j < K; j++) {
        inc_pair<TAB>(cap[j], dem[j], w, tab, a1[j], ah[j]);
        const float x = (float)a1[j];
        const float y = (float)((double)x + g.unit_wire * (double)el[j]);
        wc[j] = p0 + j < len - 1 ? y : x;
    }
}
template <int K>
__device__ __forceinline__ void track_costs(const GridDev& g, int l, int dir, int len, int p0, const float (&dem)[K],
                                            const float (&cap)[K], const float* tab, CellCost* sh, float (&wc)[K],
                                            float (&vc)[K], double (&s)[K]) {
    const int* elen = dir ? g.ylen : g.xlen;
    int el[K];                    // edge lengths, 0 from the last cell on
    if (K % 4 == 0 && p0 + K <= len - 1) {
#pragma unroll
        for (int j = 0; j < K; j += 4) {
            const int4 q = *reinterpret_cast<const int4*>(elen + p0 + j);
            el[j] = q.x; el[j + 1] = q.y; el[j + 2] = q.z; el[j + 3] = q.w;
        }
    } else {
#pragma unroll
        for (int j = 0; j < K; j++) el[j] = p0 + j < len - 1 ? elen[p0 + j] : 0;
    }
    bool q = true;
#pragma unroll
    for (int j = 0; j < K; j++) q = q && quarter_grid(cap[j], dem[j]);
    double a1[K], ah[K];
    // the exponents come from the table when every element of the wave allows
    // it, else they are computed; the values are the same either way
    if (__all(q)) own_costs<K, true>(g, l, len, p0, dem, cap, el, tab, a1, ah, wc);
    else own_costs<K, false>(g, l, len, p0, dem, cap, el, tab, a1, ah, wc);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 63) sh[wave] = CellCost{a1[K - 1], ah[K - 1], wc[K - 1]};
    __syncthreads();
    double a1p = __shfl_up(a1[K - 1], 1), ahp = __shfl_up(ah[K - 1], 1);
    float wcp = __shfl_up(wc[K - 1], 1);
    if (lane == 0 && wave > 0) {
        const CellCost c = sh[wave - 1];
        a1p = c.a1;
        ahp = c.ah;
        wcp = c.wc;
    }
#pragma unroll
    for (int j = 0; j < K; j++) {
        const int p = p0 + j;
        float v;
        if (p == 0) v = (float)a1[j];
        else if (p == len - 1) v = (float)a1p;
        else v = (float)(ah[j] + ahp);
        const bool in = p < len;
        vc[j] = in ? (float)((double)v + g.unit_via) : 0.0f;
        s[j] = in && p >= 1 ? (double)wcp : 0.0;   // exclusive prefix input
        a1p = a1[j];
        ahp = ah[j];
        wcp = wc[j];
    }
}

// Bound by the loads and stores of its ten arrays (52 bytes a cell where both
// stamps are set); every load is issued before the first use, the three integer
// scans share one barrier, and the whole update takes four.  800x800x9, every
// track dirty: 48 us a launch (54 us at the copy rate for all arrays); with a
// scan each, fourteen barriers and two counter atomics a track on shared
// addresses, 128 us.  Cost and prefix sums alone, 2500x2500x11: 429 us (542).
//
// s_c: commit stamp (0 = nothing to commit); s_r: rip-up stamp (0 = no
// rip-up); cost: recompute costs and prefix sums (and clear the dirty flag).
// stats[0] += cells of the tracks processed, stats[1] += those with rip-up.
// The workgroup is the fewest waves (at most 16) whose threads cover a track
// at K cells each.
template <int K>
__global__ void __launch_bounds__(1024) k_track_fused(GridDev g, int s_c, int s_r, int cost,
                                                      unsigned long long* stats) {
    constexpr int NWMAX = 16;
    const int nw = blockDim.x >> 6;
    __shared__ int4 sh_tot[NWMAX];
    __shared__ int2 sh_via[NWMAX];
    __shared__ CellCost sh_c[NWMAX];
    __shared__ double lds_d[NWMAX];
    __shared__ float s_exp[EXPTAB_N];
    int t = blockIdx.x;
    if (!g.dirty[t]) return;
    int l = 0;
    while (l < g.L - 1 && t >= g.tbase[l + 1]) l++;
    t -= g.tbase[l];
    const int dir = layer_dir(l, g.DIR);
    const int len = dir ? g.Y : g.X;
    const int64_t base = (int64_t)l * g.XYc + (int64_t)t * len;
    const bool v4 = (len & 3) == 0;
    const int p0 = threadIdx.x * K;
    float dem[K], cap[K];
    int ts[K], inc[K], gv[K], dec[K], cov[K], gr[K];
    uint32_t wr_dem = 0, wr_ts = 0, clr = 0;   // per-element bit masks
    // every load before the first use
    load_k<K, float, float4>(g.demand, base, p0, len, v4, dem);
    load_k<K, float, float4>(g.cap, base, p0, len, v4, cap);
    load_k<K, int, int4>(g.ts, base, p0, len, v4, ts);
    if (s_c) {
        load_k<K, int, int4>(g.pre, base, p0, len, v4, inc);
        load_k<K, int, int4>(g.vc, base, p0, len, v4, gv);
    } else {
#pragma unroll
        for (int j = 0; j < K; j++) inc[j] = gv[j] = 0;
    }
    if (s_r) {
        load_k<K, int, int4>(g.rpre, base, p0, len, v4, dec);
        load_k<K, int, int4>(g.rcov, base, p0, len, v4, cov);
        load_k<K, int, int4>(g.rvc, base, p0, len, v4, gr);
    } else {
#pragma unroll
        for (int j = 0; j < K; j++) dec[j] = cov[j] = gr[j] = 0;
    }
    if (cost)
        for (int i = threadIdx.x; i < EXPTAB_N; i += blockDim.x) s_exp[i] = g.exptab[i];
#pragma unroll
    for (int j = 0; j < K; j++)
        if (inc[j] | gv[j] | dec[j] | cov[j] | gr[j]) clr |= 1u << j;
    block_sums<K>(inc, dec, cov, sh_tot, nw);
    // commit of the wires, gate of the vias (s_c), then the rip-up's (s_r).
    // Demand that a caller set may be any float, so its sums keep the passes'
    // order too: wires and vias of the commit, then those of the rip-up.
#pragma unroll
    for (int j = 0; j < K; j++) {
        const int p = p0 + j;
        if (p <= len - 2 && inc[j] > 0) {
            dem[j] += (float)inc[j];
            wr_dem |= 1u << j;
            if (ts[j] != s_c) { ts[j] = s_c; wr_ts |= 1u << j; }
        }
        if (ts[j] >= s_c) gv[j] = 0;
        if (p <= len - 2 && dec[j] > 0) wr_dem |= 1u << j;
        else dec[j] = 0;
        if (p < len && cov[j] > 0 && ts[j] != s_r) { ts[j] = s_r; wr_ts |= 1u << j; }
        if (ts[j] >= s_r) gr[j] = 0;
        if (gv[j] | gr[j]) wr_dem |= (3u << j) >> 1;   // edges j-1 and j of this thread
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) sh_via[wave] = make_int2(gv[0], gr[0]);
    __syncthreads();
    int gvn = __shfl_down(gv[0], 1), grn = __shfl_down(gr[0], 1);
    if (lane == 63) {
        const int2 v = wave + 1 < nw ? sh_via[wave + 1] : make_int2(0, 0);
        gvn = v.x;
        grn = v.y;
    }
    if (gvn | grn) wr_dem |= 1u << (K - 1);
    apply_vias<K>(dem, gv, gvn, len, 1.0f);
#pragma unroll
    for (int j = 0; j < K; j++) dem[j] -= (float)dec[j];
    apply_vias<K>(dem, gr, grn, len, -1.0f);
#pragma unroll
    for (int j = 0; j < K; j++) {
        const int p = p0 + j;
        if (p >= len) continue;
        if (wr_dem >> j & 1) g.demand[base + p] = dem[j];
        if (wr_ts >> j & 1) g.ts[base + p] = ts[j];
        if (clr >> j & 1) {
            if (s_c) { g.pre[base + p] = 0; g.vc[base + p] = 0; }
            if (s_r) { g.rpre[base + p] = 0; g.rcov[base + p] = 0; g.rvc[base + p] = 0; }
        }
    }
    if (threadIdx.x == 0 && stats) {
        atomicAdd(&stats[0], (unsigned long long)len);
        if (s_r) atomicAdd(&stats[1], (unsigned long long)len);
    }
    if (!cost) return;
    // Costs from the new demand (src/graph.hpp:40-71), then the exclusive FP64
    // Sklansky prefix of wcost (src/graph.hpp:405-430).
    float wc[K], vc[K];
    double s[K];
    track_costs<K>(g, l, dir, len, p0, dem, cap, s_exp, sh_c, wc, vc, s);
    store_k<K>(g.wcost, base, p0, len, v4, wc);
    store_k<K>(g.vcost, base, p0, len, v4, vc);
    block_sklansky_rt<double, K>(s, lds_d, nw);
    store_k<K>(g.presum, base, p0, len, v4, s);
    if (threadIdx.x == 0) g.dirty[blockIdx.x] = 0;
}

// Cost update and prefix sums alone (no commit, no rip-up: the full sweep at
// a pass start and the timed sweep), as a persistent kernel: a grid sized to
// the workgroups the GPU holds walks the tracks, each workgroup loading its
// next dirty track's demand and capacity before it computes the current one,
// so loads stay in flight while the costs, the scan and the stores run.  The
// exp table is copied to LDS once per workgroup.  The values are those of
// k_track_fused with s_c = s_r = 0.
template <int K>
__global__ void __launch_bounds__(1024) k_track_cost(GridDev g, unsigned long long* stats) {
    constexpr int NWMAX = 16;
    const int nw = blockDim.x >> 6;
    __shared__ CellCost sh_c[2][NWMAX];
    __shared__ double lds_d[2][NWMAX];
    __shared__ float s_exp[EXPTAB_N];
    for (int i = threadIdx.x; i < EXPTAB_N; i += blockDim.x) s_exp[i] = g.exptab[i];
    __syncthreads();
    const int T = g.tbase[g.L];
    const int p0 = threadIdx.x * K;
    auto next_dirty = [&](int t) {
        while (t < T && !g.dirty[t]) t += gridDim.x;
        return t;
    };
    auto geometry = [&](int t, int& l, int& len, int64_t& base) {
        l = 0;
        while (l < g.L - 1 && t >= g.tbase[l + 1]) l++;
        len = layer_dir(l, g.DIR) ? g.Y : g.X;
        base = (int64_t)l * g.XYc + (int64_t)(t - g.tbase[l]) * len;
    };
    int t = next_dirty((int)blockIdx.x), par = 0;
    float dem[K], cap[K];
    int l = 0, len = 0;
    int64_t base = 0;
    if (t < T) {
        geometry(t, l, len, base);
        load_k<K, float, float4>(g.demand, base, p0, len, (len & 3) == 0, dem);
        load_k<K, float, float4>(g.cap, base, p0, len, (len & 3) == 0, cap);
    }
    while (t < T) {
        // the next track's loads first
        const int tn = next_dirty(t + (int)gridDim.x);
        int ln = 0, lenn = 0;
        int64_t basen = 0;
        float demn[K], capn[K];
        if (tn < T) {
            geometry(tn, ln, lenn, basen);
            load_k<K, float, float4>(g.demand, basen, p0, lenn, (lenn & 3) == 0, demn);
            load_k<K, float, float4>(g.cap, basen, p0, lenn, (lenn & 3) == 0, capn);
        }
        const bool v4 = (len & 3) == 0;
        float wc[K], vc[K];
        double sv[K];
        // the exchanges alternate between two sets of entries: the next
        // track's first write comes after this track's barriers
        track_costs<K>(g, l, layer_dir(l, g.DIR), len, p0, dem, cap, s_exp, sh_c[par], wc, vc, sv);
        store_k<K>(g.wcost, base, p0, len, v4, wc);
        store_k<K>(g.vcost, base, p0, len, v4, vc);
        block_sklansky_rt<double, K>(sv, lds_d[par], nw);
        store_k<K>(g.presum, base, p0, len, v4, sv);
        par ^= 1;
        if (threadIdx.x == 0) {
            g.dirty[t] = 0;
            if (stats) atomicAdd(&stats[0], (unsigned long long)len);
        }
        t = tn;
        l = ln;
        len = lenn;
        base = basen;
#pragma unroll
        for (int j = 0; j < K; j++) {
            dem[j] = demn[j];
            cap[j] = capn[j];
        }
    }
}

// The rip-up footprint of a list of routed nets (rip_route).
__global__ void __launch_bounds__(SB) k_rip_scatter(GridDev g, const int* nets, int64_t n, int* const* rptr,
                                                    int* bad) {
    const int64_t t = ((int64_t)blockIdx.x * SB + threadIdx.x) / RIP_LANES;
    if (t < n) rip_route(g, rptr[nets[t]], bad);
}

__global__ void k_fill_i(int* p, int64_t n, int v) {
    const int64_t i = (int64_t)blockIdx.x * SB + threadIdx.x;
    if (i < n) p[i] = v;
}

inline unsigned blocks(int64_t n) { return (unsigned)((n + SB - 1) / SB); }

} // namespace

BatchedState::BatchedState(igr_ctx* c_) : c(c_) {
    const int64_t n = c->cells();
    const int T = c->g.tbase[c->g.L];
    c->vc.zero(n, c->stream);
    c->rpre.zero(n, c->stream);
    c->rcov.zero(n, c->stream);
    c->rvc.zero(n, c->stream);
    c->bad.zero(1, c->stream);
    c->dirty.alloc(T);
    k_fill_i<<<blocks(T), SB, 0, c->stream>>>(c->dirty.p, T, 1);
    HIP_OK(hipGetLastError());
    GridDev& g = c->g;
    g.vc = c->vc.p;
    g.rpre = c->rpre.p;
    g.rcov = c->rcov.p;
    g.rvc = c->rvc.p;
    g.dirty = c->dirty.p;
}

BatchedState::~BatchedState() {
    GridDev& g = c->g;
    g.vc = g.rpre = g.rcov = g.rvc = g.dirty = nullptr;
}

void BatchedState::check() {
    int bad = 0;
    HIP_OK(hipMemcpyAsync(&bad, c->bad.p, sizeof(int), hipMemcpyDeviceToHost, c->stream));
    HIP_OK(hipStreamSynchronize(c->stream));
    if (bad) throw std::runtime_error("a ripped route has a wire across its layer's direction");
}

// Full-grid sweeps of the cost update and prefix sums, timed with events on
// the context stream: the plain form's kernels (update_wcost, update_vcost,
// presum) or the fused track kernel with every track dirty and nothing to
// commit.  Average milliseconds per sweep over reps sweeps after one warm-up.
double time_cost_sweep(igr_ctx* c, int form, int reps) {
    hipStream_t s = c->stream;
    const int T = c->g.tbase[c->g.L];
    hipEvent_t e0, e1;
    HIP_OK(hipEventCreate(&e0));
    HIP_OK(hipEventCreate(&e1));
    double ms_total = 0;
    try {
        if (form == IGR_FORM_PLAIN) {
            for (int r = 0; r <= reps; r++) {
                HIP_OK(hipEventRecord(e0, s));
                launch_update_cost(c);
                launch_presum(c);
                HIP_OK(hipEventRecord(e1, s));
                HIP_OK(hipEventSynchronize(e1));
                float ms = 0;
                HIP_OK(hipEventElapsedTime(&ms, e0, e1));
                if (r > 0) ms_total += ms;
            }
        } else {
            BatchedState bs(c);
            for (int r = 0; r <= reps; r++) {
                k_fill_i<<<blocks(T), SB, 0, s>>>(c->dirty.p, T, 1);
                HIP_OK(hipEventRecord(e0, s));
                launch_track_fused(c, 0, 0, true);
                HIP_OK(hipEventRecord(e1, s));
                HIP_OK(hipEventSynchronize(e1));
                float ms = 0;
                HIP_OK(hipEventElapsedTime(&ms, e0, e1));
                if (r > 0) ms_total += ms;
            }
            bs.check();
        }
    } catch (...) {
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
        throw;
    }
    HIP_OK(hipEventDestroy(e0));
    HIP_OK(hipEventDestroy(e1));
    return ms_total / std::max(1, reps);
}

void launch_track_fused(igr_ctx* c, int s_commit, int s_rip, bool cost) {
    KScope ks(c, K_TRACK_FUSED);
    const int T = c->g.tbase[c->g.L];
    const int ml = std::max(c->g.X, c->g.Y);
    const int cs = cost ? 1 : 0;
    // the processed-cell counters serve the byte counts of kernel timing only:
    // two atomics a workgroup on two addresses otherwise
    unsigned long long* st = c->prof.on ? c->track_stats.p : nullptr;
    hipStream_t s = c->stream;
    // Elements per thread: tuned, or 4 up to 4096-cell tracks and 8 above
    // (4 measured fastest on 800-, 1500- and 2500-cell tracks); the workgroup
    // is the fewest waves covering the longest track.
    const int K = c->tune.track_k ? c->tune.track_k : (ml <= 4096 ? 4 : 8);
    const int B = ((ml + K - 1) / K + 63) / 64 * 64;
    if (B > 1024) throw std::invalid_argument("track longer than the fused kernel's tile");
    if (!s_commit && !s_rip && cost) {
        // cost update and prefix sums only: persistent, prefetching kernel
        int cus = 0;
        HIP_OK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, c->device));
        auto go = [&](auto kern) {
            int per = 0;
            HIP_OK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kern, B, 0));
            const int grid = std::max(1, std::min(T, std::max(1, per) * cus));
            kern<<<grid, B, 0, s>>>(c->g, st);
        };
        switch (K) {
        case 4: go(k_track_cost<4>); break;
        case 8: go(k_track_cost<8>); break;
        case 16: go(k_track_cost<16>); break;
        default: throw std::invalid_argument("track_k must be 4, 8 or 16");
        }
        HIP_OK(hipGetLastError());
        return;
    }
    switch (K) {
    case 4: k_track_fused<4><<<T, B, 0, s>>>(c->g, s_commit, s_rip, cs, st); break;
    case 8: k_track_fused<8><<<T, B, 0, s>>>(c->g, s_commit, s_rip, cs, st); break;
    case 16: k_track_fused<16><<<T, B, 0, s>>>(c->g, s_commit, s_rip, cs, st); break;
    default: throw std::invalid_argument("track_k must be 4, 8 or 16");
    }
    HIP_OK(hipGetLastError());
}

void launch_rip_scatter(igr_ctx* c, const int* d_nets, int64_t n) {
    if (n == 0) return;
    KScope ks(c, K_RIP);
    k_rip_scatter<<<blocks(n * RIP_LANES), SB, 0, c->stream>>>(c->g, d_nets, n, c->nets.rptr.p, c->bad.p);
    HIP_OK(hipGetLastError());
}

} // namespace igr_dev
