// Routing order of a scheduled pass, on the device: the scheduled nets sorted
// by batch (last batch first) and, inside a batch, by a size key, with the
// per-net sizes and bases of the DAG passes in that order.  The order of nets
// inside a batch changes no result (their footprints are disjoint and their
// demand updates integer adds); the key only puts the nets that take longest
// first.  A counting sort: one pass counts every (batch, key) and keeps each
// net's rank within it, a scan turns the counts into positions.  Bound by
// launches and the counters' atomics (0.2-0.3 ms a kernel where half a million
// nets share a few hundred keys).  On the host the same preparation took 34 ms of
// a 438k-net DAG pass (205 -> 166 ms in all) and 3 ms of a 500k-net pattern
// pass (35 -> 31.6 ms), between the scheduler and the first routing kernel.
#include "igr_ctx.hpp"

namespace igr_dev {

namespace {

constexpr int TPB = 256;

inline unsigned blocks(int64_t n) { return (unsigned)((n + TPB - 1) / TPB); }

__global__ void k_zero_i32(int* p, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * TPB + threadIdx.x;
    if (i < n) p[i] = 0;
}

// List entry i is scheduler index n - 1 - i.
__global__ void k_pattern_count(const int* order, const int* batch, int64_t n, int nb, const int64_t* node_off, int* cnt,
                                int* rank) {
    const int64_t i = (int64_t)blockIdx.x * TPB + threadIdx.x;
    if (i >= n) return;
    const int net = order[i];
    const int64_t nodes = node_off[net + 1] - node_off[net];
    const int64_t key = (int64_t)(nb - 1 - batch[n - 1 - i]) * PATTERN_KEYS +
                        (nodes > LSWAVE_MAX_NODES ? 0 : PATTERN_KEYS - nodes);
    rank[i] = atomicAdd(&cnt[key], 1);
}
__global__ void k_pattern_place(const int* order, const int* batch, int64_t n, int nb, const int64_t* node_off,
                                const int64_t* off, const int* rank, int* list) {
    const int64_t i = (int64_t)blockIdx.x * TPB + threadIdx.x;
    if (i >= n) return;
    const int net = order[i];
    const int64_t nodes = node_off[net + 1] - node_off[net];
    const int64_t key = (int64_t)(nb - 1 - batch[n - 1 - i]) * PATTERN_KEYS +
                        (nodes > LSWAVE_MAX_NODES ? 0 : PATTERN_KEYS - nodes);
    list[off[key] + rank[i]] = net;
}

// Sizes of the uploaded DAGs, 16 lanes a net, and the checks the layout kernel
// relies on: edge offsets in order, depths and slot counts in range.
__global__ void __launch_bounds__(TPB) k_dag_measure(const int64_t* node_off, const int64_t* par_off,
                                                     const int* child_num, const int* depth, int64_t n, int64_t edges,
                                                     DagSize* size, int* err) {
    const int64_t i = ((int64_t)blockIdx.x * TPB + threadIdx.x) >> 4;
    const int lane = threadIdx.x & 15;
    const bool live = i < n;
    const int64_t b0 = live ? node_off[i] : 0, b1 = live ? node_off[i + 1] : 0;
    int slots = 0, deep = 0;
    bool bad = false;
    for (int64_t k = b0 + lane; k < b1; k += 16) {
        const int64_t p0 = par_off[k], p1 = par_off[k + 1];
        const int cn = child_num[k], d = depth[k];
        bad |= p1 < p0 || p0 < 0 || p1 > edges || d < 0 || d >= b1 - b0 || cn < 0 || cn > 10;
        slots += cn;
        deep = max(deep, d);
    }
    for (int o = 1; o < 16; o <<= 1) {
        slots += __shfl_xor(slots, o, 16);
        deep = max(deep, __shfl_xor(deep, o, 16));
    }
    if (live && lane == 0)
        size[i] = DagSize{(int)(b1 - b0), (int)(par_off[b1] - par_off[b0]), slots, deep + 1};
    if (bad) atomicOr(err, 1);
}

// Key of list entry i inside batch b: deep_first, the deepest DAG first; else
// the entry's span of the list, so that the keys and the ranks within them
// (k_dag_count_list) are the list's order.
__host__ __device__ constexpr int64_t list_span(int64_t n) { return (n + DAG_KEYS - 1) / DAG_KEYS; }
__device__ __forceinline__ int64_t dag_key(int b, int levels, int64_t i, int64_t n, bool deep_first) {
    return (int64_t)b * DAG_KEYS + (deep_first ? DAG_KEYS - min(levels, DAG_KEYS) : (int)(i / list_span(n)));
}
__global__ void k_dag_count(const int* batch, const DagSize* size, int64_t n, int nb, int* cnt, int* rank) {
    const int64_t i = (int64_t)blockIdx.x * TPB + threadIdx.x;
    if (i >= n) return;
    rank[i] = atomicAdd(&cnt[dag_key(nb - 1 - batch[n - 1 - i], size[i].levels, i, n, true)], 1);
}
// List order inside a batch.  A wave walks one span of the list, 64 entries a
// step, and is the only one to count its keys; entries of a step in one batch
// take their ranks by lane.  Ranks from plain counter atomics would follow the
// order in which they arrive, another one each run.  Walking the list costs what
// the counters did: 438k-net pass 155.5 ms either way.
__global__ void __launch_bounds__(64) k_dag_count_list(const int* batch, int64_t n, int nb, int* cnt, int* rank) {
    const int lane = threadIdx.x;
    const int64_t i0 = blockIdx.x * list_span(n), i1 = i0 + list_span(n) < n ? i0 + list_span(n) : n;
    for (int64_t base = i0; base < i1; base += 64) {
        const int64_t i = base + lane;
        const bool live = i < i1;
        const int b = live ? nb - 1 - batch[n - 1 - i] : -1;
        uint64_t mine = 0;                                // the step's entries of this batch
        for (uint64_t todo = __ballot(live); todo;) {
            const int of = __builtin_amdgcn_readlane(b, __builtin_ctzll(todo));
            const uint64_t m = __ballot(b == of);
            if (b == of) mine = m;
            todo &= ~m;
        }
        const int lead = live ? __builtin_ctzll(mine) : lane;
        int before = 0;
        if (live && lane == lead) before = atomicAdd(&cnt[(int64_t)b * DAG_KEYS + blockIdx.x], __popcll(mine));
        before = __shfl(before, lead);
        if (live) rank[i] = before + __popcll(mine & ((1ull << lane) - 1));
    }
}
// Per routed net: its list entry, net and sizes; per batch: the LDS its net
// kernel needs (nets beyond the largest launch raise *big instead).
__global__ void k_dag_place(const int* batch, const DagSize* size, const int* nets, int64_t n, int nb, bool deep_first,
                            int ML, const int64_t* off, const int* rank, int* rorder, int* rnets, int4* rsize,
                            int* lds, int* big) {
    const int64_t i = (int64_t)blockIdx.x * TPB + threadIdx.x;
    if (i >= n) return;
    const int b = nb - 1 - batch[n - 1 - i];
    const DagSize z = size[i];
    const int64_t r = off[dag_key(b, z.levels, i, n, deep_first)] + rank[i];
    rorder[r] = (int)i;
    rnets[r] = nets[i];
    rsize[r] = make_int4(z.nodes, z.edges, z.slots, z.levels);
    const int64_t need = dag_net_lds_bytes(z.nodes, z.slots, z.levels, ML);
    if (need > DAG_LDS_MAX) *big = 1;
    else if (need > __hip_atomic_load(&lds[b], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(&lds[b], (int)need);
}

// Exclusive prefix sums of a routed net's four sizes (nodes, edges, slots,
// levels): per-workgroup totals, a scan of those, then the bases.
constexpr int PER = 8, SPAN = TPB * PER;
struct Sum4 {
    int64_t v[4];
    __device__ __forceinline__ void add(const Sum4& o) {
        for (int k = 0; k < 4; k++) v[k] += o.v[k];
    }
};
__device__ __forceinline__ Sum4 block_excl(Sum4 x, Sum4* sh, Sum4* total) {
    // lanes of a wave by shuffles, the waves through LDS
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    Sum4 incl = x;
    for (int d = 1; d < 64; d <<= 1)
        for (int k = 0; k < 4; k++) {
            const int64_t t = __shfl_up(incl.v[k], d);
            if (lane >= d) incl.v[k] += t;
        }
    if (lane == 63) sh[wave] = incl;
    __syncthreads();
    Sum4 before{{0, 0, 0, 0}}, all{{0, 0, 0, 0}};
    for (int w = 0; w < TPB / 64; w++) {
        if (w < wave) before.add(sh[w]);
        all.add(sh[w]);
    }
    __syncthreads();
    *total = all;
    for (int k = 0; k < 4; k++) incl.v[k] += before.v[k] - x.v[k];
    return incl;
}
__device__ __forceinline__ Sum4 widen(const int4& z) { return Sum4{{z.x, z.y, z.z, z.w}}; }

__global__ void __launch_bounds__(TPB) k_sum4_totals(const int4* z, int64_t n, Sum4* tot) {
    __shared__ Sum4 sh[TPB / 64];
    const int64_t i0 = (int64_t)blockIdx.x * SPAN + (int64_t)threadIdx.x * PER;
    Sum4 s{{0, 0, 0, 0}}, all;
    for (int j = 0; j < PER; j++)
        if (i0 + j < n) s.add(widen(z[i0 + j]));
    (void)block_excl(s, sh, &all);
    if (threadIdx.x == 0) tot[blockIdx.x] = all;
}
__global__ void __launch_bounds__(TPB) k_sum4_scan(Sum4* tot, int64_t nb) {
    __shared__ Sum4 sh[TPB / 64];
    const int64_t per = (nb + TPB - 1) / TPB, b0 = threadIdx.x * per;
    Sum4 s{{0, 0, 0, 0}}, all;
    for (int64_t j = 0; j < per; j++)
        if (b0 + j < nb) s.add(tot[b0 + j]);
    Sum4 run = block_excl(s, sh, &all);
    for (int64_t j = 0; j < per; j++)
        if (b0 + j < nb) {
            const Sum4 t = tot[b0 + j];
            tot[b0 + j] = run;
            run.add(t);
        }
}
__global__ void __launch_bounds__(TPB) k_sum4_apply(const int4* z, int64_t n, const Sum4* tot, int64_t* nbase,
                                                    int64_t* ebase, int64_t* sbase, int64_t* lbase) {
    __shared__ Sum4 sh[TPB / 64];
    const int64_t i0 = (int64_t)blockIdx.x * SPAN + (int64_t)threadIdx.x * PER;
    Sum4 s{{0, 0, 0, 0}}, all;
    for (int j = 0; j < PER; j++)
        if (i0 + j < n) s.add(widen(z[i0 + j]));
    Sum4 run = block_excl(s, sh, &all);
    run.add(tot[blockIdx.x]);
    for (int j = 0; j < PER; j++) {
        const int64_t i = i0 + j;
        if (i > n) break;
        nbase[i] = run.v[0];
        ebase[i] = run.v[1];
        sbase[i] = run.v[2];
        lbase[i] = run.v[3];
        if (i < n) run.add(widen(z[i]));
    }
}

// Bounds of every batch (entry nb: the totals).
__global__ void k_dag_bounds(int nb, const int64_t* off, const int64_t* nbase, const int64_t* ebase,
                             const int64_t* sbase, const int* lds, DagBound* out) {
    const int b = blockIdx.x * TPB + threadIdx.x;
    if (b > nb) return;
    const int64_t r = off[(int64_t)b * DAG_KEYS];
    out[b] = DagBound{r, nbase[r], ebase[r], sbase[r], b < nb ? lds[b] : 0};
}

} // namespace

void launch_pattern_order(igr_ctx* c, const int* d_order, int64_t n, int nb, int* d_list, int64_t* h_off) {
    OrderDev& O = c->order;
    hipStream_t s = c->stream;
    const int64_t keys = (int64_t)nb * PATTERN_KEYS;
    O.cnt.alloc(keys);
    O.off.alloc(keys + 1);
    O.rank.alloc(n);
    k_zero_i32<<<blocks(keys), TPB, 0, s>>>(O.cnt.p, keys);
    k_pattern_count<<<blocks(n), TPB, 0, s>>>(d_order, c->sched.batch.p, n, nb, c->nets.node_off.p, O.cnt.p, O.rank.p);
    launch_exclusive_scan(c, O.cnt.p, keys, O.off.p);
    k_pattern_place<<<blocks(n), TPB, 0, s>>>(d_order, c->sched.batch.p, n, nb, c->nets.node_off.p, O.off.p, O.rank.p,
                                              d_list);
    HIP_OK(hipGetLastError());
    HIP_OK(hipMemcpyAsync(h_off, O.off.p, sizeof(int64_t) * (keys + 1), hipMemcpyDeviceToHost, s));
    HIP_OK(hipStreamSynchronize(s));
}

void launch_dag_measure(igr_ctx* c, int64_t n, int64_t edges, hipStream_t s) {
    DagDev& D = c->dag;
    D.size.alloc(n);
    D.err.alloc(1);
    k_zero_i32<<<1, TPB, 0, s>>>(D.err.p, 1);
    k_dag_measure<<<blocks(n * 16), TPB, 0, s>>>(D.r_node_off.p, D.r_par_off.p, D.r_child_num.p, D.r_depth.p, n, edges,
                                                 D.size.p, D.err.p);
    HIP_OK(hipGetLastError());
}

void launch_dag_order(igr_ctx* c, const int* d_nets, int64_t n, int nb, bool deep_first, DagBound* h_bound, int* h_big) {
    OrderDev& O = c->order;
    DagDev& D = c->dag;
    hipStream_t s = c->stream;
    const int64_t keys = (int64_t)nb * DAG_KEYS, wgs = n / SPAN + 1;   // base n is written too
    O.cnt.alloc(keys);
    O.off.alloc(keys + 1);
    O.rank.alloc(n);
    O.lds.alloc(nb + 1);
    O.rsize.alloc(n);
    O.tot.alloc(4 * wgs);
    O.bound.alloc(nb + 1);
    D.rorder.alloc(n);
    D.nets.alloc(n);
    for (DevBuf<int64_t>* b : {&D.node_off, &D.ebase, &D.sbase, &D.lbase}) b->alloc(n + 1);
    Sum4* tot = reinterpret_cast<Sum4*>(O.tot.p);
    int* big = O.lds.p + nb;
    k_zero_i32<<<blocks(keys), TPB, 0, s>>>(O.cnt.p, keys);
    k_zero_i32<<<blocks(nb + 1), TPB, 0, s>>>(O.lds.p, nb + 1);
    if (deep_first) k_dag_count<<<blocks(n), TPB, 0, s>>>(c->sched.batch.p, D.size.p, n, nb, O.cnt.p, O.rank.p);
    else k_dag_count_list<<<DAG_KEYS, 64, 0, s>>>(c->sched.batch.p, n, nb, O.cnt.p, O.rank.p);
    launch_exclusive_scan(c, O.cnt.p, keys, O.off.p);
    k_dag_place<<<blocks(n), TPB, 0, s>>>(c->sched.batch.p, D.size.p, d_nets, n, nb, deep_first, c->g.L + 1, O.off.p,
                                          O.rank.p, D.rorder.p, D.nets.p, O.rsize.p, O.lds.p, big);
    k_sum4_totals<<<(unsigned)wgs, TPB, 0, s>>>(O.rsize.p, n, tot);
    k_sum4_scan<<<1, TPB, 0, s>>>(tot, wgs);
    k_sum4_apply<<<(unsigned)wgs, TPB, 0, s>>>(O.rsize.p, n, tot, D.node_off.p, D.ebase.p, D.sbase.p, D.lbase.p);
    k_dag_bounds<<<blocks(nb + 1), TPB, 0, s>>>(nb, O.off.p, D.node_off.p, D.ebase.p, D.sbase.p, O.lds.p, O.bound.p);
    HIP_OK(hipGetLastError());
    HIP_OK(hipMemcpyAsync(h_bound, O.bound.p, sizeof(DagBound) * (nb + 1), hipMemcpyDeviceToHost, s));
    HIP_OK(hipMemcpyAsync(h_big, big, sizeof(int), hipMemcpyDeviceToHost, s));
    HIP_OK(hipStreamSynchronize(s));
}

} // namespace igr_dev
