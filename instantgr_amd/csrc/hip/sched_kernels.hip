// Conflict-free net batch scheduler (src/database_cuda.hpp:288-434,437-631).
//
// Nets compete for the cells of an X*Y ownership map by atomicMax of their
// priority index (larger hpwl = larger index wins); a net joins the current
// batch when it owns every one of its point cells.  Up to 30 rounds per batch;
// nets blocked by a committed net sit out the rest of the batch.
//
// The reference re-reads a point cell right after its own atomicMax and
// abandons the net if a higher one owns it, racing with concurrent claims
// (src/database_cuda.hpp:313-318).  Here that read is given barrier
// semantics: a round first claims every active net's point cells (kernel 1),
// then decides which nets still own all their point cells (kernel 2), and only
// those claim their neighbour cells and sampled segment cells (kernel 3).
// Every result is a pure function of the input order, identical to the CPU
// oracle's.
#include "igr_ctx.hpp"

#include <chrono>

#include <algorithm>

namespace igr_dev {

namespace {

constexpr int TPB = 256;

struct SchedArgs {
    int64_t n;
    const int* ids;              // scheduler index -> net id (segments)
    const int* pids;             // scheduler index -> row of the point arrays
    const int64_t* pt_off;
    const int* pt;
    const int64_t* hs_off;
    const int* hs;
    const int64_t* vs_off;
    const int* vs;
    int* map;                    // X*Y owner index or -1
    int* batch;                  // per scheduler index
    int* status;                 // 0 normal, 1 competing, 2 blocked for this batch
    int* viable;
    int* flags;                  // [0] = committed this round
    int X, Y, sparsity;
};

__device__ __forceinline__ bool active(const SchedArgs& a, int64_t i) { return a.status[i] != 2 && a.batch[i] == -1; }

// The kernels over nets take LPN lanes a net, a point each: a round of a few
// thousand nets is the latency of its longest net (claims of points and of the
// rest 22 and 24 us a round with a thread a net, 4 and 9 so).
constexpr int LPN = 8;
struct NetLanes {
    int64_t i;                   // scheduler index
    int lane;
    uint64_t mask;               // the net's lanes in the wave
    __device__ NetLanes()
        : i(((int64_t)blockIdx.x * TPB + threadIdx.x) / LPN), lane(threadIdx.x % LPN),
          mask(((1ull << LPN) - 1) << (threadIdx.x & 63 & ~(LPN - 1))) {}
    __device__ bool any(bool v) const { return (__ballot(v) & mask) != 0; }   // over the net's lanes
};

__global__ void __launch_bounds__(TPB) k_claim_points(SchedArgs a) {
    const NetLanes t;
    const int64_t i = t.i;
    if (i >= a.n || !active(a, i)) return;
    if (t.lane == 0) a.status[i] = 1;
    const int64_t e = a.pt_off[a.pids[i] + 1];
    for (int64_t k = a.pt_off[a.pids[i]] + t.lane; k < e; k += LPN) atomicMax(&a.map[a.pt[k]], (int)i);
}

// Whether net i has a point cell that 'bad' rejects (its lanes call together).
template <class F>
__device__ __forceinline__ bool any_point(const SchedArgs& a, const NetLanes& t, F bad) {
    const int64_t e = a.pt_off[a.pids[t.i] + 1];
    bool b = false;
    for (int64_t k = a.pt_off[a.pids[t.i]] + t.lane; k < e && !b; k += LPN) b = bad(a.map[a.pt[k]]);
    return t.any(b);
}

__global__ void __launch_bounds__(TPB) k_viable(SchedArgs a) {
    const NetLanes t;
    if (t.i >= a.n) return;
    const int ok = active(a, t.i) && !any_point(a, t, [&](int m) { return m != (int)t.i; });
    if (t.lane == 0) a.viable[t.i] = ok;
}

__global__ void __launch_bounds__(TPB) k_claim_rest(SchedArgs a) {
    const NetLanes t;
    const int64_t i = t.i;
    if (i >= a.n || !a.viable[i]) return;
    const int net = a.ids[i];
    const int X = a.X, Y = a.Y;
    const int64_t pe = a.pt_off[a.pids[i] + 1];
    for (int64_t k = a.pt_off[a.pids[i]] + t.lane; k < pe; k += LPN) {
        int p = a.pt[k], x = p / Y, y = p % Y;
        if (y - 1 >= 0) atomicMax(&a.map[x * Y + y - 1], (int)i);
        if (x - 1 >= 0) atomicMax(&a.map[(x - 1) * Y + y], (int)i);
        if (x + 1 < X) atomicMax(&a.map[(x + 1) * Y + y], (int)i);
    }
    for (int64_t k = a.hs_off[net]; k < a.hs_off[net + 1]; k++) {
        int s = a.hs[2 * k], e = a.hs[2 * k + 1], y = s % Y;
        for (int x = s / Y + t.lane * a.sparsity; x <= e / Y; x += LPN * a.sparsity) atomicMax(&a.map[x * Y + y], (int)i);
    }
    for (int64_t k = a.vs_off[net]; k < a.vs_off[net + 1]; k++) {
        int s = a.vs[2 * k], e = a.vs[2 * k + 1], x = s / Y;
        for (int y = s % Y + t.lane * a.sparsity; y <= e % Y; y += LPN * a.sparsity) atomicMax(&a.map[x * Y + y], (int)i);
    }
}

__global__ void __launch_bounds__(TPB) k_commit(SchedArgs a, int cur) {
    const NetLanes t;
    if (t.i >= a.n || !active(a, t.i)) return;
    if (any_point(a, t, [&](int m) { return m != (int)t.i; }) || t.lane != 0) return;
    a.batch[t.i] = cur;
    a.flags[0] = 1;
}

__global__ void __launch_bounds__(TPB) k_revert(SchedArgs a) {
    const NetLanes t;
    if (t.i >= a.n || a.status[t.i] != 1 || a.batch[t.i] != -1) return;
    if (any_point(a, t, [&](int m) { return m != -1 && a.batch[m] != -1; }) && t.lane == 0) a.status[t.i] = 2;
}

__global__ void __launch_bounds__(TPB) k_clear(SchedArgs a) {
    int64_t q = (int64_t)blockIdx.x * TPB + threadIdx.x;
    if (q >= (int64_t)a.X * a.Y) return;
    int m = a.map[q];
    if (m >= 0 && a.status[m] == 2) a.map[q] = -1;
}

__global__ void k_fill(int* p, int64_t n, int v) {
    int64_t i = (int64_t)blockIdx.x * TPB + threadIdx.x;
    if (i < n) p[i] = v;
}

inline unsigned blocks(int64_t n) { return (unsigned)((n + TPB - 1) / TPB); }

} // namespace

int run_schedule(igr_ctx* c, const int* h_order, int64_t n, int mode, int* h_batch_of, const int64_t* d_pt_off,
                 const int* d_pt) {
    if (n == 0) return 0;
    Sched& S = c->sched;
    NetsDev& N = c->nets;
    hipStream_t st = c->stream;
    std::vector<int> ids(n);
    for (int64_t i = 0; i < n; i++) ids[i] = h_order[n - 1 - i];
    S.ids.upload(ids.data(), n, st);
    std::vector<int> pids;
    if (d_pt_off) {
        pids.resize(n);
        for (int64_t i = 0; i < n; i++) pids[i] = (int)(n - 1 - i);
        S.pids.upload(pids.data(), n, st);
    }
    const int64_t XYc = (int64_t)c->g.X * c->g.Y;
    S.map.alloc(XYc);
    S.batch.alloc(n);
    S.status.alloc(n);
    S.viable.alloc(n);
    S.flags.alloc(4);
    SchedArgs a{n, S.ids.p, d_pt_off ? S.pids.p : S.ids.p, d_pt_off ? d_pt_off : N.pt_off.p, d_pt_off ? d_pt : N.pt.p, N.hs_off.p, N.hs.p, N.vs_off.p, N.vs.p,
                S.map.p, S.batch.p, S.status.p, S.viable.p, S.flags.p, c->g.X, c->g.Y,
                (mode == 1 || mode == 2) ? 2 : 15};
    k_fill<<<blocks(n), TPB, 0, st>>>(S.batch.p, n, -1);
    int cur = 0;
    int* h_flag = nullptr;
    HIP_OK(hipHostMalloc(&h_flag, sizeof(int)));
    const auto t_start = std::chrono::steady_clock::now();
    auto t_note = t_start;
    try {
        for (;;) {
            const auto t_now = std::chrono::steady_clock::now();
            if (std::chrono::duration<double>(t_now - t_note).count() > 20) {
                t_note = t_now;
                progress("scheduler: %d batches after %.1f s", cur,
                         std::chrono::duration<double>(t_now - t_start).count());
            }
            k_fill<<<blocks(XYc), TPB, 0, st>>>(S.map.p, XYc, -1);
            k_fill<<<blocks(n), TPB, 0, st>>>(S.status.p, n, 0);
            bool have_commit = false;
            for (int round = 0; round < 30; round++) {
                k_fill<<<1, TPB, 0, st>>>(S.flags.p, 1, 0);
                k_claim_points<<<blocks(n * LPN), TPB, 0, st>>>(a);
                k_viable<<<blocks(n * LPN), TPB, 0, st>>>(a);
                k_claim_rest<<<blocks(n * LPN), TPB, 0, st>>>(a);
                k_commit<<<blocks(n * LPN), TPB, 0, st>>>(a, cur);
                HIP_OK(hipGetLastError());
                HIP_OK(hipMemcpyAsync(h_flag, S.flags.p, sizeof(int), hipMemcpyDeviceToHost, st));
                HIP_OK(hipStreamSynchronize(st));
                if (!*h_flag) break;
                have_commit = true;
                k_revert<<<blocks(n * LPN), TPB, 0, st>>>(a);
                k_clear<<<blocks(XYc), TPB, 0, st>>>(a);
            }
            if (!have_commit) break;
            cur++;
        }
    } catch (...) {
        (void)hipHostFree(h_flag);
        throw;
    }
    HIP_OK(hipHostFree(h_flag));
    std::vector<int> b(n);
    HIP_OK(hipMemcpyAsync(b.data(), S.batch.p, sizeof(int) * n, hipMemcpyDeviceToHost, st));
    HIP_OK(hipStreamSynchronize(st));
    for (int64_t i = 0; i < n; i++) {
        if (b[i] < 0) throw std::runtime_error("scheduler left a net without a batch");
        h_batch_of[n - 1 - i] = b[i];
    }
    return cur;
}

} // namespace igr_dev
