// Routing context: device grid state, net data and the launch helpers shared
// by the kernel translation units.
#pragma once
#include "igr_dev.h"
#include "igr.h"
#include "par.hpp"

#include <hip/hip_runtime.h>

#include <cstring>
#include <memory>
#include <mutex>
#include <stdexcept>
#include <string>
#include <utility>
#include <vector>

#define HIP_OK(expr)                                                                               \
    do {                                                                                           \
        hipError_t e_ = (expr);                                                                    \
        if (e_ != hipSuccess)                                                                      \
            throw std::runtime_error(std::string(#expr) + ": " + hipGetErrorString(e_));           \
    } while (0)

namespace igr_dev {

template <typename T>
struct DevBuf {
    T* p = nullptr;
    size_t n = 0;
    DevBuf() = default;
    DevBuf(const DevBuf&) = delete;
    DevBuf& operator=(const DevBuf&) = delete;
    ~DevBuf() { release(); }
    void release() {
        if (p) (void)hipFree(p);
        p = nullptr;
        n = 0;
    }
    void alloc(size_t count) {
        if (count <= n && p) return;
        release();
        if (count == 0) count = 1;
        HIP_OK(hipMalloc(&p, count * sizeof(T)));
        n = count;
    }
    void upload(const T* h, size_t count, hipStream_t s) {
        alloc(count);
        if (count) HIP_OK(hipMemcpyAsync(p, h, count * sizeof(T), hipMemcpyHostToDevice, s));
    }
    void zero(size_t count, hipStream_t s) {
        alloc(count);
        HIP_OK(hipMemsetAsync(p, 0, count * sizeof(T), s));
    }
};

// Host memory that kernels write straight into (mapped, coherent): the route
// reads of igr_get_route.  word[0] holds the number of the last read that
// finished, the route follows from word[MAIL_HEAD].  'mu' makes one read at a
// time use it.
constexpr int MAIL_HEAD = 16, MAIL_WORDS = 16384;
struct Mailbox {
    std::mutex mu;
    int* word = nullptr;    // host address
    int* dev = nullptr;     // the same memory to the device
    int reads = 0;
    bool failed = false;    // no memory for it; not asked for again
    ~Mailbox() {
        if (word) (void)hipHostFree(word);
    }
    // Whether there is one (needs mu); without pinned memory there is none, and
    // routes are copied.
    bool open() {
        if (word || failed) return word != nullptr;
        int* w = nullptr;
        void* d = nullptr;
        failed = hipHostMalloc(reinterpret_cast<void**>(&w), sizeof(int) * (MAIL_HEAD + MAIL_WORDS),
                               hipHostMallocMapped | hipHostMallocCoherent) != hipSuccess ||
                 hipHostGetDevicePointer(&d, w, 0) != hipSuccess;
        if (failed) {
            (void)hipGetLastError();
            if (w) (void)hipHostFree(w);
            return false;
        }
        std::memset(w, 0, sizeof(int) * (MAIL_HEAD + MAIL_WORDS));
        word = w;
        dev = static_cast<int*>(d);
        return true;
    }
};

// Pinned slots for large copies to and from pageable memory (staging.hip): 16
// MiB a context, allocated by its first large copy (where that fails, copies are
// the runtime's).  'mu' lets one copy at a time use them; done[k] is the last
// copy through slot k.
struct Staging {
    static constexpr int SLOTS = 8, THREADS = 4;
    static constexpr int64_t SLOT_BYTES = 2 << 20, MIN_BYTES = 1 << 20;
    std::mutex mu;
    char* mem = nullptr;
    bool failed = false;    // no pinned memory or events; not asked for again
    hipEvent_t done[SLOTS] = {};
    ~Staging();
    bool open(int device);
    char* slot(int k) { return mem + k * SLOT_BYTES; }
};

// Net trees and footprints on the device (pattern pass).  Every net's current
// route is reached through rptr[net]: pattern routes live in 'routes' at
// route_off[net]; a rip-up-and-reroute pass moves the nets it reroutes to a
// buffer of its own (dag_routes).
struct NetsDev {
    static constexpr size_t SPARE_WORDS = 16 << 20;   // 64 MiB: what a context may hold back
    int64_t n = 0;
    DevBuf<int64_t> node_off, route_off, pt_off, hs_off, vs_off;
    DevBuf<int> node, parent, routes, pt, hs, vs;
    DevBuf<int*> rptr;
    std::vector<int64_t> h_node_off, h_route_off;
    std::vector<int> h_node;          // host copies used by the host-side batch logic
    std::vector<int*> h_rptr;
    std::vector<int64_t> h_rcap;      // capacity of each net's current route slot
    std::vector<double> h_lbytes;     // algorithmic bytes of each net's L-shape DP
    std::vector<DevBuf<int>*> dag_routes;   // freed (null) once no net's route lives there
    std::vector<int64_t> dag_live;          // nets whose route lives in dag_routes[k]
    std::vector<int> h_rbuf;                // per net: its dag_routes buffer, -1 = pattern slot
    int max_nodes = 0;
    DevBuf<int>* spare = nullptr;           // one retired buffer, for a next pass of about its size
    ~NetsDev() { clear_dag_routes(); }
    // The routes buffer of a new pass, which ends with adopt() or abandon().
    int* new_dag_routes(int64_t words) {
        const bool fits = spare && (int64_t)spare->n >= words && (int64_t)spare->n / 4 <= words;
        std::unique_ptr<DevBuf<int>> b(fits ? spare : new DevBuf<int>());
        if (fits) spare = nullptr;
        b->alloc(words);
        dag_routes.push_back(b.get());
        return b.release()->p;
    }
    // The newest retired buffer is the spare: the next pass is most likely of its size.
    void retire(DevBuf<int>* b) {
        if (b->n <= SPARE_WORDS) std::swap(spare, b);
        delete b;
    }
    // The pass of the newest buffer failed: its nets keep the routes they had.
    // Its kernels may have moved their pointers, so the device gets them back
    // before the buffer goes; a device that cannot take them keeps the buffer.
    void abandon(hipStream_t s) {
        if (dag_live.size() == dag_routes.size() && dag_live.back() > 0) return;   // adopt() failed half way
        if (hipStreamSynchronize(s) == hipSuccess &&
            hipMemcpy(rptr.p, h_rptr.data(), sizeof(int*) * h_rptr.size(), hipMemcpyHostToDevice) == hipSuccess) {
            retire(dag_routes.back());
            dag_routes.pop_back();
        } else {
            dag_live.resize(dag_routes.size(), 0);
            dag_live.back() = 1;   // of no net
        }
    }
    void clear_dag_routes() {
        delete spare;
        spare = nullptr;
        for (auto* b : dag_routes) delete b;
        dag_routes.clear();
        dag_live.clear();
        std::fill(h_rbuf.begin(), h_rbuf.end(), -1);
    }
    // Net 'net' leaves its rip-up-and-reroute buffer; an emptied buffer is
    // freed (the caller has synchronised with every kernel that used it).
    void release(int net) {
        const int k = h_rbuf[net];
        if (k < 0) return;
        h_rbuf[net] = -1;
        if (--dag_live[k] == 0) {
            retire(dag_routes[k]);
            dag_routes[k] = nullptr;
        }
    }
    // The listed nets' routes now live in the newest buffer, net rnets[r] at
    // rbase + slot(r), on 'threads' host threads.
    template <class Slot>
    void adopt(const int* rnets, int64_t n, int* rbase, int threads, Slot slot) {
        const int k = (int)dag_routes.size() - 1;
        dag_live.resize(dag_routes.size(), 0);
        // nets that leave each buffer
        std::vector<std::vector<int64_t>> left(threads, std::vector<int64_t>(dag_routes.size(), 0));
        dag_live[k] += n;
        igr::parallel_ranges(n, threads, [&](int64_t a, int64_t b, int t) {
            for (int64_t r = a; r < b; r++) {
                const int net = rnets[r];
                if (h_rbuf[net] >= 0) left[t][h_rbuf[net]]++;
                h_rptr[net] = rbase + slot(r);
                h_rcap[net] = slot(r + 1) - slot(r);
                h_rbuf[net] = k;
            }
        });
        for (const auto& v : left)
            for (size_t j = 0; j < v.size(); j++) dag_live[j] -= v[j];
        for (size_t j = 0; j < dag_routes.size(); j++)
            if (dag_routes[j] && dag_live[j] == 0) {
                retire(dag_routes[j]);
                dag_routes[j] = nullptr;
            }
    }
};

struct Sched {
    DevBuf<int> map, batch, status, viable, ids, pids, flags;
    // batched form: per-cell net lists, their heads and the round-0 map; the
    // compacted unassigned / active net lists; release-driven rounds: the
    // released cells, new owners, committed nets and their cells, with stamps
    DevBuf<int> base, cnt, c_net, ctrl, lists, rel, cand, cstamp, hits, hstamp;
    DevBuf<int64_t> head, c_off, c_end, bsum, cur;
    DevBuf<unsigned long long> stat;
    DevBuf<uint8_t> small;        // one-workgroup rounds: the nets left and their points' slots
    DevBuf<int> slot;             // X*Y slot of a cell in their map, or -1
    DevBuf<uint8_t> sn, alists;   // the nets' records; active-list rounds: their lists
    DevBuf<int> bits;             // per-net state bits (assigned, blocked in this batch)
    int* h_ctrl = nullptr;        // pinned copy of 'ctrl'
    ~Sched() {
        if (h_ctrl) (void)hipHostFree(h_ctrl);
    }
};

// Batched form: the records of a DAG's nodes and parent edges, by depth level
// within the net (16 bytes each, one load).  Positions pack x above y.
constexpr int DAG_POS_BITS = 13;
struct alignas(16) DagNode {
    uint32_t pos;                 // position, the node's layer (L: none) above it
    uint32_t loc;                 // index in the net's node order
    uint32_t slots;               // first child slot in the net, slot count in the top four bits
    uint32_t ebeg;                // first parent edge in the net (the next record's is the end)
};
struct alignas(16) DagEdge {
    uint32_t from, to;            // positions of the child and of the parent
    uint32_t slot;                // the parent's child slot in the net
    uint32_t child;               // record of the child in the net
};

struct alignas(16) DagSize {
    int nodes, edges, slots, levels;
};

// A pass's routes buffer: abandoned unless the pass gets as far as adopt().
class PassRoutes {
    NetsDev& nets;
    hipStream_t s;
    bool open = true;

public:
    int* const base;
    PassRoutes(NetsDev& nets_, hipStream_t s_, int64_t words) : nets(nets_), s(s_), base(nets.new_dag_routes(words)) {}
    PassRoutes(const PassRoutes&) = delete;
    PassRoutes& operator=(const PassRoutes&) = delete;
    ~PassRoutes() {
        if (open) nets.abandon(s);
    }
    template <class Slot>
    void adopt(const int* rnets, int64_t n, int threads, Slot slot) {
        nets.adopt(rnets, n, base, threads, slot);
        open = false;
    }
};

// One rip-up-and-reroute pass on the device: DAGs of the rerouted nets in
// routing order (batch by batch), with global node/edge/slot numbering.
struct DagDev {
    DevBuf<int> node, par, slot, child_num, loc, enode, node_net, lvl_nodes, nets;
    DevBuf<int64_t> node_off, par_off, csum, route_slot;
    DevBuf<int64_t> lvl_off;
    DevBuf<double> costs, cost_edges;
    DevBuf<uint64_t> packed, best;
    DevBuf<int> lo, best_change, emit;
    DevBuf<int> pt;
    DevBuf<int64_t> pt_off;
    // Batched form: the level-ordered records, the positions in node order,
    // the level boundaries of every net, the layer-change samples beside
    // cost_edges, and the tables of nets too large for LDS (keys in packed).
    DevBuf<DagNode> nrec;
    DevBuf<DagEdge> edge;
    DevBuf<uint32_t> npos;
    DevBuf<int> lvl;
    DevBuf<uint16_t> change;
    DevBuf<uint8_t> big_range;
    DevBuf<uint2> big_dec;
    // Batched form: the DAGs as uploaded (net list order, local parents), the
    // per-routed-net bases, and the layout kernel's level cursors, record
    // positions and slot bases.
    DevBuf<int64_t> r_node_off, r_par_off, ebase, sbase, lbase;
    DevBuf<int> r_nodes, r_par, r_slot, r_child_num, r_depth, rorder, err, lcur, lpos, lslot;
    // Batched form: the per-batch work-queue counters and the DAGs' sizes.
    DevBuf<int> queue;
    DevBuf<DagSize> size;         // per list entry
};

// Workspaces of the device routing order (order_kernels.hip).
constexpr int PATTERN_KEYS = 25;  // nets above LSWAVE_MAX_NODES, then LSWAVE_MAX_NODES .. 1 nodes
constexpr int DAG_KEYS = 64;      // 64 or more depth levels, then 63 .. 1
struct DagBound {
    int64_t net0, node0, edge0, slot0;
    int64_t lds;                  // LDS of the batch's net kernel
};
struct OrderDev {
    DevBuf<int> cnt, rank, lds;
    DevBuf<int64_t> off, tot;
    DevBuf<int4> rsize;
    DevBuf<DagBound> bound;
};
// A DAG pass's route slots, in list order: 8 ints a node and one a net.
__host__ __device__ inline int64_t dag_route_slot(int64_t nodes_before, int64_t entry) { return 8 * nodes_before + entry; }
// LDS bytes of one net's DAG tables: keys, layer ranges, decisions, levels.
__host__ __device__ inline int64_t dag_net_lds_bytes(int64_t nodes, int64_t slots, int64_t levels, int ML) {
    return 8 * slots * ML + 24 * nodes + 4 * (levels + 2);
}

// Arguments of the device DAG layout (one workgroup per routed net).
struct DagLayoutArgs {
    const int64_t* node_off;      // uploaded DAGs, net list order
    const int* nodes;
    const int64_t* par_off;
    const int* par;
    const int* slot;
    const int* child_num;
    const int* depth;
    const int* rorder;            // routed net -> list position
    const int64_t* nbase;         // per routed net: first node, edge, slot, level
    const int64_t* ebase;
    const int64_t* sbase;
    const int64_t* lbase;
    int X, Y;
    int node_limit;               // (L + 1) * X * Y
    DagNode* nrec;
    DagEdge* edge;
    uint32_t* npos;
    int* lvl;
    int* lcur;                    // per level: its fill cursor
    int* lpos;                    // per node: its record
    int* lslot;                   // per node: its first child slot in the net
    int* err;
};

struct Scratch {
    DevBuf<double> dist;
    DevBuf<int> from, lr;
    DevBuf<int> net_list;
    DevBuf<int64_t> scr_off;
    DevBuf<int> of;
    DevBuf<uint8_t> is_of;
    DevBuf<float> xsum, ysum, view;
};

// Per-kernel-class device time, measured with events on the context stream
// when enabled (igr_set_profiling).
enum KClass {
    K_COST = 0, K_PRESUM, K_LSHAPE, K_WIRE_COMMIT, K_VIA_COMMIT, K_DAG_EDGES, K_DAG_DP, K_DAG_EXTRACT, K_SCHED,
    K_TRACK_FUSED, K_RIP, K_NCLASS
};

struct KProf {
    bool on = false;
    std::vector<hipEvent_t> pool;
    size_t used = 0;
    std::vector<int> cls;
    std::vector<std::pair<hipEvent_t, hipEvent_t>> rec;
    double bytes[16] = {};         // algorithmic HBM bytes per kernel class
    hipEvent_t get() {
        if (used == pool.size()) {
            hipEvent_t e;
            HIP_OK(hipEventCreate(&e));
            pool.push_back(e);
        }
        return pool[used++];
    }
    void reset() {
        used = 0;
        cls.clear();
        rec.clear();
        for (double& b : bytes) b = 0;
    }
    ~KProf() {
        for (auto e : pool) (void)hipEventDestroy(e);
    }
};

} // namespace igr_dev

struct igr_ctx {
    igr_dev::KProf prof;
    igr_dev::GridDev g{};
    hipStream_t stream = nullptr;
    hipStream_t copy_stream = nullptr;   // uploads that overlap the compute stream
    int device = 0;
    igr_dev::DevBuf<double> w;
    igr_dev::DevBuf<int> xlen, ylen;
    igr_dev::DevBuf<float> cap, demand, wcost, vcost, exptab;
    igr_dev::DevBuf<double> presum;
    igr_dev::DevBuf<int> pre, ts;
    // Batched form: via-cut counts, rip-up differences, dirty-track flags, the
    // bad-route flag and the fused-pass cell counters (processed, ripped).
    igr_dev::DevBuf<int> vc, rpre, rcov, rvc, dirty, bad;
    igr_dev::DevBuf<unsigned long long> track_stats;
    igr_dev::NetsDev nets;
    igr_dev::Sched sched;
    igr_dev::Scratch scratch;
    igr_dev::DagDev dag;
    igr_dev::OrderDev order;
    igr_dev::Mailbox mail;
    igr_dev::Staging staging;
    std::mutex ref_mu;
    igr_dev::DevBuf<double> ref;   // a grid array in the callers' order, on its way in or out (ref_mu)
    int stamp = 0;
    igr_tuning tune{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};   // launch-shape overrides (0 = built-in)
    double last_dag_prep_s = 0;   // host preparation time of the last DAG pass
    double last_dag_prep_parts[4] = {0, 0, 0, 0};   // fill, batch metadata, upload, allocation
    int64_t cells() const { return (int64_t)g.L * g.X * g.Y; }
};

namespace igr_dev {
// Records the device time of the launches made during its lifetime and adds
// their algorithmic HBM bytes to the class total.
struct KScope {
    igr_ctx* c;
    int k;
    hipEvent_t a = nullptr;
    KScope(igr_ctx* c_, int k_, double bytes = 0) : c(c_), k(k_) {
        if (c->prof.on) {
            a = c->prof.get();
            HIP_OK(hipEventRecord(a, c->stream));
            c->prof.bytes[k] += bytes;
        }
    }
    ~KScope() {
        if (c->prof.on && a) {
            hipEvent_t b = c->prof.get();
            if (hipEventRecord(b, c->stream) == hipSuccess) {
                c->prof.cls.push_back(k);
                c->prof.rec.emplace_back(a, b);
            }
        }
    }
};

// Records msg as the calling thread's igr_last_error() and returns status.
int fail(int status, const std::string& msg);

// IGR_PROGRESS set in the environment: one line per stage on stderr, for
// long runs watched from outside.
void progress(const char* fmt, ...);

// Built-in launch-shape choices (igr_tuning fields left at 0).
// Stream launches: instantiating a graph of thousands of nodes costs more than
// its launch saves (40-net request 3.9 ms against 3.6, 20k-net run 153 against
// 150, heavy-net pass 904 against 900).
constexpr int DEF_GRAPH = 2;
constexpr int DEF_SCHED_CHUNK = 16;
constexpr int DEF_DAG_ORDER = 1;
constexpr int DEF_DAG_WAVES = 4;
constexpr int DEF_DAG_SEQ = 16;
constexpr int DEF_DAG_GRID = 2048;
// Records the work enqueued on a stream between construction and launch()
// as one graph, then launches it; inactive, the work runs as it is enqueued.
// A capture still open when the scope unwinds is ended and dropped.
struct StreamGraph {
    hipStream_t s;
    bool on;
    explicit StreamGraph(hipStream_t s_, bool on_) : s(s_), on(on_) {
        if (on) HIP_OK(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
    }
    void launch() {
        if (!on) return;
        on = false;
        hipGraph_t g = nullptr;
        HIP_OK(hipStreamEndCapture(s, &g));
        hipGraphExec_t x = nullptr;
        hipError_t e = hipGraphInstantiate(&x, g, nullptr, nullptr, 0);
        if (e == hipSuccess) e = hipGraphLaunch(x, s);
        if (x) (void)hipGraphExecDestroy(x);
        (void)hipGraphDestroy(g);
        HIP_OK(e);
    }
    ~StreamGraph() {
        if (on) {
            hipGraph_t g = nullptr;
            if (hipStreamEndCapture(s, &g) == hipSuccess && g) (void)hipGraphDestroy(g);
        }
    }
};

// Kernel launchers (defined in the .hip files).
void launch_update_cost(igr_ctx* c);
void launch_presum(igr_ctx* c);
void launch_wire_commit(igr_ctx* c, int stamp);
void launch_via_commit(igr_ctx* c, const int* d_nets, int64_t n, int stamp, int K);
void launch_lshape_plain(igr_ctx* c, const int* d_nets, const int64_t* d_scr_off, int64_t n, int stamp,
                         double bytes = 0);
// Batched form: the L-shape DP with a row of 16 lanes per net.  Nets of one
// launch have at most 'nodes' nodes (up to LSWAVE_MAX_NODES).
constexpr int LSWAVE_MAX_NODES = 24;
void launch_lshape_wave(igr_ctx* c, const int* d_nets, int64_t n, int nodes, int stamp, double bytes = 0);
void launch_to_ref(igr_ctx* c, const void* src, void* dst, int elem_bytes);
void launch_from_ref(igr_ctx* c, const void* src, void* dst, int elem_bytes);
void launch_ripup_mark(igr_ctx* c, int th, uint8_t* d_is_of, int* d_of);
void launch_congestion(igr_ctx* c, float* d_xsum, float* d_ysum);
// Its parts, on caller buffers: the per-gcell view (X*Y floats), and one
// prefix view of it (axis 0 along x, 1 along y).  No allocation, no sync.
void launch_congestion_map(igr_ctx* c, float* d_v);
void launch_view_scan(igr_ctx* c, const float* d_v, float* d_out, int axis);
// Static scratch of the no-allocation entry points: looked up once per
// device (call with that device current); the error of the lookup, if any,
// is kept for those entry points to report.
void noalloc_init(int device);
// Scheduler; with d_pt_off/d_pt given, the points of order[i] are list entry i
// of those arrays instead of the pattern footprint.
int run_schedule(igr_ctx* c, const int* h_order, int64_t n, int mode, int* h_batch_of,
                 const int64_t* d_pt_off = nullptr, const int* d_pt = nullptr);
// The same schedule computed incrementally with device-side round control
// (batched form).  The batches also stay on the device (sched.batch, by
// scheduler index); h_batch_of may be null.
int run_schedule_batched(igr_ctx* c, const int* h_order, int64_t n, int mode, int* h_batch_of,
                         const int64_t* d_pt_off = nullptr, const int* d_pt = nullptr);
void launch_rip_wire(igr_ctx* c, const int* d_nets, int64_t n, int stamp);
// Plain (reference launch structure) device work of one DAG batch, after the
// rip-up and the cost/prefix update.
struct DagBatch {
    int64_t net0, net1, node0, node1, edge0, edge1, slot0, slot1;
    int levels;
    int index = 0;              // batch number in the pass (work-queue counter)
    int64_t lvl0;               // first entry of this batch in lvl_off
    int lds = 0;                // batched form: dynamic LDS of the net kernel
    double bytes_edges = 0, bytes_dp = 0;   // algorithmic HBM bytes
};
void launch_dag_batch_plain(igr_ctx* c, const DagBatch& b, int stamp, const std::vector<int64_t>& h_lvl_off);
void launch_dag_compact(igr_ctx* c, const DagBatch& b);
// Batched form: persistent workgroups pulling the batch's nets from a work
// queue, all depth levels of a net in one workgroup; the pass's per-batch
// queue counters are zeroed first.  The batch to rip up next (or null) is
// scattered by the same launches.
void launch_dag_batch_wave(igr_ctx* c, const DagBatch& b, const DagBatch* rip, int stamp);
// The most LDS a launch of that form takes for a net's tables (a larger net's
// live in global memory).
constexpr int64_t DAG_LDS_MAX = 60 * 1024;
void launch_dag_queue_reset(igr_ctx* c, int64_t batches);
// Routing order of the last schedule's n nets (nb batches) by device kernels.
// Pattern: the net list by (batch, decreasing node count), h_off[nb *
// PATTERN_KEYS + 1] the first entry of every (batch, key).  DAG pass, after
// launch_dag_measure (sizes and checks of the uploaded DAGs; D.err): the routed
// order, nets and bases, h_bound[nb + 1] every batch's bounds, *h_big whether a
// net's tables exceed LDS.  Both wait for the stream.
void launch_pattern_order(igr_ctx* c, const int* d_order, int64_t n, int nb, int* d_list, int64_t* h_off);
void launch_dag_measure(igr_ctx* c, int64_t n, int64_t edges, hipStream_t s);
void launch_dag_order(igr_ctx* c, const int* d_nets, int64_t n, int nb, bool deep_first, DagBound* h_bound, int* h_big);
// Net's route (rc words of room, at most MAIL_WORDS) from device memory into
// the context's open mailbox, after all work on the stream; returns its host
// address.  Needs c->mail.mu.
const int* read_route(igr_ctx* c, const int* src, int64_t rc);
inline int host_threads() { return std::max(1, std::min(16, (int)std::thread::hardware_concurrency())); }
// Copies between the device and pageable memory, after all work on the stream.
// To the host: done on return.  To the device: 'src' is free on return.
void copy_to_host(igr_ctx* c, void* dst, const void* src, int64_t bytes, hipStream_t s);
void copy_to_device(igr_ctx* c, void* dst, const void* src, int64_t bytes, hipStream_t s);
template <class T>
void upload(igr_ctx* c, DevBuf<T>& b, const T* h, int64_t count, hipStream_t s) {
    b.alloc(count);
    copy_to_device(c, b.p, h, count * (int64_t)sizeof(T), s);
}
// off[i] = cnt[0] + .. + cnt[i - 1], off[n] the total (n > 0).
void launch_exclusive_scan(igr_ctx* c, const int* cnt, int64_t n, int64_t* off);
// Batched form: the device layout of a pass's DAGs.
void launch_dag_layout(igr_ctx* c, const DagLayoutArgs& a, int64_t n);
void launch_expf(const float* in, float* out, int64_t n, hipStream_t s);
// Fills the cost kernels' exp table (EXPTAB_N floats, GridDev::exptab).
void launch_exptab(float* t, hipStream_t s);
// Device-to-device copy of 'bytes' repeated 'reps' times; returns GB/s
// (bytes read + written).
double copy_probe(int64_t bytes, int reps, hipStream_t s);

// Batched-form grid state for the lifetime of one pass: clears the scatter
// arrays, flags every track dirty and points the grid at them; the plain
// kernels see null pointers outside it.
struct BatchedState {
    igr_ctx* c;
    explicit BatchedState(igr_ctx* c_);
    ~BatchedState();
    BatchedState(const BatchedState&) = delete;
    BatchedState& operator=(const BatchedState&) = delete;
    void check();   // throws if a ripped route could not be scattered
};
// Fused per-track pass: commit of the routed batch (s_commit > 0), rip-up of
// the next one (s_rip > 0), then costs and prefix sums when 'cost' is set.
void launch_track_fused(igr_ctx* c, int s_commit, int s_rip, bool cost);
double time_cost_sweep(igr_ctx* c, int form, int reps);
// Every net's route into d_out at d_off[i] (slices of the nets' route capacities).
void gather_routes(igr_ctx* c, const int64_t* d_off, int* d_out);
// The GPU evaluator (eval_kernels.hip).
void evaluate_routes_dev(igr_ctx* c, const igr_eval_nets* e, const int64_t* h_route_off, const int* h_routes,
                         igr_score* out);
void launch_rip_scatter(igr_ctx* c, const int* d_nets, int64_t n);
} // namespace igr_dev
