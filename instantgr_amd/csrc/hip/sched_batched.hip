// Batched form of the conflict-free net batch scheduler: the same batches as
// the round-by-round scheduler (src/database_cuda.hpp:288-434,437-631, with
// the deterministic claim semantics stated in sched_kernels.hip), with less
// work and no host synchronisation per round.
//
//  * Round 0 of every batch starts from the map every unassigned net claims
//    with its point cells: per cell, the highest-priority unassigned net that
//    lists the cell.  It is kept across batches from a per-cell list of nets
//    sorted by priority (built once per pass) and a head index per cell that
//    moves past assigned nets at the end of each batch, so round 0 claims
//    nothing.
//  * Within a batch a cell's value only grows (claims are maxima) except where
//    the end of a round releases the cells of blocked nets, so a later point
//    claim can only change a released cell.
//  * Two ways to run the later rounds give the same batches at different
//    costs per round:
//    - active-list rounds (kernels k_a_*): the nets still active in the batch
//      form a compacted list rebuilt after each round that committed; they
//      claim their points where the map holds a lower value, and the revert
//      tests each of them against the owners of its points.  Work per round
//      follows the active nets' point counts.
//    - release-driven rounds (kernels k_r_*): the end of a round lists the
//      cells it released; each goes to its highest-priority active lister (the
//      first active entry of the cell's list, scanned by a lane group), and
//      only those new owners are tested for viability (a net can only turn
//      viable by taking a released cell).  A net is blocked when one of its
//      points is owned by a net committed in this batch; owners committed in
//      earlier rounds already blocked every active net they could (their
//      cells only shrink), so the revert lists the cells of the nets committed
//      in this round and blocks the active nets in those cells' lists.  Work
//      per round follows the released cells and committed nets.
//    On a 640k-cell grid with 0.5M nets the active-list rounds cost less; on a
//    2.25M-cell grid with 3M-10M nets the release-driven ones do.
//  * Short lists, and the last batches of long ones, run in one workgroup
//    (k_small_rounds) unless the tuning asks for a kind of rounds.
//  * List orders are free: every decision is an atomic maximum or a test
//    against the map.
//  * The round and batch control lives in a device word block; the host
//    enqueues rounds in chunks and reads back one flag per chunk.  Kernels of
//    rounds after the end return at once.
#include "igr_ctx.hpp"

#include <algorithm>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <type_traits>

namespace igr_dev {

namespace {

constexpr int TPB = 256;
// Threads of the kernels that append to a list or count: a workgroup's appends
// cost one returning atomic on one counter, and those serialise at some 20 ns
// each, so at most 512 large workgroups.  Average launch on a 1500x1500 grid,
// 1.6M nets (release-driven), against 256 threads with an atomic per append or
// per 256-thread workgroup: viability 11 us (76), commit 18 (93), round end 27
// (46), released-cell claims 22 (28).
constexpr int LTPB = 1024;
constexpr int ROUNDS = 30;        // rounds per batch (src/database_cuda.hpp:612)
// Release-driven rounds where the cells' lists hold this many nets on average
// and the nets are this many, active-list rounds elsewhere.  Their rounds cost
// more each but follow the released cells, so they pay where a congested design
// needs many batches.  Scheduler ms of the active-list rounds against the
// release-driven ones, by (nets, list length).  Detour footprints of congested
// designs: (133k, 43) 285 / 289, (181k, 41) 473 / 439, (207k, 42) 545 / 495,
// (254k, 40) 678 / 589, (386k, 34) 535 / 463, (390k, 28) 383 / 372, (401k, 46)
// 929 / 746, (497k, 28) 410 / 393.  Pattern footprints of such designs: (171k, 42)
// 58 / 68, (225k, 34) 82 / 91, (448k, 37) 213 / 208, (602k, 32) 227 / 223, (604k,
// 26) 155 / 166, (609k, 28) 170 / 176, (611k, 38) 304 / 281, (716k, 39) 330 / 298,
// (2.1M, 27) 207 / 209.  Even designs have long lists but few batches and lose a
// tenth above the line: (314k, 48) 158 / 175, (405k, 43) 63 / 74, (474k, 48) 192 /
// 212; below it (219k, 24) 73 / 98, (438k, 24) 97 / 122.
constexpr int64_t SCHED_RELEASE_NETS = 175000, SCHED_RELEASE_LIST = 28;

// control state words (two slots of C_WORDS, then the placed-net counter).
// C_NU / C_UL: length and buffer of the nets round 0 tests.  Active-list
// rounds: the unassigned list, and C_NA / C_AL the same for the batch's
// active list (C_NA < 0: the unassigned list itself).  Release-driven rounds:
// the round-0 candidates (below); C_NV0, the nets round 0 found viable (list
// v0); C_NR, cells the previous round released (list rel); C_NK, new owners
// of those cells (list cand); C_NC, nets committed in this round;
// C_NH, cells those nets own (list hits).
// C_LASTC, nets placed when the lists were last compacted.  C_LEFT (active-list
// rounds): some net of the active list is still active after the round.
enum { C_DONE = 0, C_CUR, C_ROUND, C_COMMIT, C_HAVE, C_NVIABLE, C_NU, C_UL, C_NA, C_AL, C_NR, C_NK, C_NC, C_NH,
       C_NV0, C_LASTC, C_LEFT, C_WORDS };
constexpr int NLISTS = 3;         // net list buffers of n entries each
constexpr int COMPACT_DIV = 64;   // release-driven rounds: compact the cell lists every n/64 placed nets

// A net by scheduler index: its points.  One load where the index, the row and
// two offsets were a chain of three.
struct alignas(16) SNet {
    int64_t pt0;
    int npt, pad;
};
// An entry of the active-list rounds' net lists: the net with its points, so
// that a round's kernels read a list and then points, not a record between.
struct alignas(16) ANet {
    int i, npt;
    int64_t pt0;
};
// Its segments, read beside it by the kernels that walk a net's rest cells.
struct alignas(8) SSeg {
    int64_t h0, v0;
    int nh, nv;
};

struct BArgs {
    int64_t n;
    const SNet* sn;
    const SSeg* sg;
    const int* pt;
    const int* hs;
    const int* vs;
    int* map;                     // X*Y owner or -1
    int* base;                    // X*Y highest unassigned net listing the cell, or -1
    const int64_t* c_off;         // X*Y+1 per-cell list offsets
    int64_t* c_end;               // X*Y end of each list (below c_off[q+1] once compacted)
    int* c_net;                   // per-cell lists, highest index first
    int64_t* head;                // X*Y first unassigned entry of each list
    int* batch;
    int* ctrl;
    int* lists;                   // release-driven rounds: NLISTS buffers of n net indices
    ANet* alists;                 // active-list rounds: NLISTS buffers of n nets
    int small_at;                 // a batch that leaves this many nets or fewer stops the rounds (C_DONE 2)
    // release-driven rounds only
    int* rel;                     // X*Y cells released by the previous round
    int* cand;                    // nets that took a released cell this round
    int* cstamp;                  // per net: 1 + the round that listed it in cand, -(1 + g) when the
                                  // end of round g listed it as a round-0 candidate
    int* v0;                      // nets viable in round 0 of the batch
    int* hits;                    // X*Y cells owned by the nets committed this round
    int* hstamp;                  // per cell: 1 + the round that listed it in hits
    int64_t* cur;                 // X*Y: no active net before this entry of the cell's list in this batch
    unsigned long long* stat;     // rounds run, nets tested for viability, unassigned at batch starts
    // per net two bits, 16 nets a word (a few MB even at 10M nets, so the
    // random lookups of the list scans stay in L2): bit 0 assigned, bit 1
    // blocked in this batch; a net is active while both are clear
    uint32_t* nst;
    int64_t nwords;
    int X, Y, sparsity;
    // optional per-round record (IGR_SCHED_TRACE): TR_WORDS per round
    long long* trace;
    int64_t trace_cap;
    // kernel timing only: bytes the release-driven round kernels read and
    // write, one slot per workgroup index modulo BYTE_SLOTS
    unsigned long long* bytes;
};
constexpr int BYTE_SLOTS = 4096;

// Adds a wave's byte count to its workgroup's slot (profiling only; every
// lane of the wave calls it together, at the kernel's end).
__device__ __forceinline__ void flush_bytes(const BArgs& a, unsigned long long nb) {
    if (!a.bytes) return;
    for (int off = 32; off > 0; off >>= 1) nb += __shfl_xor(nb, off);
    if ((threadIdx.x & 63) == 0 && nb) atomicAdd(&a.bytes[blockIdx.x % BYTE_SLOTS], nb);
}

// Per-round record: batch, round in the batch, nets tested, viable,
// committed, cells those own, cells released by the previous round, new
// owners, device wall clock at the round's last kernel.
enum { TR_CUR = 0, TR_ROUND, TR_TESTED, TR_VIABLE, TR_COMM, TR_HITS, TR_REL, TR_NEWOWN, TR_CLOCK, TR_WORDS };

__device__ __forceinline__ uint32_t nstate(const BArgs& a, int64_t i) {
    return (a.nst[i >> 4] >> (2 * (i & 15))) & 3u;
}
__device__ __forceinline__ bool assigned(const BArgs& a, int64_t i) { return nstate(a, i) & 1u; }
__device__ __forceinline__ bool blocked(const BArgs& a, int64_t i) { return nstate(a, i) & 2u; }
__device__ __forceinline__ void set_assigned(const BArgs& a, int64_t i) {
    atomicOr(&a.nst[i >> 4], 1u << (2 * (i & 15)));
}
__device__ __forceinline__ void set_blocked(const BArgs& a, int64_t i) {
    atomicOr(&a.nst[i >> 4], 2u << (2 * (i & 15)));
}
// batch end: every blocked net is active again (assigned bits kept)
constexpr uint32_t NST_ASSIGNED = 0x55555555u;

// Active-list rounds: the batch's active list of the round whose state is st.
__device__ __forceinline__ const ANet* a_list(const BArgs& a, const int* st, int64_t& na) {
    na = st[C_NA] < 0 ? st[C_NU] : st[C_NA];
    return a.alists + (int64_t)st[C_AL] * a.n;
}

// Release-driven rounds: the nets whose viability the round whose state is st
// tests: the round-0 candidates in round 0 (every net in the first batch), the
// new owners of released cells later.
__device__ __forceinline__ const int* r_list(const BArgs& a, const int* st, int64_t& na) {
    if (st[C_ROUND] == 0) {
        na = st[C_NU];
        return a.lists + (int64_t)st[C_UL] * a.n;
    }
    na = st[C_NK];
    return a.cand;
}

// not assigned and not blocked in this batch
__device__ __forceinline__ bool active(const BArgs& a, int64_t i) { return nstate(a, i) == 0; }

// ---- per-cell lists -------------------------------------------------------
__global__ void k_cell_count(int64_t n, const SNet* sn, const int* pt, int* cnt) {
    const int64_t i = (int64_t)blockIdx.x * TPB + threadIdx.x;
    if (i >= n) return;
    const SNet s = sn[i];
    for (int64_t k = s.pt0; k < s.pt0 + s.npt; k++) atomicAdd(&cnt[pt[k]], 1);
}

__global__ void k_cell_fill(BArgs a, int* fillc) {
    const int64_t i = (int64_t)blockIdx.x * TPB + threadIdx.x;
    if (i >= a.n) return;
    const SNet s = a.sn[i];
    for (int64_t k = s.pt0; k < s.pt0 + s.npt; k++) {
        const int p = a.pt[k];
        const int pos = atomicAdd(&fillc[p], 1);
        a.c_net[a.c_off[p] + pos] = (int)i;
    }
}

// Heap sort of one cell's list into decreasing order (min-heap), then the
// initial head and base.
__device__ void sift_min(int* v, int64_t root, int64_t n) {
    for (;;) {
        int64_t c = 2 * root + 1;
        if (c >= n) return;
        if (c + 1 < n && v[c + 1] < v[c]) c++;
        if (v[c] >= v[root]) return;
        const int t = v[c];
        v[c] = v[root];
        v[root] = t;
        root = c;
    }
}

__global__ void k_cell_sort(BArgs a, int64_t cells) {
    const int64_t q = (int64_t)blockIdx.x * TPB + threadIdx.x;
    if (q >= cells) return;
    const int64_t b = a.c_off[q], m = a.c_off[q + 1] - b;
    int* v = a.c_net + b;
    for (int64_t r = m / 2 - 1; r >= 0; r--) sift_min(v, r, m);
    for (int64_t e = m - 1; e > 0; e--) {
        const int t = v[0];
        v[0] = v[e];
        v[e] = t;
        sift_min(v, 0, e);
    }
    a.head[q] = b;
    a.c_end[q] = b + m;
    if (a.cur) a.cur[q] = b;
    const int top = m > 0 ? v[0] : -1;
    a.base[q] = top;
    a.map[q] = top;
}

// ---- exclusive scan of the per-cell counts into int64 offsets ------------
constexpr int SCAN_PER = 16;
constexpr int SCAN_BLOCK = TPB * SCAN_PER;

__device__ int64_t block_excl_scan(int64_t v, int64_t* sh, int64_t* total) {
    sh[threadIdx.x] = v;
    __syncthreads();
    for (int d = 1; d < TPB; d <<= 1) {
        const int64_t t = threadIdx.x >= d ? sh[threadIdx.x - d] : 0;
        __syncthreads();
        sh[threadIdx.x] += t;
        __syncthreads();
    }
    const int64_t incl = sh[threadIdx.x];
    *total = sh[TPB - 1];
    __syncthreads();
    return incl - v;
}

__global__ void k_scan_reduce(const int* cnt, int64_t n, int64_t* bsum) {
    __shared__ int64_t sh[TPB];
    const int64_t b0 = (int64_t)blockIdx.x * SCAN_BLOCK + (int64_t)threadIdx.x * SCAN_PER;
    int64_t s = 0;
    for (int j = 0; j < SCAN_PER; j++)
        if (b0 + j < n) s += cnt[b0 + j];
    int64_t tot;
    block_excl_scan(s, sh, &tot);
    if (threadIdx.x == 0) bsum[blockIdx.x] = tot;
}

__global__ void k_scan_bsums(int64_t* bsum, int64_t nb) {
    __shared__ int64_t sh[TPB];
    const int64_t per = (nb + TPB - 1) / TPB;
    const int64_t b0 = (int64_t)threadIdx.x * per;
    int64_t s = 0;
    for (int64_t j = 0; j < per; j++)
        if (b0 + j < nb) s += bsum[b0 + j];
    int64_t tot;
    int64_t run = block_excl_scan(s, sh, &tot);
    for (int64_t j = 0; j < per; j++)
        if (b0 + j < nb) {
            const int64_t v = bsum[b0 + j];
            bsum[b0 + j] = run;
            run += v;
        }
}

__global__ void k_scan_apply(const int* cnt, int64_t n, const int64_t* bsum, int64_t* off) {
    __shared__ int64_t sh[TPB];
    const int64_t b0 = (int64_t)blockIdx.x * SCAN_BLOCK + (int64_t)threadIdx.x * SCAN_PER;
    int64_t s = 0;
    for (int j = 0; j < SCAN_PER; j++)
        if (b0 + j < n) s += cnt[b0 + j];
    int64_t tot;
    int64_t run = block_excl_scan(s, sh, &tot) + bsum[blockIdx.x];
    for (int j = 0; j < SCAN_PER; j++)
        if (b0 + j < n) {
            off[b0 + j] = run;
            run += cnt[b0 + j];
        }
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == TPB - 1) off[n] = run;
}

// ---- rounds -----------------------------------------------------------------
// Round g reads the control state in slot g & 1; its last kernel writes the
// successor state into the other slot, so no kernel reads a word another
// kernel of the same round rewrites.  A net's point list is walked by a group
// of G lanes (one step covers G points), with wave ballots for the early
// exits; a viable net's neighbour and segment claims are spread over a whole
// wave.
__device__ __forceinline__ uint64_t group_bits(uint64_t m, int G) {
    const int base = (int)(threadIdx.x & 63) & ~(G - 1);
    const uint64_t mask = G == 64 ? ~0ull : ((1ull << G) - 1);
    return (m >> base) & mask;
}

// Appends v to list for every thread with want, one counter atomic per
// workgroup (a returning atomic per wave on one counter serialises thousands
// of waves).  Every thread of the workgroup calls it; s holds LTPB/64+1 ints.
template <class T>
__device__ __forceinline__ void block_append(bool want, const T& v, int* counter, T* list, int* s) {
    constexpr int NW = LTPB / 64;
    const uint64_t m = __ballot(want);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    if (lane == 0) s[wv] = __popcll(m);
    __syncthreads();
    if (threadIdx.x == 0) {
        int tot = 0;
        for (int w = 0; w < NW; w++) {
            const int c = s[w];
            s[w] = tot;
            tot += c;
        }
        s[NW] = tot ? atomicAdd(counter, tot) : 0;
    }
    __syncthreads();
    if (want) list[s[NW] + s[wv] + __popcll(m & ((1ull << lane) - 1))] = v;
    __syncthreads();   // s is reused by the next call
}

// A workgroup's appends to one list, gathered in LDS over the whole kernel
// and written with one counter atomic at the end: counter atomics per wave or
// per pass serialise thousands of waves on the one address each round.  add()
// may be called by diverged lanes (the ballot covers the active lanes, and the
// lane that takes the offsets is one of them); entries beyond the LDS
// capacity go out at once.  Every thread of the workgroup calls init() and
// flush().
constexpr int GL_CAP = 4096;
struct GroupList {
    int* buf;                     // LDS, GL_CAP entries
    int* hdr;                     // LDS: count, then the list offset
    int* counter;
    int* list;
    __device__ __forceinline__ void init() {
        if (threadIdx.x == 0) hdr[0] = 0;
        __syncthreads();
    }
    __device__ __forceinline__ void add(bool want, int v) {
        const uint64_t m = __ballot(want);
        if (m == 0) return;
        const int lane = threadIdx.x & 63;
        const int leader = __builtin_ctzll(m);
        int off = 0;
        if (lane == leader) off = atomicAdd(&hdr[0], __popcll(m));
        off = __shfl(off, leader);
        const int pos = off + __popcll(m & ((1ull << lane) - 1));
        if (want) {
            if (pos < GL_CAP) buf[pos] = v;
            else list[atomicAdd(counter, 1)] = v;
        }
    }
    // U candidates a lane with one counter update.
    template <int U>
    __device__ __forceinline__ void add(const bool (&want)[U], const int (&v)[U]) {
        uint64_t m[U];
        int total = 0;
#pragma unroll
        for (int u = 0; u < U; u++) {
            m[u] = __ballot(want[u]);
            total += __popcll(m[u]);
        }
        if (total == 0) return;
        const int lane = threadIdx.x & 63;
        const uint64_t here = __ballot(true);
        const int leader = __builtin_ctzll(here);
        int off = 0;
        if (lane == leader) off = atomicAdd(&hdr[0], total);
        off = __shfl(off, leader);
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int pos = off + __popcll(m[u] & ((1ull << lane) - 1));
            if (want[u]) {
                if (pos < GL_CAP) buf[pos] = v[u];
                else list[atomicAdd(counter, 1)] = v[u];
            }
            off += __popcll(m[u]);
        }
    }
    __device__ __forceinline__ void flush() {
        __syncthreads();
        const int nb = hdr[0] < GL_CAP ? hdr[0] : GL_CAP;
        if (threadIdx.x == 0) hdr[1] = nb ? atomicAdd(counter, nb) : 0;
        __syncthreads();
        for (int i = threadIdx.x; i < nb; i += blockDim.x) list[hdr[1] + i] = buf[i];
    }
};

// Calls f(valid, q) with U cells per lane at a time, over the sampled cells of
// a net's segments (every sparsity-th cell from each segment's start,
// src/database_cuda.hpp:320-352), the cells of up to W segments at a time
// spread evenly over the W lanes of the net's group (a lane per segment would
// walk a long segment alone).  Every lane of the wave calls it together; valid
// is false on the lanes past the last cell, and f may use ballots.  The ends of
// the first W segments come from segment_ends, called ahead of other work: its
// loads then wait beside that work's.
struct SegEnds {
    int b, e;
};
__device__ __forceinline__ SegEnds segment_ends(const BArgs& a, const SSeg& g, int k) {
    if (k >= g.nh + g.nv) return SegEnds{0, 0};
    const int* seg = k < g.nh ? a.hs + 2 * (g.h0 + k) : a.vs + 2 * (g.v0 + k - g.nh);
    return SegEnds{seg[0], seg[1]};
}
template <int W, int U, class F>
__device__ __forceinline__ void group_segment_cells(const BArgs& a, const SSeg& g, SegEnds se, F f) {
    const int lane = threadIdx.x & (W - 1);
    const int Y = a.Y, sp = a.sparsity;
    const int ns = g.nh + g.nv;
    for (int sb = 0; __ballot(sb < ns); sb += W) {
        const int k = sb + lane;
        int cnt = 0, first = 0, step = 0;
        if (sb > 0) se = segment_ends(a, g, k);
        if (k < ns) {
            const bool hor = k < g.nh;
            const int b = se.b, e = se.e;
            const int bx = b / Y, by = b - bx * Y, ex = e / Y, ey = e - ex * Y;
            const int span = hor ? ex - bx : ey - by;   // along x at y = by, or along y at x = bx
            cnt = span >= 0 ? span / sp + 1 : 0;
            first = b;
            step = hor ? sp * Y : sp;
        }
        int incl = cnt;                  // inclusive scan of the cell counts
        for (int d = 1; d < W; d <<= 1) {
            const int v = __shfl_up(incl, d, W);
            if (lane >= d) incl += v;
        }
        const int total = __shfl(incl, W - 1, W);
        const int excl = incl - cnt;
        for (int cb = 0; __ballot(cb < total); cb += W * U) {
            bool valid[U];
            int q[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int c = cb + W * u + lane;
                int sg = 0;              // the first lane whose inclusive count exceeds c
                for (int b2 = W / 2; b2 > 0; b2 >>= 1)
                    if (__shfl(incl, sg + b2 - 1, W) <= c) sg += b2;
                const int f0 = __shfl(first, sg, W), st0 = __shfl(step, sg, W), ex = __shfl(excl, sg, W);
                valid[u] = c < total;
                q[u] = valid[u] ? f0 + (c - ex) * st0 : 0;
            }
            f(valid, q);
        }
    }
}
template <int U, class F>
__device__ __forceinline__ void wave_segment_cells(const BArgs& a, const SSeg& g, SegEnds se, F f) {
    group_segment_cells<64, U>(a, g, se, f);
}

// The neighbour cells (0,-1), (-1,0), (1,0) of a point.
__device__ __forceinline__ void point_neighbours(const BArgs& a, bool in, int p, bool (&valid)[3], int (&q)[3]) {
    const int x = p / a.Y, y = p - x * a.Y;
    valid[0] = in && y > 0;
    valid[1] = in && x > 0;
    valid[2] = in && x + 1 < a.X;
    q[0] = p - 1;
    q[1] = p - a.Y;
    q[2] = p + a.Y;
}

// 3. (both) a wave per viable net claims the neighbour cells (0,-1), (-1,0),
//    (1,0) of its points and every sparsity-th cell of its segments
__global__ void __launch_bounds__(TPB) k_b_claim_rest(BArgs a, int64_t g, const int* vlist) {
    const int* st = a.ctrl + (g & 1) * C_WORDS;
    if (st[C_DONE]) return;
    const int nv = st[C_NVIABLE];
    unsigned long long nb = 0;
    for (int w = (threadIdx.x >> 6) * gridDim.x + blockIdx.x; w < nv; w += (gridDim.x * TPB) >> 6) {
        const int i = vlist[w];
        const SNet s = a.sn[i];
        const SSeg sg = a.sg[i];
        const int lane = threadIdx.x & 63;
        const SegEnds se = segment_ends(a, sg, lane);
        if (lane == 0) nb += 4 + 16 + 24;   // list entry, net and segment records
        for (int k = lane; k < s.npt; k += 64) {
            bool valid[3];
            int q[3];
            point_neighbours(a, true, a.pt[s.pt0 + k], valid, q);
            for (int u = 0; u < 3; u++)
                if (valid[u]) {
                    atomicMax(&a.map[q[u]], i);
                    nb += 4;
                }
        }
        wave_segment_cells<1>(a, sg, se, [&](bool(&valid)[1], int(&q)[1]) {
            if (valid[0]) {
                atomicMax(&a.map[q[0]], i);
                nb += 4;
            }
        });
    }
    flush_bytes(a, nb);
}

// A workgroup's commits of the round, counted once (after a barrier).
__device__ __forceinline__ void count_commits(const BArgs& a, int* st, int won) {
    if (threadIdx.x != 0 || won == 0) return;
    atomicAdd(&st[C_NC], won);
    atomicAdd(&a.ctrl[2 * C_WORDS], won);   // nets placed so far
    st[C_COMMIT] = 1;
}

// ---- active-list rounds -----------------------------------------------------
// 1. point claims of the active nets (from round 1; round 0 starts from the
//    kept map): only cells holding a lower value can change
template <int G>
__global__ void __launch_bounds__(TPB) k_a_claim(BArgs a, int64_t g) {
    const int* st = a.ctrl + (g & 1) * C_WORDS;
    if (st[C_DONE] || st[C_ROUND] == 0) return;
    int64_t na;
    const ANet* al = a_list(a, st, na);
    const int64_t nth = (int64_t)gridDim.x * TPB / G;
    const int lg = threadIdx.x & (G - 1);
    for (int64_t t = ((int64_t)blockIdx.x * TPB + threadIdx.x) / G; t < na; t += nth) {
        const ANet s = al[t];   // every listed net is active
        for (int k = lg; k < s.npt; k += G) {
            int* m = &a.map[a.pt[s.pt0 + k]];
            if (*m < s.i) atomicMax(m, s.i);
        }
    }
}

// 2. active nets owning every point cell go to the viable list
template <int G>
__global__ void __launch_bounds__(LTPB) k_a_viable(BArgs a, int64_t g, int* vlist) {
    __shared__ int s_buf[GL_CAP], s_hdr[2];
    int* st = a.ctrl + (g & 1) * C_WORDS;
    if (st[C_DONE]) return;
    GroupList gl{s_buf, s_hdr, &st[C_NVIABLE], vlist};
    gl.init();
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        // the successor lists' counters, filled by this round's last kernel
        int* nx = a.ctrl + ((g + 1) & 1) * C_WORDS;
        nx[C_NA] = 0;
        nx[C_NU] = 0;
    }
    int64_t na;
    const ANet* al = a_list(a, st, na);
    const int64_t nth = (int64_t)gridDim.x * LTPB / G;
    const int lg = threadIdx.x & (G - 1);
    const int64_t rounds = (na + nth - 1) / nth;   // the same for every lane of the wave
    for (int64_t r = 0; r < rounds; r++) {
        const int64_t t = ((int64_t)blockIdx.x * LTPB + threadIdx.x) / G + r * nth;
        const bool live = t < na;   // every listed net is active
        const ANet s = live ? al[t] : ANet{0, 0, 0};
        bool fail = !live;
        for (int k = lg;; k += G) {
            const bool f = !fail && k < s.npt && a.map[a.pt[s.pt0 + k]] != s.i;
            fail = fail || group_bits(__ballot(f), G) != 0;
            if (__ballot(!fail && k + G < s.npt) == 0) break;
        }
        gl.add(lg == 0 && !fail, s.i);
    }
    gl.flush();
}

// 4. a wave per viable net: commit it if it still owns every point cell
__global__ void __launch_bounds__(LTPB) k_a_commit(BArgs a, int64_t g, const int* vlist) {
    __shared__ int s_won;
    int* st = a.ctrl + (g & 1) * C_WORDS;
    if (st[C_DONE]) return;
    if (threadIdx.x == 0) s_won = 0;
    __syncthreads();
    const int nv = st[C_NVIABLE];
    const int lane = threadIdx.x & 63;
    for (int w = (blockIdx.x * LTPB + threadIdx.x) >> 6; w < nv; w += (gridDim.x * LTPB) >> 6) {
        const int i = vlist[w];
        const SNet s = a.sn[i];
        bool lost = false;
        for (int k = lane; k < s.npt; k += 64) lost = lost || a.map[a.pt[s.pt0 + k]] != i;
        if (__ballot(lost) == 0 && lane == 0) {
            a.batch[i] = st[C_CUR];
            set_assigned(a, i);
            atomicAdd(&s_won, 1);
        }
    }
    __syncthreads();
    count_commits(a, st, s_won);
}

// 5. after a commit: active nets with a point cell owned by a committed net
//    sit out the batch
template <int G>
__global__ void __launch_bounds__(TPB) k_a_revert(BArgs a, int64_t g) {
    int* st = a.ctrl + (g & 1) * C_WORDS;
    if (st[C_DONE] || !st[C_COMMIT]) return;
    int64_t na;
    const ANet* al = a_list(a, st, na);
    const int64_t nth = (int64_t)gridDim.x * TPB / G;
    const int lg = threadIdx.x & (G - 1);
    const int64_t rounds = (na + nth - 1) / nth;
    bool left = false;
    for (int64_t r = 0; r < rounds; r++) {
        const int64_t t = ((int64_t)blockIdx.x * TPB + threadIdx.x) / G + r * nth;
        ANet s = t < na ? al[t] : ANet{0, 0, 0};
        const bool live = t < na && !assigned(a, s.i);
        if (!live) s.npt = 0;
        bool hit = false;
        for (int k = lg;; k += G) {
            bool h = false;
            if (!hit && k < s.npt) {
                const int pre = a.map[a.pt[s.pt0 + k]];
                h = pre != -1 && assigned(a, pre);
            }
            hit = hit || group_bits(__ballot(h), G) != 0;
            if (__ballot(!hit && k + G < s.npt) == 0) break;
        }
        if (lg == 0 && live && hit) set_blocked(a, s.i);
        left = left || (live && !hit);
    }
    if (__ballot(left) != 0 && (threadIdx.x & 63) == 0) st[C_LEFT] = 1;
}

// 6. end of the round.  The batch goes on after a commit that left active
//    nets, below the round limit: cells of blocked nets are released.
//    Otherwise the batch ends (without active nets the next round would commit
//    nothing and end it; that round's six kernels took 17 us):
//    each cell's list moves past assigned nets, the next batch starts from
//    the kept map with every unassigned net active.  The successor lists go
//    to a buffer neither current list uses.  Thread 0 writes the successor
//    control state.
__global__ void __launch_bounds__(LTPB) k_a_clear_end(BArgs a, int64_t g, int64_t cells) {
    __shared__ int s_app[LTPB / 64 + 1];
    const int* st = a.ctrl + (g & 1) * C_WORDS;
    int* nx = a.ctrl + ((g + 1) & 1) * C_WORDS;
    const int64_t t = (int64_t)blockIdx.x * LTPB + threadIdx.x;
    const int64_t stride = (int64_t)gridDim.x * LTPB;   // grid-stride over cells and list entries
    const bool done = st[C_DONE] != 0;
    const bool commit = st[C_COMMIT] != 0;
    const int round = st[C_ROUND];
    const bool end = !commit || !st[C_LEFT] || round + 1 >= ROUNDS;
    int fresh = 0;   // the first list buffer neither current list uses
    while (fresh == st[C_AL] || fresh == st[C_UL]) fresh++;
    ANet* nl = a.alists + (int64_t)fresh * a.n;
    if (!done) {
        if (end) {
            for (int64_t q = t; q < cells; q += stride) {
                int64_t h = a.head[q];
                const int64_t e = a.c_end[q];
                while (h < e && assigned(a, a.c_net[h])) h++;
                a.head[q] = h;
                const int b = h < e ? a.c_net[h] : -1;
                a.base[q] = b;
                a.map[q] = b;
            }
            const ANet* ul = a.alists + (int64_t)st[C_UL] * a.n;
            const int64_t nu = st[C_NU], passes = (nu + stride - 1) / stride;   // the same for every thread
            for (int64_t ps = 0; ps < passes; ps++) {
                const int64_t u = ps * stride + t;
                const ANet s = u < nu ? ul[u] : ANet{0, 0, 0};
                block_append(u < nu && !assigned(a, s.i), s, &nx[C_NU], nl, s_app);
            }
            // every unassigned net is active again in the next batch
            for (int64_t w = t; w < a.nwords; w += stride) a.nst[w] &= NST_ASSIGNED;
        } else {
            for (int64_t q = t; q < cells; q += stride) {
                const int m = a.map[q];
                if (m >= 0 && blocked(a, m)) a.map[q] = -1;
            }
            int64_t na;
            const ANet* al = a_list(a, st, na);
            const int64_t passes = (na + stride - 1) / stride;   // the same for every thread
            for (int64_t ps = 0; ps < passes; ps++) {
                const int64_t u = ps * stride + t;
                const ANet s = u < na ? al[u] : ANet{0, 0, 0};
                block_append(u < na && active(a, s.i), s, &nx[C_NA], nl, s_app);
            }
        }
    }
    if (t == 0) {
        if (!done) {
            int64_t na;
            (void)a_list(a, st, na);
            if (a.trace && g < a.trace_cap) {
                long long* rec = a.trace + g * TR_WORDS;
                rec[TR_CUR] = st[C_CUR];
                rec[TR_ROUND] = round;
                rec[TR_TESTED] = na;
                rec[TR_VIABLE] = st[C_NVIABLE];
                rec[TR_COMM] = st[C_NC];
                rec[TR_HITS] = st[C_NH];
                rec[TR_REL] = st[C_NR];
                rec[TR_NEWOWN] = st[C_NK];
                rec[TR_CLOCK] = (long long)wall_clock64();
            }
            a.stat[0] += 1;
            a.stat[1] += (unsigned long long)na;
            if (round == 0) a.stat[2] += (unsigned long long)st[C_NU];
        }
        int d = st[C_DONE], cur = st[C_CUR], r = st[C_ROUND], have = st[C_HAVE] | (commit ? 1 : 0);
        if (!d) {
            if (!end) {
                r = round + 1;
            } else if (!have) {
                d = 1;                       // a batch without commits: nothing left to place
            } else {
                cur += 1;
                r = 0;
                have = 0;
                const int64_t rest = a.n - a.ctrl[2 * C_WORDS];
                d = rest == 0 ? 1 : rest <= a.small_at ? 2 : 0;
            }
        }
        nx[C_DONE] = d;
        nx[C_CUR] = cur;
        nx[C_ROUND] = r;
        nx[C_HAVE] = have;
        nx[C_COMMIT] = 0;
        nx[C_LEFT] = 0;
        nx[C_NC] = 0;
        nx[C_NVIABLE] = 0;
        if (done) {
            nx[C_NA] = st[C_NA];
            nx[C_AL] = st[C_AL];
            nx[C_NU] = st[C_NU];
            nx[C_UL] = st[C_UL];
        } else if (end) {
            nx[C_NA] = -1;           // the new unassigned list is the active list
            nx[C_AL] = fresh;
            nx[C_UL] = fresh;
        } else {
            nx[C_AL] = fresh;        // C_NA counted above
            nx[C_NU] = st[C_NU];
            nx[C_UL] = st[C_UL];
        }
    }
}

// ---- release-driven rounds --------------------------------------------------
// 1. from round 1: each cell the previous round released goes to its
//    highest-priority active lister (the first active entry of its list),
//    which joins the viability test.  A group of G lanes scans a cell's list
//    G entries a step.
template <int G>
__global__ void __launch_bounds__(LTPB) k_r_claim(BArgs a, int64_t g) {
    __shared__ int s_buf[GL_CAP], s_hdr[2];
    int* st = a.ctrl + (g & 1) * C_WORDS;
    if (st[C_DONE] || st[C_ROUND] == 0) return;
    GroupList gl{s_buf, s_hdr, &st[C_NK], a.cand};
    gl.init();
    const int64_t nr = st[C_NR];
    const int64_t nth = (int64_t)gridDim.x * LTPB / G;
    const int lg = threadIdx.x & (G - 1);
    const int64_t rounds = (nr + nth - 1) / nth;   // the same for every thread
    unsigned long long nb = 0;
    for (int64_t r = 0; r < rounds; r++) {
        const int64_t t = ((int64_t)blockIdx.x * LTPB + threadIdx.x) / G + r * nth;
        const bool live = t < nr;
        const int q = live ? a.rel[t] : 0;
        int64_t h = live ? a.cur[q] : 0;
        const int64_t e = live ? a.c_end[q] : 0;
        if (live && lg == 0) nb += 4 + 16;   // cell, its cursor and list end
        bool found = !live;
        bool fresh = false;   // this lane took the cell for a net not yet listed this round
        int owner = 0;
        for (;;) {
            const int64_t k = h + lg;
            int j = -1;
            bool act = false;
            if (!found && k < e) {
                j = a.c_net[k];
                act = active(a, j);
                nb += 8;   // list entry, state word
            }
            const uint64_t m = group_bits(__ballot(act), G);
            if (m != 0 && lg == __builtin_ctzll(m)) {
                a.map[q] = j;
                a.cur[q] = k;   // the entries before k stay inactive for the rest of the batch
                owner = j;
                fresh = atomicExch(&a.cstamp[j], (int)g + 1) != (int)g + 1;
                nb += 4 + 8 + 8 + (fresh ? 4 : 0);   // map, cursor, stamp, new-owner entry
            }
            found = found || m != 0;
            h += G;
            if (__ballot(!found && h < e) == 0) break;
        }
        gl.add(fresh, owner);
    }
    gl.flush();
    flush_bytes(a, nb);
}

// 2. the nets under test (every unassigned net in round 0, the new owners of
//    released cells later) that own every point cell go to the viable list
template <int G>
__global__ void __launch_bounds__(LTPB) k_r_viable(BArgs a, int64_t g, int* vlist) {
    __shared__ int s_buf[GL_CAP], s_hdr[2];
    int* st = a.ctrl + (g & 1) * C_WORDS;
    if (st[C_DONE]) return;
    GroupList gl{s_buf, s_hdr, &st[C_NVIABLE], vlist};
    gl.init();
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        // the successor lists' counters, filled by this round's last kernel
        int* nx = a.ctrl + ((g + 1) & 1) * C_WORDS;
        nx[C_NU] = 0;
        nx[C_NR] = 0;
    }
    int64_t na;
    const int* al = r_list(a, st, na);
    const int64_t nth = (int64_t)gridDim.x * LTPB / G;
    const int lg = threadIdx.x & (G - 1);
    const int64_t rounds = (na + nth - 1) / nth;   // the same for every lane of the wave
    unsigned long long nb = 0;
    for (int64_t r = 0; r < rounds; r++) {
        const int64_t t = ((int64_t)blockIdx.x * LTPB + threadIdx.x) / G + r * nth;
        const int64_t i = t < na ? al[t] : 0;
        const bool live = t < na && active(a, i);
        if (t < na && lg == 0) nb += 4 + 4 + 16;   // entry, state, net record
        SNet s = t < na ? a.sn[i] : SNet{0, 0, 0};   // beside the state word, not after it
        if (!live) s.npt = 0;
        bool fail = !live;
        for (int k = lg;; k += G) {
            const bool chk = !fail && k < s.npt;
            const bool f = chk && a.map[a.pt[s.pt0 + k]] != (int)i;
            if (chk) nb += 8;   // point, map cell
            fail = fail || group_bits(__ballot(f), G) != 0;
            if (__ballot(!fail && k + G < s.npt) == 0) break;
        }
        if (lg == 0 && !fail) nb += 4;
        gl.add(lg == 0 && !fail, (int)i);
    }
    gl.flush();
    flush_bytes(a, nb);
}

// Lists the cells not yet listed in the round of this stamp.
template <int U>
__device__ __forceinline__ void hit(const BArgs& a, GroupList& gl, int stamp, const bool (&own)[U], const int (&q)[U],
                                    unsigned long long& nb) {
    bool h[U];
#pragma unroll
    for (int u = 0; u < U; u++) h[u] = own[u] && atomicExch(&a.hstamp[q[u]], stamp) != stamp;
#pragma unroll
    for (int u = 0; u < U; u++) nb += (own[u] ? 8 : 0) + (h[u] ? 4 : 0);   // stamp, hit entry
    gl.add(h, q);
}

// 4. a wave per viable net: commit it if it still owns every point cell;
//    a committed net's wave then lists the cells it owns (points, their
//    neighbours, sampled segment cells), once each.  Commits do not change
//    the map, so a net's cells are the same whichever nets of the round
//    commit around it.
__global__ void __launch_bounds__(LTPB) k_r_commit(BArgs a, int64_t g, const int* vlist) {
    __shared__ int s_buf[GL_CAP], s_hdr[2], s_won;
    int* st = a.ctrl + (g & 1) * C_WORDS;
    if (st[C_DONE]) return;
    GroupList gl{s_buf, s_hdr, &st[C_NH], a.hits};
    if (threadIdx.x == 0) s_won = 0;
    gl.init();
    const int nv = st[C_NVIABLE];
    const int lane = threadIdx.x & 63;
    const int stamp = (int)g + 1;
    unsigned long long nb = 0;
    for (int w = (threadIdx.x >> 6) * gridDim.x + blockIdx.x; w < nv; w += (gridDim.x * LTPB) >> 6) {
        const int i = vlist[w];
        const SNet s = a.sn[i];
        const SSeg sg = a.sg[i];
        // round 0's viable nets: the batch end lists those still unassigned
        if (lane == 0 && st[C_ROUND] == 0) a.v0[w] = i;
        if (lane == 0) nb += 4 + 16 + 24;   // list entry, net and segment records
        // the first 64 points' neighbours and the segments are read beside the
        // points, whatever comes of the net
        const SegEnds se = segment_ends(a, sg, lane);
        const bool in0 = lane < s.npt;
        const int p0 = in0 ? a.pt[s.pt0 + lane] : 0;
        bool valid0[3];
        int q0[4], m0[3];
        {
            int nq[3];
            point_neighbours(a, in0, p0, valid0, nq);
            for (int u = 0; u < 3; u++) q0[u] = nq[u];
            q0[3] = p0;
        }
#pragma unroll
        for (int u = 0; u < 3; u++) m0[u] = valid0[u] ? a.map[q0[u]] : -1;
        bool lost = in0 && a.map[p0] != i;
        if (in0) nb += 8;   // point, map cell
        for (int k = lane + 64; k < s.npt; k += 64) {
            lost = lost || a.map[a.pt[s.pt0 + k]] != i;
            nb += 8;
        }
        if (__ballot(lost) != 0) continue;
        if (lane == 0) {
            a.batch[i] = st[C_CUR];
            set_assigned(a, i);
            atomicAdd(&s_won, 1);
            nb += 8;   // batch, state word
        }
        // several cells a lane at a time: their map loads, then their stamp
        // exchanges, overlap
        {
            const bool own[4] = {m0[0] == i, m0[1] == i, m0[2] == i, in0};
            hit<4>(a, gl, stamp, own, q0, nb);
        }
        for (int k = lane + 64; k - lane < s.npt; k += 64) {
            const bool in = k < s.npt;
            const int p = in ? a.pt[s.pt0 + k] : 0;
            bool valid[3], own[4];
            int nq[3], q[4];
            point_neighbours(a, in, p, valid, nq);
            own[3] = in;
            q[3] = p;
#pragma unroll
            for (int u = 0; u < 3; u++) {
                q[u] = nq[u];
                own[u] = valid[u] && a.map[nq[u]] == i;
            }
            hit<4>(a, gl, stamp, own, q, nb);
        }
        wave_segment_cells<2>(a, sg, se, [&](bool(&valid)[2], int(&q)[2]) {
            bool own[2];
#pragma unroll
            for (int u = 0; u < 2; u++) own[u] = valid[u] && a.map[q[u]] == i;
            nb += 4 * (valid[0] + valid[1]);
            hit<2>(a, gl, stamp, own, q, nb);
        });
    }
    gl.flush();
    count_commits(a, st, s_won);
    flush_bytes(a, nb);
}

// 5. every active net listing one of those cells sits out the batch (a net
//    is blocked when one of its point cells is owned by a net committed in
//    this batch; owners committed in earlier rounds blocked their listers
//    then, and their cells only shrink).  A group of G lanes per cell (a
//    wave: the lists of cells in dense regions run to thousands of nets).
template <int G>
__global__ void __launch_bounds__(TPB) k_r_block(BArgs a, int64_t g) {
    const int* st = a.ctrl + (g & 1) * C_WORDS;
    if (st[C_DONE] || !st[C_COMMIT]) return;
    const int64_t nh = st[C_NH];
    const int64_t nth = (int64_t)gridDim.x * TPB / G;
    const int lg = threadIdx.x & (G - 1);
    unsigned long long nb = 0;
    for (int64_t t = ((int64_t)blockIdx.x * TPB + threadIdx.x) / G; t < nh; t += nth) {
        const int q = a.hits[t];
        const int64_t e = a.c_end[q];
        for (int64_t k = a.cur[q] + lg; k < e; k += G) {
            const int j = a.c_net[k];
            nb += 8;   // list entry, state word
            if (active(a, j)) {
                set_blocked(a, j);
                nb += 4;
            }
        }
        // every entry from the cursor on is now inactive for the rest of the
        // batch (a later release or hit of the cell finds no active lister)
        if (lg == 0) {
            a.cur[q] = e;
            nb += 4 + 24;   // hit entry, list end, cursor read and write
        }
    }
    flush_bytes(a, nb);
}

// 6. end of the round.  The batch goes on after a commit below the round
//    limit: cells of blocked nets are released.  Otherwise the batch ends:
//    each cell's list moves past assigned nets, the next batch starts from
//    the kept map with every unassigned net active.  The successor lists go
//    to a buffer neither current list uses.  Thread 0 writes the successor
//    control state.
__global__ void __launch_bounds__(LTPB) k_r_clear_end(BArgs a, int64_t g, int64_t cells) {
    __shared__ int s_buf[GL_CAP], s_hdr[2];
    const int* st = a.ctrl + (g & 1) * C_WORDS;
    int* nx = a.ctrl + ((g + 1) & 1) * C_WORDS;
    const int64_t t = (int64_t)blockIdx.x * LTPB + threadIdx.x;
    const int64_t stride = (int64_t)gridDim.x * LTPB;   // grid-stride over cells and list entries
    const bool done = st[C_DONE] != 0;
    const bool commit = st[C_COMMIT] != 0;
    const int round = st[C_ROUND];
    const bool end = !commit || round + 1 >= ROUNDS;
    const int fresh = 1 - st[C_UL];   // the candidate-list buffer not in use
    int* nl = a.lists + (int64_t)fresh * a.n;
    unsigned long long nb = 0;
    if (!done) {
        if (end) {
            // Round 0 of the next batch tests only nets that may own every
            // point cell of the kept map: a net viable in round 0 of this
            // batch and still unassigned keeps its cells (a list's head moves
            // past assigned nets only), and any other net can only become
            // viable by taking a cell whose head moved.
            // Every COMPACT_DIV-th of the nets placed since the last time,
            // the lists drop their assigned entries (order kept): the scans
            // of the later rounds then skip no dead entries.
            GroupList gl{s_buf, s_hdr, &nx[C_NU], nl};
            gl.init();
            const int stamp = -(int)(g + 1);
            const bool compact = (int64_t)(a.ctrl[2 * C_WORDS] - st[C_LASTC]) * COMPACT_DIV >= a.n;
            if (compact) {
                // a group of CG lanes per cell compacts its list in place:
                // every lane reads its entry before the group's ballot, and
                // an entry moves to a slot at or below its own
                constexpr int CG = 16;
                const int lg = threadIdx.x & (CG - 1);
                const int64_t ng = stride / CG;
                const int64_t gpasses = (cells + ng - 1) / ng;
                for (int64_t ps = 0; ps < gpasses; ps++) {
                    const int64_t q = ps * ng + t / CG;
                    const bool live = q < cells;
                    const int64_t s0 = live ? a.c_off[q] : 0, e = live ? a.c_end[q] : 0;
                    int64_t w = s0;
                    for (int64_t k = live ? a.head[q] : 0;; k += CG) {
                        const int64_t kk = k + lg;
                        int j = -1;
                        bool keep = false;
                        if (kk < e) nb += 12;   // entry read, state word, entry written
                        if (kk < e) {
                            j = a.c_net[kk];
                            keep = !assigned(a, j);
                        }
                        const uint64_t m = group_bits(__ballot(keep), CG);
                        if (keep) a.c_net[w + __popcll(m & ((1ull << lg) - 1))] = j;
                        w += __popcll(m);
                        if (__ballot(k + CG < e) == 0) break;
                    }
                    int b = -1;
                    bool want = false;
                    if (live && lg == 0) {
                        a.c_end[q] = w;
                        a.head[q] = s0;
                        a.cur[q] = s0;
                        b = w > s0 ? a.c_net[s0] : -1;
                        const bool moved = b != a.base[q];
                        if (moved) a.base[q] = b;
                        a.map[q] = b;
                        want = moved && b >= 0 && atomicExch(&a.cstamp[b], stamp) != stamp;
                    }
                    gl.add(want, b);
                }
            } else {
                const int64_t passes = (cells + stride - 1) / stride;
                for (int64_t ps = 0; ps < passes; ps++) {
                    const int64_t q = ps * stride + t;
                    bool want = false;
                    int b = -1;
                    if (q < cells) {
                        const int64_t h0 = a.head[q], e = a.c_end[q];
                        int64_t h = h0;
                        while (h < e && assigned(a, a.c_net[h])) h++;
                        nb += 16 + 8 * (h - h0 + (h < e ? 1 : 0)) + 8 + 12;   // head, end; entries; cur, base, map
                        if (h != h0) a.head[q] = h;
                        b = h < e ? a.c_net[h] : -1;
                        // the first unassigned lister changed exactly where
                        // the previous one was assigned
                        const bool moved = b != a.base[q];
                        a.cur[q] = h;
                        if (moved) a.base[q] = b;
                        a.map[q] = b;
                        want = moved && b >= 0 && atomicExch(&a.cstamp[b], stamp) != stamp;
                    }
                    gl.add(want, b);
                }
            }
            const int64_t nv0 = round == 0 ? st[C_NVIABLE] : st[C_NV0], vpasses = (nv0 + stride - 1) / stride;
            for (int64_t ps = 0; ps < vpasses; ps++) {
                const int64_t u = ps * stride + t;
                const int i = u < nv0 ? a.v0[u] : 0;
                const bool want = u < nv0 && !assigned(a, i) && atomicExch(&a.cstamp[i], stamp) != stamp;
                gl.add(want, i);
            }
            gl.flush();
            // every unassigned net is active again in the next batch
            for (int64_t w = t; w < a.nwords; w += stride) {
                a.nst[w] &= NST_ASSIGNED;
                nb += 8;
            }
        } else {
            // UNR independent cells per lane and pass
            GroupList gl{s_buf, s_hdr, &nx[C_NR], a.rel};
            gl.init();
            constexpr int UNR = 4;
            const int64_t per = stride * UNR;
            for (int64_t ps = 0; ps * per < cells; ps++) {
                int m[UNR];
                for (int u = 0; u < UNR; u++) {
                    const int64_t q = ps * per + u * stride + t;
                    m[u] = q < cells ? a.map[q] : -1;
                }
                bool rl[UNR];
                for (int u = 0; u < UNR; u++) rl[u] = m[u] >= 0 && blocked(a, m[u]);
                for (int u = 0; u < UNR; u++)
                    nb += (ps * per + u * stride + t < cells ? 4 : 0) + (m[u] >= 0 ? 4 : 0) + (rl[u] ? 8 : 0);
                for (int u = 0; u < UNR; u++) {
                    const int64_t q = ps * per + u * stride + t;
                    if (rl[u]) a.map[q] = -1;
                    gl.add(rl[u], (int)q);
                }
            }
            gl.flush();
        }
    }
    if (t == 0) {
        if (!done) {
            int64_t na;
            (void)r_list(a, st, na);
            if (a.trace && g < a.trace_cap) {
                long long* rec = a.trace + g * TR_WORDS;
                rec[TR_CUR] = st[C_CUR];
                rec[TR_ROUND] = round;
                rec[TR_TESTED] = na;
                rec[TR_VIABLE] = st[C_NVIABLE];
                rec[TR_COMM] = st[C_NC];
                rec[TR_HITS] = st[C_NH];
                rec[TR_REL] = st[C_NR];
                rec[TR_NEWOWN] = st[C_NK];
                rec[TR_CLOCK] = (long long)wall_clock64();
            }
            a.stat[0] += 1;
            a.stat[1] += (unsigned long long)na;
            // unassigned nets at the batch start (placed now, less round 0's commits)
            if (round == 0) a.stat[2] += (unsigned long long)(a.n - (a.ctrl[2 * C_WORDS] - st[C_NC]));
        }
        int d = st[C_DONE], cur = st[C_CUR], r = st[C_ROUND], have = st[C_HAVE] | (commit ? 1 : 0);
        if (!d) {
            if (!end) {
                r = round + 1;
            } else if (!have) {
                d = 1;                       // a batch without commits: nothing left to place
            } else {
                cur += 1;
                r = 0;
                have = 0;
                const int64_t rest = a.n - a.ctrl[2 * C_WORDS];
                d = rest == 0 ? 1 : rest <= a.small_at ? 2 : 0;
            }
        }
        nx[C_DONE] = d;
        nx[C_CUR] = cur;
        nx[C_ROUND] = r;
        nx[C_HAVE] = have;
        nx[C_COMMIT] = 0;
        nx[C_NVIABLE] = 0;
        nx[C_NV0] = done ? st[C_NV0] : end ? 0 : round == 0 ? st[C_NVIABLE] : st[C_NV0];
        nx[C_LASTC] = !done && end && (int64_t)(a.ctrl[2 * C_WORDS] - st[C_LASTC]) * COMPACT_DIV >= a.n
                          ? a.ctrl[2 * C_WORDS]
                          : st[C_LASTC];
        nx[C_NK] = 0;
        nx[C_NC] = 0;
        nx[C_NH] = 0;
        if (done) {
            nx[C_NU] = st[C_NU];
            nx[C_UL] = st[C_UL];
            nx[C_NR] = st[C_NR];
        } else if (end) {
            nx[C_UL] = fresh;        // C_NU counted above
        } else {
            nx[C_NU] = st[C_NU];     // C_NR counted above
            nx[C_UL] = st[C_UL];
        }
    }
    flush_bytes(a, nb);
}

// ---- few nets: all rounds in one workgroup ----------------------------------
// With few nets left a round's six kernels are launches and load chains (26 us
// whatever they do).  Here one workgroup runs the remaining batches with the
// owner map in LDS.  Only the point cells of the nets left can decide
// anything, so the map has a slot per such cell: k_small_mark leaves at each
// one of its points' positions in the list of all of them (any one serves),
// and the points that find their own number there take the slots.  The points'
// slots follow the map in LDS.  Owners are
// ranks in the nets' order, which keeps the priorities.  The rounds are the active-list rounds: point
// claims, viability, the viable nets' neighbour and segment claims, commits,
// block, release.  Bound by one CU's instruction issue: a pass over a batch's
// first 1000 nets of 33 points takes some 3 us, a late round 3 us in all, so
// beyond 2000 nets the kernels win (pattern pass of 20k nets with its last 512,
// 1024, 2048, 4096 nets here: 8.3, 8.2, 8.1, 8.7 ms, without 8.95).  Schedules
// of 1000 nets (81 batches) 10.5 -> 3.4 ms, of 40 nets 0.46 -> 0.15 ms.
constexpr int SMALL_NETS = 2048, SMALL_PTS = 65535;
constexpr int SMALL_LDS = 144 << 10;   // of the 160 KB: the map (4 bytes a cell), then the points' slots (2 each)
constexpr int SLOT_BASE = 1 << 17;   // a cell's slot in the map is its entry less this
struct SmallNet {
    ANet net;
    SSeg seg;
};

// The unassigned nets in index order with their points' offsets; *res is how
// many they are, -1 if they or their points exceed the limits.
__global__ void __launch_bounds__(LTPB) k_small_list(BArgs a, SmallNet* sl, int* soff, int* res) {
    __shared__ int s_w[LTPB / 64];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    // exclusive scan over the workgroup; *total: its sum (the same everywhere)
    const auto scan = [&](int v, int* total) {
        int incl = v;
        for (int d = 1; d < 64; d <<= 1) {
            const int u = __shfl_up(incl, d);
            if (lane >= d) incl += u;
        }
        if (lane == 63) s_w[wv] = incl;
        __syncthreads();
        int before = 0, all = 0;
        for (int w = 0; w < LTPB / 64; w++) {
            if (w < wv) before += s_w[w];
            all += s_w[w];
        }
        __syncthreads();
        *total = all;
        return before + incl - v;
    };
    int n = 0;
    for (int64_t w0 = 0; w0 < a.nwords; w0 += LTPB) {
        const int64_t w = w0 + tid;
        uint32_t m = w < a.nwords ? ~a.nst[w] & NST_ASSIGNED : 0;
        if (w == a.nwords - 1 && (a.n & 15)) m &= (1u << (2 * (a.n & 15))) - 1;
        int total;
        int pos = n + scan(__popc(m), &total);
        for (; m; m &= m - 1, pos++)
            if (pos < SMALL_NETS) sl[pos].net.i = (int)(w * 16 + (__builtin_ctz(m) >> 1));
        n += total;
    }
    __syncthreads();   // sl is read by other threads below
    int64_t pts = 0;
    if (n <= SMALL_NETS)
        for (int r0 = 0; r0 < n; r0 += LTPB) {
            const int r = r0 + tid;
            SNet s{0, 0, 0};
            if (r < n) s = a.sn[sl[r].net.i];
            // a net of more points than the limit counts as the limit and one
            int total;
            const int off = (int)pts + scan(s.npt <= SMALL_PTS ? s.npt : SMALL_PTS + 1, &total);
            if (r < n) {
                sl[r].net.npt = s.npt;
                sl[r].net.pt0 = s.pt0;
                sl[r].seg = a.sg[sl[r].net.i];
                soff[r] = off;
            }
            pts += total;
            if (pts > SMALL_PTS) break;
        }
    if (tid == 0) {
        const bool fits = n <= SMALL_NETS && pts <= SMALL_PTS;
        if (fits) soff[n] = (int)pts;
        *res = fits ? n : -1;
    }
}

__global__ void k_small_fill(int* slot, int64_t cells) {
    const int64_t q = (int64_t)blockIdx.x * TPB + threadIdx.x;
    if (q < cells) slot[q] = -1;
}

// Sixteen lanes a net: the cells' slots.
__global__ void __launch_bounds__(TPB) k_small_mark(BArgs a, const SmallNet* sl, const int* soff, int* slot, const int* res) {
    const int r = (int)(((int64_t)blockIdx.x * TPB + threadIdx.x) >> 4);
    if (r >= *res) return;
    const ANet s = sl[r].net;
    const int off = soff[r];
    for (int k = threadIdx.x & 15; k < s.npt; k += 16) slot[a.pt[s.pt0 + k]] = off + k;
}

__global__ void __launch_bounds__(LTPB) k_small_rounds(BArgs a, int64_t g, const SmallNet* sl,
                                                       const int* soff, int* slot, int* res) {
    __shared__ __align__(16) int s_map[SMALL_LDS / 4];
    __shared__ uint16_t s_off[SMALL_NETS + 2], s_act[SMALL_NETS], s_via[SMALL_NETS];
    __shared__ uint8_t s_st[SMALL_NETS];   // 0 active, 1 assigned, 2 blocked in this batch
    __shared__ int s_na, s_nv, s_won, s_cells;
    constexpr int PER = SMALL_NETS / LTPB;
    const int nu = *res;
    if (nu < 0) return;
    const int tid = threadIdx.x, lane = tid & 63;
    const int grp = tid >> 4, lg = tid & 15;
    constexpr int GROUPS = LTPB / 16, U = 4, CHUNK_NETS = GROUPS * U, KEEP = 1;
    if (tid == 0) s_cells = 0;
    for (int r = tid; r <= nu; r += LTPB) s_off[r] = (uint16_t)soff[r];
    for (int r = tid; r < nu; r += LTPB) s_st[r] = 0;
    __syncthreads();
    // slots: f(point's position, cell) over all points, sixteen lanes a net
    const auto points = [&](auto f) {
        for (int r0 = 0; r0 < nu; r0 += GROUPS) {
            const int r = r0 + grp;
            const ANet s = r < nu ? sl[r].net : ANet{0, 0, 0};
            const int off = r < nu ? s_off[r] : 0;
            for (int k = lg; __ballot(k < s.npt); k += 16) f(k < s.npt, off + k, k < s.npt ? a.pt[s.pt0 + k] : 0);
        }
    };
    points([&](bool in, int e, int q) {
        const bool mine = in && slot[q] == e;
        const uint64_t m = __ballot(mine);
        if (m == 0) return;
        int base = 0;
        if (lane == 0) base = atomicAdd(&s_cells, __popcll(m));
        base = __shfl(base, 0);
        if (mine) slot[q] = SLOT_BASE + base + __popcll(m & ((1ull << lane) - 1));
    });
    __threadfence();
    __syncthreads();
    const int ne = s_cells, ne4 = (ne + 3) / 4 * 4;
    if (4 * ne4 + 2 * s_off[nu] > SMALL_LDS) {
        if (tid == 0) *res = -1;
        return;
    }
    uint16_t* const pid = reinterpret_cast<uint16_t*>(s_map + ne4);
    points([&](bool in, int e, int q) {
        if (in) pid[e] = (uint16_t)(slot[q] - SLOT_BASE);
    });
    __syncthreads();
    // A chunk: 256 listed nets, sixteen lanes a net, U nets a group, with the
    // lanes' first two points' slots.  A round's first KEEP chunks stay in
    // registers from pass to pass: the loads of a pass, not its work, are its
    // time.
    struct Chunk {
        int net[U];      // rank, -1: none
        int cnt[U];      // points
        int slot[U];     // two slots, 0xffff: none
        int live;        // steps of GROUPS nets that hold any
    };
    const auto load = [&](const uint16_t* list, int n, int t0) {
        Chunk c;
        c.live = (n - t0 + GROUPS - 1) / GROUPS;
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (u >= c.live) break;
            const int t = t0 + u * GROUPS + grp;
            const int r = t < n ? list[t] : -1;
            const int beg = r >= 0 ? s_off[r] : 0;
            c.cnt[u] = r >= 0 ? s_off[r + 1] - beg : 0;
            c.net[u] = r;
            const int p0 = lg < c.cnt[u] ? pid[beg + lg] : 0xffff;
            const int p1 = lg + 16 < c.cnt[u] ? pid[beg + lg + 16] : 0xffff;
            c.slot[u] = p0 | p1 << 16;
        }
        return c;
    };
    // test(rank, slot) over the points of a chunk's nets for which begin(rank)
    // holds; end(rank, whether any of the lane's points gave true).
    const auto apply = [&](const Chunk& c, auto begin, auto test, auto end) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (u >= c.live) break;   // the same for every thread
            const int r = c.net[u];
            const bool on = r >= 0 && begin(r);
            const int p0 = c.slot[u] & 0xffff, p1 = c.slot[u] >> 16 & 0xffff;
            bool f = on && p0 != 0xffff && test(r, p0);
            if (on && p1 != 0xffff) f |= test(r, p1);
            if (on && c.cnt[u] > 32) {
                const int beg = s_off[r];
                for (int k = lg + 32; k < c.cnt[u]; k += 16) f |= test(r, (int)pid[beg + k]);
            }
            end(r, f);
        }
    };
    Chunk kept[KEEP];
    const auto over = [&](int n, auto begin, auto point, auto end) {
#pragma unroll
        for (int k = 0; k < KEEP; k++)
            if (k * CHUNK_NETS < n) apply(kept[k], begin, point, end);
        for (int t0 = KEEP * CHUNK_NETS; t0 < n; t0 += CHUNK_NETS) apply(load(s_act, n, t0), begin, point, end);
    };
    const auto all = [](int) { return true; };
    // appends rank v for every lane with want (all lanes of the wave call)
    const auto append = [&](bool want, int v, uint16_t* list, int* counter) {
        const uint64_t m = __ballot(want);
        if (m == 0) return;
        int base = 0;
        if (lane == 0) base = atomicAdd(counter, __popcll(m));
        base = __shfl(base, 0);
        if (want) list[base + __popcll(m & ((1ull << lane) - 1))] = (uint16_t)v;
    };
    int cur = a.ctrl[(g & 1) * C_WORDS + C_CUR];
    int placed = 0;
    unsigned long long rounds = 0, tested = 0, starts = 0;
    while (placed < nu) {
        // every unassigned net is active again, the map empty
        __syncthreads();
        if (tid == 0) s_na = s_nv = s_won = 0;
        for (int e = 4 * tid; e < ne; e += 4 * LTPB) *reinterpret_cast<int4*>(s_map + e) = make_int4(-1, -1, -1, -1);
        __syncthreads();
        for (int r0 = 0; r0 < nu; r0 += LTPB) {
            const int r = nu - 1 - r0 - tid;   // the highest priority claims first: most others then only look
            const bool live = r >= 0 && s_st[r] != 1;
            if (live) s_st[r] = 0;
            append(live, r, s_act, &s_na);
        }
        __syncthreads();
        int na = s_na;
        starts += na;
        bool have = false;
        for (int round = 0; round < ROUNDS; round++) {
            rounds++;
            tested += na;
#pragma unroll
            for (int k = 0; k < KEEP; k++)
                if (k * CHUNK_NETS < na) kept[k] = load(s_act, na, k * CHUNK_NETS);
            // point claims
            over(na, all,
                 [&](int r, int p) {
                     if (s_map[p] < r) atomicMax(&s_map[p], r);
                     return false;
                 },
                 [](int, bool) {});
            __syncthreads();
            // the nets that own every point cell
            over(na, all, [&](int r, int p) { return s_map[p] != r; },
                 [&](int r, bool lost) {
                     const bool any = group_bits(__ballot(lost), 16) != 0;
                     append(lg == 0 && r >= 0 && !any, r, s_via, &s_nv);
                 });
            __syncthreads();
            const int nv = s_nv;
            // their neighbour and segment claims
            for (int w0 = 0; w0 < nv; w0 += GROUPS) {
                const int r = w0 + grp < nv ? s_via[w0 + grp] : -1;
                const SmallNet s = r >= 0 ? sl[r] : SmallNet{};
                const auto claim = [&](bool in, int q) {
                    const int p = in ? slot[q] - SLOT_BASE : -1;
                    if (p >= 0) atomicMax(&s_map[p], r);
                };
                const SegEnds se = segment_ends(a, s.seg, lg);
                for (int k = lg; k < s.net.npt; k += 16) {
                    bool valid[3];
                    int q[3], p[3];
                    point_neighbours(a, true, a.pt[s.net.pt0 + k], valid, q);
                    for (int u = 0; u < 3; u++) p[u] = slot[valid[u] ? q[u] : 0];
                    for (int u = 0; u < 3; u++)
                        if (valid[u] && p[u] >= 0) atomicMax(&s_map[p[u] - SLOT_BASE], r);
                }
                group_segment_cells<16, 1>(a, s.seg, se, [&](bool(&valid)[1], int(&q)[1]) { claim(valid[0], q[0]); });
            }
            __syncthreads();
            // commits
            for (int t0 = 0; t0 < nv; t0 += CHUNK_NETS)
                apply(load(s_via, nv, t0), all, [&](int r, int p) { return s_map[p] != r; },
                      [&](int r, bool lost) {
                          const bool any = group_bits(__ballot(lost), 16) != 0;
                          if (lg == 0 && r >= 0 && !any) {
                              s_st[r] = 1;
                              a.batch[sl[r].net.i] = cur;
                              atomicAdd(&s_won, 1);
                          }
                      });
            __syncthreads();
            const int won = s_won;
            if (won == 0) break;
            have = true;
            placed += won;
            // active nets with a point cell of a committed net sit out the batch
            over(na, [&](int r) { return s_st[r] == 0; },
                 [&](int, int p) {
                     const int o = s_map[p];
                     return o >= 0 && s_st[o] == 1;
                 },
                 [&](int r, bool hit) {
                     const bool any = group_bits(__ballot(hit), 16) != 0;
                     if (lg == 0 && r >= 0 && any) s_st[r] = 2;
                 });
            int keep[PER];
            for (int j = 0; j < PER; j++) keep[j] = j * LTPB + tid < na ? s_act[j * LTPB + tid] : -1;
            __syncthreads();
            if (tid == 0) s_na = s_nv = s_won = 0;
            // their cells are free again; the nets still active
            for (int e = 4 * tid; e < ne; e += 4 * LTPB) {   // past ne: -1 since the batch start
                const int4 m = *reinterpret_cast<const int4*>(s_map + e);
                const int bx = s_st[max(m.x, 0)], by = s_st[max(m.y, 0)], bz = s_st[max(m.z, 0)], bw = s_st[max(m.w, 0)];
                const bool fx = (m.x >= 0) & (bx == 2), fy = (m.y >= 0) & (by == 2);
                const bool fz = (m.z >= 0) & (bz == 2), fw = (m.w >= 0) & (bw == 2);
                if (fx | fy | fz | fw)
                    *reinterpret_cast<int4*>(s_map + e) =
                        make_int4(fx ? -1 : m.x, fy ? -1 : m.y, fz ? -1 : m.z, fw ? -1 : m.w);
            }
            __syncthreads();
            for (int j = 0; j < PER; j++)
                if (j * LTPB < na) append(keep[j] >= 0 && s_st[keep[j]] == 0, keep[j], s_act, &s_na);
            __syncthreads();
            na = s_na;
            if (na == 0) break;
        }
        if (!have) break;   // cannot happen while nets are left: the host reports it
        cur++;
    }
    if (tid == 0) {
        for (int k = 0; k < 2; k++) {
            a.ctrl[k * C_WORDS + C_DONE] = 1;
            a.ctrl[k * C_WORDS + C_CUR] = cur;
        }
        a.ctrl[2 * C_WORDS] += placed;
        a.stat[0] += rounds;
        a.stat[1] += tested;
        a.stat[2] += starts;
    }
}

// The nets left do not fit: the rounds go on from the batch start they stopped at.
__global__ void k_small_resume(BArgs a) {
    a.ctrl[C_DONE] = 0;
    a.ctrl[C_WORDS + C_DONE] = 0;
}

// Net records.  Scheduler index i is entry n - 1 - i of the order (its net
// 'order' and, where the points come per entry, its row of the point arrays).
__global__ void k_nets(int64_t n, const int* order, const int64_t* pt_off, bool by_entry, const int64_t* hs_off,
                       const int64_t* vs_off, SNet* sn, SSeg* sg) {
    const int64_t i = (int64_t)blockIdx.x * TPB + threadIdx.x;
    if (i >= n) return;
    const int net = order[n - 1 - i];
    const int64_t row = by_entry ? n - 1 - i : net;
    const int64_t p0 = pt_off[row];
    sn[i] = SNet{p0, (int)(pt_off[row + 1] - p0), 0};
    const int64_t h0 = hs_off[net], v0 = vs_off[net];
    sg[i] = SSeg{h0, v0, (int)(hs_off[net + 1] - h0), (int)(vs_off[net + 1] - v0)};
}

// Start state: every net unassigned and active, listed in buffer 0.
__global__ void k_start(BArgs a) {
    const int64_t i = (int64_t)blockIdx.x * TPB + threadIdx.x;
    if (i < a.n) {
        if (a.alists) a.alists[i] = ANet{(int)i, a.sn[i].npt, a.sn[i].pt0};
        else a.lists[i] = (int)i;
        a.batch[i] = -1;
    }
    if (i == 0) {
        a.ctrl[C_NU] = (int)a.n;
        a.ctrl[C_UL] = 0;
        a.ctrl[C_NA] = -1;   // active-list rounds: the unassigned list is the active list
        a.ctrl[C_AL] = 0;
    }
}

inline unsigned blocks(int64_t n) { return (unsigned)((n + TPB - 1) / TPB); }

} // namespace

void launch_exclusive_scan(igr_ctx* c, const int* cnt, int64_t n, int64_t* off) {
    const int64_t nb = (n + SCAN_BLOCK - 1) / SCAN_BLOCK;
    c->sched.bsum.alloc(nb);
    k_scan_reduce<<<(unsigned)nb, TPB, 0, c->stream>>>(cnt, n, c->sched.bsum.p);
    k_scan_bsums<<<1, TPB, 0, c->stream>>>(c->sched.bsum.p, nb);
    k_scan_apply<<<(unsigned)nb, TPB, 0, c->stream>>>(cnt, n, c->sched.bsum.p, off);
    HIP_OK(hipGetLastError());
}

int run_schedule_batched(igr_ctx* c, const int* h_order, int64_t n, int mode, int* h_batch_of,
                         const int64_t* d_pt_off, const int* d_pt) {
    if (n == 0) return 0;
    if (n >= 0x7fffffff) throw std::invalid_argument("too many nets for the scheduler");
    KScope ks(c, K_SCHED);
    Sched& S = c->sched;
    NetsDev& N = c->nets;
    hipStream_t st = c->stream;
    S.ids.upload(h_order, n, st);
    S.sn.alloc((sizeof(SNet) + sizeof(SSeg)) * (size_t)n);
    SNet* sn = reinterpret_cast<SNet*>(S.sn.p);
    SSeg* sg = reinterpret_cast<SSeg*>(sn + n);
    k_nets<<<blocks(n), TPB, 0, st>>>(n, S.ids.p, d_pt_off ? d_pt_off : N.pt_off.p, d_pt_off != nullptr, N.hs_off.p,
                                      N.vs_off.p, sn, sg);
    HIP_OK(hipGetLastError());
    const int64_t XYc = (int64_t)c->g.X * c->g.Y;
    S.map.alloc(XYc);
    S.base.alloc(XYc);
    S.head.alloc(XYc);
    S.c_off.alloc(XYc + 1);
    S.c_end.alloc(XYc);
    S.cnt.zero(XYc, st);
    S.batch.alloc(n);
    S.viable.alloc(n);
    S.stat.zero(3, st);
    S.ctrl.zero(2 * C_WORDS + 2, st);   // the last word: k_small_list's result
    const int64_t nwords = (n + 15) / 16;
    S.bits.zero(nwords, st);
    const char* trace_path = std::getenv("IGR_SCHED_TRACE");
    const bool tracing = trace_path && *trace_path;
    if (!S.h_ctrl) HIP_OK(hipHostMalloc(&S.h_ctrl, sizeof(int) * (2 * C_WORDS + 2)));
    int* h_ctrl = S.h_ctrl;
    const auto read_ctrl = [&] {
        HIP_OK(hipMemcpyAsync(h_ctrl, S.ctrl.p, sizeof(int) * (2 * C_WORDS + 2), hipMemcpyDeviceToHost, st));
        HIP_OK(hipStreamSynchronize(st));
    };
    // The one-workgroup rounds for the nets that are left, where they fit.
    const bool small_ok = c->tune.sched_kind == 0 && !tracing;
    const auto small_rounds = [&](const BArgs& b, int64_t g) {
        S.small.alloc(sizeof(SmallNet) * SMALL_NETS + sizeof(int) * (SMALL_NETS + 4));
        S.slot.alloc(XYc);
        SmallNet* sl = reinterpret_cast<SmallNet*>(S.small.p);
        int* soff = reinterpret_cast<int*>(sl + SMALL_NETS);
        int* res = S.ctrl.p + 2 * C_WORDS + 1;
        k_small_list<<<1, LTPB, 0, st>>>(b, sl, soff, res);
        k_small_fill<<<blocks(XYc), TPB, 0, st>>>(S.slot.p, XYc);
        k_small_mark<<<blocks((int64_t)SMALL_NETS * 16), TPB, 0, st>>>(b, sl, soff, S.slot.p, res);
        k_small_rounds<<<1, LTPB, 0, st>>>(b, g, sl, soff, S.slot.p, res);
        HIP_OK(hipGetLastError());
        read_ctrl();
        return h_ctrl[2 * C_WORDS + 1] >= 0;
    };
    BArgs a{};
    a.n = n;
    a.sn = sn;
    a.sg = sg;
    a.pt = d_pt_off ? d_pt : N.pt.p;
    a.hs = N.hs.p;
    a.vs = N.vs.p;
    a.batch = S.batch.p;
    a.ctrl = S.ctrl.p;
    a.stat = S.stat.p;
    a.nst = (uint32_t*)S.bits.p;
    a.nwords = nwords;
    a.X = c->g.X;
    a.Y = c->g.Y;
    a.sparsity = (mode == 1 || mode == 2) ? 2 : 15;
    const auto finish = [&](const char* kind) {
        const int nbatch = h_ctrl[C_CUR];
        const int64_t placed = h_ctrl[2 * C_WORDS];
        unsigned long long sv[3] = {0, 0, 0};
        HIP_OK(hipMemcpyAsync(sv, S.stat.p, sizeof(sv), hipMemcpyDeviceToHost, st));
        HIP_OK(hipStreamSynchronize(st));
        progress("scheduler (%s rounds): %d batches, %llu rounds, %.0f nets tested per round, %.0f unassigned per "
                 "batch", kind, nbatch, sv[0], sv[0] ? (double)sv[1] / (double)sv[0] : 0.0,
                 nbatch ? (double)sv[2] / nbatch : 0.0);
        if (placed != n) throw std::runtime_error("scheduler left a net without a batch");
        if (!h_batch_of) return nbatch;
        std::vector<int> b(n);
        HIP_OK(hipMemcpyAsync(b.data(), S.batch.p, sizeof(int) * n, hipMemcpyDeviceToHost, st));
        HIP_OK(hipStreamSynchronize(st));
        for (int64_t i = 0; i < n; i++) h_batch_of[n - 1 - i] = b[i];
        return nbatch;
    };
    if (small_ok && n <= SMALL_NETS && small_rounds(a, 0)) return finish("one-workgroup");
    // Per-cell lists of the nets' point cells, highest priority first.
    k_cell_count<<<blocks(n), TPB, 0, st>>>(n, sn, d_pt_off ? d_pt : N.pt.p, S.cnt.p);
    launch_exclusive_scan(c, S.cnt.p, XYc, S.c_off.p);
    int64_t entries = 0;
    HIP_OK(hipMemcpyAsync(&entries, S.c_off.p + XYc, sizeof(int64_t), hipMemcpyDeviceToHost, st));
    HIP_OK(hipStreamSynchronize(st));
    S.c_net.alloc(std::max<int64_t>(1, entries));
    const bool release = c->tune.sched_kind ? c->tune.sched_kind == 2
                                            : n >= SCHED_RELEASE_NETS && entries >= SCHED_RELEASE_LIST * XYc;
    if (!release) S.alists.alloc(sizeof(ANet) * NLISTS * (size_t)n);
    if (release) {
        S.lists.alloc(NLISTS * n);
        S.rel.alloc(XYc);
        S.cand.alloc(n);
        S.cstamp.zero(n, st);
        S.hits.alloc(XYc);
        S.hstamp.zero(XYc, st);
        S.cur.alloc(XYc);
    }
    a.map = S.map.p;
    a.base = S.base.p;
    a.c_off = S.c_off.p;
    a.c_end = S.c_end.p;
    a.c_net = S.c_net.p;
    a.head = S.head.p;
    if (release) {
        a.lists = S.lists.p;
        a.rel = S.rel.p;
        a.cand = S.cand.p;
        a.cstamp = S.cstamp.p;
        a.v0 = S.lists.p + 2 * n;
        a.hits = S.hits.p;
        a.hstamp = S.hstamp.p;
        a.cur = S.cur.p;
    } else {
        a.alists = reinterpret_cast<ANet*>(S.alists.p);
    }
    // Nets that fit the one-workgroup rounds if they are like the others, with
    // two points a cell (4 bytes a point).
    if (small_ok) a.small_at = (int)std::min<int64_t>(SMALL_NETS, SMALL_LDS / 4 * n / std::max<int64_t>(1, entries));
    // kernel timing on: the round kernels count the bytes they move
    DevBuf<unsigned long long> byte_slots;
    if (c->prof.on && release) {
        byte_slots.zero(BYTE_SLOTS, st);
        a.bytes = byte_slots.p;
    }
    // IGR_SCHED_TRACE=<file>: append one line per round (the TR_* record)
    DevBuf<long long> trace;
    if (tracing) {
        a.trace_cap = 1 << 20;
        trace.zero(a.trace_cap * TR_WORDS, st);
        a.trace = trace.p;
    }
    HIP_OK(hipMemsetAsync(S.cnt.p, 0, sizeof(int) * XYc, st));
    k_cell_fill<<<blocks(n), TPB, 0, st>>>(a, S.cnt.p);
    k_cell_sort<<<blocks(XYc), TPB, 0, st>>>(a, XYc);
    k_start<<<blocks(n), TPB, 0, st>>>(a);
    HIP_OK(hipGetLastError());
    // Lanes per net: about half the average point count, at most 16.
    const int64_t entries_total = entries;
    const double avg = (double)entries_total / (double)n;
    const int G = c->tune.sched_group ? c->tune.sched_group : avg <= 6 ? 4 : avg <= 16 ? 8 : 16;
    const int CHUNK = c->tune.sched_chunk ? c->tune.sched_chunk : DEF_SCHED_CHUNK;
    const unsigned ggrid = (unsigned)std::min<int64_t>(2048, blocks(n * G));
    const unsigned vgrid = (unsigned)std::min<int64_t>(512, (n * G + LTPB - 1) / LTPB);
    // a wave per viable net, as many as a round of this many nets may find
    const unsigned wgrid = (unsigned)std::min<int64_t>(1024, std::max<int64_t>(16, n / 64));
    const unsigned cgrid = (wgrid + 3) / 4;
    const unsigned gm = (unsigned)std::min<int64_t>(512, (std::max(XYc, n) + LTPB - 1) / LTPB);   // grid-stride
    const int64_t max_rounds = (int64_t)ROUNDS * (n + 1) + CHUNK;
    int64_t g = 0;
    const auto t_start = std::chrono::steady_clock::now();
    auto t_note = t_start;
    for (;;) {
        if (g > max_rounds) throw std::runtime_error("scheduler did not finish");
        const auto t_now = std::chrono::steady_clock::now();
        if (std::chrono::duration<double>(t_now - t_note).count() > 20) {
            t_note = t_now;
            progress("scheduler: %d batches after %.1f s", h_ctrl[(g & 1) * C_WORDS + C_CUR],
                     std::chrono::duration<double>(t_now - t_start).count());
        }
        auto round = [&](auto gv) {
            constexpr int GV = decltype(gv)::value;
            if (release) {
                k_r_claim<GV><<<vgrid, LTPB, 0, st>>>(a, g);
                k_r_viable<GV><<<vgrid, LTPB, 0, st>>>(a, g, S.viable.p);
                k_b_claim_rest<<<wgrid, TPB, 0, st>>>(a, g, S.viable.p);
                k_r_commit<<<cgrid, LTPB, 0, st>>>(a, g, S.viable.p);
                k_r_block<64><<<ggrid, TPB, 0, st>>>(a, g);
                k_r_clear_end<<<gm, LTPB, 0, st>>>(a, g, XYc);
                return;
            }
            k_a_claim<GV><<<ggrid, TPB, 0, st>>>(a, g);
            k_a_viable<GV><<<vgrid, LTPB, 0, st>>>(a, g, S.viable.p);
            k_b_claim_rest<<<wgrid, TPB, 0, st>>>(a, g, S.viable.p);
            k_a_commit<<<cgrid, LTPB, 0, st>>>(a, g, S.viable.p);
            k_a_revert<GV><<<ggrid, TPB, 0, st>>>(a, g);
            k_a_clear_end<<<gm, LTPB, 0, st>>>(a, g, XYc);
        };
        for (int r = 0; r < CHUNK; r++, g++) {
            if (G == 4) round(std::integral_constant<int, 4>{});
            else if (G == 8) round(std::integral_constant<int, 8>{});
            else round(std::integral_constant<int, 16>{});
        }
        HIP_OK(hipGetLastError());
        read_ctrl();
        const int done = h_ctrl[(g & 1) * C_WORDS + C_DONE];
        if (done == 1) break;
        if (done == 2) {
            const int64_t rest = n - h_ctrl[2 * C_WORDS];
            if (small_rounds(a, g)) break;
            a.small_at = (int)(rest / 2);
            k_small_resume<<<1, 1, 0, st>>>(a);
        }
    }
    h_ctrl[C_CUR] = h_ctrl[(g & 1) * C_WORDS + C_CUR];
    if (a.bytes) {
        std::vector<unsigned long long> slots(BYTE_SLOTS);
        HIP_OK(hipMemcpyAsync(slots.data(), a.bytes, sizeof(unsigned long long) * BYTE_SLOTS, hipMemcpyDeviceToHost,
                              st));
        HIP_OK(hipStreamSynchronize(st));
        double tot = 0;
        for (unsigned long long v : slots) tot += (double)v;
        c->prof.bytes[K_SCHED] += tot;
    }
    if (a.trace) {
        const int64_t nrec = std::min<int64_t>(g, a.trace_cap);
        std::vector<long long> rec((size_t)(nrec * TR_WORDS));
        HIP_OK(hipMemcpyAsync(rec.data(), a.trace, sizeof(long long) * rec.size(), hipMemcpyDeviceToHost, st));
        HIP_OK(hipStreamSynchronize(st));
        int khz = 0;
        HIP_OK(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, c->device));
        if (FILE* f = std::fopen(trace_path, "a")) {
            std::fprintf(f, "# nets %lld rounds %s lanes %d clock_khz %d\n", (long long)n,
                         release ? "release-driven" : "active-list", G, khz);
            std::fprintf(f, "g batch round tested viable committed hits released new_owners clock\n");
            for (int64_t r = 0; r < nrec; r++) {
                const long long* q = rec.data() + r * TR_WORDS;
                if (r > 0 && q[TR_CLOCK] == 0) break;   // rounds after the last batch record nothing
                std::fprintf(f, "%lld %lld %lld %lld %lld %lld %lld %lld %lld %lld\n", (long long)r, q[0], q[1], q[2],
                             q[3], q[4], q[5], q[6], q[7], q[8]);
            }
            std::fclose(f);
        }
    }
    return finish(release ? "release-driven" : "active-list");
}

} // namespace igr_dev
