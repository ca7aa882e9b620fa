// Route buffers of rip-up-and-reroute passes (NetsDev, PassRoutes) without a
// GPU: the HIP calls they make are defined here over host memory, with the
// live blocks counted, so that every pointer the device would follow can be
// checked.  Prints one line per finding; exits 0 when there is none.
#include "igr_ctx.hpp"

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>

static std::map<char*, size_t> live;
static int fail_malloc = 0, fail_copy = 0;   // the next so many calls fail

hipError_t hipMalloc(void** p, size_t n) {
    if (fail_malloc > 0) return fail_malloc--, hipErrorOutOfMemory;
    *p = std::calloc(1, n);
    live[(char*)*p] = n;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    live.erase((char*)p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
    if (fail_copy > 0) return fail_copy--, hipErrorInvalidValue;
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t) { return hipMemcpy(d, s, n, k); }
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { return std::memset(d, v, n), hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipHostFree(void*) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "failed"; }

using namespace igr_dev;

static int findings = 0;
static void expect(bool ok, const char* what) {
    if (ok) return;
    findings++;
    std::printf("%s\n", what);
}

constexpr int NETS = 8, WORDS = 64;   // words a net

static void open_nets(NetsDev& N) {
    N.n = NETS;
    N.routes.alloc(NETS * WORDS);
    for (int i = 0; i < NETS; i++) {
        N.h_rptr.push_back(N.routes.p + i * WORDS);
        N.h_rcap.push_back(WORDS);
        N.h_rbuf.push_back(-1);
    }
    N.rptr.upload(N.h_rptr.data(), NETS, nullptr);
}

// A pass over 'nets': its kernels move the device pointers and mark the routes
// with 'mark'; 'fails' ends it before it is adopted.
static void pass(NetsDev& N, const std::vector<int>& nets, int mark, bool fails) {
    try {
        PassRoutes r(N, nullptr, (int64_t)nets.size() * WORDS);
        for (size_t k = 0; k < nets.size(); k++) {
            r.base[k * WORDS] = mark;
            N.rptr.p[nets[k]] = r.base + k * WORDS;
        }
        if (fails) throw std::runtime_error("pass");
        r.adopt(nets.data(), (int64_t)nets.size(), 2, [](int64_t i) { return i * WORDS; });
    } catch (const std::runtime_error&) {
    }
}

// What the device reads for a net: the mark, or -1 where its memory is gone.
static int seen(const NetsDev& N, int net) {
    char* p = (char*)N.rptr.p[net];
    auto it = live.upper_bound(p);
    if (it == live.begin()) return -1;
    --it;
    return p + WORDS * sizeof(int) <= it->first + it->second ? *N.rptr.p[net] : -1;
}

int main() {
    {   // a failed pass, then passes that free and reuse buffers
        NetsDev N;
        open_nets(N);
        pass(N, {0, 1, 2}, 1, false);
        pass(N, {0, 1, 2, 3}, 2, true);
        for (int k = 0; k < 4; k++) pass(N, {4, 5, 6}, 3 + k, false);
        for (int i = 0; i < 3; i++) expect(seen(N, i) == 1, "a net of a failed pass lost its route");
        expect(seen(N, 3) == 0, "a net of a failed pass lost its pattern route");
        for (int i = 4; i < 7; i++) expect(seen(N, i) == 6, "a later pass's route is not read");
        for (int i = 0; i < NETS; i++) expect(N.h_rptr[i] == N.rptr.p[i], "host and device read different routes");
    }
    {   // the same where the pointers cannot be put back
        NetsDev N;
        open_nets(N);
        try {
            PassRoutes r(N, nullptr, 4 * WORDS);
            r.base[0] = 7;
            N.rptr.p[3] = r.base;
            fail_copy = 1;
            throw std::runtime_error("pass");
        } catch (const std::runtime_error&) {
        }
        fail_copy = 0;
        for (int k = 0; k < 4; k++) pass(N, {4, 5, 6}, 3 + k, false);
        expect(seen(N, 3) == 7, "a buffer the device still points to went away");
    }
    {   // no memory for a pass's buffer
        NetsDev N;
        open_nets(N);
        fail_malloc = 1;
        pass(N, {0, 1}, 1, false);
        expect(N.dag_routes.empty(), "a buffer without memory stayed");
        pass(N, {0, 1}, 2, false);
        pass(N, {0, 1}, 3, false);
        expect(N.spare && N.spare->p, "no spare buffer after two passes");
        int* p = N.spare ? N.spare->p : nullptr;
        pass(N, {0, 1}, 4, false);
        expect(N.rptr.p[0] == p, "the spare buffer was not used");
        // a spare of another size makes way for the next one retired
        pass(N, {0, 1, 2, 3, 4, 5, 6, 7}, 5, false);
        pass(N, {0, 1, 2, 3, 4, 5, 6, 7}, 6, false);
        p = N.spare ? N.spare->p : nullptr;
        pass(N, {0, 1, 2, 3, 4, 5, 6, 7}, 7, false);
        expect(p && N.rptr.p[0] == p, "a spare that does not fit blocks the next one");
    }
    expect(live.empty(), "a buffer was not freed");
    return findings != 0;
}
