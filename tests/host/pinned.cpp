// Large copies (staging.hip) and the route mailbox where pinned memory can and
// cannot be had, without a GPU: the HIP calls are defined here over host memory.
// Prints one line per finding; exits 0 when there is none.
#include "igr_ctx.hpp"

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

static bool no_pinned = false;      // pinned allocations fail
static bool no_device_address = false;
static int asked = 0, held = 0;     // pinned allocations asked for, and not freed
static hipError_t last = hipSuccess;

hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    asked++;
    if (no_pinned) return last = hipErrorOutOfMemory;
    held++;
    return *p = std::malloc(n), hipSuccess;
}
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned) {
    if (no_device_address) return last = hipErrorInvalidValue;
    return *d = h, hipSuccess;
}
hipError_t hipHostFree(void* p) { return held--, std::free(p), hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) { return *p = std::calloc(1, n), hipSuccess; }
hipError_t hipFree(void* p) { return std::free(p), hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { return std::memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t) { return hipMemcpy(d, s, n, k); }
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { return std::memset(d, v, n), hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return *e = reinterpret_cast<hipEvent_t>(8), hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* t, hipEvent_t, hipEvent_t) { return *t = 0, hipSuccess; }
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() {
    const hipError_t e = last;
    return last = hipSuccess, e;
}
const char* hipGetErrorString(hipError_t) { return "failed"; }

using namespace igr_dev;

static int findings = 0;
static void expect(bool ok, const char* what) {
    if (ok) return;
    findings++;
    std::printf("%s\n", what);
}

// One array to the device and back.
static bool round_trip(igr_ctx& c, int64_t bytes, int seed) {
    std::vector<char> a(bytes), dev(bytes, 0), b(bytes, 0);
    for (int64_t i = 0; i < bytes; i++) a[i] = (char)(i * 7 + i / 4099 + seed);
    copy_to_device(&c, dev.data(), a.data(), bytes, nullptr);
    copy_to_host(&c, b.data(), dev.data(), bytes, nullptr);
    return a == b;
}

int main() {
    constexpr int64_t M = 1 << 20;
    const int64_t sizes[] = {0, 1, M - 1, M, 2 * M, 2 * M + 1, 3 * M, 16 * M, 16 * M + 1, 35 * M};
    for (bool pinned : {true, false}) {
        no_pinned = !pinned;
        asked = 0;
        igr_ctx c;
        for (int64_t n : sizes) {
            bool same = false;
            try {
                same = round_trip(c, n, 1);
            } catch (const std::exception& e) {
                std::printf("%s\n", e.what());
            }
            expect(same, pinned ? "a copy differs" : "a copy fails without pinned memory");
        }
        expect(asked == 1, "pinned memory is asked for again and again");
        expect(last == hipSuccess, "a failed allocation is left for the next call");
        expect(held == (pinned ? 1 : 0), "pinned memory is not kept once");
    }
    no_pinned = false;
    expect(held == 0, "a context's pinned memory is not freed");
    for (int k = 0; k < 3; k++) {
        no_pinned = k == 1;
        no_device_address = k == 2;
        asked = 0;
        {
            igr_ctx c;
            for (int t = 0; t < 3; t++) expect(c.mail.open() == (k == 0), "the mailbox opens without its memory, or not with it");
            expect(asked == 1, "the mailbox asks again and again");
            expect(last == hipSuccess, "the mailbox leaves an error for the next call");
        }
        expect(held == 0, "the mailbox is not freed");
    }
    return findings != 0;
}
