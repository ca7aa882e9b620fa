// parallel_ranges, and with an argument where threads cannot be created: the
// address space is limited so that no thread stack fits.  Prints one line per
// finding; exits 0 when there is none.
#include "par.hpp"

#include <sys/resource.h>

#include <cstdio>
#include <cstring>
#include <stdexcept>
#include <vector>

static int findings = 0;
static void expect(bool ok, const char* what) {
    if (ok) return;
    findings++;
    std::printf("%s\n", what);
}

static void check(const char* where) {
    for (int64_t n : {0, 1, 2, 7, 1000}) {
        std::vector<int> seen((size_t)n, 0);
        igr::parallel_ranges(n, 8, [&](int64_t a, int64_t b, int t) {
            expect(t >= 0 && t < 8, "a range's thread index is out of range");
            for (int64_t i = a; i < b; i++) seen[(size_t)i]++;
        });
        for (int s : seen) expect(s == 1, where);
    }
    bool thrown = false;
    try {
        igr::parallel_ranges(100, 8, [&](int64_t a, int64_t, int) {
            if (a > 50) throw std::runtime_error("range");
        });
    } catch (const std::runtime_error& e) {
        thrown = !std::strcmp(e.what(), "range");
    }
    expect(thrown, "a range's exception is not passed on");
}

int main(int argc, char**) {
    if (argc == 1) {
        check("an element is not visited once");
        return findings != 0;
    }
    rlimit lim{};
    long pages = 0;
    if (FILE* f = std::fopen("/proc/self/statm", "r")) {
        if (std::fscanf(f, "%ld", &pages) != 1) pages = 0;
        std::fclose(f);
    }
    lim.rlim_cur = lim.rlim_max = (rlim_t)pages * 4096 + (4 << 20);
    setrlimit(RLIMIT_AS, &lim);
    bool created = true;
    try {
        std::thread th([] {});
        th.join();
    } catch (const std::system_error&) {
        created = false;
    }
    expect(!created, "threads can still be created: nothing is tested");
    check("without threads an element is not visited once");
    return findings != 0;
}
