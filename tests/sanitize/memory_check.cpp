// Device memory that runs out, on a stand-in for the HIP allocator with 1000 bytes: buffers that
// grow, and calls after calls that left their buffers behind. Built and run by
// tests/test_device_memory.py; exits non-zero on a failed check.
#include <cstdio>
#include <cstdlib>
#include <map>
#include <thread>

#include "lease.hpp"

#define CHECK(c)                                                                 \
    do {                                                                         \
        if (!(c)) {                                                              \
            std::fprintf(stderr, "check failed: %s (line %d)\n", #c, __LINE__);  \
            std::exit(1);                                                        \
        }                                                                        \
    } while (0)

namespace {
constexpr size_t kMemory = 1000;
std::map<void*, size_t> g_blocks;
size_t g_used = 0;
hipError_t g_last = hipSuccess;
}  // namespace

extern "C" {
hipError_t hipMalloc(void** p, size_t bytes) {
    if (g_used + bytes > kMemory) return g_last = hipErrorOutOfMemory;
    *p = std::malloc(bytes);
    g_blocks[*p] = bytes;
    g_used += bytes;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    g_used -= g_blocks.at(p);
    g_blocks.erase(p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipGetLastError() {
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}
hipError_t hipGetDevice(int* d) {
    *d = 0;
    return hipSuccess;
}
const char* hipGetErrorString(hipError_t) { return "error"; }
}

using namespace kahip;

struct Buffers {
    DevBuf<char> a, b, c;
};
using BufLease = Lease<Buffers>;

// A call that needs so many bytes of each buffer; how often it ran.
int call(long long a, long long b, long long c) {
    int runs = 0;
    run_giving_back<Buffers>([&] {
        ++runs;
        BufLease l;
        if (a) l->a.reserve(a);
        if (b) l->b.reserve(b);
        if (c) l->c.reserve(c);
    });
    CHECK(hipGetLastError() == hipSuccess);
    return runs;
}

int main() {
    {  // the margin of a growing buffer is given up when it does not fit
        DevBuf<char> x;
        x.reserve(100);
        x.reserve(400);
        CHECK(x.cap == 450);
        x.reserve(950);
        CHECK(x.cap == 950);
        CHECK(hipGetLastError() == hipSuccess);
        bool refused = false;
        try {
            x.reserve(1001);
        } catch (const OutOfMemory&) {
            refused = true;
        }
        CHECK(refused && x.cap == 0 && x.p == nullptr && g_used == 0);
        CHECK(hipGetLastError() == hipSuccess);
        x.reserve(1000);
    }
    CHECK(call(10, 10, 0) == 1);
    CHECK(call(10, 10, 0) == 1);
    CHECK(call(480, 500, 0) == 2);  // fits without the margins
    CHECK(call(480, 500, 0) == 1);
    CHECK(call(0, 0, 600) == 2);    // fits without the buffers of the calls before
    run_giving_back<Buffers>([&] {  // a call without a lease
        DevBuf<char> graph;
        graph.reserve(900);
    });
    CHECK(g_used == 0);
    CHECK(call(300, 0, 0) == 1);
    bool refused = false;
    try {
        call(900, 200, 0);  // does not fit at all
    } catch (const OutOfMemory&) {
        refused = true;
    }
    CHECK(refused && hipGetLastError() == hipSuccess);
    CHECK(call(100, 0, 0) == 1);
    {  // what another call holds is not given back
        BufLease held;
        held->a.reserve(600);
        refused = false;
        std::thread other([&] {
            try {
                call(0, 500, 0);
            } catch (const OutOfMemory&) {
                refused = true;
            }
        });
        other.join();
        CHECK(refused && held->a.cap >= 600);
    }
    CHECK(call(0, 300, 0) == 1);
    CHECK(BufLease::release_idle() && g_used == 0 && !BufLease::release_idle());
    std::puts("memory_check ok");
    return 0;
}
