// The initial partitioner when the system has only so many threads to give: pthread_create fails
// after the first `allowed` ones. Prints the partition's checksum. Built and run by
// tests/test_thread_limit.py.
#include <dlfcn.h>
#include <pthread.h>

#include <atomic>
#include <cerrno>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "initial_partition.hpp"

static std::atomic<int> g_allowed{1 << 30};

extern "C" int pthread_create(pthread_t* t, const pthread_attr_t* a, void* (*f)(void*), void* x) {
    using Create = int (*)(pthread_t*, const pthread_attr_t*, void* (*)(void*), void*);
    static const Create create = (Create)dlsym(RTLD_NEXT, "pthread_create");
    return g_allowed-- > 0 ? create(t, a, f, x) : EAGAIN;
}

int main(int argc, char** argv) {
    const int allowed = argc > 1 ? std::atoi(argv[1]) : 0;
    kahip::HostGraph g;  // a torus of 96 x 96 nodes
    const int side = 96;
    g.n = side * side;
    for (int v = 0; v < g.n; ++v) {
        const int x = v % side, y = v / side;
        g.xadj.push_back((int)g.adjncy.size());
        for (int u : {y * side + (x + 1) % side, y * side + (x + side - 1) % side,
                      (y + 1) % side * side + x, (y + side - 1) % side * side + x}) {
            g.adjncy.push_back(u);
            g.adjwgt.push_back(1);
        }
        g.vwgt.push_back(1);
    }
    g.xadj.push_back((int)g.adjncy.size());
    kahip::IpParams p;
    p.k = 16;
    p.block_bound = (int)(1.03 * g.n / 16);
    p.repetitions = 4;
    p.bisection_tries = 4;
    p.threads = 16;
    p.seed = 5;
    if (allowed >= 0) g_allowed = allowed;
    std::vector<int> part;
    kahip::initial_partition(g, p, part);
    unsigned long long h = 1469598103934665603ull;
    for (int b : part) h = (h ^ (unsigned)b) * 1099511628211ull;
    std::printf("%llx\n", h);
    return 0;
}
