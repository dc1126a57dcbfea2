#include "mail.hpp"

#include <atomic>

namespace kahip {

namespace {

struct Pieces {
    Mail::Piece p[Mail::kMaxPieces];
};

constexpr int kMailThreads = 1024;

// Every thread's words are on the host (system-scope fence) before the number is.
__global__ __launch_bounds__(kMailThreads) void send_mail(Pieces m, int* box, int seq) {
    int at = 1;
#pragma unroll
    for (int i = 0; i < Mail::kMaxPieces; ++i) {
        for (int j = threadIdx.x; j < m.p[i].n; j += kMailThreads) box[at + j] = m.p[i].p[j];
        at += m.p[i].n;
    }
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0)
        __hip_atomic_store(box, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

}  // namespace

void MappedBuf::alloc(size_t bytes) {
    KH_CHECK(hipHostMalloc(&p, bytes, hipHostMallocMapped | hipHostMallocCoherent));
    KH_CHECK(hipHostGetDevicePointer(&dev, p, 0));
}

MappedBuf::~MappedBuf() {
    if (p) (void)hipHostFree(p);
}

void Mail::init() {
    if (host_) return;
    buf_.alloc(sizeof(int) * (kInts + 1));
    dev_ = static_cast<int*>(buf_.dev);
    host_ = static_cast<volatile int*>(buf_.p);
    host_[0] = 0;
}

int* Mail::box() {
    init();
    return dev_;
}

int Mail::next() {
    init();
    seq_ = (int)((unsigned)seq_ + 1u);  // (wraps)
    return seq_;
}

void Mail::post(hipStream_t s, Piece a, Piece b, Piece c, Piece d) {
    KH_REQUIRE((long long)a.n + b.n + c.n + d.n <= kInts, "mail too long");
    const int seq = next();
    hipLaunchKernelGGL(send_mail, dim3(1), dim3(kMailThreads), 0, s, Pieces{{a, b, c, d}}, dev_,
                       seq);
    KH_CHECK(hipGetLastError());
}

const int* Mail::wait(hipStream_t s) {
    for (unsigned spin = 1; host_[0] != seq_; ++spin) {
        __builtin_ia32_pause();
        if (spin % (1u << 16)) continue;
        const hipError_t e = hipStreamQuery(s);
        if (e == hipErrorNotReady) {
            (void)hipGetLastError();  // not an error of ours
            continue;
        }
        KH_CHECK(e);
        KH_REQUIRE(host_[0] == seq_, "the GPU finished without its answer");
    }
    std::atomic_thread_fence(std::memory_order_acquire);
    return const_cast<const int*>(host_) + 1;
}

}  // namespace kahip
