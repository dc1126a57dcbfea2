// Small results from the GPU to the waiting host without a copy engine or a stream
// synchronisation.
#pragma once

#include "common.hpp"

namespace kahip {

// Host memory that kernels read and write in place.
struct MappedBuf {
    void* p = nullptr;    // for the host
    void* dev = nullptr;  // for kernels
    MappedBuf() = default;
    MappedBuf(const MappedBuf&) = delete;
    MappedBuf& operator=(const MappedBuf&) = delete;
    ~MappedBuf();
    void alloc(size_t bytes);
};

// A kernel writes a few words into mapped host memory, then their sequence number; the host polls
// for it. The answer is there about 6 us after the kernels before it; a pageable
// device-to-host copy and its synchronisation take 20 to 40 us (blit kernel, signal, wake-up), and
// a level of the multilevel pipeline waits about ten times. Used by one thread at a time.
class Mail {
public:
    static constexpr int kInts = 1 << 18;  // capacity in words (1 MB of pinned memory)
    struct Piece {
        const int* p;
        int n;
    };
    static constexpr int kMaxPieces = 4;

    Mail() = default;
    // Enqueues the sending of the pieces, one after the other, on s.
    void post(hipStream_t s, Piece a, Piece b = {nullptr, 0}, Piece c = {nullptr, 0},
              Piece d = {nullptr, 0});
    // For kernels that write the answer themselves (words 1.. of box(), then the number to word 0).
    int next();
    int* box();
    // Waits for the last post() or next() and returns its words. s is the stream it was enqueued
    // on: a failed launch ends the wait with an error.
    const int* wait(hipStream_t s);

private:
    void init();
    MappedBuf buf_;
    volatile int* host_ = nullptr;
    int* dev_ = nullptr;
    int seq_ = 0;
};

}  // namespace kahip
