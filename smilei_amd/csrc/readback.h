// readback.h -- device arrays to pageable host memory through pinned staging.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace smi {

// Staging of one context (one host thread at a time).  From 4 MiB on, 1 MiB
// blocks arrive in pinned memory and are copied out by four threads while the
// next ones are under way: hipMemcpy into pageable memory moves 15 GB/s, one
// host thread copying out of the runtime's own staging, and 10 into pages that
// were never touched (8.4 MB: 557 -> 335 us, 33.6 MB into fresh memory: 3,440
// -> 1,390).  Smaller arrays keep hipMemcpy: in whole runs of 0.26 and 2 MB
// fields staging gained nothing and its allocation cost 1.3 ms per context.
class Readback {
public:
    // for arrays of up to `bytes`: 8 MiB of pinned memory, or none
    void init(size_t bytes);
    void release();
    // copies n bytes from src, ordered after the work on st; returns when done
    void copy(void *dst, const void *src, size_t n, hipStream_t st);

private:
    static constexpr size_t kLarge = 4u << 20, kBlock = 1u << 20;
    static constexpr int kSlots = 8, kThreads = 4;
    void copy_threads(char *dst, const char *src, size_t n, hipStream_t st);
    char *buf_ = nullptr;
    hipEvent_t ev_[kSlots] = {};
};

}  // namespace smi
