// readback.cpp -- pinned staging of device-to-host copies.
#include "readback.h"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <system_error>
#include <thread>
#include <vector>

#include "common.h"

namespace smi {

void Readback::init(size_t bytes)
{
    if (bytes < kLarge) return;
    if (hipHostMalloc((void **)&buf_, kSlots * kBlock, 0) != hipSuccess) {
        buf_ = nullptr;
        (void)hipGetLastError();  // copy() does without
        return;
    }
    for (auto &e : ev_) SMI_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
}

void Readback::release()
{
    for (auto &e : ev_) {
        if (e) (void)hipEventDestroy(e);
        e = nullptr;
    }
    (void)hipHostFree(buf_);
    buf_ = nullptr;
}

void Readback::copy(void *dst, const void *src, size_t n, hipStream_t st)
{
    if (n == 0) return;
    if (buf_ && n >= kLarge) {
        copy_threads((char *)dst, (const char *)src, n, st);
    } else {
        SMI_HIP(hipStreamSynchronize(st));
        SMI_HIP(hipMemcpy(dst, src, n, hipMemcpyDeviceToHost));
    }
}

// Block b waits in slot b % kSlots: arrived[b] is set once it is there, done[b]
// once it has been copied out (helper t takes the blocks b with b % kThreads ==
// t, in order).  Every wait ends: the calling thread marks all
// blocks, on an error as arrived too (gone: nothing is copied any more).
void Readback::copy_threads(char *dst, const char *src, size_t n, hipStream_t st)
{
    const int nb = (int)((n + kBlock - 1) / kBlock);
    std::vector<std::atomic<int>> arrived(nb), done(nb);
    for (int b = 0; b < nb; ++b) {
        arrived[b].store(0, std::memory_order_relaxed);
        done[b].store(0, std::memory_order_relaxed);
    }
    std::atomic<int> gone{0};
    auto helper = [&](int t) {
        for (int b = t; b < nb; b += kThreads) {
            while (!arrived[b].load(std::memory_order_acquire)) std::this_thread::yield();
            if (gone.load(std::memory_order_acquire)) return;
            const size_t o = (size_t)b * kBlock;
            std::memcpy(dst + o, buf_ + (size_t)(b % kSlots) * kBlock, std::min(kBlock, n - o));
            done[b].store(1, std::memory_order_release);
        }
    };
    std::vector<std::thread> team;
    auto finish = [&](bool failed) {
        if (failed) {
            gone.store(1, std::memory_order_release);
            for (int b = 0; b < nb; ++b) arrived[b].store(1, std::memory_order_release);
        }
        for (auto &th : team) th.join();
    };
    try {
        team.reserve(kThreads);
        for (int t = 0; t < kThreads; ++t) team.emplace_back(helper, t);
    } catch (const std::system_error &) {  // no more threads on this host
        finish(true);
        SMI_HIP(hipStreamSynchronize(st));
        SMI_HIP(hipMemcpy(dst, src, n, hipMemcpyDeviceToHost));
        return;
    }
    try {
        int issued = 0;
        for (int b = 0; b < nb; ++b) {
            // two blocks under way while the helpers copy the earlier ones out
            for (; issued < nb && issued < b + 2; ++issued) {
                if (issued >= kSlots)
                    while (!done[issued - kSlots].load(std::memory_order_acquire)) std::this_thread::yield();
                const size_t o = (size_t)issued * kBlock;
                SMI_HIP(hipMemcpyAsync(buf_ + (size_t)(issued % kSlots) * kBlock, src + o, std::min(kBlock, n - o),
                                       hipMemcpyDeviceToHost, st));
                SMI_HIP(hipEventRecord(ev_[issued % kSlots], st));
            }
            SMI_HIP(hipEventSynchronize(ev_[b % kSlots]));
            arrived[b].store(1, std::memory_order_release);
        }
    } catch (...) {
        finish(true);
        (void)hipStreamSynchronize(st);
        throw;
    }
    finish(false);
}

}  // namespace smi
