// readback.cpp -- pinned staging of device-to-host copies.
#include "readback.h"

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <mutex>
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

namespace {

// Flags of the blocks: set once, waited for by a short spin (the next block of a
// running copy is tens of microseconds away) and then asleep.
class Flags {
public:
    explicit Flags(int n) : set_(n) {}
    void set(int b)
    {
        {
            std::lock_guard<std::mutex> hold(lock_);
            set_[b].store(1, std::memory_order_release);
        }
        changed_.notify_all();
    }
    void wait(int b, bool spin)
    {
        for (int k = 0; spin && k < 200; ++k) {
            if (set_[b].load(std::memory_order_acquire)) return;
            std::this_thread::yield();
        }
        std::unique_lock<std::mutex> hold(lock_);
        changed_.wait(hold, [&] { return set_[b].load(std::memory_order_acquire) != 0; });
    }

private:
    std::vector<std::atomic<int>> set_;
    std::mutex lock_;
    std::condition_variable changed_;
};

}  // namespace

// Block b waits in slot b % kSlots: it is marked arrived once it is there and
// done once it has been copied out (helper t takes the blocks b with b %
// kThreads == t, in order).  Before its first block a helper sleeps while the
// stream has other work: it may have a long way to go to the copy (on an idle
// stream the spin saves 15 us of 340 for 8.4 MB).  Every wait ends: the calling
// thread marks all blocks, on an error as arrived too (gone: nothing is copied
// any more).
void Readback::copy_threads(char *dst, const char *src, size_t n, hipStream_t st)
{
    const int nb = (int)((n + kBlock - 1) / kBlock);
    Flags arrived(nb), done(nb);
    std::atomic<int> gone{0};
    const bool idle = hipStreamQuery(st) == hipSuccess;
    if (!idle) (void)hipGetLastError();  // not ready; a fault is found by the copy
    auto helper = [&](int t) {
        for (int b = t; b < nb; b += kThreads) {
            arrived.wait(b, idle || b != t);
            if (gone.load(std::memory_order_acquire)) return;
            const size_t o = (size_t)b * kBlock;
            std::memcpy(dst + o, buf_ + (size_t)(b % kSlots) * kBlock, std::min(kBlock, n - o));
            done.set(b);
        }
    };
    std::vector<std::thread> team;
    auto finish = [&](bool failed) {
        if (failed) {
            gone.store(1, std::memory_order_release);
            for (int b = 0; b < nb; ++b) arrived.set(b);
        }
        for (auto &th : team) th.join();
    };
    try {
        team.reserve(kThreads);
        for (int t = 0; t < kThreads; ++t) team.emplace_back(helper, t);
    } catch (const std::exception &) {  // no more threads or memory on this host
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
                if (issued >= kSlots) done.wait(issued - kSlots, true);
                const size_t o = (size_t)issued * kBlock;
                SMI_HIP(hipMemcpyAsync(buf_ + (size_t)(issued % kSlots) * kBlock, src + o, std::min(kBlock, n - o),
                                       hipMemcpyDeviceToHost, st));
                SMI_HIP(hipEventRecord(ev_[issued % kSlots], st));
            }
            SMI_HIP(hipEventSynchronize(ev_[b % kSlots]));
            arrived.set(b);
        }
    } catch (...) {
        finish(true);
        (void)hipStreamSynchronize(st);
        throw;
    }
    finish(false);
}

}  // namespace smi
