// workspace.cpp -- the stream-ordered pools behind Workspace.
#include "workspace.h"

#include <cstdint>
#include <mutex>
#include <vector>

namespace smi {

namespace {


std::mutex g_lock;
std::vector<hipMemPool_t> g_pool;  // by device; made at the first use, held until the process ends

hipMemPool_t device_pool(int dev)
{
    std::lock_guard<std::mutex> hold(g_lock);
    if ((int)g_pool.size() <= dev) g_pool.resize(dev + 1, nullptr);
    if (!g_pool[dev]) {
        hipMemPoolProps props{};
        props.allocType = hipMemAllocationTypePinned;
        props.location.type = hipMemLocationTypeDevice;
        props.location.id = dev;
        hipMemPool_t pool = nullptr;
        if (hipMemPoolCreate(&pool, &props) != hipSuccess) return nullptr;
        uint64_t keep = kWorkspaceKeep;
        (void)hipMemPoolSetAttribute(pool, hipMemPoolAttrReleaseThreshold, &keep);
        g_pool[dev] = pool;
    }
    return g_pool[dev];
}

}  // namespace

Workspace::Workspace(size_t bytes, hipStream_t stream) : st(stream)
{
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &status) != hipSuccess || status != hipStreamCaptureStatusNone) return;
    int dev = 0;
    hipMemPool_t pool = hipGetDevice(&dev) == hipSuccess ? device_pool(dev) : nullptr;
    if (pool && hipMallocFromPoolAsync(&p, bytes, pool, stream) != hipSuccess) {
        p = nullptr;
        (void)hipGetLastError();  // out of memory: the caller does without
    }
}

Workspace::~Workspace()
{
    if (p) (void)hipFreeAsync(p, st);
}

}  // namespace smi
