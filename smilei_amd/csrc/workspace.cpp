// workspace.cpp -- the stream-ordered pools behind Workspace.
#include "workspace.h"

#include <cstdint>
#include <mutex>
#include <vector>

namespace smi {

namespace {

// A device's pool: made at the first use, held until the process ends.
struct DevicePool {
    hipMemPool_t pool = nullptr;
    bool tried = false;  // a device without pools is not asked again
};

std::mutex g_lock;
std::vector<DevicePool> g_pool;  // by device

hipMemPool_t device_pool(int dev)
{
    std::lock_guard<std::mutex> hold(g_lock);
    if ((int)g_pool.size() <= dev) g_pool.resize(dev + 1);
    DevicePool &d = g_pool[dev];
    if (!d.tried) {
        d.tried = true;
        hipMemPoolProps props{};
        props.allocType = hipMemAllocationTypePinned;
        props.location.type = hipMemLocationTypeDevice;
        props.location.id = dev;
        hipMemPool_t pool = nullptr;
        if (hipMemPoolCreate(&pool, &props) != hipSuccess) return nullptr;
        uint64_t keep = kWorkspaceKeep;
        // (without its threshold a pool only gives everything back)
        if (hipMemPoolSetAttribute(pool, hipMemPoolAttrReleaseThreshold, &keep) != hipSuccess) (void)hipGetLastError();
        d.pool = pool;
    }
    return d.pool;
}

bool allocate(void **p, size_t bytes, hipStream_t st)
{
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(st, &status) != hipSuccess || status != hipStreamCaptureStatusNone) return false;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return false;
    const hipMemPool_t pool = device_pool(dev);
    return pool && hipMallocFromPoolAsync(p, bytes, pool, st) == hipSuccess;
}

}  // namespace

Workspace::Workspace(size_t bytes, hipStream_t stream) : st(stream)
{
    if (allocate(&p, bytes, stream)) return;
    p = nullptr;
    // the caller does without: what failed here must not be taken for a
    // failure of the launches that follow
    (void)hipGetLastError();
}

Workspace::~Workspace()
{
    if (p && hipFreeAsync(p, st) != hipSuccess) (void)hipGetLastError();
}

}  // namespace smi
