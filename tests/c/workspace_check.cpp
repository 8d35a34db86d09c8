// Workspace over a HIP runtime of stubs: every way to fail leaves p null and no
// error behind, and a device without pools is asked once.
#include <cstdio>

#include "workspace.h"

namespace {
hipError_t last = hipSuccess;
hipError_t create_rc, attribute_rc, capturing_rc, device_rc, malloc_rc, free_rc;
hipStreamCaptureStatus status;
int device, created, mallocs, frees;
char block;

hipError_t result(hipError_t e)
{
    if (e != hipSuccess) last = e;  // kept across successful calls
    return e;
}
void reset()
{
    last = create_rc = attribute_rc = capturing_rc = device_rc = malloc_rc = free_rc = hipSuccess;
    status = hipStreamCaptureStatusNone;
    created = mallocs = frees = 0;
    ++device;  // one without a pool yet
}
int failures = 0;
void check(bool ok, const char *what)
{
    if (!ok) {
        std::printf("FAILED: %s\n", what);
        ++failures;
    }
}
bool null_and_clean()
{
    smi::Workspace w(64, nullptr);
    return w.p == nullptr && last == hipSuccess;
}
}  // namespace

extern "C" {
hipError_t hipGetLastError()
{
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
hipError_t hipMemPoolCreate(hipMemPool_t *pool, const hipMemPoolProps *)
{
    ++created;
    if (create_rc == hipSuccess) *pool = (hipMemPool_t)&block;
    return result(create_rc);
}
hipError_t hipMemPoolSetAttribute(hipMemPool_t, hipMemPoolAttr, void *) { return result(attribute_rc); }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *s)
{
    *s = status;
    return result(capturing_rc);
}
hipError_t hipGetDevice(int *d)
{
    *d = device;
    return result(device_rc);
}
hipError_t hipMallocFromPoolAsync(void **p, size_t, hipMemPool_t, hipStream_t)
{
    ++mallocs;
    if (malloc_rc == hipSuccess) *p = &block;
    return result(malloc_rc);
}
hipError_t hipFreeAsync(void *, hipStream_t)
{
    ++frees;
    return result(free_rc);
}
}

int main()
{
    reset();
    create_rc = hipErrorNotSupported;
    check(null_and_clean(), "no pool");
    create_rc = hipSuccess;
    check(null_and_clean() && created == 1, "a device without a pool is asked once");
    reset();
    capturing_rc = hipErrorStreamCaptureImplicit;
    check(null_and_clean() && created == 0, "capture of another stream");
    reset();
    status = hipStreamCaptureStatusActive;
    check(null_and_clean() && created == 0 && mallocs == 0, "captured stream");
    reset();
    device_rc = hipErrorInvalidDevice;
    check(null_and_clean() && created == 0, "no device");
    reset();
    malloc_rc = hipErrorOutOfMemory;
    check(null_and_clean() && created == 1, "no memory");
    malloc_rc = hipSuccess;
    {
        smi::Workspace w(64, nullptr);
        check(w.p == &block && created == 1 && last == hipSuccess, "memory");
    }
    check(frees == 1, "given back once");
    reset();
    free_rc = hipErrorInvalidValue;
    {
        smi::Workspace w(64, nullptr);
    }
    check(frees == 1 && last == hipSuccess, "a failed free leaves nothing behind");
    reset();
    attribute_rc = hipErrorInvalidValue;
    {
        smi::Workspace w(64, nullptr);
        check(w.p == &block, "a pool without its threshold");
        check(last == hipSuccess, "... leaves no error");
    }
    std::printf(failures ? "%d checks failed\n" : "ok\n", failures);
    return failures != 0;
}
