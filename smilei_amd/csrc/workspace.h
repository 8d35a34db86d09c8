// workspace.h -- scratch memory of one call, ordered on its stream.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace smi {

// Bytes that a device's pool holds between calls.
constexpr size_t kWorkspaceKeep = size_t(256) << 20;

// Device memory taken from the library's pool of the current device in the
// order of a stream and given back in that order when the object goes out of
// scope, so a call can be repeated from any number of threads and streams
// without waiting.  The pool keeps at most kWorkspaceKeep between calls; what is
// above goes back to the device at the next synchronisation.  p stays null
// where the stream is being captured (a graph would keep the address) and
// where the device has no pool or no memory left.
struct Workspace {
    void *p = nullptr;
    hipStream_t st;
    Workspace(size_t bytes, hipStream_t stream);
    ~Workspace();
    Workspace(const Workspace &) = delete;
    Workspace &operator=(const Workspace &) = delete;
};

}  // namespace smi
