// Results from the device to pageable host memory.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace lbm_dev
{

struct HostPiece
{
    void *dst;        // host
    const void *src;  // device
    size_t bytes;
};

// Copies the pieces once the work enqueued on `stream` is done; returns when
// they have arrived.  Any thread, any stream.
hipError_t download(const HostPiece *pieces, size_t count, hipStream_t stream);

// The objects that may call download() (contexts, batches, networks) hold its
// staging memory between them: it is given back with the last of them.
void hold_staging();
void release_staging();

}  // namespace lbm_dev
