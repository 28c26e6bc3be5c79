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
// they have arrived.  Any thread, any stream.  Its pinned staging, 16 MiB, is
// made at the first call and kept for the process.
hipError_t download(const HostPiece *pieces, size_t count, hipStream_t stream);

}  // namespace lbm_dev
