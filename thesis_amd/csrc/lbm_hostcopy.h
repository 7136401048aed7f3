// Device-to-host copies of whole fields into the caller's (pageable) memory.
#pragma once
#include <hip/hip_runtime.h>
#include <cstddef>

namespace lbm {

struct OutCopy {
    void* dst;
    const void* src;
    size_t bytes;
};

// Enqueues the copies after the work on st and waits for all of them.
hipError_t copy_to_host(const OutCopy* c, int n, int dev, hipStream_t st);

// Every context holds the staging buffers while it lives; they are freed with
// the last one.
void host_staging_retain();
void host_staging_release();

}  // namespace lbm
