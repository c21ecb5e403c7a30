// transfer.hpp -- copies between host memory and the device: through pinned
// staging buffers that are kept from call to call where that is faster than
// hipMemcpy, and refused where hipMemcpy refuses them.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace st {

struct UploadPart {
    void *dst;         // device
    const void *src;   // host
    size_t bytes;
};

// Copies the parts to the current device; on return they are there.  The order
// to other work is hipMemcpy's: that of the null stream.
hipError_t upload(const UploadPart *parts, int n);

// Copies device memory to the host; on return it is there (same ordering).
hipError_t download(void *dst, const void *src, size_t bytes);

// Gives the kept staging buffers back.
void staging_shutdown();

}  // namespace st
