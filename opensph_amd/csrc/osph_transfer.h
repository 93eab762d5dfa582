// Device results to the host (osph_transfer.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace osph {

// Copies device memory written by earlier work on `stream` into pageable host memory, and returns when it is there.
// Safe from several threads and for several streams and devices (the calling thread's current one).
hipError_t copy_to_host(hipStream_t stream, void* host, const void* dev, size_t bytes);
// Every context that copies is attached while it lives; the pinned buffers go with the last one.
void transfer_attach();
void transfer_detach();

}  // namespace osph
