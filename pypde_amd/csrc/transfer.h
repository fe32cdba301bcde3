// Copies between pageable host arrays and the device, and idle streams kept
// for the next context.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

namespace pypde {

// Both return when `host` may be read or reused and the copy has completed.  It
// may also be pinned, managed or device memory, which is copied without staging;
// work queued on `stream` before the call is complete too.
hipError_t copy_to_device(void* dev, const void* host, size_t n, int device, hipStream_t stream);
hipError_t copy_to_host(void* host, const void* dev, size_t n, int device, hipStream_t stream);

// A default-priority stream of the current device, and its return (idle).
hipError_t take_stream(int device, hipStream_t* s);
void give_stream(int device, hipStream_t s);

// Frees the staging buffers and streams that nothing is using.
void release_idle_transfer();

}  // namespace pypde
