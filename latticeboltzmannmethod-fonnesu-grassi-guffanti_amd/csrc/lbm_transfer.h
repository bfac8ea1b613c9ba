// Large copies between device memory and a caller's ordinary (pageable)
// host memory.  Internal.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace lbm {

// Copies `bytes` on stream s: what hipMemcpyAsync does, and done by it for
// small copies and for page-locked host memory.  To the host the copy is
// waited for; to the device it may be in flight, and the caller waits for the
// stream before the memory may change.  `device` is the stream's; soon: what
// is queued before the copy is known to be short.
hipError_t copy_to_host(int device, void *dst, const void *src, size_t bytes, hipStream_t s, bool soon = false);
hipError_t copy_to_device(int device, void *dst, const void *src, size_t bytes, hipStream_t s);

// The device's view of `bytes` of page-locked host memory (nullptr unless the
// first and the last byte lie in one).
void *device_view(const void *host, size_t bytes);

// Contexts alive: the page-locked chunks the copies go through are shared by
// all of them and freed with the last one.
void transfer_retain();
void transfer_release();

}  // namespace lbm
