// mkde_copy.h -- large copies between the caller's pageable memory and the
// device (mkde_copy.cpp).
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>

namespace mkde_copy {

// Copies below this many bytes go through one hipMemcpyAsync: of a context on
// its own, of one that shares the device with others (the job server's).
constexpr size_t MIN_BYTES = (size_t)1 << 20;
constexpr size_t SHARED_MIN_BYTES = (size_t)16 << 20;

// One per context: the lanes are freed when the last user is gone.
void retain();
void release();

// Copies bytes between host (pageable) and device memory of `device` with
// several lanes and returns when all has arrived; the caller has made the
// device current and has waited for every queued use of the device memory.
// shared non-null: the transfers go through that stream.  *done = false (and
// hipSuccess) when no lane is free or can be made: nothing was copied then.
hipError_t run(int device, hipStream_t shared, void *dst, const void *src, size_t bytes, bool to_host, bool *done);

}  // namespace mkde_copy
