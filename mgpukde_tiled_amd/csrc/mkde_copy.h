// mkde_copy.h -- large copies between the caller's pageable memory and the
// device (mkde_copy.cpp).
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>

namespace mkde_copy {

// Copies below this many bytes go through one hipMemcpyAsync.  To the device the
// runtime reads the caller's pages in place and needs no staging: lanes win only
// where several threads' worth of copying is to be had (repeated copies of
// 8 / 16 / 64 MB: 326 / 617 / 2400 us without, 260 / 455 / 1440 us with lanes, but a
// single 16 MB mask on a new context 790 against 960 us; a 21 MB tile mask a call,
// warm, 300 us less with lanes).  From the device: 2 / 4 / 16 / 64 MB 131 / 252 /
// 1030 / 6750 us without, 127 / 190 / 446 / 1890 us with lanes.
constexpr size_t MIN_TO_DEVICE = (size_t)20 << 20;
constexpr size_t MIN_TO_HOST = (size_t)1 << 20;
// Contexts that share the device with others (the job server's), either way.
constexpr size_t MIN_SHARED = (size_t)32 << 20;
inline size_t least(bool shared, bool to_host) { return shared ? MIN_SHARED : to_host ? MIN_TO_HOST : MIN_TO_DEVICE; }
// Lanes are made once such copies on the device have come to this many bytes.
// Eight cost 2.5 ms (their streams 1.1, the pinned memory 0.6, its first touches
// 0.8), what copies of 4 to 16 MB save in 30 to 100 MB and a larger one by itself.
constexpr size_t MIN_MOVED = (size_t)32 << 20;

// Copies bytes between host (pageable) and device memory of `device` with
// several lanes and returns when all has arrived; the caller has made the
// device current and has waited for every queued use of the device memory.
// shared non-null: the transfers go through that stream.  *done = false (and
// hipSuccess) when the copy is not one for lanes, or none is free or can be made:
// nothing was copied then.
hipError_t run(int device, hipStream_t shared, void *dst, const void *src, size_t bytes, bool to_host, bool *done);

// Frees the device's lanes that no copy is using; later copies make them anew.
void give_back(int device);

}  // namespace mkde_copy
