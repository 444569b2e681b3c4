// mkde_copy.h -- large copies between the caller's pageable memory and the
// device (mkde_copy.cpp).
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>

namespace mkde_copy {

// Copies below this many bytes go through one hipMemcpyAsync.  From the device 1 /
// 1.5 / 2 / 4 / 16 MB take 73 / 92 / 120 / 244 / 950 us that way into warm pages and
// 237 / 340 / 475 / 980 / 3900 us into fresh ones, 68 / 82 / 104 / 185 / 545 and 240 /
// 325 / 450 / 690 / 1230 us with lanes.  To the device the runtime pins the caller's
// pages in place and keeps them so for a while.  Masks of 8 / 12 / 16 / 20 / 24 / 32 MB
// (the whole upload), new ones in new contexts: 385 / 506 / 615 / 742 / 850 / 1240 us
// that way, 400 / 525 / 630 / 710 / 785 / 1050 us with lanes; new ones in a kept context
// 335 / 452 / 562 / 689 / 801 / 1132 and 355 / 490 / 540 / 630 / 725 / 890 us; three in
// turn 337 / 515 / 690 / 850 / 1003 / 1325 and 330 / 460 / 520 / 610 / 700 / 840 us.  Lanes
// win in all three from 20 MB on.
constexpr size_t MIN_TO_HOST = (size_t)3 << 19;
constexpr size_t MIN_TO_DEVICE = (size_t)20 << 20;
// Contexts that share the device with others (the job server's), either way: a burst
// of 12 jobs on rasters of 4 / 8.6 / 16 / 32 / 64 MB takes 5.4 / 7.6 / 11.5 / 23.9 / 43.4 ms
// without lanes and 5.8 / 7.6 / 12.0 / 21.7 / 42.0 ms with them.
constexpr size_t MIN_SHARED = (size_t)32 << 20;
inline size_t least(bool shared, bool to_host) { return shared ? MIN_SHARED : to_host ? MIN_TO_HOST : MIN_TO_DEVICE; }
// Lanes are made once such copies on the device have come to this many bytes.
// Eight cost 2.5 ms (their streams 1.1, the pinned memory 0.6, its first touches
// 0.8), what copies of 4 to 16 MB save in 30 to 100 MB and a larger one by itself;
// 9 ms more where their streams are the first to open the device's other three
// hardware queues.
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
