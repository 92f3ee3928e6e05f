// hostcopy.hpp -- large copies between pageable host arrays and the device.
//
// One hipMemcpy of a pageable array is bound by the calling thread (pinning,
// page faults of a fresh destination, staging): 29 GB/s to the device, 17 from
// it, 10 into pages not yet touched, on a link that carries 57 each way. A few
// threads that each copy pieces of 4 MB on a stream of their own reach 50 and
// more (512 MB to the device 18 -> 10 ms, to a fresh array 50 -> 12 ms).
#pragma once

#include <functional>
#include <vector>

#include "common.hpp"

namespace erm {

// Pieces and threads of a large copy. Smaller arrays go in one hipMemcpy: to
// the device 36 MB took 1.2 ms that way against 1.5 from six threads, to the
// host 3.5 against 1.6 (the first use of the streams in a process costs about
// 14 ms more, hardware queues and staging buffers being set up).
constexpr size_t kCopyPiece = size_t(4) << 20;
constexpr size_t kLargeToDevice = size_t(96) << 20;
constexpr size_t kLargeToHost = size_t(16) << 20;
constexpr int kCopyThreads = 6;

// n bytes between host and device memory, done on return. The device side
// must be idle (its producers finished).
int copy_to_device(void* dst, const void* src, size_t n);
int copy_to_host(void* dst, const void* src, size_t n);

// Runs work(k, stream) for k = 0..n-1 on n threads (at most kLanes), each with a
// stream of its own. Calls may run at the same time, on one device or several;
// idle streams, at most kLanes a device, are kept for the next calls until
// release_copy_lanes(). Where a thread cannot be started its work
// runs on the calling thread after the others. Returns the first error.
constexpr int kLanes = 8;
int with_copy_lanes(int n, const std::function<int(int, hipStream_t)>& work);
void release_copy_lanes();

}  // namespace erm
