// hostcopy.hip -- see hostcopy.hpp.
#include "hostcopy.hpp"

#include <algorithm>
#include <atomic>
#include <mutex>
#include <string>
#include <thread>

namespace erm {

namespace {

// Streams of the copy threads: one set per process, on the device of its last
// use, used by one call at a time (concurrent calls share one link anyway).
std::mutex g_lanes_mu;
std::vector<hipStream_t> g_lanes;
int g_lanes_dev = -1;

void drop_lanes() {
  for (hipStream_t s : g_lanes) (void)hipStreamDestroy(s);
  g_lanes.clear();
  g_lanes_dev = -1;
}

int get_lanes(int n, int dev) {
  if (g_lanes_dev != dev) drop_lanes();
  g_lanes_dev = dev;
  while ((int)g_lanes.size() < n) {
    hipStream_t s;
    HIPCHK(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
    g_lanes.push_back(s);
  }
  return OK;
}

int copy(void* dst, const void* src, size_t n, hipMemcpyKind kind) {
  if (n == 0) return OK;
  if (n < (kind == hipMemcpyHostToDevice ? kLargeToDevice : kLargeToHost)) {
    HIPCHK(hipMemcpy(dst, src, n, kind));
    return OK;
  }
  const size_t pieces = (n + kCopyPiece - 1) / kCopyPiece;
  std::atomic<size_t> next{0};
  return with_copy_lanes((int)std::min<size_t>(pieces, kCopyThreads), [&](int, hipStream_t st) -> int {
    for (size_t k = next++; k < pieces; k = next++) {
      const size_t o = k * kCopyPiece, m = std::min(kCopyPiece, n - o);
      HIPCHK(hipMemcpyAsync(static_cast<char*>(dst) + o, static_cast<const char*>(src) + o, m, kind, st));
      HIPCHK(hipStreamSynchronize(st));
    }
    return OK;
  });
}

}  // namespace

int with_copy_lanes(int n, const std::function<int(int, hipStream_t)>& work) {
  n = std::min(std::max(n, 1), kLanes);
  int dev = 0;
  HIPCHK(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lock(g_lanes_mu);
  STCHK(get_lanes(n, dev));
  std::vector<int> rc(n, OK);
  std::vector<std::string> msg(n);
  auto run = [&](int k) {
    rc[k] = hipSetDevice(dev) == hipSuccess ? work(k, g_lanes[k]) : E_HIP;
    if (rc[k] != OK) msg[k] = last_error();  // the message is the thread's own
  };
  std::vector<std::thread> th;
  th.reserve(n);
  int started = 0;
  try {
    for (; started < n; ++started) th.emplace_back(run, started);
  } catch (const std::exception&) {  // no more threads: the rest runs below
  }
  for (int k = started; k < n; ++k) run(k);
  for (std::thread& t : th) t.join();
  for (int k = 0; k < n; ++k)
    if (rc[k] != OK) {
      set_error("%s", msg[k].c_str());
      return rc[k];
    }
  return OK;
}

void release_copy_lanes() {
  std::lock_guard<std::mutex> lock(g_lanes_mu);
  drop_lanes();
}

int copy_to_device(void* dst, const void* src, size_t n) { return copy(dst, src, n, hipMemcpyHostToDevice); }
int copy_to_host(void* dst, const void* src, size_t n) { return copy(dst, src, n, hipMemcpyDeviceToHost); }

}  // namespace erm
