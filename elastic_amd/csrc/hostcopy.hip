// hostcopy.hip -- see hostcopy.hpp.
#include "hostcopy.hpp"

#include <algorithm>
#include <atomic>
#include <map>
#include <mutex>
#include <string>
#include <thread>

namespace erm {

namespace {

// Idle streams of the copy threads, by device. A call takes those it finds,
// creates the rest and gives them back, so calls at the same time (also on other
// devices) have streams of their own and wait for nothing but the link.
std::mutex g_idle_mu;
std::map<int, std::vector<hipStream_t>> g_idle;

// The streams of one call.
struct Lanes {
  int dev;
  std::vector<hipStream_t> st;
  bool sound = true;  // false: a lane failed, its stream may hold work

  explicit Lanes(int device) : dev(device) {}
  int get(int n) {
    st.reserve(n);
    {
      std::lock_guard<std::mutex> lock(g_idle_mu);
      std::vector<hipStream_t>& idle = g_idle[dev];
      for (; (int)st.size() < n && !idle.empty(); idle.pop_back()) st.push_back(idle.back());
      idle.reserve(kLanes);  // giving back does not allocate
    }
    while ((int)st.size() < n) {
      hipStream_t s;
      HIPCHK(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
      st.push_back(s);
    }
    return OK;
  }
  ~Lanes() {
    if (!sound)
      for (hipStream_t s : st) (void)hipStreamSynchronize(s);
    if (sound) {
      std::lock_guard<std::mutex> lock(g_idle_mu);
      std::vector<hipStream_t>& idle = g_idle[dev];
      for (; !st.empty() && (int)idle.size() < kLanes; st.pop_back()) idle.push_back(st.back());
    }
    for (hipStream_t s : st) (void)hipStreamDestroy(s);
  }
};

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
  Lanes lanes(dev);
  STCHK(lanes.get(n));
  std::vector<int> rc(n, OK);
  std::vector<std::string> msg(n);
  auto run = [&](int k) {
    rc[k] = hipSetDevice(dev) == hipSuccess ? work(k, lanes.st[k]) : E_HIP;
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
      lanes.sound = false;
      set_error("%s", msg[k].c_str());
      return rc[k];
    }
  return OK;
}

void release_copy_lanes() {
  std::map<int, std::vector<hipStream_t>> idle;
  {
    std::lock_guard<std::mutex> lock(g_idle_mu);
    idle.swap(g_idle);
  }
  for (auto& d : idle)
    for (hipStream_t s : d.second) (void)hipStreamDestroy(s);
}

int copy_to_device(void* dst, const void* src, size_t n) { return copy(dst, src, n, hipMemcpyHostToDevice); }
int copy_to_host(void* dst, const void* src, size_t n) { return copy(dst, src, n, hipMemcpyDeviceToHost); }

}  // namespace erm
