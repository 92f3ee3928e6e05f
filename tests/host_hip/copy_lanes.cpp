// copy_lanes.cpp -- hostcopy.hip on the CPU: calls at the same time, calls on
// several devices, what is kept and given back, failing lanes, and the pieces
// of large copies.
#include "check.hpp"

#include "../../elastic_amd/csrc/hostcopy.hip"

#include <chrono>
#include <condition_variable>

using namespace erm;

// Two calls (on devices d0 and d1) whose lanes all wait until every lane of both
// runs: they meet only if neither call waits for the other to end.
static void at_the_same_time(int d0, int d1) {
  std::mutex mu;
  std::condition_variable cv;
  int in = 0, met = 0;
  auto call = [&](int dev) {
    (void)hipSetDevice(dev);
    const int rc = with_copy_lanes(4, [&](int, hipStream_t s) -> int {
      CHECK(s->dev == dev);
      std::unique_lock<std::mutex> lk(mu);
      ++in;
      cv.notify_all();
      met += cv.wait_for(lk, std::chrono::seconds(5), [&] { return in == 8; });
      return OK;
    });
    CHECK(rc == OK);
  };
  std::thread a(call, d0), b(call, d1);
  a.join();
  b.join();
  CHECK(met == 8);
}

static void devices_in_turn() {
  release_copy_lanes();
  const int before = host_hip::created;
  for (int i = 0; i < 10; ++i) {
    (void)hipSetDevice(i & 1);
    CHECK(with_copy_lanes(6, [&](int, hipStream_t s) -> int { return s->dev == (i & 1) ? OK : E_HIP; }) == OK);
  }
  (void)hipSetDevice(0);
  CHECK(host_hip::created - before == 12);  // six a device, kept
}

static void bounded_and_given_back() {
  std::vector<std::thread> th;
  for (int i = 0; i < 6; ++i)
    th.emplace_back([] { CHECK(with_copy_lanes(kLanes, [](int, hipStream_t) -> int { return OK; }) == OK); });
  for (std::thread& t : th) t.join();
  CHECK(host_hip::streams <= 2 * kLanes);  // device 1's of the test before, device 0's
  release_copy_lanes();
  CHECK(host_hip::streams == 0);
}

static void failing_lane() {
  for (int bad = 0; bad < 3; ++bad) {
    const int rc = with_copy_lanes(3, [&](int k, hipStream_t) -> int {
      if (k != bad) return OK;
      set_error("lane %d", k);
      return E_NOMEM;
    });
    CHECK(rc == E_NOMEM && std::string(last_error()) == "lane " + std::to_string(bad));
    CHECK(host_hip::streams == 0);  // those of a failed call are not kept
  }
}

static void large_copies() {
  for (size_t n : {size_t(0), size_t(5), kLargeToDevice - 1, kLargeToDevice, kLargeToDevice + 3, 25 * kCopyPiece + 4097,
                   26 * kCopyPiece - 1}) {
    std::vector<unsigned char> a(n + 1), b(n + 1, 7), c(n + 1, 9);
    for (size_t i = 0; i < n; ++i) a[i] = (unsigned char)(i * 2654435761u >> 13);
    CHECK(copy_to_device(b.data(), a.data(), n) == OK && std::equal(a.begin(), a.end() - 1, b.begin()) && b[n] == 7);
    CHECK(copy_to_host(c.data(), b.data(), n) == OK && std::equal(a.begin(), a.end() - 1, c.begin()) && c[n] == 9);
  }
  std::vector<unsigned char> a(kLargeToDevice), b(kLargeToDevice);
  host_hip::copies = 0;
  host_hip::fail_copy = 11;
  CHECK(copy_to_device(b.data(), a.data(), a.size()) == E_HIP);
  host_hip::fail_copy = -1;
}

int main() {
  at_the_same_time(0, 0);
  at_the_same_time(0, 1);
  devices_in_turn();
  bounded_and_given_back();
  failing_lane();
  large_copies();
  std::printf("OK\n");
  return 0;
}
