// op3_chunks.cpp -- the chunked passage of the drop-in's histories on the CPU,
// with a recursion of whole numbers in place of the stencils (every field of a
// level reads all fields of the next and its own of the one after), against the
// same recursion over the whole history.
#include "check.hpp"

#include "../../elastic_amd/csrc/hostcopy.hip"
#include "../../elastic_amd/csrc/op3_chunks.hpp"

using namespace erm;

using History = std::vector<std::vector<float>>;  // five fields of nt levels

static void recursion(float* const* f, size_t n2, int L) {
  for (int k = 0; k < 5; ++k)
    for (size_t i = 0; i < n2; ++i) {
      float s = f[k][L * n2 + i] + f[k][(L + 2) * n2 + i];
      for (int j = 0; j < 5; ++j) s += (float)(1 + (j + k) % 3) * f[j][(L + 1) * n2 + i];
      f[k][L * n2 + i] = s - 1024.f * (float)(int)(s / 1024.f);  // exact: stays small
    }
}

static History start(int nt, size_t n2) {
  History h(5);
  for (int k = 0; k < 5; ++k)
    for (size_t i = 0; i < nt * n2; ++i) h[k].push_back((float)((i * 7 + k * 13) % 101));
  return h;
}

// alias: bit f set: field f's result goes into its input. Returns the status.
static int run(int nt, size_t n2, unsigned alias, bool threads, int fail_level, History& in, History& out) {
  in = start(nt, n2);
  out.assign(5, std::vector<float>(nt * n2, -5.f));
  std::vector<float> dev(5 * nt * n2);
  const float* ip[5];
  float* op[5];
  float* dp[5];
  for (int f = 0; f < 5; ++f) {
    ip[f] = in[f].data();
    op[f] = alias >> f & 1 ? in[f].data() : out[f].data();
    dp[f] = dev.data() + f * nt * n2;
  }
  Op3Run r;
  r.nt = nt; r.n2 = n2; r.in = ip; r.out = op; r.dev = dev.data(); r.st = nullptr;
  r.split();
  r.step = [&](int L) -> int {
    if (L == fail_level) {
      set_error("level %d", L);
      return E_HIP;
    }
    recursion(dp, n2, L);
    return OK;
  };
  for (int i = 0; i < 2 * r.nchunk; ++i) r.ev.push_back(new int(0));
  int rc;
  if (threads) {
    rc = with_copy_lanes(kLanes, [&](int k, hipStream_t lane) { return r.work(k, lane); });
  } else {
    hipStream_t lane;
    (void)hipStreamCreateWithFlags(&lane, 0);
    r.nup = 1;
    rc = r.work(0, lane);
    (void)hipStreamDestroy(lane);
  }
  for (hipEvent_t e : r.ev) (void)hipEventDestroy(e);
  for (int f = 0; f < 5; ++f)
    if (alias >> f & 1) out[f] = in[f];
  return rc;
}

int main() {
  const struct { int nt; size_t n2; } sizes[] = {{3, 40}, {4, 144}, {37, 900}, {700, 60}, {61, 30000}, {5, 1200000}};
  for (auto [nt, n2] : sizes) {
    History want = start(nt, n2);
    float* wp[5];
    for (int f = 0; f < 5; ++f) wp[f] = want[f].data();
    for (int L = nt - 3; L >= 0; --L) recursion(wp, n2, L);
    for (bool threads : {false, true})
      for (unsigned alias : {0u, 31u, 1u, 16u, 22u}) {
        History in, out;
        CHECK(run(nt, n2, alias, threads, -1, in, out) == OK);
        const History given = start(nt, n2);
        for (int f = 0; f < 5; ++f) {
          if (out[f] != want[f]) std::printf("field %d of %d levels of %zu cells, alias %u\n", f, nt, n2, alias);
          CHECK(out[f] == want[f]);
          if (!(alias >> f & 1)) CHECK(in[f] == given[f]);
        }
      }
  }
  // a step or a copy up that fails leaves histories that are worked on in place as
  // they were: the first step, one on the way, the last; copies of every chunk
  for (bool threads : {false, true})
    for (unsigned alias : {31u, 1u}) {
      const int nt = 61;
      const size_t n2 = 30000;
      const History given = start(nt, n2);
      History in, out;
      for (int level : {nt - 3, nt / 2, 0}) {
        CHECK(run(nt, n2, alias, threads, level, in, out) == E_HIP);
        CHECK(std::string(last_error()) == "level " + std::to_string(level));
        CHECK(in == given);
      }
      for (int copy : {0, 7, 10, 14}) {  // 15 go up: five fields of three chunks
        host_hip::copies = 0;
        host_hip::fail_copy = copy;
        CHECK(run(nt, n2, alias, threads, -1, in, out) == E_HIP);
        host_hip::fail_copy = -1;
        CHECK(in == given);
      }
    }
  std::printf("OK\n");
  return 0;
}
