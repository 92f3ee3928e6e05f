// op3_chunks.hpp -- the drop-in adjoint's histories between host and device.
//
// The host link bounds it: every level goes up and comes down once. The
// histories pass in chunks of levels, from the top; each chunk's pieces go up
// from several threads, whichever completes a chunk launches its steps, and
// finished levels come down from other threads while later ones go up (the
// link carries both directions at once). 390 x 690 x 100 levels (1.08 GB both
// ways): 51 ms one after the other from one thread, 19 to 22 ms like this; 21 to 25
// in place, where the levels come down after the last step (see split()).
#pragma once

#include <algorithm>
#include <condition_variable>
#include <functional>
#include <mutex>
#include <vector>

#include "hostcopy.hpp"

namespace erm {

struct Op3Run {
  int nt, nup;
  size_t n2;
  const float* const* in;
  float* const* out;
  float* dev;                         // field f of level L at dev + (f*nt + L)*n2
  int chunk;                          // levels per chunk; chunk 0 ends at level nt
  int nchunk;
  std::function<int(int)> step;       // launches the step of a level
  hipStream_t st;
  std::vector<hipEvent_t> ev;         // 2c: before, 2c+1: after the steps of chunk c
  std::mutex mu;
  std::condition_variable cv;
  std::vector<size_t> left;           // bytes of chunk c still to go up
  size_t up_task = 0, down_task = 0;  // next tasks, chunk by chunk
  int launched = 0;                   // chunks whose steps are queued
  bool failed = false;
  bool hold = false;                  // results wait for the last step

  // chunks of about 16 MB, at most 256 of them; the first holds a stepped level
  void split() {
    const size_t level = 5 * n2 * sizeof(float);
    chunk = (int)std::max<size_t>({(kCopyPiece * 4 + level - 1) / level, ((size_t)nt + 255) / 256, 3});
    nchunk = (nt + chunk - 1) / chunk;
    left.resize(nchunk);
    for (int c = 0; c < nchunk; ++c) left[c] = 5 * field_bytes(c, 0, false);
    // A result that goes into an input: nothing is written until every step has
    // run, so that a call that fails on the way leaves the caller's histories as
    // they were.
    const std::less<const float*> before;
    for (int f = 0; f < 5; ++f)
      for (int g = 0; g < 5; ++g)
        hold |= before(out[f], in[g] + (size_t)nt * n2) && before(in[g], out[f] + (size_t)nt * n2);
    nup = hold ? kLanes : kLanes / 2;
  }
  int hi(int c) const { return nt - c * chunk; }
  int lo(int c) const { return std::max(0, hi(c) - chunk); }
  size_t field_bytes(int c, int f, bool down) const {
    // in place the field's top two levels are as they were
    const int h = down && in[f] == out[f] ? std::min(hi(c), nt - 2) : hi(c);
    return h > lo(c) ? (size_t)(h - lo(c)) * n2 * sizeof(float) : 0;
  }
  size_t pieces() const { return ((size_t)chunk * n2 * sizeof(float) + kCopyPiece - 1) / kCopyPiece; }
  size_t tasks() const { return (size_t)nchunk * 5 * pieces(); }
  // task -> chunk, field and bytes [o, o+m) of the chunk's run of that field
  bool piece(size_t task, bool down, int* c, int* f, size_t* o, size_t* m) const {
    const size_t np = pieces();
    *c = (int)(task / (5 * np));
    *f = (int)(task / np % 5);
    *o = task % np * kCopyPiece;
    const size_t n = field_bytes(*c, *f, down);
    *m = *o < n ? std::min(kCopyPiece, n - *o) : 0;
    return *m > 0;
  }
  char* at(float* base, int c, size_t o) const { return reinterpret_cast<char*>(base + (size_t)lo(c) * n2) + o; }

  // with mu held: queues the steps of every chunk that is complete
  int advance() {
    while (launched < nchunk && left[launched] == 0) {
      const int c = launched;
      HIPCHK(hipEventRecord(ev[2 * c], st));
      for (int L = std::min(hi(c), nt - 2) - 1; L >= lo(c); --L) STCHK(step(L));
      HIPCHK(hipEventRecord(ev[2 * c + 1], st));
      ++launched;
      cv.notify_all();
    }
    return OK;
  }
  int up(hipStream_t lane) {
    for (;;) {
      int c, f;
      size_t o, m;
      {
        std::lock_guard<std::mutex> lk(mu);
        if (failed || up_task == tasks()) return OK;
        if (!piece(up_task++, false, &c, &f, &o, &m)) continue;
      }
      HIPCHK(hipMemcpyAsync(at(dev + (size_t)f * nt * n2, c, o), at(const_cast<float*>(in[f]), c, o), m,
                            hipMemcpyHostToDevice, lane));
      HIPCHK(hipStreamSynchronize(lane));
      std::lock_guard<std::mutex> lk(mu);
      left[c] -= m;
      STCHK(advance());
    }
  }
  int down(hipStream_t lane) {
    for (;;) {
      int c, f;
      size_t o, m;
      {
        std::unique_lock<std::mutex> lk(mu);
        if (failed || down_task == tasks()) return OK;
        if (!piece(down_task++, true, &c, &f, &o, &m)) continue;
        const int last = hold ? nchunk - 1 : c;
        cv.wait(lk, [&] { return failed || launched > last; });
        if (failed) return OK;
      }
      if (hold)
        HIPCHK(hipEventSynchronize(ev[2 * nchunk - 1]));
      else
        HIPCHK(hipStreamWaitEvent(lane, ev[2 * c + 1], 0));
      HIPCHK(hipMemcpyAsync(at(out[f], c, o), at(dev + (size_t)f * nt * n2, c, o), m, hipMemcpyDeviceToHost, lane));
      HIPCHK(hipStreamSynchronize(lane));
    }
  }
  // thread k: the first nup upload until all is up, then download too
  int work(int k, hipStream_t lane) {
    int rc = k < nup ? up(lane) : OK;
    if (rc == OK) rc = down(lane);
    if (rc != OK) {
      std::lock_guard<std::mutex> lk(mu);
      failed = true;
      cv.notify_all();
    }
    return rc;
  }
};

}  // namespace erm
