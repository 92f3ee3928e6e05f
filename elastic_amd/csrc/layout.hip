// layout.hip -- device rearrangement between the callers' array layouts and
// the engine's (see layout.hpp).
//
// The copies over the host link bound these paths: about 27 GB/s to the
// device and 17 GB/s from it for pageable arrays, in contiguous pieces of a
// megabyte and more. A pitched copy of nx columns is nx small transfers of
// about 5 us each (the three images of twelve 290 x 490 grids took 110 ms,
// their bytes 3 ms), and the host's transposing loop of a record ran at 0.5
// GB/s (the 24 MB record of 600 traces x 2000 samples: 52 ms). The kernels
// here run at HBM rates, so they only have to be launched over enough
// workgroups; the scratch is allocated per call (under 50 us for 32 MiB).
#include "layout.hpp"
#include "hostcopy.hpp"

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <vector>

namespace erm {

namespace {

constexpr size_t kScratch = size_t(32) << 20;
constexpr int TT = 64;  // transpose tile: 64 x 64 through LDS, rows padded by one bank

__device__ __forceinline__ void flag_nonfinite(bool bad, int* flag) {
  if (flag && __any(bad) && (threadIdx.x & 63) == 0) atomicOr(flag, 1);
}

// Matrices blockIdx.z: dst[c][r] = src[r][c] for r < rows, c < cols.
__global__ __launch_bounds__(256) void k_transpose(const float* __restrict__ src, float* __restrict__ dst, int rows,
                                                   int cols, long long src_ld, long long dst_ld, long long src_bs,
                                                   long long dst_bs, int* flag) {
  __shared__ float t[TT][TT + 1];
  const float* s = src + blockIdx.z * src_bs;
  float* d = dst + blockIdx.z * dst_bs;
  const int c0 = blockIdx.x * TT, r0 = blockIdx.y * TT;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  bool bad = false;
#pragma unroll
  for (int i = 0; i < TT / 4; ++i) {
    const int r = r0 + w + 4 * i, c = c0 + lane;
    const float v = r < rows && c < cols ? s[r * src_ld + c] : 0.f;
    bad |= !isfinite(v);
    t[w + 4 * i][lane] = v;
  }
  flag_nonfinite(bad, flag);
  __syncthreads();
#pragma unroll
  for (int i = 0; i < TT / 4; ++i) {
    const int c = c0 + w + 4 * i, r = r0 + lane;
    if (r < rows && c < cols) d[c * dst_ld + r] = t[lane][w + 4 * i];
  }
}

// One field's columns ix0 .. ix0+ncol-1: packed (nz rows) -> padded (ldz rows).
__global__ __launch_bounds__(256) void k_pad(const float* __restrict__ src, float* __restrict__ dst, int nz, int ldz,
                                             int ix0, long long n, FieldBox b) {
  for (long long i = blockIdx.x * 256LL + threadIdx.x; i < n; i += gridDim.x * 256LL) {
    const unsigned c = (unsigned)i / (unsigned)ldz;  // a field stays below 2^31 cells
    const int iz = (int)((unsigned)i - c * (unsigned)ldz), ix = ix0 + (int)c;
    const bool in = iz >= b.iz0 && iz <= b.iz1 && ix >= b.ix0 && ix <= b.ix1;
    dst[i] = in ? src[(long long)c * nz + iz] : 0.f;
  }
}

// nf fields, padded -> packed, one after the other.
__global__ __launch_bounds__(256) void k_unpad(const float* __restrict__ src, float* __restrict__ dst, int nz, int ldz,
                                               long long n, long long src_fs, long long dst_fs, int* flag) {
  const float* s = src + blockIdx.y * src_fs;
  float* d = dst + blockIdx.y * dst_fs;
  bool bad = false;
  for (long long i = blockIdx.x * 256LL + threadIdx.x; i < n; i += gridDim.x * 256LL) {
    const unsigned c = (unsigned)i / (unsigned)nz;
    const int iz = (int)((unsigned)i - c * (unsigned)nz);
    const float v = s[(long long)c * ldz + iz];
    bad |= !isfinite(v);
    d[i] = v;
  }
  flag_nonfinite(bad, flag);
}

__global__ __launch_bounds__(256) void k_round(const double* __restrict__ src, float* __restrict__ dst, size_t n) {
  for (size_t i = blockIdx.x * (size_t)256 + threadIdx.x; i < n; i += gridDim.x * (size_t)256) dst[i] = (float)src[i];
}

__global__ void k_clear_flag(int* flag) { *flag = 0; }

unsigned blocks_of(size_t n) { return (unsigned)std::min<size_t>((n + 255) / 256, 16384); }

// Scratch of `want` bytes, at least `least`, at most kScratch (or least), with
// 256 bytes behind it for the flag. False: none is to be had (RTM_SCRATCH=0, for
// tests: as if).
struct Scratch {
  DevBuf b;
  size_t bytes = 0;
  int* flag = nullptr;
  bool get(size_t want, size_t least) {
    bytes = std::max(std::min(want, kScratch), least);
    bytes = (bytes + 255) / 256 * 256;
    void* p = nullptr;
    const char* e = getenv("RTM_SCRATCH");
    if (e && atoi(e) == 0) return false;
    if (hipMalloc(&p, bytes + 256) != hipSuccess) {
      (void)hipGetLastError();
      return false;
    }
    b.p = p;
    b.bytes = bytes + 256;
    flag = reinterpret_cast<int*>(static_cast<char*>(p) + bytes);
    return true;
  }
  float* data() const { return b.as<float>(); }
};

int start_flag(const Scratch& s, bool on, hipStream_t st) {
  if (!on) return OK;
  hipLaunchKernelGGL(k_clear_flag, dim3(1), dim3(1), 0, st, s.flag);
  HIPCHK(hipGetLastError());
  return OK;
}
int read_flag(const Scratch& s, bool* out, hipStream_t st) {
  if (!out) return OK;
  int f = 0;
  HIPCHK(hipMemcpyAsync(&f, s.flag, sizeof f, hipMemcpyDeviceToHost, st));
  HIPCHK(hipStreamSynchronize(st));
  *out = f != 0;
  return OK;
}
bool host_nonfinite(const float* p, size_t n) {
  for (size_t i = 0; i < n; ++i)
    if (!std::isfinite(p[i])) return true;
  return false;
}

// Copy from the scratch to a caller's array behind the stream's kernels; a large
// one from several threads.
int to_host(void* dst, const void* src, size_t n, hipStream_t st) {
  if (n < kLargeToHost) {
    HIPCHK(hipMemcpyAsync(dst, src, n, hipMemcpyDeviceToHost, st));
    return OK;
  }
  HIPCHK(hipStreamSynchronize(st));
  return copy_to_host(dst, src, n);
}

int transpose(const float* src, float* dst, int rows, int cols, long long src_ld, long long dst_ld, int nb,
              long long src_bs, long long dst_bs, int* flag, hipStream_t st) {
  // grid.y counts blocks of rows: 65535 of them hold 4.19 million levels or traces
  const long long step = 65535LL * TT;
  for (long long r = 0; r < rows; r += step) {
    const int n = (int)std::min<long long>(step, rows - r);
    hipLaunchKernelGGL(k_transpose, dim3((cols + TT - 1) / TT, (n + TT - 1) / TT, nb), dim3(256), 0, st,
                       src + r * src_ld, dst + r, n, cols, src_ld, dst_ld, src_bs, dst_bs, flag);
    HIPCHK(hipGetLastError());
  }
  return OK;
}

}  // namespace

int store_fields(const float* const* src, int nf, int nz, int nx, int ldz, float* dst, size_t fs, const FieldBox* box,
                 hipStream_t st) {
  if (nf <= 0) return OK;
  const FieldBox whole{0, nz - 1, 0, nx - 1};
  const size_t col = (size_t)nz * sizeof(float);
  Scratch s;
  if (!s.get(col * nx * nf, col)) {
    std::vector<float> h((size_t)ldz * nx);
    for (int f = 0; f < nf; ++f) {
      const FieldBox b = box ? box[f] : whole;
      std::fill(h.begin(), h.end(), 0.f);
      for (int ix = std::max(b.ix0, 0); ix <= b.ix1; ++ix)
        for (int iz = b.iz0; iz <= b.iz1; ++iz) h[iz + (size_t)ldz * ix] = src[f][iz + (size_t)nz * ix];
      HIPCHK(hipMemcpyAsync(dst + f * fs, h.data(), h.size() * sizeof(float), hipMemcpyHostToDevice, st));
      HIPCHK(hipStreamSynchronize(st));
    }
    return OK;
  }
  // pieces of whole columns; consecutive pieces use consecutive parts of the
  // scratch while they fit, else its start again (stream order protects it)
  const int most = (int)std::min<size_t>(s.bytes / col, nx);
  size_t used = 0;
  for (int f = 0; f < nf; ++f)
    for (int ix = 0; ix < nx; ix += most) {
      const int nc = std::min(most, nx - ix);
      if (used + nc * col > s.bytes) used = 0;
      float* t = s.data() + used / sizeof(float);
      used += nc * col;
      HIPCHK(hipMemcpyAsync(t, src[f] + (size_t)nz * ix, nc * col, hipMemcpyHostToDevice, st));
      const long long n = (long long)ldz * nc;
      hipLaunchKernelGGL(k_pad, dim3(blocks_of(n)), dim3(256), 0, st, t, dst + f * fs + (size_t)ldz * ix, nz, ldz, ix, n,
                         box ? box[f] : whole);
      HIPCHK(hipGetLastError());
    }
  HIPCHK(hipStreamSynchronize(st));
  return OK;
}

int fetch_fields(float* dst, int nf, int nz, int nx, int ldz, const float* src, size_t fs, bool* nonfinite,
                 hipStream_t st) {
  if (nonfinite) *nonfinite = false;
  if (nf <= 0) return OK;
  const size_t col = (size_t)nz * sizeof(float), all = (size_t)nz * nx;
  Scratch s;
  if (!s.get(col * nx * nf, col)) {
    for (int f = 0; f < nf; ++f)
      HIPCHK(hipMemcpy2DAsync(dst + f * all, col, src + f * fs, ldz * sizeof(float), col, nx, hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    if (nonfinite) *nonfinite = host_nonfinite(dst, nf * all);
    return OK;
  }
  STCHK(start_flag(s, nonfinite != nullptr, st));
  int* flag = nonfinite ? s.flag : nullptr;
  if (col * nx * nf <= s.bytes) {  // all fields at once
    hipLaunchKernelGGL(k_unpad, dim3(blocks_of(all), nf), dim3(256), 0, st, src, s.data(), nz, ldz, (long long)all,
                       (long long)fs, (long long)all, flag);
    HIPCHK(hipGetLastError());
    STCHK(to_host(dst, s.data(), nf * all * sizeof(float), st));
  } else {
    const int most = (int)std::min<size_t>(s.bytes / col, nx);
    for (int f = 0; f < nf; ++f)
      for (int ix = 0; ix < nx; ix += most) {
        const int nc = std::min(most, nx - ix);
        const long long n = (long long)nz * nc;
        hipLaunchKernelGGL(k_unpad, dim3(blocks_of(n), 1), dim3(256), 0, st, src + f * fs + (size_t)ldz * ix, s.data(),
                           nz, ldz, n, 0LL, 0LL, flag);
        HIPCHK(hipGetLastError());
        STCHK(to_host(dst + f * all + (size_t)nz * ix, s.data(), nc * col, st));
      }
  }
  STCHK(read_flag(s, nonfinite, st));
  HIPCHK(hipStreamSynchronize(st));
  return OK;
}

int store_records(const float* src, int nc, int nt, int nrx, float* dst, hipStream_t st) {
  const size_t tr = (size_t)nt * sizeof(float), comp = (size_t)nt * nrx;
  if (comp == 0 || nc <= 0) return OK;
  Scratch s;
  if (!s.get(tr * nrx * nc, tr)) {
    std::vector<float> t(comp);
    for (int f = 0; f < nc; ++f) {
      const float* h = src + f * comp;
      for (int ix = 0; ix < nrx; ++ix)
        for (int it = 0; it < nt; ++it) t[(size_t)it * nrx + ix] = h[it + (size_t)nt * ix];
      HIPCHK(hipMemcpyAsync(dst + f * comp, t.data(), comp * sizeof(float), hipMemcpyHostToDevice, st));
      HIPCHK(hipStreamSynchronize(st));
    }
    return OK;
  }
  if (tr * nrx * nc <= s.bytes) {
    HIPCHK(hipMemcpyAsync(s.data(), src, nc * comp * sizeof(float), hipMemcpyHostToDevice, st));
    STCHK(transpose(s.data(), dst, nrx, nt, nt, nrx, nc, comp, comp, nullptr, st));
  } else {
    const int most = (int)std::min<size_t>(s.bytes / tr, nrx);
    for (int f = 0; f < nc; ++f)
      for (int ix = 0; ix < nrx; ix += most) {
        const int n = std::min(most, nrx - ix);
        HIPCHK(hipMemcpyAsync(s.data(), src + f * comp + (size_t)nt * ix, n * tr, hipMemcpyHostToDevice, st));
        STCHK(transpose(s.data(), dst + f * comp + ix, n, nt, nt, nrx, 1, 0, 0, nullptr, st));
      }
  }
  HIPCHK(hipStreamSynchronize(st));
  return OK;
}

int fetch_records(float* dst, int nc, int nt, int nrx, const float* src, bool* nonfinite, hipStream_t st) {
  if (nonfinite) *nonfinite = false;
  const size_t tr = (size_t)nt * sizeof(float), comp = (size_t)nt * nrx;
  if (comp == 0 || nc <= 0) return OK;
  Scratch s;
  if (!s.get(tr * nrx * nc, tr)) {
    std::vector<float> t(comp);
    for (int f = 0; f < nc; ++f) {
      float* h = dst + f * comp;
      HIPCHK(hipMemcpyAsync(t.data(), src + f * comp, comp * sizeof(float), hipMemcpyDeviceToHost, st));
      HIPCHK(hipStreamSynchronize(st));
      for (int ix = 0; ix < nrx; ++ix)
        for (int it = 0; it < nt; ++it) h[it + (size_t)nt * ix] = t[(size_t)it * nrx + ix];
    }
    if (nonfinite) *nonfinite = host_nonfinite(dst, nc * comp);
    return OK;
  }
  STCHK(start_flag(s, nonfinite != nullptr, st));
  int* flag = nonfinite ? s.flag : nullptr;
  if (tr * nrx * nc <= s.bytes) {
    STCHK(transpose(src, s.data(), nt, nrx, nrx, nt, nc, comp, comp, flag, st));
    STCHK(to_host(dst, s.data(), nc * comp * sizeof(float), st));
  } else {
    const int most = (int)std::min<size_t>(s.bytes / tr, nrx);
    for (int f = 0; f < nc; ++f)
      for (int ix = 0; ix < nrx; ix += most) {
        const int n = std::min(most, nrx - ix);
        STCHK(transpose(src + f * comp + ix, s.data(), nt, n, nrx, nt, 1, 0, 0, flag, st));
        STCHK(to_host(dst + f * comp + (size_t)nt * ix, s.data(), n * tr, st));
      }
  }
  STCHK(read_flag(s, nonfinite, st));
  HIPCHK(hipStreamSynchronize(st));
  return OK;
}

int fetch_rounded(float* dst, const double* src, size_t n, hipStream_t st) {
  if (n == 0) return OK;
  Scratch s;
  if (!s.get(n * sizeof(float), 256)) {
    std::vector<double> h(n);
    HIPCHK(hipMemcpyAsync(h.data(), src, n * sizeof(double), hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    for (size_t i = 0; i < n; ++i) dst[i] = (float)h[i];
    return OK;
  }
  const size_t most = s.bytes / sizeof(float);
  for (size_t i = 0; i < n; i += most) {
    const size_t m = std::min(most, n - i);
    hipLaunchKernelGGL(k_round, dim3(blocks_of(m)), dim3(256), 0, st, src + i, s.data(), m);
    HIPCHK(hipGetLastError());
    STCHK(to_host(dst + i, s.data(), m * sizeof(float), st));
  }
  HIPCHK(hipStreamSynchronize(st));
  return OK;
}

}  // namespace erm
