// acoustic3d.hip -- 3D acoustic 10th-order (radius 5) propagator and
// cross-correlation imaging on one GPU's subdomain (gfx950).
//
// The reference's multi-GPU acoustic RTM (W/wave_fkernel.3d8o.cu:31-106,
// :183-210; W/gpu_funcs_3d.cu:64-131) is 8th order with separate damping,
// injection and imaging kernels. Here one kernel does a whole step:
//   p_next = K (2 p - p_prev + c lap p),  c = (v dt/dx)^2,  K = kz kx ky
// for the interior (5 cells from every face), then the point source or the
// receiver-plane injection, the receiver recording, the per-snapshot max-abs
// of the source wavefield and, in the receiver pass, the image update.
// Layout: (n1, n2, n3) = (z fastest, x, y slowest); on the device each z-row is
// padded so that the first interior cell, and with it every wave's row of 64,
// starts on a cache line (see Layout). A workgroup owns a 64 x 16
// tile of the (z, x) plane and marches along y over a chunk of planes; the
// y-neighbours live in an 11-deep register queue, the (z, x) halo of the
// current plane in LDS. Each step moves 16 algorithmic bytes per cell
// (read p, p_prev, c; write p_next): HBM-bound.

#include "../../include/acoustic3d.h"
#include "buffer.hpp"
#include "common.hpp"
#include "engine2d.hpp"
#include "hostcopy.hpp"
#include "layout.hpp"

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <vector>

namespace erm {

namespace {

constexpr float W0 = -5269.0f / 1800.0f, W1 = 5.0f / 3.0f, W2 = -5.0f / 21.0f, W3 = 5.0f / 126.0f,
                W4 = -5.0f / 1008.0f, W5 = 1.0f / 3150.0f;
constexpr int AZ = 64;     // tile along n1 (one wave64)
constexpr int AWY = 4;     // waves along n2
constexpr int ATXR = 4;    // n2 cells per thread
constexpr int AX = AWY * ATXR;
constexpr int AH = 5;
constexpr int AC3_MAX_CHUNK = 128;  // planes a workgroup marches at most
constexpr int ALZ = AZ + 2 * AH, ALX = AX + 2 * AH;

struct Ac3Args {
  int n1, n2, n3;
  long long s2, s3;          // strides of axes 2 and 3
  const float* p;            // current level
  float* pp;                 // previous level in, next level out
  const float* c;
  const float* kz; const float* kx; const float* ky;  // null = no sponge
  int mode;                  // 0 source pass, 1 receiver pass
  int sz, sx, sy;
  float amp;                 // source amplitude of this level (mode 0)
  int zr;
  float* rec_out;            // plane record of this level (mode 0), [i3][i2]
  const float* rec_in;       // plane injection of this level (mode 1)
  unsigned* smax;            // per-snapshot max-abs (float bits) (mode 0 snapshot level)
  const void* snap;          // source snapshot of this level (mode 1 image level)
  float snap_scale;
  int snap_bf16;
  void* snap_out;            // snapshot of the current level p to write (mode 0)
  const unsigned* snap_max;  // its max-abs (float bits)
  float* img;                // image (mode 1 image level)
  int ychunk;
};

__device__ __forceinline__ float bf16_to_f(unsigned short h) { return __uint_as_float(((unsigned)h) << 16); }

// Halo cells of the (z, x) plane tile that are not owned by a thread of the
// block: 10 z-halo rows of the 16 interior columns, then the 10 x-halo
// columns over the full 74 rows.
constexpr int AHALO = 2 * AH * AX + 2 * AH * ALZ;
constexpr int ANH = (AHALO + 255) / 256;

__device__ __forceinline__ void halo_cell(int h, int& lx, int& lz) {
  if (h < 2 * AH * AX) {
    lx = AH + h / (2 * AH);
    const int r = h % (2 * AH);
    lz = r < AH ? r : AZ + r;
  } else {
    const int h2 = h - 2 * AH * AX;
    const int cc = h2 / ALZ;
    lx = cc < AH ? cc : AX + cc;
    lz = h2 % ALZ;
  }
}

// Global loads through address-space-1 pointers (GLOBAL, not FLAT,
// instructions: FLAT ones also count against the LDS wait counter).
template <class T>
__device__ __forceinline__ T g1(const T* p, int i) {
  return ((const __attribute__((address_space(1))) T*)p)[i];
}

// The march along y is software-pipelined: the global loads of plane y+1
// (its new queue entry, and the own-cell p_prev, c, snapshot and image
// operands) are issued before plane y is computed, so their latency hides
// behind the arithmetic of the current plane. The plane tile is
// double-buffered in LDS with one barrier per plane whose fences cover LDS
// only, so those loads stay in flight across it.
// A plane is addressed as a raw buffer, so the offsets of a thread's cells stay
// the same through the march; what a plane needs besides (image, injected row)
// is loaded at its start. us a step, 203 x 181 x 247 (bound by latency and
// vector instructions) and 522^3 (bound by memory: the step moves 2.6 GB, 5.4
// TB/s, of which 0.5 GB are halo lines fetched twice): through pointers 42 and
// 526, with the image 60 and 970; now 33 and 480, 56 and 767.
// The halo cells of a plane are loaded with the queue entry of the same
// plane, five planes before it is computed: that is when the neighbouring
// tiles load those cells as their own queue entries, so the second read of
// each line is an L2 hit rather than a second fetch. Each thread keeps its
// halo cells of the five planes ahead in a ring in LDS (slot = plane % 5)
// that only it reads.
// What a step does besides: nothing, update the image (receiver pass at an
// imaging level), or store the snapshot of the level it reads (source pass: the
// level's max-abs is complete and its cells are at hand in the queue, so the
// snapshot costs its own bytes only; a pass of its own read the field again).
enum StepKind { STEP_PLAIN, STEP_IMAGE, STEP_SNAP };

// The max-abs of a snapshot is kept in SMAX_SLOTS partial maxima, each on a cache
// line of its own: thousands of waves that end together would queue at one
// address (203 x 181 x 247: 66 us a step against 33 without the maximum).
constexpr int SMAX_SLOTS = 32, SMAX_STRIDE = 32, SMAX_SNAP = SMAX_SLOTS * SMAX_STRIDE;
__device__ __forceinline__ float snap_max(const unsigned* m) {
  float v = __uint_as_float(m[(threadIdx.x & (SMAX_SLOTS - 1)) * SMAX_STRIDE]);
#pragma unroll
  for (int o = SMAX_SLOTS / 2; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  return v;
}
__device__ __forceinline__ float snap_inv(const unsigned* m) {
  const float v = snap_max(m);
  return v > 1e-30f ? 1.f / v : 0.f;  // subnormal maxima would overflow 1/v
}
__device__ __forceinline__ unsigned short snap_bf16(float v, float inv) {
  unsigned u = __float_as_uint(v * inv);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (unsigned short)(u >> 16);
}

template <int KIND>
__global__ __launch_bounds__(256, 4) void k_ac3_step(const Ac3Args a) {
  __shared__ float sh[2][ALX * ALZ + 1];  // the last one takes the threads without a halo cell
  __shared__ float hring[5][ANH][256];
  const int nbz = (a.n1 - 10 + AZ - 1) / AZ;
  const int nbx = (a.n2 - 10 + AX - 1) / AX;
  // z-fastest tile order, renumbered so each XCD gets a contiguous range:
  // the z- and x-neighbours whose halos a tile reads share its L2
  int b = xcd_tile(blockIdx.x, gridDim.x);
  const int bz = b % nbz;
  b /= nbz;
  const int bx = b % nbx;
  const int by = b / nbx;
  const int z0 = AH + bz * AZ, x0 = AH + bx * AX;
  const int y0 = AH + by * a.ychunk;
  const int y1 = min(y0 + a.ychunk, a.n3 - AH);
  // ty is wave-uniform (a wave is one row of 64 threads), so values indexed
  // by it and by the plane come from scalar loads
  const int tz = threadIdx.x, ty = __builtin_amdgcn_readfirstlane(threadIdx.y);
  const int tid = tz + AZ * ty;
  const int gz = z0 + tz;
  const bool zok = gz < a.n1 - AH;
  const int s2 = (int)a.s2;
  const unsigned plane = 4u * (unsigned)a.s3;  // bytes of a plane, which a buffer covers
  constexpr bool imaging = KIND == STEP_IMAGE;
  const float inv = KIND == STEP_SNAP && a.snap_bf16 ? snap_inv(a.snap_max) : 0.f;
  auto at = [&](const float* f, int y) { return Buf(f + (long long)y * a.s3, plane); };
  // per-thread halo cells (plane independent): LDS slot and byte
  // offset in a plane (kOutside: outside the grid, staged as zero)
  int hlds[ANH];
  unsigned hoff[ANH];
#pragma unroll
  for (int k = 0; k < ANH; ++k) {
    const int h = tid + 256 * k;
    int lx = 0, lz = 0;
    hlds[k] = ALX * ALZ;
    hoff[k] = kOutside;
    if (h < AHALO) {
      halo_cell(h, lx, lz);
      hlds[k] = lx * ALZ + lz;
      const int gx = x0 - AH + lx, g1v = z0 - AH + lz;
      if (gx >= 0 && gx < a.n2 && g1v >= 0 && g1v < a.n1) hoff[k] = 4u * (unsigned)(g1v + gx * s2);
    }
  }
  // own columns (kOutside: outside the interior, where every value is zero and
  // nothing is written), and their sponge factors of row and column
  unsigned coff[ATXR];
  float kzx[ATXR];
  auto sc = [](const float* p, int i) { return ((const __attribute__((address_space(4))) float*)p)[i]; };
  const float kzv = (a.kz && zok) ? g1(a.kz, gz) : 1.f;
#pragma unroll
  for (int j = 0; j < ATXR; ++j) {
    const int gx = x0 + ty * ATXR + j;
    coff[j] = (zok && gx < a.n2 - AH) ? 4u * (unsigned)(gz + gx * s2) : kOutside;
    kzx[j] = a.kz ? kzv * sc(a.kx, min(gx, a.n2 - 1)) : 1.f;
  }
  // register queue: q[k][j] = p at plane y-5+k
  float q[11][ATXR];
#pragma unroll
  for (int k = 0; k < 10; ++k) {
    const Buf p = at(a.p, y0 - AH + k);
#pragma unroll
    for (int j = 0; j < ATXR; ++j) q[k][j] = p.get(coff[j]);
  }
  float hv[ANH], ppv[ATXR], cv[ATXR], snv[ATXR], qn[ATXR];
  // loads of plane y: own cells, and with the queue entry of plane y+5 its halo
  auto load_plane = [&](int y, float (&h)[ANH], float (&qv)[ATXR], float (&pv)[ATXR], float (&c)[ATXR],
                        float (&sn)[ATXR]) {
    const Buf p5 = at(a.p, y + AH), pp = at(a.pp, y), cc = at(a.c, y);
#pragma unroll
    for (int j = 0; j < ATXR; ++j) {
      qv[j] = p5.get(coff[j]);
      pv[j] = pp.get(coff[j]);
      c[j] = cc.get(coff[j]);
    }
    if (imaging) {
      const Buf sb(static_cast<const char*>(a.snap) + (long long)y * (a.snap_bf16 ? plane / 2 : plane), plane);
#pragma unroll
      for (int j = 0; j < ATXR; ++j) {
        sn[j] = a.snap_bf16 ? bf16_to_f(sb.get16(coff[j] / 2)) * a.snap_scale : sb.get(coff[j]);
      }
    }
#pragma unroll
    for (int k = 0; k < ANH; ++k) h[k] = p5.get(hoff[k]);
  };
  // halo cells of the first five planes into the ring
#pragma unroll
  for (int j = 0; j < AH; ++j) {
    const Buf p = at(a.p, y0 + j);
#pragma unroll
    for (int k = 0; k < ANH; ++k) hring[(y0 + j) % 5][k][tid] = p.get(hoff[k]);
  }
  if (y0 < y1) load_plane(y0, hv, qn, ppv, cv, snv);
  float mx = 0.f;
  // receiver row: recorded (source pass), or injected from loads issued before
  // the plane's arithmetic
  const bool row = gz == a.zr && a.mode == 0 && a.rec_out;
  const bool inject = a.mode != 0 && a.rec_in && a.zr >= z0 && a.zr < z0 + AZ;  // uniform over the workgroup
  for (int y = y0; y < y1; ++y) {
    const int bb = (y - y0) & 1;
    float* const sp = sh[bb];
    // the image and the injected row: loaded here, not a plane ahead (registers)
    float rv[ATXR], imv[ATXR];
    if (imaging) {
      const Buf ib = at(a.img, y);
#pragma unroll
      for (int j = 0; j < ATXR; ++j) imv[j] = ib.get(coff[j]);
    }
    if (inject) {
      const Buf r(a.rec_in + (long long)y * a.n2, 4u * (unsigned)a.n2);
#pragma unroll
      for (int j = 0; j < ATXR; ++j) rv[j] = r.get(gz == a.zr ? 4u * (unsigned)(x0 + ty * ATXR + j) : kOutside);
    }
#pragma unroll
    for (int j = 0; j < ATXR; ++j) q[10][j] = qn[j];
#pragma unroll
    for (int j = 0; j < ATXR; ++j) sp[(ty * ATXR + j + AH) * ALZ + tz + AH] = q[5][j];
    // this plane's halo cells from the ring; the slot then takes plane y+5's
    const int slot = y % 5;
#pragma unroll
    for (int k = 0; k < ANH; ++k) {
      sp[hlds[k]] = hring[slot][k][tid];
      hring[slot][k][tid] = hv[k];
    }
    // the tile of plane y is complete; plane y-1's buffer is free again
    // once every wave has passed this barrier
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    // issue the next plane's loads before this plane's arithmetic
    float hv2[ANH], pp2[ATXR], c2[ATXR], sn2[ATXR];
    load_plane(y + 1 < y1 ? y + 1 : y, hv2, qn, pp2, c2, sn2);
    const float kyv = a.kz ? sc(a.ky, y) : 1.f;
    const Buf out = at(a.pp, y);
    float v[ATXR];
#pragma unroll
    for (int j = 0; j < ATXR; ++j) {
      const int p0 = (ty * ATXR + j + AH) * ALZ + tz + AH;
      float lap = 3.f * W0 * q[5][j];
      lap += W1 * ((sp[p0 + 1] + sp[p0 - 1]) + (sp[p0 + ALZ] + sp[p0 - ALZ]) + (q[6][j] + q[4][j]));
      lap += W2 * ((sp[p0 + 2] + sp[p0 - 2]) + (sp[p0 + 2 * ALZ] + sp[p0 - 2 * ALZ]) + (q[7][j] + q[3][j]));
      lap += W3 * ((sp[p0 + 3] + sp[p0 - 3]) + (sp[p0 + 3 * ALZ] + sp[p0 - 3 * ALZ]) + (q[8][j] + q[2][j]));
      lap += W4 * ((sp[p0 + 4] + sp[p0 - 4]) + (sp[p0 + 4 * ALZ] + sp[p0 - 4 * ALZ]) + (q[9][j] + q[1][j]));
      lap += W5 * ((sp[p0 + 5] + sp[p0 - 5]) + (sp[p0 + 5 * ALZ] + sp[p0 - 5 * ALZ]) + (q[10][j] + q[0][j]));
      v[j] = kzx[j] * kyv * (2.f * q[5][j] - ppv[j] + cv[j] * lap);
    }
    if (a.mode == 0 && y == a.sy) {
#pragma unroll
      for (int j = 0; j < ATXR; ++j)
        if (gz == a.sz && x0 + ty * ATXR + j == a.sx) v[j] += a.amp;
    }
    if (inject) {
#pragma unroll
      for (int j = 0; j < ATXR; ++j) v[j] = gz == a.zr ? v[j] + rv[j] : v[j];
    }
    if (row) {
#pragma unroll
      for (int j = 0; j < ATXR; ++j)
        if (coff[j] != kOutside) a.rec_out[(long long)y * a.n2 + x0 + ty * ATXR + j] = v[j];
    }
#pragma unroll
    for (int j = 0; j < ATXR; ++j) out.put(coff[j], 0, v[j]);
    if (KIND == STEP_SNAP) {
      const Buf so(static_cast<char*>(a.snap_out) + (long long)y * (a.snap_bf16 ? plane / 2 : plane), plane);
#pragma unroll
      for (int j = 0; j < ATXR; ++j) {
        if (a.snap_bf16)
          so.put16(coff[j] / 2, snap_bf16(q[5][j], inv));
        else
          so.put(coff[j], 0, q[5][j]);
      }
    }
    if (imaging) {
      const Buf io = at(a.img, y);
#pragma unroll
      for (int j = 0; j < ATXR; ++j) io.put(coff[j], 0, imv[j] + snv[j] * v[j]);
    }
    if (a.smax) {
#pragma unroll
      for (int j = 0; j < ATXR; ++j) mx = coff[j] != kOutside ? fmaxf(mx, fabsf(v[j])) : mx;
    }
#pragma unroll
    for (int k = 0; k < 10; ++k)
#pragma unroll
      for (int j = 0; j < ATXR; ++j) q[k][j] = q[k + 1][j];
#pragma unroll
    for (int k = 0; k < ANH; ++k) hv[k] = hv2[k];
#pragma unroll
    for (int j = 0; j < ATXR; ++j) {
      ppv[j] = pp2[j];
      cv[j] = c2[j];
      snv[j] = sn2[j];
    }
  }
  if (a.mode == 0 && a.smax) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
    if (tz == 0) atomicMax(a.smax + ((blockIdx.x * AWY + ty) & (SMAX_SLOTS - 1)) * SMAX_STRIDE, __float_as_uint(mx));
  }
}

// Snapshot of the last level (no later step reads it): bf16 with the level's
// max-abs scale, or fp32 copy.
__global__ void k_ac3_snap(const float* p, void* out, size_t n, const unsigned* smax, int bf16) {
  const float inv = snap_inv(smax);
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x) {
    if (bf16)
      static_cast<unsigned short*>(out)[i] = snap_bf16(p[i], inv);
    else
      static_cast<float*>(out)[i] = p[i];
  }
}

// The max-abs of every snapshot.
__global__ void k_ac3_scales(const unsigned* smax, float* out) {
  const float v = snap_max(smax + (size_t)blockIdx.x * SMAX_SNAP);
  if (threadIdx.x == 0) out[blockIdx.x] = v;
}

// Rows of n1 cells, contiguous on one side and ld apart on the other.
__global__ void k_ac3_rows(const float* in, float* out, int n1, long long rows, int ld_in, int ld_out) {
  for (long long r = blockIdx.x * (long long)blockDim.y + threadIdx.y; r < rows; r += (long long)gridDim.x * blockDim.y)
    for (int z = threadIdx.x; z < n1; z += blockDim.x) out[r * ld_out + z] = in[r * ld_in + z];
}

__global__ void k_fill3(float* p, size_t n) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    p[i] = 0.f;
}

__global__ void k_sub_rec(float* a, const float* b, size_t n) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    a[i] -= b[i];
}

int fill0(float* p, size_t n, hipStream_t st) {
  size_t blocks = std::min<size_t>((n + 255) / 256, 65536);
  hipLaunchKernelGGL(k_fill3, dim3((unsigned)blocks), dim3(256), 0, st, p, n);
  HIPCHK(hipGetLastError());
  return OK;
}

// Sponge taper of W/abc-mod.f90:35-50 applied per axis (1 inside).
std::vector<float> taper(int n, int abc) {
  std::vector<float> k(n, 1.f);
  if (abc <= 0) return k;
  std::vector<float> f(abc + 5);
  for (int i = 1; i <= abc; ++i) {
    const float aux = (1.0f * (float)i) / (1.0f * (float)abc);
    f[i - 1] = std::exp(-0.09f * aux * aux);
  }
  for (int i = abc + 1; i <= abc + 5; ++i) f[i - 1] = f[abc - 1];
  const int abc2 = abc + 5;
  for (int i1 = 1; i1 <= abc2; ++i1) {
    const int top = i1 - 1, bot = n - abc2 + i1 - 1;
    if (top < n) k[top] *= f[abc2 - i1];
    if (bot >= 0 && bot < n) k[bot] *= f[i1 - 1];
  }
  return k;
}

// Step workgroups resident at once on the current device (122 VGPRs without
// imaging: 4 waves per SIMD, so 4 workgroups a CU, 1024 on the chip).
int resident_workgroups() {
  static const int n = [] {
    int dev = 0, cus = 0, per = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, k_ac3_step<STEP_PLAIN>, AZ * AWY, 0) != hipSuccess ||
        cus * per <= 0)
      return 1024;
    return cus * per;
  }();
  return n;
}

// Planes a workgroup marches along y. A plane costs a workgroup about 1.2 us
// whatever the grid (the latency of its loads), and a chunk some six planes
// more for its first loads, so the step takes (rounds of resident workgroups)
// x (planes + 6): the number of chunks that minimises it. Both sides,
// source-pass step: 203 x 181 x 247 (44 tiles) 64 planes 83 us, 11 planes (the
// rule's) 35 us; 266^3 (64 tiles) 64 planes 83 us, 16 planes (the rule's, one
// whole round) 52, 8 planes (two) 50; 64^3 (4 tiles) 64 planes 67 us, 8 planes 13,
// one plane (the rule's) 5.8. At 522^3 (256 tiles), where memory bounds the step,
// 128 planes (the rule's) 483 us, 103 494, 86 488, 64 504, 32 506.
int planes_per_workgroup(int tiles, int n) {
  const int resident = resident_workgroups();
  long long best = -1;
  int ych = n;
  for (int chunks = 1; chunks <= n; ++chunks) {
    const int c = (n + chunks - 1) / chunks;
    if (c > AC3_MAX_CHUNK) continue;
    const long long rounds = ((long long)tiles * ((n + c - 1) / c) + resident - 1) / resident;
    const long long cost = rounds * (c + 6);
    if (best < 0 || cost < best) {
      best = cost;
      ych = c;
    }
  }
  return ych;
}

}  // namespace

}  // namespace erm

using namespace erm;

struct ac3d {
  ac3d_cfg_t cfg{};
  size_t n = 0;         // cells
  // Device layout of a field: cell (z, x, y) at lead + z + ld (x + n2 y). With
  // lead 27 and ld a multiple of 64 the first interior cell of every row (z = 5)
  // lies on a 128-byte line, so a wave's row is two lines instead of three; a
  // snapshot starts 32 elements later (slead), which does the same for its
  // 16-bit rows (522^3: 10% fewer L2 requests, step 565 -> 526 us, with the image
  // 1064 -> 970). Where that takes much memory or 32-bit offsets do not allow it,
  // rows are contiguous (lead 0).
  int lead = 0, slead = 0, ld = 0;
  size_t np = 0;  // elements of a field and of a snapshot
  long long plane = 0;
  int ychunk = 0;  // planes per step workgroup
  DevBuf c, c_alt, k, f0, f1, rec, rec_tmp, snap, smax, img, amp_h_dummy;
  std::vector<float> amp;
  std::vector<float> scales;  // per snapshot (host copy after the source pass)
  hipStream_t st = nullptr;
  hipEvent_t ev[2] = {};
  double timings[6] = {0, 0, 0, 0, 0, 0};
  void* snap_at(int k) const {  // snapshot k, as the step kernel indexes it
    const size_t esz = cfg.snap_prec == 1 ? 2 : 4;
    return snap.as<char>() + ((size_t)k * np + slead) * esz;
  }
  ~ac3d() {
    for (auto& e : ev)
      if (e) (void)hipEventDestroy(e);
    if (st) (void)hipStreamDestroy(st);
  }
};

static int ac3_launch(ac3d* a, const float* p, float* pp, const float* c, int mode, int level, bool record,
                      bool inject, unsigned* smax, const void* snap, float scale, float* img,
                      void* snap_out = nullptr, const unsigned* snap_max = nullptr) {
  const ac3d_cfg_t& g = a->cfg;
  Ac3Args x{};
  x.n1 = g.n1; x.n2 = g.n2; x.n3 = g.n3;
  x.s2 = a->ld;
  x.s3 = (long long)a->ld * g.n2;
  x.p = p; x.pp = pp; x.c = c;
  if (g.abc > 0) {
    x.kz = a->k.as<float>();
    x.kx = x.kz + g.n1;
    x.ky = x.kx + g.n2;
  }
  x.mode = mode;
  x.sz = g.sz; x.sx = g.sx; x.sy = g.sy;
  x.amp = mode == 0 ? a->amp[level - 1] : 0.f;
  x.zr = g.zr;
  x.rec_out = record ? a->rec.as<float>() + (long long)(level - 1) * a->plane : nullptr;
  x.rec_in = inject ? a->rec.as<float>() + (long long)(level - 1) * a->plane : nullptr;
  x.smax = smax;
  x.snap = snap;
  x.snap_scale = scale;
  x.snap_bf16 = g.snap_prec == 1;
  x.img = img;
  x.snap_out = snap_out;
  x.snap_max = snap_max;
  x.ychunk = a->ychunk;
  const int nbz = (g.n1 - 10 + AZ - 1) / AZ, nbx = (g.n2 - 10 + AX - 1) / AX;
  const int nby = (g.n3 - 10 + x.ychunk - 1) / x.ychunk;
  if (mode == 1 && img)
    hipLaunchKernelGGL(k_ac3_step<STEP_IMAGE>, dim3(nbz * nbx * nby), dim3(AZ, AWY), 0, a->st, x);
  else if (snap_out)
    hipLaunchKernelGGL(k_ac3_step<STEP_SNAP>, dim3(nbz * nbx * nby), dim3(AZ, AWY), 0, a->st, x);
  else
    hipLaunchKernelGGL(k_ac3_step<STEP_PLAIN>, dim3(nbz * nbx * nby), dim3(AZ, AWY), 0, a->st, x);
  HIPCHK(hipGetLastError());
  return OK;
}

// Rows between the caller's layout and the device's.
static int ac3_rows(const float* in, float* out, int n1, long long rows, int ld_in, int ld_out, hipStream_t st) {
  hipLaunchKernelGGL(k_ac3_rows, dim3((unsigned)std::min<long long>((rows + 3) / 4, 65536)), dim3(64, 4), 0, st, in, out,
                     n1, rows, ld_in, ld_out);
  HIPCHK(hipGetLastError());
  return OK;
}
// To the device: the source field of the passes, which begin with a fill of their
// own, carries the contiguous side.
static int ac3_upload(ac3d* a, const float* host, float* dev) {
  if (a->ld == a->cfg.n1) return copy_to_device(dev + a->lead, host, a->n * 4);
  STCHK(copy_to_device(a->f0.p, host, a->n * 4));
  STCHK(ac3_rows(a->f0.as<float>(), dev + a->lead, a->cfg.n1, a->plane, a->cfg.n1, a->ld, a->st));
  HIPCHK(hipStreamSynchronize(a->st));
  return OK;
}
// From the device, where a run may be using the fields: through scratch of its
// own. Large arrays in pieces of whole rows, a piece of each copy thread at a time.
static int ac3_fetch(ac3d* a, const float* dev, float* host) {
  const int n1 = a->cfg.n1;
  const size_t row = (size_t)n1 * 4;
  const long long most = std::max<long long>(kCopyPiece / row, 1), pieces = (a->plane + most - 1) / most;
  const int lanes = (int)std::min<long long>(pieces, kCopyThreads);
  DevBuf t;
  if (a->n * 4 < kLargeToHost || t.alloc(lanes * most * row, "scratch") != OK) {
    (void)hipGetLastError();  // no scratch: fetch_fields does without
    return fetch_fields(host, 1, n1, (int)a->plane, a->ld, dev, 0, nullptr, a->st);
  }
  std::atomic<long long> next{0};
  return with_copy_lanes(lanes, [&](int lane, hipStream_t st) -> int {
    float* const s = t.as<float>() + lane * most * n1;
    for (long long k = next++; k < pieces; k = next++) {
      const long long r0 = k * most, rows = std::min(most, a->plane - r0);
      STCHK(ac3_rows(dev + r0 * a->ld, s, n1, rows, a->ld, n1, st));
      HIPCHK(hipMemcpyAsync(host + r0 * n1, s, rows * row, hipMemcpyDeviceToHost, st));
      HIPCHK(hipStreamSynchronize(st));
    }
    return OK;
  });
}

// Source pass: levels 1..nt with the model c; records the receiver plane
// (subtracting when sub) and, with snapshots, stores every j-th level.
static int ac3_source_pass(ac3d* a, const float* c, int record, int sub, int snaps) {
  const ac3d_cfg_t& g = a->cfg;
  STCHK(fill0(a->f0.as<float>(), a->np, a->st));
  STCHK(fill0(a->f1.as<float>(), a->np, a->st));
  float* p = a->f0.as<float>() + a->lead;
  float* pp = a->f1.as<float>() + a->lead;
  float* rec_dst = nullptr;
  if (record) {
    if (sub) {
      std::swap(a->rec, a->rec_tmp);  // record into the scratch, subtract afterwards
    }
    STCHK(fill0(a->rec.as<float>(), (size_t)g.nt * a->plane, a->st));
    rec_dst = a->rec.as<float>();
  }
  const int j = g.snap_every;
  const int nsnap = g.nt / j;
  if (snaps) HIPCHK(hipMemsetAsync(a->smax.p, 0, sizeof(unsigned) * SMAX_SNAP * std::max(nsnap, 1), a->st));
  for (int t = 1; t <= g.nt; ++t) {
    const bool sl = snaps && t % j == 0;
    unsigned* sm = sl ? a->smax.as<unsigned>() + (size_t)(t / j - 1) * SMAX_SNAP : nullptr;
    // the snapshot of the level this step reads
    const int k = snaps && t > 1 && (t - 1) % j == 0 ? (t - 1) / j - 1 : -1;
    STCHK(ac3_launch(a, p, pp, c, 0, t, record != 0, false, sm, nullptr, 0.f, nullptr, k < 0 ? nullptr : a->snap_at(k),
                     k < 0 ? nullptr : a->smax.as<unsigned>() + (size_t)k * SMAX_SNAP));
    if (sl && t == g.nt) {
      const size_t cells = (size_t)a->ld * a->plane;
      size_t blocks = std::min<size_t>((cells + 255) / 256, 65536);
      hipLaunchKernelGGL(k_ac3_snap, dim3((unsigned)blocks), dim3(256), 0, a->st, pp, a->snap_at(t / j - 1), cells, sm,
                         g.snap_prec == 1);
      HIPCHK(hipGetLastError());
    }
    std::swap(p, pp);
  }
  (void)rec_dst;
  if (record && sub) {
    std::swap(a->rec, a->rec_tmp);  // a->rec is the first record again
    size_t cnt = (size_t)g.nt * a->plane;
    size_t blocks = std::min<size_t>((cnt + 255) / 256, 65536);
    hipLaunchKernelGGL(k_sub_rec, dim3((unsigned)blocks), dim3(256), 0, a->st, a->rec.as<float>(),
                       a->rec_tmp.as<float>(), cnt);
    HIPCHK(hipGetLastError());
  }
  return OK;
}

RTM_EXPORT int ac3d_create(ac3d** out, const ac3d_cfg_t* cfg, const float* c, const float* amp) {
  if (!out || !cfg || !c || !amp) { set_error("null argument"); return E_ARG; }
  const ac3d_cfg_t& g = *cfg;
  if (g.n1 < 11 || g.n2 < 11 || g.n3 < 11 || g.nt < 1 || g.snap_every < 1) {
    set_error("ac3d: grid must exceed the 5-cell halo on every axis; nt, snap_every >= 1");
    return E_ARG;
  }
  if (g.sz < 5 || g.sz >= g.n1 - 5 || g.sx < 5 || g.sx >= g.n2 - 5 || g.sy < 5 || g.sy >= g.n3 - 5 ||
      g.zr < 5 || g.zr >= g.n1 - 5) {
    set_error("ac3d: source or receiver plane outside the interior");
    return E_ARG;
  }
  if (g.abc > 0 && (2 * (g.abc + 5) > g.n1 || 2 * (g.abc + 5) > g.n2 || 2 * (g.abc + 5) > g.n3)) {
    set_error("ac3d: sponge does not fit");
    return E_ARG;
  }
  STCHK(ensure_device());
  std::unique_ptr<ac3d> a(new ac3d());
  a->cfg = g;
  a->n = (size_t)g.n1 * g.n2 * g.n3;
  if (a->n >= (size_t)1 << 31) {  // the step kernel addresses a field with 32-bit offsets
    set_error("3D grid of %zu cells exceeds 2^31 cells per field", a->n);
    return E_ARG;
  }
  a->plane = (long long)g.n2 * g.n3;
  const int nsnap = std::max(g.nt / g.snap_every, 1);
  const size_t esz = g.snap_prec == 1 ? 2 : 4;
  a->ld = g.n1;
  a->np = a->n;
  {
    const int ld = round_up(g.n1, 64);
    const size_t np = (size_t)ld * a->plane + 64;
    const size_t fixed = 2 * (size_t)g.nt * a->plane * 4, cell = 5 * 4 + (size_t)nsnap * esz;
    size_t freeb = 0, totb = 0;
    HIPCHK(hipMemGetInfo(&freeb, &totb));
    // Padding is to cost little memory, which other handles may be counting on:
    // at most a third more than contiguous rows take, and at most a sixteenth of
    // what is free. RTM_AC3_PAD (tests): 0 contiguous rows, 1 padded ones.
    const char* pad = getenv("RTM_AC3_PAD");
    const bool fits = np * cell + fixed < freeb / 10 * 9;
    const bool little = 3LL * ld <= 4LL * g.n1 && (np - a->n) * cell <= freeb / 16;
    if (np < (size_t)1 << 31 && fits && (pad ? atoi(pad) != 0 : little)) {
      a->ld = ld;
      a->lead = 27;
      a->slead = 59;
      a->np = np;
    }
  }
  // RTM_AC3_YCHUNK overrides the planes per workgroup (experiments)
  const char* fixed = getenv("RTM_AC3_YCHUNK");
  a->ychunk = fixed && atoi(fixed) > 0
                  ? atoi(fixed)
                  : planes_per_workgroup(((g.n1 - 10 + AZ - 1) / AZ) * ((g.n2 - 10 + AX - 1) / AX), g.n3 - 10);
  HIPCHK(hipStreamCreateWithFlags(&a->st, hipStreamNonBlocking));
  for (auto& e : a->ev) HIPCHK(hipEventCreate(&e));
  STCHK(a->c.alloc(a->np * 4, "velocity term"));
  STCHK(a->f0.alloc(a->np * 4, "wavefield"));
  STCHK(a->f1.alloc(a->np * 4, "wavefield"));
  STCHK(ac3_upload(a.get(), c, a->c.as<float>()));
  STCHK(a->k.alloc((size_t)(g.n1 + g.n2 + g.n3) * 4, "sponge"));
  std::vector<float> k1 = taper(g.n1, g.abc), k2 = taper(g.n2, g.abc), k3 = taper(g.n3, g.abc);
  HIPCHK(hipMemcpy(a->k.p, k1.data(), g.n1 * 4, hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(a->k.as<float>() + g.n1, k2.data(), g.n2 * 4, hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(a->k.as<float>() + g.n1 + g.n2, k3.data(), g.n3 * 4, hipMemcpyHostToDevice));
  STCHK(a->rec.alloc((size_t)g.nt * a->plane * 4, "receiver data"));
  STCHK(fill0(a->rec.as<float>(), (size_t)g.nt * a->plane, a->st));
  STCHK(a->img.alloc(a->np * 4, "image"));
  STCHK(a->snap.alloc((size_t)nsnap * a->np * esz, "snapshots"));
  STCHK(a->smax.alloc(sizeof(unsigned) * (SMAX_SNAP + 1) * nsnap, "snapshot scales"));
  a->amp.assign(amp, amp + g.nt);
  HIPCHK(hipStreamSynchronize(a->st));
  *out = a.release();
  return OK;
}

RTM_EXPORT int ac3d_model_data(ac3d* a, const float* c_true) {
  if (!a) { set_error("null handle"); return E_ARG; }
  // observed = data(true model) - data(migration model) when c_true is given,
  // else the migration-model data
  HIPCHK(hipEventRecord(a->ev[0], a->st));
  if (c_true) {
    STCHK(a->c_alt.alloc(a->np * 4, "true model"));
    STCHK(ac3_upload(a, c_true, a->c_alt.as<float>()));
    if (!a->rec_tmp.p) STCHK(a->rec_tmp.alloc((size_t)a->cfg.nt * a->plane * 4, "receiver scratch"));
    STCHK(ac3_source_pass(a, a->c_alt.as<float>() + a->lead, 1, 0, 0));
    STCHK(ac3_source_pass(a, a->c.as<float>() + a->lead, 1, 1, 0));
    a->c_alt.release();
  } else {
    STCHK(ac3_source_pass(a, a->c.as<float>() + a->lead, 1, 0, 0));
  }
  HIPCHK(hipEventRecord(a->ev[1], a->st));
  HIPCHK(hipStreamSynchronize(a->st));
  float ms = 0;
  HIPCHK(hipEventElapsedTime(&ms, a->ev[0], a->ev[1]));
  a->timings[4] = ms;
  return OK;
}

RTM_EXPORT int ac3d_migrate(ac3d* a) {
  if (!a) { set_error("null handle"); return E_ARG; }
  const ac3d_cfg_t& g = a->cfg;
  HIPCHK(hipEventRecord(a->ev[0], a->st));
  STCHK(ac3_source_pass(a, a->c.as<float>() + a->lead, 0, 0, 1));
  HIPCHK(hipEventRecord(a->ev[1], a->st));
  HIPCHK(hipStreamSynchronize(a->st));
  float ms_src = 0;
  HIPCHK(hipEventElapsedTime(&ms_src, a->ev[0], a->ev[1]));
  const int j = g.snap_every;
  const int nsnap = g.nt / j;
  a->scales.assign(std::max(nsnap, 1), 0.f);
  if (nsnap > 0) {
    float* scales = reinterpret_cast<float*>(a->smax.as<unsigned>() + (size_t)nsnap * SMAX_SNAP);
    hipLaunchKernelGGL(k_ac3_scales, dim3(nsnap), dim3(64), 0, a->st, a->smax.as<unsigned>(), scales);
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(a->st));
    HIPCHK(hipMemcpy(a->scales.data(), scales, sizeof(float) * nsnap, hipMemcpyDeviceToHost));
  }
  // receiver pass, levels nt..1
  STCHK(fill0(a->f0.as<float>(), a->np, a->st));
  STCHK(fill0(a->f1.as<float>(), a->np, a->st));
  STCHK(fill0(a->img.as<float>(), a->np, a->st));
  float* q = a->f0.as<float>() + a->lead;
  float* qq = a->f1.as<float>() + a->lead;
  HIPCHK(hipEventRecord(a->ev[0], a->st));
  for (int t = g.nt; t >= 1; --t) {
    const bool il = t % j == 0;
    const void* sp = il ? a->snap_at(t / j - 1) : nullptr;
    const float sc = il ? a->scales[t / j - 1] : 0.f;
    STCHK(ac3_launch(a, q, qq, a->c.as<float>() + a->lead, 1, t, false, true, nullptr, sp, sc,
                     il ? a->img.as<float>() + a->lead : nullptr));
    std::swap(q, qq);
  }
  HIPCHK(hipEventRecord(a->ev[1], a->st));
  HIPCHK(hipStreamSynchronize(a->st));
  float ms_rcv = 0;
  HIPCHK(hipEventElapsedTime(&ms_rcv, a->ev[0], a->ev[1]));
  a->timings[0] = ms_src;
  a->timings[1] = g.nt;
  a->timings[2] = ms_rcv;
  a->timings[3] = g.nt;
  return OK;
}

RTM_EXPORT int ac3d_set_data(ac3d* a, const float* rec) {
  if (!a || !rec) { set_error("null argument"); return E_ARG; }
  return copy_to_device(a->rec.p, rec, (size_t)a->cfg.nt * a->plane * 4);
}

RTM_EXPORT int ac3d_get_data(ac3d* a, float* rec) {
  if (!a || !rec) { set_error("null argument"); return E_ARG; }
  HIPCHK(hipStreamSynchronize(a->st));
  return copy_to_host(rec, a->rec.p, (size_t)a->cfg.nt * a->plane * 4);
}

RTM_EXPORT int ac3d_get_image(ac3d* a, float* img) {
  if (!a || !img) { set_error("null argument"); return E_ARG; }
  HIPCHK(hipStreamSynchronize(a->st));
  if (a->ld == a->cfg.n1) return copy_to_host(img, a->img.as<float>() + a->lead, a->n * 4);
  return ac3_fetch(a, a->img.as<float>() + a->lead, img);
}

RTM_EXPORT int ac3d_get_snapshot_scales(ac3d* a, float* out, int n) {
  if (!a || !out) { set_error("null argument"); return E_ARG; }
  for (int i = 0; i < n && i < (int)a->scales.size(); ++i) out[i] = a->scales[i];
  return OK;
}

RTM_EXPORT int ac3d_timings(ac3d* a, double* out6) {
  if (!a || !out6) { set_error("null argument"); return E_ARG; }
  for (int i = 0; i < 6; ++i) out6[i] = a->timings[i];
  return OK;
}

RTM_EXPORT int ac3d_destroy(ac3d* a) {
  delete a;
  return OK;
}
