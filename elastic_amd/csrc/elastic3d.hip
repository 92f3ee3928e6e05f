// elastic3d.hip -- 9-field 3D elastic adjoint time step (gfx950).
//
// The reference's 3D elastic kernel test (K3/rtmlib-modC.c:277-589 CPU loop,
// K3/rtmlib-modC-gpu.cu:374-690 CUDA kernel) advances the adjoint of the
// staggered-grid velocity-stress system by one level:
//   out = out + in1 + sum of 10-tap gathers of coefficient * field
// over 9 fields (Vy, Vx, Vz, syy, sxx, szz, sxy, sxz, syz) and 6 coefficient
// arrays (m1_y, m1_x, m1_z, m2, m3, m2m3), every array padded by 5 cells per
// face, (nz+10) x (nx+10) x (ny+10), z fastest. Each output is a sum of
// 1 to 5 gathers along one axis with tap set A (offsets -5..4) or B (-4..5).
//
// Here the gathers of one output along one axis are merged: the products
// coefficient * field that share an axis and a tap set are summed first
// (e.g. m2m3 sxx + m2 syy + m2 szz for Vx along x), which leaves 18 gathers
// over 9 distinct product arrays. The step falls into two halves that read
// nothing in common: the velocity outputs come from the six stresses and m2,
// m3, m2m3, the stress outputs from the three velocities and m1_x, m1_y, m1_z.
// A workgroup of 16 waves computes one half of a tz (z) x tx (x) tile of the
// (z, x) plane, at most 1024 cells, marching along y over a chunk of planes:
//   * the 3 products gathered along x, over the tile plus its 5-column
//     x-halo, and the 3 gathered along z, over the tile plus its 5-row
//     z-halo, go to LDS;
//   * the 3 products gathered along y live in an 11-deep register queue of
//     the thread's own column (planes y-5 .. y+5), refilled 5 planes ahead.
// Each step moves 168 algorithmic bytes per cell (in, in1, out and the 6
// coefficients read, out written): HBM-bound once the loads of a plane are in
// flight while the plane before it is computed (see el3_march).

#include "../../include/elastic3d.h"
#include "common.hpp"
#include "elastic2d.hpp"
#include "engine2d.hpp"

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <mutex>

namespace erm {

namespace {

enum { VY, VX, VZ, SYY, SXX, SZZ, SXY, SXZ, SYZ };
enum { M1Y, M1X, M1Z, M2, M3, M2M3 };

constexpr int EH = 5;                // stencil radius
constexpr int ENT = 1024;            // threads of a workgroup: 16 waves
constexpr int EZ = 64;               // tile rows (z) at most
constexpr int EX = 22;               // tile columns (x) at most
constexpr int EHN = 832;             // halo cells at most
constexpr int EP = EZ + 2 * EH;      // rows of one product's column in LDS
constexpr int EC = 3 * EP;           // a column's three products
constexpr int EBAND = (2 * EX + 2 * EH) * EC;  // x-band (EX + 10 columns), z-band (EX)

struct El3Args {
  int ny, nz, nx;
  int sx, sy;  // element strides of x and y (z is 1)
  const float* in[9];
  const float* in1[9];
  float* out[9];
  const float* m[6];
  int tz, tx;  // tile: tz <= EZ, tx <= EX, tz * tx <= ENT, 10 (tz + tx) <= EHN
  int nbz, nbx, ych, nblk;
  int xcd;
};

// Element at byte offset o of a plane: a scalar base and a 32-bit lane offset.
// (opaque() keeps the compiler from hoisting the sums of 33 array bases and a
// lane's offset out of the march as 66 vector registers.)
__device__ __forceinline__ unsigned opaque(unsigned o) {
  asm volatile("" : "+v"(o));
  return o;
}
__device__ __forceinline__ float gl(const float* plane, unsigned o) {
  return *(const __attribute__((address_space(1))) float*)((const __attribute__((address_space(1))) char*)plane + o);
}
__device__ __forceinline__ void gs(float* plane, unsigned o, float v) {
  *(__attribute__((address_space(1))) float*)((__attribute__((address_space(1))) char*)plane + o) = v;
}

// The 9 distinct products of one cell that the 18 gathers read:
//   PX = m2m3 sxx + m2 (syy + szz)  (x, set A, Vx)   Pxy = m3 sxy (x: Vy, y: Vx)
//   PY = m2m3 syy + m2 (szz + sxx)  (y, set A, Vy)   Pxz = m3 sxz (x: Vz, z: Vx)
//   PZ = m2m3 szz + m2 (sxx + syy)  (z, set A, Vz)   Pyz = m3 syz (z: Vy, y: Vz)
//   Qx = m1_x Vx (x: sxx, y: sxy, z: sxz)   Qy = m1_y Vy (x: sxy, y: syy, z: syz)
//   Qz = m1_z Vz (x: sxz, y: syz, z: szz); every other gather uses set B.
enum { PX, PY, PZ, PXY, PXZ, PYZ, QX, QY, QZ };

// Gathers at cell i of products P along one axis, P(k) = product at i + k:
//   set A: sum_d c_(6-d) (P(-d) - P(d-1))     set B: sum_d c_(6-d) (P(1-d) - P(d))
template <class F>
__device__ __forceinline__ float gather_a(F P) {
  float s = C5 * (P(-1) - P(0));
  s = fmaf(C4, P(-2) - P(1), s);
  s = fmaf(C3, P(-3) - P(2), s);
  s = fmaf(C2, P(-4) - P(3), s);
  return fmaf(C1, P(-5) - P(4), s);
}
template <class F>
__device__ __forceinline__ float gather_b(F P) {
  float s = C5 * (P(0) - P(1));
  s = fmaf(C4, P(-1) - P(2), s);
  s = fmaf(C3, P(-2) - P(3), s);
  s = fmaf(C2, P(-3) - P(4), s);
  return fmaf(C1, P(-4) - P(5), s);
}

// Workgroup barrier whose fences cover LDS only: global loads issued before
// it stay in flight.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// The two halves. own(): the raw operands of a cell of the thread's own column;
// halo(): those of a cell of the x-band (x) or of the z-band, whose three
// products differ in two operands; queue(): the products along y; band slots
// of the x- and z-band (the own cell's products that are not in the queue wait
// 5 planes in registers, keep()).
struct Velocity {  // outputs Vx, Vy, Vz
  static constexpr int NO = 9, NH = 8, NK = 3, NF = 3;
  static constexpr int OUT[NF] = {VX, VY, VZ};
  static __device__ __forceinline__ void own(const El3Args& a, long long py, unsigned o, float (&w)[NO]) {
    constexpr int f[6] = {SXX, SYY, SZZ, SXY, SXZ, SYZ};
#pragma unroll
    for (int k = 0; k < 6; ++k) w[k] = gl(a.in[f[k]] + py, o);
    w[6] = gl(a.m[M2] + py, o);
    w[7] = gl(a.m[M3] + py, o);
    w[8] = gl(a.m[M2M3] + py, o);
  }
  static __device__ __forceinline__ void products(const float (&w)[NO], float (&p)[9]) {
    p[PX] = fmaf(w[8], w[0], w[6] * (w[1] + w[2]));
    p[PY] = fmaf(w[8], w[1], w[6] * (w[2] + w[0]));
    p[PZ] = fmaf(w[8], w[2], w[6] * (w[0] + w[1]));
    p[PXY] = w[7] * w[3];
    p[PXZ] = w[7] * w[4];
    p[PYZ] = w[7] * w[5];
  }
  static constexpr int QUEUE[3] = {PY, PXY, PYZ};
  static constexpr int KEEP[3] = {PX, PZ, PXZ};
  static constexpr int XB[3] = {PX, PXY, PXZ};
  static constexpr int ZB[3] = {PZ, PYZ, PXZ};
  // the band's own shear stress differs: x-band sxy, z-band syz
  static __device__ __forceinline__ const float* split(const El3Args& a, bool x) { return x ? a.in[SXY] : a.in[SYZ]; }
  static __device__ __forceinline__ void halo(const El3Args& a, const float* sp, long long py, unsigned o, float (&w)[NH]) {
    w[0] = gl(a.in[SXX] + py, o);
    w[1] = gl(a.in[SYY] + py, o);
    w[2] = gl(a.in[SZZ] + py, o);
    w[3] = gl(sp + py, o);
    w[4] = gl(a.in[SXZ] + py, o);
    w[5] = gl(a.m[M2] + py, o);
    w[6] = gl(a.m[M3] + py, o);
    w[7] = gl(a.m[M2M3] + py, o);
  }
  static __device__ __forceinline__ void halo_products(const float (&w)[NH], bool x, float (&p)[3]) {
    const float d = x ? w[0] : w[2], e = x ? w[2] : w[0];
    p[0] = fmaf(w[7], d, w[5] * (w[1] + e));
    p[1] = w[6] * w[3];
    p[2] = w[6] * w[4];
  }
  template <class FX, class FY, class FZ>
  static __device__ __forceinline__ void gather(FX X, FY Y, FZ Z, float (&g)[NF]) {
    g[0] = gather_a(X(0)) + gather_b(Y(1)) + gather_b(Z(2));
    g[1] = gather_a(Y(0)) + gather_b(Z(1)) + gather_b(X(1));
    g[2] = gather_a(Z(0)) + gather_b(Y(2)) + gather_b(X(2));
  }
};
struct Stress {  // the six stress outputs
  static constexpr int NO = 6, NH = 6, NK = 0, NF = 6;
  static constexpr int OUT[NF] = {SXX, SYY, SZZ, SXY, SXZ, SYZ};
  static __device__ __forceinline__ void own(const El3Args& a, long long py, unsigned o, float (&w)[NO]) {
    w[0] = gl(a.in[VX] + py, o);
    w[1] = gl(a.in[VY] + py, o);
    w[2] = gl(a.in[VZ] + py, o);
    w[3] = gl(a.m[M1X] + py, o);
    w[4] = gl(a.m[M1Y] + py, o);
    w[5] = gl(a.m[M1Z] + py, o);
  }
  static __device__ __forceinline__ void products(const float (&w)[NO], float (&p)[9]) {
    p[QX] = w[3] * w[0];
    p[QY] = w[4] * w[1];
    p[QZ] = w[5] * w[2];
  }
  static constexpr int QUEUE[3] = {QX, QY, QZ};
  static constexpr int KEEP[1] = {QX};  // none kept
  static constexpr int XB[3] = {QX, QY, QZ};
  static constexpr int ZB[3] = {QX, QY, QZ};
  static __device__ __forceinline__ const float* split(const El3Args&, bool) { return nullptr; }
  static __device__ __forceinline__ void halo(const El3Args& a, const float*, long long py, unsigned o, float (&w)[NH]) {
    own(a, py, o, w);
  }
  static __device__ __forceinline__ void halo_products(const float (&w)[NH], bool, float (&p)[3]) {
    p[0] = w[3] * w[0];
    p[1] = w[4] * w[1];
    p[2] = w[5] * w[2];
  }
  template <class FX, class FY, class FZ>
  static __device__ __forceinline__ void gather(FX X, FY Y, FZ Z, float (&g)[NF]) {
    g[0] = gather_b(X(0));
    g[1] = gather_b(Y(1));
    g[2] = gather_b(Z(2));
    g[3] = gather_b(X(1)) + gather_b(Y(0));
    g[4] = gather_b(Z(0)) + gather_b(X(2));
    g[5] = gather_b(Z(1)) + gather_b(Y(2));
  }
};

// One half of a tile's chunk. Every input column is loaded once per plane by
// its owner, 5 planes ahead (plane y+5), so plane y's own cells reach the bands
// from registers. The halo cells, at most one per thread, are loaded with the
// own column's plane y+5 too, which is when the neighbouring tiles load them as
// theirs (so the second read is an L2 hit), and their products wait in a
// 5-plane ring in LDS that only the thread reads. All loads of a plane are
// issued while the plane before it is computed, and the bands are
// double-buffered (one barrier a plane, whose fences cover LDS only).
template <class H>
__device__ __forceinline__ void el3_march(const El3Args& a, int b, float* lds, float* ring) {
  const int bz = b % a.nbz;
  const int r = b / a.nbz;
  const int bx = r % a.nbx;
  const int yc = r / a.nbx;
  const int tz = a.tz, tx = a.tx;
  const int z0 = bz * tz, x0 = bx * tx, y0 = yc * a.ych;
  const int y1 = min(y0 + a.ych, a.ny);
  const int t = threadIdx.x;
  const int lx = t / tz, lz = t - lx * tz;
  const int gz = z0 + lz, gx = x0 + lx;
  const bool act = lx < tx;
  const bool own = act && gz < a.nz && gx < a.nx;
  // the own column's products are needed (as halo of valid cells) up to nz+5 /
  // nx+5; beyond that the padded array ends, and the lanes load its first cell,
  // whose products no valid cell reads (so nothing is masked)
  const bool ownp = act && gz < a.nz + EH && gx < a.nx + EH;
  const unsigned oo0 = ownp ? 4u * (unsigned)((gz + EH) + a.sx * (gx + EH)) : 0u;
  // halo cells: 10 columns of tz rows beside the tile (x-band), then 10 rows
  // above and below its tx columns (z-band)
  const int h2 = t - 2 * EH * tz;
  const bool hx = h2 < 0, hact = h2 < 2 * EH * tx;
  int hcol, hrow, hz, hc;
  if (hx) {
    const int c = t / tz;
    hcol = c < EH ? c : c + tx;
    hrow = t - c * tz;
    hz = z0 + hrow;
    hc = x0 - EH + hcol;
  } else {
    const int c = h2 / (2 * EH), rr = h2 - c * (2 * EH);
    hrow = rr < EH ? rr : rr + tz;
    hz = z0 - EH + hrow;
    hc = x0 + c;
    hcol = c + EX + 2 * EH;  // the z-band follows the x-band
  }
  const unsigned ho0 = hact && hz < a.nz + EH && hc < a.nx + EH ? 4u * (unsigned)((hz + EH) + a.sx * (hc + EH)) : 0u;
  const int hdst = hact ? hcol * EC + hrow : 0;
  const float* const hsp = H::split(a, hx);
  // waves without halo cells skip their loads (EHN is whole waves: every lane
  // of the others has a place in the ring)
  const bool halo_wave = __builtin_amdgcn_readfirstlane(t) < 2 * EH * (tz + tx);
  const int xo = (lx + EH) * EC + lz, zo = (EX + 2 * EH + lx) * EC + lz + EH;
  const long long sy = a.sy;
  auto plane = [&](int y) { return sy * (y + EH); };

  float q[3][11];                  // QUEUE products, slot j = plane y-5+j
  float keep[H::NK > 0 ? H::NK : 1][6];  // KEEP products, slot j = plane y+j
  // prime planes y0-5 .. y0+4 (the loop shifts the queue first)
#pragma unroll
  for (int j = 0; j < 10; ++j) {
    float w[H::NO], p[9];
    H::own(a, plane(y0 - 5 + j), opaque(oo0), w);
    H::products(w, p);
#pragma unroll
    for (int k = 0; k < 3; ++k) q[k][j + 1] = p[H::QUEUE[k]];
#pragma unroll
    for (int k = 0; k < H::NK; ++k)
      if (j >= 5) keep[k][j - 4] = p[H::KEEP[k]];
  }
  // halo products of planes y0 .. y0+4 into the ring
  if (halo_wave) {
#pragma unroll
    for (int j = 0; j < 5; ++j) {
      float h[H::NH], e[3];
      H::halo(a, hsp, plane(min(y0 + j, a.ny + EH - 1)), opaque(ho0), h);
      H::halo_products(h, hx, e);
#pragma unroll
      for (int k = 0; k < 3; ++k) ring[(j * 3 + k) * EHN + t] = e[k];
    }
  }
  float w[H::NO], h[H::NH];
  auto load_next = [&](int y) {
    H::own(a, plane(y + 5), opaque(oo0), w);
    if (halo_wave) H::halo(a, hsp, plane(y + 5), opaque(ho0), h);
  };
  load_next(y0);
  int slot = 0;  // (y - y0) % 5

  for (int y = y0; y < y1; ++y) {
    float* const bd = lds + ((y - y0) & 1) * EBAND;
    {
      float p[9], c[9];
      H::products(w, p);
#pragma unroll
      for (int k = 0; k < 3; ++k) {
#pragma unroll
        for (int j = 0; j < 10; ++j) q[k][j] = q[k][j + 1];
        q[k][10] = p[H::QUEUE[k]];
        c[H::QUEUE[k]] = q[k][5];
      }
#pragma unroll
      for (int k = 0; k < H::NK; ++k) {
#pragma unroll
        for (int j = 0; j < 5; ++j) keep[k][j] = keep[k][j + 1];
        keep[k][5] = p[H::KEEP[k]];
        c[H::KEEP[k]] = keep[k][0];
      }
      if (act) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          bd[xo + k * EP] = c[H::XB[k]];
          bd[zo + k * EP] = c[H::ZB[k]];
        }
      }
      if (halo_wave) {
        float e[3];
        H::halo_products(h, hx, e);
        float* const rg = ring + slot * 3 * EHN + t;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          if (hact) bd[hdst + k * EP] = rg[k * EHN];
          rg[k * EHN] = e[k];
        }
      }
      slot = slot == 4 ? 0 : slot + 1;
    }
    lds_barrier();
    // this plane's out and in1, added after the gathers, then the next plane's
    // operands
    const unsigned oo = opaque(oo0);
    float u[H::NF], v[H::NF], g[H::NF];
#pragma unroll
    for (int f = 0; f < H::NF; ++f) {
      u[f] = gl(a.out[H::OUT[f]] + plane(y), oo);
      v[f] = gl(a.in1[H::OUT[f]] + plane(y), oo);
    }
    load_next(y + 1 < y1 ? y + 1 : y);
    if (own) {
      H::gather([&](int k) { return [&, k](int d) { return bd[xo + d * EC + k * EP]; }; },
                [&](int k) { return [&, k](int d) { return q[k][5 + d]; }; },
                [&](int k) { return [&, k](int d) { return bd[zo + d + k * EP]; }; }, g);
#pragma unroll
      for (int f = 0; f < H::NF; ++f) gs(a.out[H::OUT[f]] + plane(y), oo, (u[f] + v[f]) + g[f]);
    }
  }
}

// Both halves in one launch, the two of a tile next to each other; 16 waves and
// 146 KB of LDS, one workgroup a CU. What bounds a step is the traffic beyond
// the L2 (171 + 37 B a cell against 168 algorithmic at 4.4 TB/s). Step at 200^3
// (us, algorithmic GB/s): 64 x 8 tiles of 8 waves for both halves at once, a
// plane's loads issued and awaited in that plane, 530 (2540; 267 + 39 B a
// cell); next plane's loads in flight, 768 threads for both halves, 451; halves
// apart, two workgroups of 512 threads a CU, 446; 1024 threads with the halo
// loaded at plane y+5, 376 (3580). 64^3: 18 us; 260^3: 830 us (3560).
__global__ __launch_bounds__(ENT) __attribute__((amdgpu_waves_per_eu(4))) void k_el3_adj(const El3Args a) {
  __shared__ float lds[2 * EBAND];
  __shared__ float ring[5 * 3 * EHN];
  const int b = a.xcd ? xcd_tile(blockIdx.x, 2 * a.nblk) : (int)blockIdx.x;
  if (b & 1)
    el3_march<Stress>(a, b >> 1, lds, ring);
  else
    el3_march<Velocity>(a, b >> 1, lds, ring);
}

// Workgroups resident at once: one per CU.
int el3_resident() {
  static const int n = [] {
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
      return 256;
    return cus;
  }();
  return n;
}

// Tile and planes per workgroup: the tiles along z as even as they come, as
// many columns as the workgroup's threads and LDS take (RTM_EL3_W fixes them),
// and the number of chunks along y (RTM_EL3_YCHUNK: their planes) that
// minimises rounds of resident workgroups x (planes + EPRIME); a chunk's first
// loads cost about that many planes.
constexpr int EPRIME = 8;
void el3_partition(El3Args& a) {
  const char* ws = std::getenv("RTM_EL3_W");
  const char* ys = std::getenv("RTM_EL3_YCHUNK");
  const int wfix = ws ? std::min(std::max(std::atoi(ws), 0), EX) : 0, yfix = ys ? std::atoi(ys) : 0;
  const int res = el3_resident();
  long long best = -1;
  const int nbz0 = (a.nz + EZ - 1) / EZ;
  for (int nbz = nbz0; nbz < nbz0 + 3 && nbz <= a.nz; ++nbz) {
    const int tz = (a.nz + nbz - 1) / nbz;
    int tx = std::min(wfix > 0 ? wfix : EX, std::min(ENT / tz, EHN / 10 - tz));
    const int nbx = (a.nx + tx - 1) / tx;
    if (wfix <= 0) tx = (a.nx + nbx - 1) / nbx;
    for (int chunks = 1; chunks <= a.ny; ++chunks) {
      const int ych = yfix > 0 ? std::min(yfix, a.ny) : (a.ny + chunks - 1) / chunks;
      const long long blocks = 2LL * nbz * nbx * ((a.ny + ych - 1) / ych);
      const long long cost = (blocks + res - 1) / res * (ych + EPRIME);
      if (best < 0 || cost < best) {
        best = cost;
        a.tz = tz; a.tx = tx; a.nbz = (a.nz + tz - 1) / tz; a.nbx = nbx; a.ych = ych;
      }
      if (yfix > 0) break;
    }
  }
  a.nblk = a.nbz * a.nbx * ((a.ny + a.ych - 1) / a.ych);
}

struct El3Timing {
  double ms = 0, launches = 0, cells = 0, ych = 0;
};
thread_local El3Timing g_el3_timing;

}  // namespace

// nsteps with the reference's rotation (K3/rtmlib-modC-gpu.cu:273-372):
// after a step that is not the last, (out, in, in1) <- (in1, out, in).
static int el3_steps(int ny, int nz, int nx, float* in[9], float* in1[9], float* out[9], const float* const m[6],
                     int nsteps, hipStream_t st) {
  if (ny < 1 || nz < 1 || nx < 1 || nsteps < 0) {
    set_error("elastic3d: grid %d x %d x %d or %d steps out of range", ny, nz, nx, nsteps);
    return E_ARG;
  }
  const long long n = (long long)(nz + 10) * (nx + 10) * (ny + 10);
  if (n >= (1LL << 31)) {
    set_error("elastic3d: %lld padded cells per field exceed 2^31", n);
    return E_ARG;
  }
  for (int f = 0; f < 9; ++f)
    if (!in[f] || !in1[f] || !out[f]) { set_error("elastic3d: null field pointer"); return E_ARG; }
  for (int k = 0; k < 6; ++k)
    if (!m[k]) { set_error("elastic3d: null coefficient pointer"); return E_ARG; }
  El3Args a{};
  a.ny = ny; a.nz = nz; a.nx = nx;
  a.sx = nz + 10;
  a.sy = (nz + 10) * (nx + 10);
  for (int k = 0; k < 6; ++k) a.m[k] = m[k];
  el3_partition(a);
  a.xcd = default_xcd();
  hipEvent_t e0, e1;
  HIPCHK(hipEventCreate(&e0));
  HIPCHK(hipEventCreate(&e1));
  struct EvGuard {
    hipEvent_t a, b;
    ~EvGuard() { (void)hipEventDestroy(a); (void)hipEventDestroy(b); }
  } eg{e0, e1};
  HIPCHK(hipEventRecord(e0, st));
  for (int s = 0; s < nsteps; ++s) {
    for (int f = 0; f < 9; ++f) {
      a.in[f] = in[f];
      a.in1[f] = in1[f];
      a.out[f] = out[f];
    }
    hipLaunchKernelGGL(k_el3_adj, dim3(2 * a.nblk), dim3(ENT), 0, st, a);
    HIPCHK(hipGetLastError());
    if (s < nsteps - 1) {
      for (int f = 0; f < 9; ++f) {
        float* t = out[f];
        out[f] = in1[f];
        in1[f] = in[f];
        in[f] = t;
      }
    }
  }
  HIPCHK(hipEventRecord(e1, st));
  HIPCHK(hipEventSynchronize(e1));
  float ms = 0;
  HIPCHK(hipEventElapsedTime(&ms, e0, e1));
  g_el3_timing.ms = ms;
  g_el3_timing.launches = nsteps;
  g_el3_timing.cells = (double)nz * nx * ny;
  g_el3_timing.ych = a.ych;
  return OK;
}

}  // namespace erm

using namespace erm;

RTM_EXPORT int rtm3d_adj_steps_dev(int ny, int nz, int nx, float* in[9], float* in1[9], float* out[9],
                                   const float* const coef[6], int nsteps) {
  if (!in || !in1 || !out || !coef) { set_error("elastic3d: null pointer array"); return E_ARG; }
  STCHK(ensure_device());
  return el3_steps(ny, nz, nx, in, in1, out, coef, nsteps, nullptr);
}

RTM_EXPORT int rtm3d_timings(double* out4) {
  if (!out4) { set_error("null argument"); return E_ARG; }
  out4[0] = g_el3_timing.ms;
  out4[1] = g_el3_timing.launches;
  out4[2] = g_el3_timing.cells;
  out4[3] = g_el3_timing.ych;
  return OK;
}

// --- the reference's host interface (K3/gpu.h:39-50) ------------------------
namespace {
struct El3Ctx {
  int ny = 0, nz = 0, nx = 0;
  size_t n = 0;
  DevBuf buf;  // 27 fields (in, in1, out) then 6 coefficients
};
std::mutex g_el3_mu;
El3Ctx* g_el3 = nullptr;
}  // namespace

RTM_EXPORT int rtm3d_gpu_init(int ny, int nz, int nx) {
  std::lock_guard<std::mutex> lk(g_el3_mu);
  if (ny < 1 || nz < 1 || nx < 1) { set_error("elastic3d: grid %d x %d x %d out of range", ny, nz, nx); return E_ARG; }
  STCHK(ensure_device());
  delete g_el3;
  g_el3 = new El3Ctx;
  g_el3->ny = ny; g_el3->nz = nz; g_el3->nx = nx;
  g_el3->n = (size_t)(nz + 10) * (nx + 10) * (ny + 10);
  const int s = g_el3->buf.alloc(33 * g_el3->n * sizeof(float), "3D elastic fields");
  if (s != OK) { delete g_el3; g_el3 = nullptr; }
  return s;
}

RTM_EXPORT int rtm3d_gpu_final(void) {
  std::lock_guard<std::mutex> lk(g_el3_mu);
  delete g_el3;
  g_el3 = nullptr;
  return OK;
}

// Copies the 27 fields and 6 coefficients in, runs one step (the reference's
// Steps_write_back = 1, K3/gpu.h:11), copies the 9 out fields back.
// gpu_kernel_time (may be null): seconds of copy-in, compute, copy-out.
RTM_EXPORT int rtm3d_gpu_func(int ny, int nz, int nx, float* Vy0_in, float* Vx0_in, float* Vz0_in, float* syy0_in,
                              float* sxx0_in, float* szz0_in, float* sxy0_in, float* sxz0_in, float* syz0_in,
                              float* Vy0_in1, float* Vx0_in1, float* Vz0_in1, float* syy0_in1, float* sxx0_in1,
                              float* szz0_in1, float* sxy0_in1, float* sxz0_in1, float* syz0_in1, float* Vy0_out,
                              float* Vx0_out, float* Vz0_out, float* syy0_out, float* sxx0_out, float* szz0_out,
                              float* sxy0_out, float* sxz0_out, float* syz0_out, float* m1_y, float* m1_x,
                              float* m1_z, float* m2, float* m3, float* m2m3, float* debug,
                              float* gpu_kernel_time) {
  (void)debug;
  std::lock_guard<std::mutex> lk(g_el3_mu);
  if (!g_el3) { set_error("elastic3d: rtm3d_gpu_init was not called"); return E_ARG; }
  if (g_el3->ny != ny || g_el3->nz != nz || g_el3->nx != nx) {
    set_error("elastic3d: grid %d x %d x %d differs from rtm3d_gpu_init's %d x %d x %d", ny, nz, nx, g_el3->ny,
              g_el3->nz, g_el3->nx);
    return E_ARG;
  }
  float* host[33] = {Vy0_in,  Vx0_in,  Vz0_in,  syy0_in,  sxx0_in,  szz0_in,  sxy0_in,  sxz0_in,  syz0_in,
                     Vy0_in1, Vx0_in1, Vz0_in1, syy0_in1, sxx0_in1, szz0_in1, sxy0_in1, sxz0_in1, syz0_in1,
                     Vy0_out, Vx0_out, Vz0_out, syy0_out, sxx0_out, szz0_out, sxy0_out, sxz0_out, syz0_out,
                     m1_y,    m1_x,    m1_z,    m2,       m3,       m2m3};
  for (float* p : host)
    if (!p) { set_error("elastic3d: null array argument"); return E_ARG; }
  const size_t n = g_el3->n;
  float* d = g_el3->buf.as<float>();
  hipEvent_t ev[4];
  for (auto& e : ev) HIPCHK(hipEventCreate(&e));
  struct EvGuard {
    hipEvent_t* e;
    ~EvGuard() { for (int i = 0; i < 4; ++i) (void)hipEventDestroy(e[i]); }
  } eg{ev};
  HIPCHK(hipEventRecord(ev[0], nullptr));
  for (int k = 0; k < 33; ++k)
    HIPCHK(hipMemcpyAsync(d + k * n, host[k], n * sizeof(float), hipMemcpyHostToDevice, nullptr));
  HIPCHK(hipEventRecord(ev[1], nullptr));
  float *in[9], *in1[9], *out[9];
  const float* m[6];
  for (int f = 0; f < 9; ++f) {
    in[f] = d + f * n;
    in1[f] = d + (9 + f) * n;
    out[f] = d + (18 + f) * n;
  }
  for (int k = 0; k < 6; ++k) m[k] = d + (27 + k) * n;
  STCHK(el3_steps(ny, nz, nx, in, in1, out, m, 1, nullptr));
  HIPCHK(hipEventRecord(ev[2], nullptr));
  for (int f = 0; f < 9; ++f)
    HIPCHK(hipMemcpyAsync(host[18 + f], out[f], n * sizeof(float), hipMemcpyDeviceToHost, nullptr));
  HIPCHK(hipEventRecord(ev[3], nullptr));
  HIPCHK(hipEventSynchronize(ev[3]));
  if (gpu_kernel_time) {
    for (int i = 0; i < 3; ++i) {
      float ms = 0;
      HIPCHK(hipEventElapsedTime(&ms, ev[i], ev[i + 1]));
      gpu_kernel_time[i] = ms / 1000.f;
    }
  }
  return OK;
}
