// elastic2d_device.hpp -- device helpers shared by the 2D elastic step kernels.
#pragma once

#include "elastic2d.hpp"

namespace erm {

// Staggered differences on an LDS tile; S is the element stride of the axis.
template <int S>
__device__ __forceinline__ float sp(const float* f, int p) {
  float r = C1 * (f[p + 5 * S] - f[p - 4 * S]);
  r = fmaf(C2, f[p + 4 * S] - f[p - 3 * S], r);
  r = fmaf(C3, f[p + 3 * S] - f[p - 2 * S], r);
  r = fmaf(C4, f[p + 2 * S] - f[p - S], r);
  r = fmaf(C5, f[p + S] - f[p], r);
  return r;
}
template <int S>
__device__ __forceinline__ float sm(const float* f, int p) {
  float r = C1 * (f[p + 4 * S] - f[p - 5 * S]);
  r = fmaf(C2, f[p + 3 * S] - f[p - 4 * S], r);
  r = fmaf(C3, f[p + 2 * S] - f[p - 3 * S], r);
  r = fmaf(C4, f[p + S] - f[p - 2 * S], r);
  r = fmaf(C5, f[p] - f[p - S], r);
  return r;
}

__device__ __forceinline__ void neumaier(float& s, float& c, float t) {
#pragma clang fp contract(off)
  const float u = s + t;
  if (fabsf(s) >= fabsf(t))
    c += (s - u) + t;
  else
    c += (t - u) + s;
  s = u;
}

// Global-memory accesses through address-space-1 pointers. The descriptor's
// pointers are generic; read through them the compiler emits FLAT
// instructions, which also count against the LDS wait counter, so waiting
// for an LDS read would wait for every global load in flight as well.
template <class T>
__device__ __forceinline__ T gld(const T* p, int i) {
  return ((const __attribute__((address_space(1))) T*)p)[i];
}
template <class T>
__device__ __forceinline__ void gst(T* p, int i, T v) {
  ((__attribute__((address_space(1))) T*)p)[i] = v;
}
template <class T>
__device__ __forceinline__ void gst_nt(T* p, int i, T v) {
  __builtin_nontemporal_store(v, (__attribute__((address_space(1))) T*)p + i);
}
// Load of an element whose index is the same in every lane, of an array no
// kernel writes while it runs: through the constant address space it is
// one scalar load into a scalar register (a divergent index would still be
// served correctly, by vector loads).
template <class T>
__device__ __forceinline__ T gldu(const T* p, int i) {
  return ((const __attribute__((address_space(4))) T*)p)[i];
}
// Masked load without a branch: lanes outside read element 0 (a valid
// address) and return zero.
template <class T>
__device__ __forceinline__ T gldm(const T* p, int i, bool in) {
  const T v = gld(p, in ? i : 0);
  return in ? v : T(0);
}

// Born scattering sources of one cell of level L (image_op2's forward branch,
// W/image-mod-rtm.f90:146-162) from the background Vx, Vz tiles hx, hz at LDS
// position p, the next level's Vx, Vz (next) and the perturbation d. Fused only
// where written, so that every caller rounds it the same way.
template <int SX, class Shot>
__device__ __forceinline__ void born_sources(const Shot& S, const float* hx, const float* hz, int p, int gz, int gx,
                                             bool has_next, const float (&next)[2], const float (&d)[3],
                                             float (&q)[5]) {
#pragma clang fp contract(off)
  const int nz = S.nz, nx = S.nx;
  float s1 = 0.f, s2 = 0.f, s4 = 0.f, s5 = 0.f, s6 = 0.f;
  if (has_next) {
    s1 = S.inv_dt * (next[0] - hx[p]);
    s2 = S.inv_dt * (next[1] - hz[p]);
  }
  if (gz >= 4 && gz <= nz - 6 && gx >= 4 && gx <= nx - 6) {
    s4 = sp<SX>(hx, p) * S.inv_dx;
    s5 = sp<1>(hz, p) * S.inv_dx;
  }
  if (gz >= 5 && gz <= nz - 6 && gx >= 5 && gx <= nx - 6) {
    s6 = sm<1>(hx, p) * S.inv_dx;
    s6 = fmaf(sm<SX>(hz, p), S.inv_dx, s6);
  }
  const float s3 = s4 + s5;
  q[0] = d[0] * s1;
  q[1] = d[0] * s2;
  q[2] = fmaf(-(d[2] * 2.f), s4, -(d[1] * s3));
  q[3] = fmaf(-(d[2] * 2.f), s5, -(d[1] * s3));
  q[4] = -(d[2] * s6);
}

}  // namespace erm
