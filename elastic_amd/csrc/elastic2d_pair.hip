// elastic2d_pair.hip -- two levels of the 2D elastic step in one launch, for
// one shot on a grid too small to fill the GPU.
//
// On such a grid a one-level launch is a chain of latencies, not of bytes or
// arithmetic: dispatch and the end of the kernel (about 2 us), one memory
// latency for the operands, the stencils of one wave, the stores. Two levels
// in one launch pay that chain once. A workgroup owns a TZ x TX tile; its
// threads stage level L-1 with a radius-10 halo, compute level L on the tile
// plus a radius-5 halo -- one cell per thread, so that what a thread loaded for
// its cell (coefficients, sponge factors) stays in registers for the second
// level -- pass it through LDS, and compute level L+1 on the tile. Everything
// the first loads depend on is a kernel argument held in scalar registers from
// the dispatch on; there is no descriptor or tile table to wait for.
//
// us a level, one level a launch -> two, forward / adjoint: 64 x 64 3.65 / 5.62
// -> 1.98 / 3.24, 150 x 300 3.89 / 5.81 -> 2.62 / 4.13, 300 x 300 4.10 / 6.19 ->
// 3.28 / 5.18, 330 x 420 5.25 / 8.05 -> 3.89 / 6.04, forward of 390 x 690 6.62 ->
// 5.72. What bounds it now is a CU's LDS reads and vector instructions (a
// workgroup more than doubles the cells of its tile), hence the choice of the
// tile by waves per CU in pair_tile(). Two columns per thread share a fifth of
// the LDS reads, but halve the waves: slower (300 x 300: 3.55 / 5.86).
//
// Every cell of both levels gets exactly the arithmetic of k_fwd / k_adj, so
// results are bitwise those of two one-level launches.
#include "buffer.hpp"
#include "elastic2d_device.hpp"

#include <cstdlib>

namespace erm {

namespace {

// What a launch needs of its shot beyond the scalar arguments; read while the
// operands are in flight.
struct PairArgs {
  int nz, nx, nt;
  int zs, xs, zr, rx0, nrx;
  float amp0, amp1;  // source terms of the first and the second level
  float inv_dx, inv_dt, img_w;
  int k0, k1;        // fp32 snapshots: the one a step belongs to
  float* rec;
  float* snap;
  float* img;
  float* imgc;
  const float* dm;
};

// OCC: waves a SIMD is to hold (512 / OCC registers; Born modelling would spill).
template <int TZ_, int TX_, int NT_, int CX_, int OCC_>
struct PairTile {
  static constexpr int TZ = TZ_, TX = TX_, H = 5, NT = NT_, CX = CX_, OCC = OCC_;
  static constexpr int LZ1 = TZ + 4 * H, N1 = LZ1 * (TX + 4 * H);           // the level read
  static constexpr int LZ0 = TZ + 2 * H, LX0 = TX + 2 * H, N0 = LZ0 * LX0;  // the first level computed
  static constexpr int NIT = (N1 + NT - 1) / NT;
  static_assert(LX0 % CX == 0 && N0 <= NT * CX, "CX cells of the first level per thread");
};
using PairS = PairTile<22, 6, 512, 1, 6>;
using PairM = PairTile<22, 14, 768, 1, 6>;
using PairL = PairTile<22, 22, 1024, 1, 4>;
using PairX = PairTile<54, 22, 1024, 2, 4>;

// launch flags beside F_* and A_*
constexpr int P_XCD = 1 << 20;   // XCD-aware tile numbering
constexpr int P_HIST = 1 << 21;  // fp32 history of every level (SNAP_HIST): write / image both levels

// The cells of a thread: CX columns of one row of the tile and its halo.
template <class T>
struct PairCells {
  static constexpr int CX = T::CX;
  int z0, x0, tid, lz, lx, gz, gx;  // of the first cell (a thread without cells: the last ones)
  unsigned gi[CX];       // byte offset of a cell in a field (kOutside: none)
  bool in[CX], own[CX];  // a cell is in the grid; and belongs to the tile
  bool any, some;        // the thread has cells; and some of the tile

  __device__ __forceinline__ PairCells(int nz, int nx, int ldz, int ntiles, int nbz, int flags) {
    const int b = (flags & P_XCD) ? xcd_tile(blockIdx.x, ntiles) : (int)blockIdx.x;
    const int bx = b / nbz;
    z0 = (b - bx * nbz) * T::TZ;
    x0 = bx * T::TX;
    tid = threadIdx.x;
    any = tid < T::N0 / CX;
    const int c = any ? tid : T::N0 / CX - 1;
    lx = c / T::LZ0;
    lz = c - lx * T::LZ0;
    lx *= CX;
    gx = x0 - T::H + lx;
    gz = z0 - T::H + lz;
    some = false;
#pragma unroll
    for (int i = 0; i < CX; ++i) {
      in[i] = any && gx + i >= 0 && gx + i < nx && gz >= 0 && gz < nz;
      own[i] = in[i] && lx + i >= T::H && lx + i < T::H + T::TX && lz >= T::H && lz < T::H + T::TZ;
      gi[i] = in[i] ? 4u * (unsigned)(gz + ldz * (gx + i)) : kOutside;
      some |= own[i];
    }
  }
  __device__ __forceinline__ int p1(int i) const { return (lx + i + T::H) * T::LZ1 + lz + T::H; }
  __device__ __forceinline__ int p0(int i) const { return (lx + i) * T::LZ0 + lz; }
};

// Staged cell k of this thread: byte offset (kOutside: none).
template <class T>
__device__ __forceinline__ unsigned staged(const PairCells<T>& pc, int k, int nz, int nx, int ldz) {
  const int c = pc.tid + T::NT * k;
  const int lx = c / T::LZ1, lz = c - lx * T::LZ1;
  const int gx = pc.x0 - 2 * T::H + lx, gz = pc.z0 - 2 * T::H + lz;
  const bool in = c < T::N1 && gx >= 0 && gx < nx && gz >= 0 && gz < nz;
  return in ? 4u * (unsigned)(gz + ldz * gx) : kOutside;
}

// One forward cell-update: v holds the level before the last (plus Born
// sources), the differences are those of the level in h at position p.
template <int SX>
__device__ __forceinline__ void fwd_cell(const float* h, int n, int p, const float (&m)[5], bool src, float amp,
                                         float kz, float kx, float (&v)[5]) {
  const float *vx = h, *vz = h + n, *xx = h + 2 * n, *zz = h + 3 * n, *xz = h + 4 * n;
  v[0] = fmaf(m[0], sm<SX>(xx, p), v[0]);
  v[0] = fmaf(m[0], sp<1>(xz, p), v[0]);
  v[1] = fmaf(m[1], sp<SX>(xz, p), v[1]);
  v[1] = fmaf(m[1], sm<1>(zz, p), v[1]);
  v[2] = src ? v[2] + amp : v[2];
  v[3] = src ? v[3] + amp : v[3];
  const float dx = sp<SX>(vx, p), dz = sp<1>(vz, p);
  v[2] = fmaf(m[4], dx, v[2]);
  v[2] = fmaf(m[2], dz, v[2]);
  v[3] = fmaf(m[2], dx, v[3]);
  v[3] = fmaf(m[4], dz, v[3]);
  v[4] = fmaf(m[3], sm<1>(vx, p), v[4]);
  v[4] = fmaf(m[3], sm<SX>(vz, p), v[4]);
#pragma unroll
  for (int f = 0; f < 5; ++f) v[f] = (v[f] * kz) * kx;  // factors of one without a sponge
}

__device__ __forceinline__ void record(const PairArgs& a, int L, int gx, int flags, const float (&v)[5]) {
  float* r = a.rec + (long long)(L - 1) * a.nrx + (gx - a.rx0);
  const long long rs = (long long)a.nt * a.nrx;
#pragma unroll
  for (int f = 0; f < 5; ++f) {
    if (flags & F_RECSUB)
      gst(r + f * rs, 0, gld(r + f * rs, 0) - v[f]);
    else
      gst(r + f * rs, 0, v[f]);
  }
}

// Levels L and L+1. lev: the four-level ring (level l in slot l & 3), kfac:
// sponge factors of the rows, then of the columns.
template <class T, bool BORN>
__global__ __launch_bounds__(T::NT, BORN ? 4 : T::OCC) void k_fwd_pair(float* lev, const float* coef, const float* kfac, int nz, int nx,
                                                    int ntiles, int nbz, int L, int flags, PairArgs a) {
  constexpr int CX = T::CX;
  // a thread whose first or last cell lies beside the tile reads one column
  // more than the halo at the second level: s0 has room on both sides
  __shared__ struct {
    float s1[(BORN ? 7 : 5) * T::N1];  // level L-1 (and the background of level L)
    float s0[(BORN ? 7 : 5) * T::N0];  // level L (and the background of level L+1)
    float room[CX * T::LZ0];
  } lds;
  float *const s1 = lds.s1, *const s0 = lds.s0;
  const int ldz = (nz + 31) / 32 * 32, n2 = ldz * nx;
  const unsigned fs = 4u * n2;  // bytes of a field
  const Buf x2(lev + ((L + 2) & 3) * 5 * n2, 5 * fs), y1(lev + ((L + 3) & 3) * 5 * n2, 5 * fs);
  const Buf out0(lev + (L & 3) * 5 * n2, 5 * fs), out1(lev + ((L + 1) & 3) * 5 * n2, 5 * fs);
  const Buf co(coef, 5 * fs), ks(kfac, 4u * (nz + nx));
  const PairCells<T> k(nz, nx, ldz, ntiles, nbz, flags);

  float st[T::NIT][5], bs[BORN ? T::NIT : 1][2];
  // Born: background Vx, Vz of levels L, L+1 and L+2 (past the last one: zero)
  const bool has2 = BORN && L + 2 <= a.nt;
  const Buf bg(a.snap + (long long)(L - 1) * 2 * n2, BORN ? (has2 ? 6 : 4) * fs : 0);
#pragma unroll
  for (int j = 0; j < T::NIT; ++j) {
    const unsigned gi = staged<T>(k, j, nz, nx, ldz);
#pragma unroll
    for (int f = 0; f < 5; ++f) st[j][f] = y1.get(gi, f * fs);
    if (BORN) {
#pragma unroll
      for (int f = 0; f < 2; ++f) bs[j][f] = bg.get(gi, f * fs);
    }
  }
  float v[CX][5], m[CX][5], kx[CX], b1[CX][2], b2[CX][2], d[CX][3];
  const bool sponge = flags & F_K;
  const float kz = sponge ? ks.get(4u * k.gz, 0) : 1.f;
  const Buf dm(a.dm, BORN ? 3 * fs : 0);
#pragma unroll
  for (int i = 0; i < CX; ++i) {
    kx[i] = sponge ? ks.get(4u * (k.gx + i), 4u * nz) : 1.f;
#pragma unroll
    for (int f = 0; f < 5; ++f) {
      v[i][f] = x2.get(k.gi[i], f * fs);
      m[i][f] = co.get(k.gi[i], f * fs);
    }
    if (BORN) {
#pragma unroll
      for (int f = 0; f < 2; ++f) {
        b1[i][f] = bg.get(k.gi[i], (2 + f) * fs);
        b2[i][f] = bg.get(k.gi[i], (4 + f) * fs);
      }
#pragma unroll
      for (int f = 0; f < 3; ++f) d[i][f] = dm.get(k.gi[i], f * fs);
    }
  }
#pragma unroll
  for (int j = 0; j < T::NIT; ++j) {
    const int c = k.tid + T::NT * j;
    if (c < T::N1) {
#pragma unroll
      for (int f = 0; f < 5; ++f) s1[f * T::N1 + c] = st[j][f];
      if (BORN) {
#pragma unroll
        for (int f = 0; f < 2; ++f) s1[(5 + f) * T::N1 + c] = bs[j][f];
      }
    }
  }
  __syncthreads();

  float y[CX][5];  // the own cells of level L-1
  bool src[CX], receiver[CX];
#pragma unroll
  for (int i = 0; i < CX; ++i) {
    const int p = k.p1(i), gx = k.gx + i;
    src[i] = (flags & F_SRC) && k.gz == a.zs && gx == a.xs;
    receiver[i] = (flags & (F_REC | F_RECSUB)) && k.own[i] && k.gz == a.zr && gx >= a.rx0 && gx < a.rx0 + a.nrx;
#pragma unroll
    for (int f = 0; f < 5; ++f) y[i][f] = s1[f * T::N1 + p];
    if (BORN) {
      float q[5];
      born_sources<T::LZ1>(a, s1 + (BORN ? 5 : 0) * T::N1, s1 + (BORN ? 6 : 0) * T::N1, p, k.gz, gx, true, b1[i], d[i], q);
#pragma unroll
      for (int f = 0; f < 5; ++f) v[i][f] = q[f] + v[i][f];
    }
    fwd_cell<T::LZ1>(s1, T::N1, p, m[i], src[i], a.amp0, kz, kx[i], v[i]);
  }
  if (k.any) {
#pragma unroll
    for (int i = 0; i < CX; ++i) {
#pragma unroll
      for (int f = 0; f < 5; ++f) s0[f * T::N0 + k.p0(i)] = k.in[i] ? v[i][f] : 0.f;
      if (BORN) {
#pragma unroll
        for (int f = 0; f < 2; ++f) s0[(5 + f) * T::N0 + k.p0(i)] = b1[i][f];
      }
    }
  }
  unsigned go[CX];  // the cells to store: those of the tile
#pragma unroll
  for (int i = 0; i < CX; ++i) {
    go[i] = k.own[i] ? k.gi[i] : kOutside;
#pragma unroll
    for (int f = 0; f < 5; ++f) out0.put(go[i], f * fs, v[i][f]);
  }
  __syncthreads();
  if (!k.some) return;

  float w[CX][5];
#pragma unroll
  for (int i = 0; i < CX; ++i) {
    const int p = k.p0(i);
#pragma unroll
    for (int f = 0; f < 5; ++f) w[i][f] = y[i][f];
    if (BORN) {
      float q[5];
      born_sources<T::LZ0>(a, s0 + (BORN ? 5 : 0) * T::N0, s0 + (BORN ? 6 : 0) * T::N0, p, k.gz, k.gx + i, has2, b2[i], d[i],
                           q);
#pragma unroll
      for (int f = 0; f < 5; ++f) w[i][f] = q[f] + w[i][f];
    }
    fwd_cell<T::LZ0>(s0, T::N0, p, m[i], src[i], a.amp1, kz, kx[i], w[i]);
  }
#pragma unroll
  for (int i = 0; i < CX; ++i) {
#pragma unroll
    for (int f = 0; f < 5; ++f) out1.put(go[i], f * fs, w[i][f]);
    if (receiver[i]) {
      record(a, L, k.gx + i, flags, v[i]);
      record(a, L + 1, k.gx + i, flags, w[i]);
    }
    if (flags & P_HIST) {
      const Buf h(a.snap + (long long)(L - 1) * 2 * n2, 4 * fs);
#pragma unroll
      for (int f = 0; f < 2; ++f) {
        h.put(go[i], f * fs, v[i][f]);
        h.put(go[i], (2 + f) * fs, w[i][f]);
      }
    }
    if (flags & F_SNAP) {  // of level L-1
      const Buf h(a.snap + (long long)a.k0 * 4 * n2, 4 * fs);
#pragma unroll
      for (int f = 0; f < 2; ++f) {
        h.put(go[i], f * fs, y[i][f]);
        h.put(go[i], (2 + f) * fs, v[i][f] - y[i][f]);
      }
    }
    if (flags & F_SNAP2) {  // of level L
      const Buf h(a.snap + (long long)a.k1 * 4 * n2, 4 * fs);
#pragma unroll
      for (int f = 0; f < 2; ++f) {
        h.put(go[i], f * fs, v[i][f]);
        h.put(go[i], (2 + f) * fs, w[i][f] - v[i][f]);
      }
    }
  }
}

// Products of the adjoint stencils at one cell.
__device__ __forceinline__ void adj_products(const float (&y)[5], const float (&m)[5], float (&q)[5]) {
  q[0] = fmaf(m[4], y[2], m[2] * y[3]);
  q[1] = fmaf(m[2], y[2], m[4] * y[3]);
  q[2] = m[3] * y[4];
  q[3] = m[0] * y[0];
  q[4] = m[1] * y[1];
}

// One adjoint cell-update: b holds the level after the next (plus the receiver
// row), h the products of the next level (stride n per product) at p.
template <int SX>
__device__ __forceinline__ void adj_cell(const float* h, int n, int p, float kz, float kx,
                                         const float (&b)[5], float (&v)[5]) {
  v[0] = b[0] - sm<SX>(h, p);
  v[0] -= sp<1>(h + 2 * n, p);
  v[1] = b[1] - sm<1>(h + n, p);
  v[1] -= sp<SX>(h + 2 * n, p);
  v[2] = b[2] - sp<SX>(h + 3 * n, p);
  v[3] = b[3] - sp<1>(h + 4 * n, p);
  v[4] = b[4] - sm<1>(h + 3 * n, p);
  v[4] -= sm<SX>(h + 4 * n, p);
#pragma unroll
  for (int f = 0; f < 5; ++f) v[f] = (v[f] * kz) * kx;  // factors of one without a sponge
}

// Imaging terms of one cell: adjoint fields v, source Vx, Vz in sx, sz at p and
// S1, S2 (image-mod-rtm.f90:154-162). Fused only where written, as in k_adj.
template <int SX>
__device__ __forceinline__ void image_terms(const PairArgs& a, const float* sx, const float* sz, int p, int gz, int gx,
                                            float s1, float s2, const float (&v)[5], float (&t)[3]) {
#pragma clang fp contract(off)
  const bool in4 = gz >= 4 && gz <= a.nz - 6 && gx >= 4 && gx <= a.nx - 6, in5 = in4 && gz >= 5 && gx >= 5;
  const float s4 = in4 ? sp<SX>(sx, p) * a.inv_dx : 0.f;
  const float s5 = in4 ? sp<1>(sz, p) * a.inv_dx : 0.f;
  float s6 = sm<1>(sx, p) * a.inv_dx;
  s6 = in5 ? fmaf(sm<SX>(sz, p), a.inv_dx, s6) : 0.f;
  const float s3 = s4 + s5;
  t[0] = a.img_w * fmaf(v[0], s1, v[1] * s2);
  t[1] = -a.img_w * fmaf(v[2], s3, v[3] * s3);
  t[2] = -a.img_w * fmaf(v[4], s6, fmaf(v[3] * 2.f, s5, v[2] * 2.f * s4));
}

// Levels L and L-1 of the adjoint, from L+1 and L+2, with the imaging of
// either (A_IMG: level L, A_IMG2: level L-1); an image is read and written once
// for both. Layout of snap: with P_HIST Vx, Vz of every level, else Vx, Vz, dVx,
// dVz of the imaged level (one of the two at most).
template <class T>
__global__ __launch_bounds__(T::NT, T::OCC) void k_adj_pair(float* lev, const float* coef, const float* kfac, int nz, int nx,
                                                    int ntiles, int nbz, int L, int flags, PairArgs a) {
  constexpr int H = T::H, CX = T::CX;
  __shared__ struct {  // room on both sides of s0 and sv, see k_fwd_pair
    float s1[5 * T::N1];  // products of level L+1
    float s0[5 * T::N0];  // products of level L
    float sv[4 * T::N0];  // source Vx, Vz of levels L and L-1
    float room[CX * T::LZ0];
  } lds;
  float *const s1 = lds.s1, *const s0 = lds.s0, *const sv = lds.sv;
  const int ldz = (nz + 31) / 32 * 32, n2 = ldz * nx;
  const unsigned fs = 4u * n2;  // bytes of a field
  const Buf x2(lev + ((L + 2) & 3) * 5 * n2, 5 * fs), y1(lev + ((L + 1) & 3) * 5 * n2, 5 * fs);
  const Buf out0(lev + (L & 3) * 5 * n2, 5 * fs), out1(lev + ((L + 3) & 3) * 5 * n2, 5 * fs);
  const Buf co(coef, 5 * fs), ks(kfac, 4u * (nz + nx));
  const PairCells<T> k(nz, nx, ldz, ntiles, nbz, flags);

  float st[T::NIT][5];
#pragma unroll
  for (int j = 0; j < T::NIT; ++j) {
    const unsigned gi = staged<T>(k, j, nz, nx, ldz);
    float y[5], m[5];
#pragma unroll
    for (int f = 0; f < 5; ++f) {
      y[f] = y1.get(gi, f * fs);
      m[f] = co.get(gi, f * fs);
    }
    adj_products(y, m, st[j]);  // zero outside
  }
  float b[CX][5], m[CX][5], y[CX][5], kx[CX];
  const bool sponge = flags & A_K;
  const float kz = sponge ? ks.get(4u * k.gz, 0) : 1.f;
#pragma unroll
  for (int i = 0; i < CX; ++i) {
    kx[i] = sponge ? ks.get(4u * (k.gx + i), 4u * nz) : 1.f;
#pragma unroll
    for (int f = 0; f < 5; ++f) {
      b[i][f] = x2.get(k.gi[i], f * fs);
      m[i][f] = co.get(k.gi[i], f * fs);
      y[i][f] = y1.get(k.gi[i], f * fs);
    }
  }
  // imaging operands: source Vx, Vz of level L (g0) and L-1 (g1), of level L+1
  // or the differences at the own cells (gn), the images
  const bool hist = flags & P_HIST, imaging = flags & (A_IMG | A_IMG2), next = flags & A_NEXT;
  const Buf img(a.img, 3 * fs), imgc(a.imgc, (flags & A_COMP) ? 3 * fs : 0);
  float g0[CX][2], g1[CX][2], gn[CX][2], im[CX][3], imc[CX][3];
  if (imaging) {
    // history: levels L-1, L and L+1 (past the last one: zero); else the
    // snapshot serves whichever level is imaged
    const Buf h(hist ? a.snap + (long long)(L - 2) * 2 * n2 : a.snap + (long long)a.k0 * 4 * n2, (hist && next ? 6 : 4) * fs);
#pragma unroll
    for (int i = 0; i < CX; ++i) {
#pragma unroll
      for (int f = 0; f < 2; ++f) {
        g1[i][f] = h.get(k.gi[i], f * fs);
        g0[i][f] = h.get(k.gi[i], hist ? (2 + f) * fs : f * fs);
        gn[i][f] = h.get(k.gi[i], (hist ? 4 + f : 2 + f) * fs);
      }
#pragma unroll
      for (int f = 0; f < 3; ++f) {
        im[i][f] = img.get(k.gi[i], f * fs);
        imc[i][f] = imgc.get(k.gi[i], f * fs);
      }
    }
  }
  // receiver rows of both levels
  bool receiver[CX];
  float r0[CX][5], r1[CX][5];
  const bool tile_row = (flags & A_INJ) && a.zr >= k.z0 - H && a.zr < k.z0 + T::TZ + H;
#pragma unroll
  for (int i = 0; i < CX; ++i) {
    const int gx = k.gx + i;
    receiver[i] = tile_row && k.in[i] && k.gz == a.zr && gx >= a.rx0 && gx < a.rx0 + a.nrx;
    if (tile_row) {
      const float* r = a.rec + (long long)(L - 2) * a.nrx + (receiver[i] ? gx - a.rx0 : 0);
      const long long rs = (long long)a.nt * a.nrx;
#pragma unroll
      for (int f = 0; f < 5; ++f) {
        r0[i][f] = gld(r + f * rs, receiver[i] ? a.nrx : 0);
        r1[i][f] = gld(r + f * rs, 0);
      }
    }
  }
#pragma unroll
  for (int j = 0; j < T::NIT; ++j) {
    const int c = k.tid + T::NT * j;
    if (c < T::N1) {
#pragma unroll
      for (int f = 0; f < 5; ++f) s1[f * T::N1 + c] = st[j][f];
    }
  }
  if (imaging && k.any) {
#pragma unroll
    for (int i = 0; i < CX; ++i)
#pragma unroll
      for (int f = 0; f < 2; ++f) {
        sv[f * T::N0 + k.p0(i)] = g0[i][f];
        sv[(2 + f) * T::N0 + k.p0(i)] = g1[i][f];
      }
  }
  __syncthreads();

  if (tile_row) {
#pragma unroll
    for (int i = 0; i < CX; ++i)
#pragma unroll
      for (int f = 0; f < 5; ++f) b[i][f] = receiver[i] ? r0[i][f] + b[i][f] : b[i][f];
  }
  float v[CX][5];
#pragma unroll
  for (int i = 0; i < CX; ++i) adj_cell<T::LZ1>(s1, T::N1, k.p1(i), kz, kx[i], b[i], v[i]);
  if (k.any) {
#pragma unroll
    for (int i = 0; i < CX; ++i) {
      float q[5];
      adj_products(v[i], m[i], q);
#pragma unroll
      for (int f = 0; f < 5; ++f) s0[f * T::N0 + k.p0(i)] = k.in[i] ? q[f] : 0.f;
    }
  }
  unsigned go[CX];  // the cells to store: those of the tile
#pragma unroll
  for (int i = 0; i < CX; ++i) {
    go[i] = k.own[i] ? k.gi[i] : kOutside;
#pragma unroll
    for (int f = 0; f < 5; ++f) out0.put(go[i], f * fs, v[i][f]);
  }
  __syncthreads();
  if (!k.some) return;

  if (tile_row) {
#pragma unroll
    for (int i = 0; i < CX; ++i)
#pragma unroll
      for (int f = 0; f < 5; ++f) y[i][f] = receiver[i] ? r1[i][f] + y[i][f] : y[i][f];
  }
  float w[CX][5];
#pragma unroll
  for (int i = 0; i < CX; ++i) adj_cell<T::LZ0>(s0, T::N0, k.p0(i), kz, kx[i], y[i], w[i]);
#pragma unroll
  for (int i = 0; i < CX; ++i)
#pragma unroll
    for (int f = 0; f < 5; ++f) out1.put(go[i], f * fs, w[i][f]);
  if (!imaging) return;

  // level L, then level L-1; d: forward time differences
  auto add = [&](int i, const float* src, float d1, float d2, const float (&u)[5]) {
    float t[3];
    image_terms<T::LZ0>(a, src, src + T::N0, k.p0(i), k.gz, k.gx + i, d1, d2, u, t);
#pragma unroll
    for (int f = 0; f < 3; ++f) {
      if (flags & A_COMP)
        neumaier(im[i][f], imc[i][f], t[f]);
      else
        im[i][f] = im[i][f] + t[f];
    }
  };
  if (flags & A_IMG) {
#pragma unroll
    for (int i = 0; i < CX; ++i) {
      const float d1 = a.inv_dt * (hist ? gn[i][0] - g0[i][0] : gn[i][0]);
      const float d2 = a.inv_dt * (hist ? gn[i][1] - g0[i][1] : gn[i][1]);
      add(i, sv, next ? d1 : 0.f, next ? d2 : 0.f, v[i]);
    }
  }
  if (flags & A_IMG2) {
#pragma unroll
    for (int i = 0; i < CX; ++i)
      add(i, sv + 2 * T::N0, a.inv_dt * (hist ? g0[i][0] - g1[i][0] : gn[i][0]),
          a.inv_dt * (hist ? g0[i][1] - g1[i][1] : gn[i][1]), w[i]);
  }
#pragma unroll
  for (int i = 0; i < CX; ++i)
#pragma unroll
    for (int f = 0; f < 3; ++f) {
      img.put(go[i], f * fs, im[i][f]);
      if (flags & A_COMP) imgc.put(go[i], f * fs, imc[i][f]);
    }
}

PairArgs pair_args(const ShotDev& s) {
  PairArgs a{};
  a.nz = s.nz; a.nx = s.nx; a.nt = s.nt;
  a.zs = s.zs; a.xs = s.xs; a.zr = s.zr; a.rx0 = s.rx0; a.nrx = s.nrx;
  a.inv_dx = s.inv_dx; a.inv_dt = s.inv_dt; a.img_w = s.img_w;
  a.rec = s.rec; a.snap = static_cast<float*>(s.snap); a.img = s.img; a.imgc = s.imgc; a.dm = s.dm;
  return a;
}

// The kernels take the ring, the sponge factors and the stride as the engine
// lays them out.
int check_layout(const ShotDev& s) {
  if (s.lev_mod != 4 || s.lev_off % 4 != 0 || s.lev_stride != 5 * s.n2 || s.fstride != s.n2 || s.ldz != device_ldz(s.nz) ||
      s.n2 != (long long)s.ldz * s.nx || s.n2 > kPairCells || (s.kz && s.kx != s.kz + s.nz)) {
    set_error("two-level step: unexpected layout of the shot");
    return E_ARG;
  }
  return OK;
}

template <class T>
struct Grid {
  int nbz, n;
  explicit Grid(const ShotDev& s) : nbz((s.nz + T::TZ - 1) / T::TZ), n(nbz * ((s.nx + T::TX - 1) / T::TX)) {}
};

template <class T, bool BORN>
int fwd_pair(const ShotDev& s, const PairArgs& a, int L, int flags, hipStream_t st) {
  const Grid<T> g(s);
  hipLaunchKernelGGL((k_fwd_pair<T, BORN>), dim3(g.n), dim3(T::NT), 0, st, s.lev, s.coef, s.kz, s.nz, s.nx, g.n, g.nbz, L,
                     flags, a);
  HIPCHK(hipGetLastError());
  return OK;
}

template <class T>
int adj_pair(const ShotDev& s, const PairArgs& a, int L, int flags, hipStream_t st) {
  const Grid<T> g(s);
  hipLaunchKernelGGL(k_adj_pair<T>, dim3(g.n), dim3(T::NT), 0, st, s.lev, s.coef, s.kz, s.nz, s.nx, g.n, g.nbz, L, flags,
                     a);
  HIPCHK(hipGetLastError());
  return OK;
}

// RTM_PAIR (tests, experiments): 0 one level a launch, 1 to 4 the S, M, L or X
// tile whatever the grid.
int pair_forced() {
  const char* e = getenv("RTM_PAIR");
  const int v = e ? atoi(e) : -1;
  return v <= PAIR_X ? v : -1;
}

}  // namespace

// The tile of a launch. A CU that holds w waves of the S, M or L tile takes
// about 2.8 + 0.19 w us for two forward levels (measured: 4.2 us at w = 8, 5.1
// at 12, 5.9 at 16, 7.2 to 7.6 at 24, 9.0 to 9.7 at 32) and 4.0 + 0.31 w for two
// adjoint levels (6.5, 7.6, 9.0, 11.8, 15.3), so the tile is the one with the
// fewest waves on the busiest CU. Two one-level launches take 8.2 and 12.3 us at
// 300 x 300 (w = 16: 6.5 and 10.3), 11.1 and 17.0 at 390 x 500 (w = 32: 9.7 and
// 15.3) and 13.2 and 21.3 at 390 x 690 (w = 48: 13.0 and 22.0): up to w = 36 two
// levels a launch are faster. Above that the forward still gains with the X tile
// where its tiles fit one round (390 x 690: 11.4 us); its halo is smaller against
// the tile, and each thread computes two columns.
int pair_tile(int nz, int nx, bool forward, bool born) {
  const int forced = pair_forced();
  if (forced >= 0) return forced == PAIR_X && (!forward || born) ? PAIR_L : forced;
  const int cus = device_cus();
  if (cus <= 0 || (long long)device_ldz(nz) * nx > kPairCells) return PAIR_ONE;
  auto waves = [&](int tz, int tx, int w) {
    const long long n = (long long)((nz + tz - 1) / tz) * ((nx + tx - 1) / tx);
    return (n + cus - 1) / cus * w;
  };
  const long long w[3] = {waves(PairS::TZ, PairS::TX, PairS::NT / 64), waves(PairM::TZ, PairM::TX, PairM::NT / 64),
                          waves(PairL::TZ, PairL::TX, PairL::NT / 64)};
  const int best = w[0] <= w[1] && w[0] <= w[2] ? 0 : w[1] <= w[2] ? 1 : 2;
  if (w[best] <= 36) return PAIR_S + best;
  if (forward && !born && waves(PairX::TZ, PairX::TX, 1) == 1) return PAIR_X;
  return PAIR_ONE;
}

int launch_fwd_pair(const ShotDev& s, int tile, int L, int flags, float amp0, float amp1, int xcd, hipStream_t st) {
  STCHK(check_layout(s));
  PairArgs a = pair_args(s);
  a.amp0 = amp0;
  a.amp1 = amp1;
  if (s.snap_fmt == SNAP_HIST && (flags & F_SNAP)) flags = (flags & ~F_SNAP) | P_HIST;
  a.k0 = (L - 1) / s.snap_every - 1;
  a.k1 = L / s.snap_every - 1;
  if (xcd) flags |= P_XCD;
  const bool born = flags & F_BORN;
  switch (tile) {
    case PAIR_S: return born ? fwd_pair<PairS, true>(s, a, L, flags, st) : fwd_pair<PairS, false>(s, a, L, flags, st);
    case PAIR_M: return born ? fwd_pair<PairM, true>(s, a, L, flags, st) : fwd_pair<PairM, false>(s, a, L, flags, st);
    case PAIR_L: return born ? fwd_pair<PairL, true>(s, a, L, flags, st) : fwd_pair<PairL, false>(s, a, L, flags, st);
    case PAIR_X:
      if (!born) return fwd_pair<PairX, false>(s, a, L, flags, st);
  }
  set_error("two-level forward step: no tile %d", tile);
  return E_ARG;
}

int launch_adj_pair(const ShotDev& s, int tile, int L, int flags, int xcd, hipStream_t st) {
  STCHK(check_layout(s));
  PairArgs a = pair_args(s);
  if (s.snap_fmt == SNAP_HIST && (flags & (A_IMG | A_IMG2))) flags |= P_HIST;
  a.k0 = ((flags & A_IMG) ? L : L - 1) / s.snap_every - 1;
  if (xcd) flags |= P_XCD;
  switch (tile) {
    case PAIR_S: return adj_pair<PairS>(s, a, L, flags, st);
    case PAIR_M: return adj_pair<PairM>(s, a, L, flags, st);
    case PAIR_L: return adj_pair<PairL>(s, a, L, flags, st);
  }
  set_error("two-level adjoint step: no tile %d", tile);
  return E_ARG;
}

}  // namespace erm
