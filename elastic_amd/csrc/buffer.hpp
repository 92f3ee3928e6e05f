// buffer.hpp -- fields read and written as raw buffers (gfx950).
#pragma once

#include "common.hpp"

namespace erm {

// The base is a scalar descriptor, the array (or its offset from the base) a
// scalar offset and the cell one vector register for all arrays: through
// pointers the compiler forms a 64-bit vector address per access, a seventh of
// the vector instructions of the 2D pair kernels and a third of the 3D acoustic
// step's. An offset past the buffer reads zero and writes nothing, which masks
// cells outside the grid.
struct Buf {
  __amdgpu_buffer_rsrc_t r;
  __device__ __forceinline__ Buf(const void* p, unsigned bytes)
      : r(__builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, 0x00020000)) {}
  __device__ __forceinline__ float get(unsigned cell, unsigned array = 0) const {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, cell, array, 0));
  }
  __device__ __forceinline__ unsigned short get16(unsigned cell, unsigned array = 0) const {
    return __builtin_amdgcn_raw_buffer_load_b16(r, cell, array, 0);
  }
  __device__ __forceinline__ void put(unsigned cell, unsigned array, float v) const {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, cell, array, 0);
  }
  __device__ __forceinline__ void put_nt(unsigned cell, unsigned array, float v) const {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, cell, array, 2);
  }
  __device__ __forceinline__ void put16(unsigned cell, unsigned short v) const {
    __builtin_amdgcn_raw_buffer_store_b16(v, r, cell, 0, 0);
  }
};
constexpr unsigned kOutside = 0x80000000u;  // past every buffer (all are smaller than 2 GiB)

// a + b, no less than either (kOutside stays outside).
__device__ __forceinline__ unsigned add_sat(unsigned a, unsigned b) { return __builtin_elementwise_add_sat(a, b); }

// Five fields n2 floats apart (one buffer, the field a scalar offset), or, FAR,
// fs apart (a buffer each: the fields of a drop-in history span gigabytes).
template <bool FAR>
struct Fields {
  const float* p;
  long long fs;
  unsigned bytes;  // of one field
  __device__ __forceinline__ Fields(const float* p_, long long fs_, int n2) : p(p_), fs(fs_), bytes(4u * (unsigned)n2) {}
  __device__ __forceinline__ float get(int f, unsigned cell) const {
    return FAR ? Buf(p + f * fs, bytes).get(cell) : Buf(p, 5u * bytes).get(cell, f * bytes);
  }
  __device__ __forceinline__ void put(int f, unsigned cell, float v) const {
    if (FAR)
      Buf(p + f * fs, bytes).put(cell, 0, v);
    else
      Buf(p, 5u * bytes).put(cell, f * bytes, v);
  }
};

}  // namespace erm
