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
  __device__ __forceinline__ unsigned short get16(unsigned cell) const {
    return __builtin_amdgcn_raw_buffer_load_b16(r, cell, 0, 0);
  }
  __device__ __forceinline__ void put(unsigned cell, unsigned array, float v) const {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, cell, array, 0);
  }
  __device__ __forceinline__ void put16(unsigned cell, unsigned short v) const {
    __builtin_amdgcn_raw_buffer_store_b16(v, r, cell, 0, 0);
  }
};
constexpr unsigned kOutside = 0x80000000u;  // past every buffer (all are smaller than 2 GiB)

}  // namespace erm
