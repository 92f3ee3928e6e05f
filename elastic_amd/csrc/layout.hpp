// layout.hpp -- host arrays to and from the device layouts of the 2D engine.
//
// Callers hold unpadded (nz, nx) fields and (nt, nrx) records (time fastest);
// the device keeps fields with padded columns (ldz) and records with the
// traces fastest ([5][nt][nrx], one contiguous row per level). Each function
// moves the caller's array in contiguous copies through a device scratch of
// at most 32 MiB and rearranges it there. They return when the caller's
// array may be used. Where the scratch cannot be allocated they fall back to
// pitched copies or a host loop.
#pragma once

#include "common.hpp"

namespace erm {

// Cells of a field that are stored; the others are zeroed.
struct FieldBox {
  int iz0, iz1, ix0, ix1;  // inclusive
};

// nf host fields (nz, nx) -> device fields of column stride ldz, fs elements
// apart, rows nz..ldz-1 and cells outside box[f] (null: the whole grid) zero.
int store_fields(const float* const* src, int nf, int nz, int nx, int ldz, float* dst, size_t fs, const FieldBox* box,
                 hipStream_t st);
// Device fields -> nf host fields, one after the other in dst. nonfinite (may
// be null) is set when a value is not finite.
int fetch_fields(float* dst, int nf, int nz, int nx, int ldz, const float* src, size_t fs, bool* nonfinite,
                 hipStream_t st);
// nc components (nt, nrx) of a record, to and from device [nc][nt][nrx].
int store_records(const float* src, int nc, int nt, int nrx, float* dst, hipStream_t st);
int fetch_records(float* dst, int nc, int nt, int nrx, const float* src, bool* nonfinite, hipStream_t st);
// n doubles on the device -> n host floats (rounded once).
int fetch_rounded(float* dst, const double* src, size_t n, hipStream_t st);

}  // namespace erm
