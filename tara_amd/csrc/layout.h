// Conversions between the reference's kx-fastest half spectra (Nh, Ny[, Nz])
// and the device's ky-major layout (element (i, j) at i*Ny + j per z plane).
#pragma once
#include "common.h"

namespace tara {

// dst[i*ny + j] = src[j*nh + i] for each of nplanes planes of nh*ny elements.
// zero, one: ints that the launch sets to 0 and 1 besides (null: none).
int to_kymajor(const double2* src, double2* dst, int nh, int ny, int nplanes, hipStream_t st, int* zero = nullptr,
               int* one = nullptr);
// dst[j*nh + i] = src[i*ny + j], the inverse.
int from_kymajor(const double2* src, double2* dst, int nh, int ny, int nplanes, hipStream_t st);

// Fields whose rows are padded from nh to ld elements <-> packed rows, for the
// host boundary (at most 8 fields per launch).  A host copy of padded rows
// (hipMemcpy2D) moves one row of at most 2 KB at a time, about 7 us each: the
// 270 MB state of a 256 x 128 x 128 run took 0.93 s, against 0.04 s packed here
// first and copied whole.
struct RowFields {
    const double2* src[8];
    double2* dst[8];
};
// dst[r*nh + i] = src[r*ld + i], i < nh.
int pack_rows(const RowFields& f, int nfields, int nh, int ld, size_t rows, hipStream_t st);
// dst[r*ld + i] = src[r*nh + i] for i < nh, 0 in the padding.
int unpack_rows(const RowFields& f, int nfields, int nh, int ld, size_t rows, hipStream_t st);
// nfields host arrays of rows x nh elements <-> device fields of pitch ld,
// through the device buffer pack (at least nfields * rows * nh elements, ordered
// on st).  The copies are enqueued; the caller synchronises st.
int rows_from_host(double2* const dev[], const double* const host[], int nfields, int nh, int ld, size_t rows,
                   const DevBuf& pack, hipStream_t st);
int rows_to_host(double* const host[], const double2* const dev[], int nfields, int nh, int ld, size_t rows,
                 const DevBuf& pack, hipStream_t st);

}  // namespace tara
