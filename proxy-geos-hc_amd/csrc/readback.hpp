// readback.hpp -- padded device fields from and into dense host arrays.
#pragma once

#include <hip/hip_runtime.h>

#include "fd_kernels.hpp"
#include "phc_common.hpp"

namespace phc {

// Sponge product a level still owes (FDTDkernels.hpp:115): per-axis face
// factors, the face-slab rule of the FD step.
struct FieldDamping {
    int sw = 0;  // 0: none
    const float *fx = nullptr, *fy = nullptr, *fz = nullptr;
};

// Points [-lx, nx+lx) x [-ly, ny+ly) x [-lz, nz+lz) of `field` (layout L) into
// host, last axis fastest, the owed damping applied to interior points.  The
// rows are packed on the device, in pieces of at most READ_PIECE bytes (one
// row at least) through `scratch`, and each piece is one copy.  `scratch` is no
// larger than a piece or the field, and is kept for the next call; without
// memory for it the planes are copied row by row.  Repacking the whole array on
// the host cost 0.4 ms more for a 101^3 field.  Pieces of 16 and 8 MiB took 4
// and 6% longer to read a 401^3 field (15.6 ms), 64 MiB no less.
constexpr size_t READ_PIECE = (size_t)32 << 20;
phc_status read_field(hipStream_t stream, DevBuf &scratch, const float *field, const FdLayout &L, int lx, int ly,
                      int lz, const FieldDamping &damping, const float *const host_factors[3], float *host);

// The reverse: host into those points of `field`, everything else left as it is.
phc_status write_field(hipStream_t stream, DevBuf &scratch, float *field, const FdLayout &L, int lx, int ly, int lz,
                       const float *host);

// Every float of an array.
phc_status fill_field(hipStream_t stream, float *field, int64_t n, float value);

// The slice host[k * nx + i] = field(i, j, k) (interior, damping applied),
// gathered on the device in pieces of at most READ_PIECE bytes: 0.05 ms at
// 150^3, 2.0 ms through the whole field.
phc_status read_slice_xz(hipStream_t stream, DevBuf &scratch, const float *field, const FdLayout &L, int j,
                         const FieldDamping &damping, const float *const host_factors[3], float *host);

} // namespace phc
