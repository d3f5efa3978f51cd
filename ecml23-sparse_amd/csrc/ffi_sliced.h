// Sample-sliced copies of a gathered operand that does not fit in LDS: layout, and how work is dealt to the XCDs.
//
// A gather of a row costs what its cache lines cost where they are found.  Measured (rows of 128 bytes at random places,
// eight lanes of 16 bytes per row): 31 TB/s out of an XCD's own 4-MB L2, 15 TB/s from a table of 8 MB per XCD, 10 from
// 17 MB, 8.4 from 34 MB, 7.4 from 100 MB; rows of 64 bytes move half of that, rows of 256 bytes and more the same.  So
// the samples are cut into slices whose rows are one cache line (32 fp32 or 64 bf16 samples), every slice is a table of
// its own -- a row of a plain [N][B] matrix at a fixed sample offset would use only some of the L2 channels -- and an XCD
// works on one slice at a time: its L2 sees one table, not all of them.
#ifndef FFI_SLICED_H
#define FFI_SLICED_H

#include "ffi_internal.h"

namespace ffi {

constexpr int kXcds = 8;
constexpr size_t kXcdL2Bytes = 4u << 20;

// Samples per slice: a lane holds 16 bytes of a row; as many lanes per row as the batch needs, eight (one cache line) at most.
inline int slice_lanes(int B, int per_lane) {
    const int lanes = (B + per_lane - 1) / per_lane;
    return lanes <= 1 ? 1 : lanes <= 2 ? 2 : lanes <= 4 ? 4 : 8;
}

#if defined(__HIPCC__)
// Units of work in slice-major order are dealt to the XCDs in eight consecutive ranges; workgroups go round-robin over the
// XCDs.  The unit of this workgroup, or -1.
__device__ __forceinline__ int xcd_unit(int block, int units) {
    const int per = (units + kXcds - 1) / kXcds;
    const int xcd = block & (kXcds - 1), t = block / kXcds;
    const int u = xcd * per + t;
    return (t < per && u < units) ? u : -1;
}
#endif
inline unsigned xcd_grid(int units) { return (unsigned)((units + kXcds - 1) / kXcds) * kXcds; }

// dst[slice][row][SL] = the samples of every row of a matrix given as [rows, B] (tp) or [B, rows]; zeros behind sample B.
int launch_slices_f32(const float* src, float* dst, int rows, int B, int sl, bool tp, hipStream_t s);

}  // namespace ffi

#endif  // FFI_SLICED_H
