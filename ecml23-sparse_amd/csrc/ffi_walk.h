// Which stream of a plan's global form a wavefront of the kernel that walks them takes (ffi_wide.hip).  Plain C++.
#ifndef FFI_WALK_H
#define FFI_WALK_H

namespace ffi {

constexpr int kWalkWaves = 8;        // wavefronts of a workgroup

// The wavefronts of a launch take the streams of one slice of the samples after those of the other, `units` of each: the place of wavefront
// `wave` of workgroup `workgroup` among the `all` of them (behind the last one: the last one's).
constexpr int walk_place(int workgroup, int wave, int all) {
    const int place = workgroup * kWalkWaves + wave;
    return place < all ? place : all - 1;
}

// The stream at that place, whichever slice it is of: with few streams a workgroup spans several slices.
constexpr int walk_stream(int workgroup, int wave, int units, int all) {
    return (int)((unsigned)walk_place(workgroup, wave, all) % (unsigned)units);
}

}  // namespace ffi

#endif  // FFI_WALK_H
