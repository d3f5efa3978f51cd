// Device helpers shared by the kernels that keep a [rows][32] fp32 tile in LDS and gather whole
// 128-byte rows from it, one row per lane (gfx950: 160 KB of LDS per CU, 64 banks x 4 bytes, of
// which a row covers one half; measured delivery to registers: 128 bytes per clock per CU).
#ifndef FFI_LDS_TILE_H
#define FFI_LDS_TILE_H

#include "ffi_internal.h"

#include <type_traits>
#include <utility>

namespace ffi {

constexpr int kTileBatch = 32;        // batch entries per LDS row: 128 bytes = one pass over the banks
constexpr int kTileThreads = 1024;    // 16 wavefronts per workgroup, one workgroup per CU
constexpr size_t kTileLdsBudget = 152 * 1024;   // of the 160 KB per CU

__host__ __device__ inline size_t tile_lds_bytes(int rows) { return (size_t)rows * kTileBatch * sizeof(float); }
inline bool tile_path_fits(int rows) { return tile_lds_bytes(rows) <= kTileLdsBudget; }

#if defined(__HIPCC__)

// Workgroups are dealt round-robin to the 8 XCDs; this renumbers them so that consecutive logical
// ids share an XCD (and its L2), however many there are (left in round-robin order where their number is no multiple of eight, the
// 255 workgroups of 160 or 192 samples fetched every label's ids and weights in each of three batch tiles' XCDs: 192 x 600 x 200,000 x 40,
// forward by tiles of 64 198 us, 104 so, by tiles of 32 144 and 98).
__device__ __forceinline__ int xcd_contiguous_block(int block, int nblocks) {
    const int xcd = block & 7, per = nblocks >> 3, more = nblocks & 7;
    return xcd * per + min(xcd, more) + (block >> 3);
}

// xs[r][c] = src[r*ld + c0 + c] for c < 32 (zero beyond column `ld`), r < rows.  src rows are read
// in 128-byte pieces, LDS writes are conflict-free.  All of a thread's loads are issued before its
// first LDS write, so the staging costs one memory round trip, not one per row.
// thread -> (row, 16-byte chunk): 8 threads per row, whose rows start at any float (the memory system serves them; element by
// element, one in flight, a tile of 768 rows took some 12 us instead of 2: all passes at 127 x 768 x 131,072 x 32 208 us, at 127 x 767 x
// 131,072 x 4 130, at 163 x 797 x 10,774 x 4 114; 165, 87 and 82 so).
typedef float f32x4_unaligned __attribute__((ext_vector_type(4), aligned(4)));
typedef int i32x4_unaligned __attribute__((ext_vector_type(4), aligned(4)));
template <int THREADS, int INFLIGHT = 4>
__device__ __forceinline__ void stage_rows32(float* __restrict__ xs, const float* __restrict__ src, int rows,
                                             int ld, int c0) {
    constexpr int kRowsPerIter = THREADS / 8;
    constexpr int kInFlight = INFLIGHT;
    const int q = threadIdx.x & 7;
    const int there = ld - (c0 + 4 * q);                                  // elements of the chunk, if fewer than four
    const float* p = src + c0 + 4 * q;
    for (int r0 = threadIdx.x >> 3; r0 < rows; r0 += kRowsPerIter * kInFlight) {
        float4 v[kInFlight];
#pragma unroll
        for (int i = 0; i < kInFlight; ++i) {
            const int r = r0 + i * kRowsPerIter;
            v[i] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (r >= rows) continue;
            const float* from = p + (size_t)r * ld;
            if (there >= 4) {
                const f32x4_unaligned u = *reinterpret_cast<const f32x4_unaligned*>(from);
                v[i] = make_float4(u.x, u.y, u.z, u.w);
            } else {
                if (there > 0) v[i].x = from[0];
                if (there > 1) v[i].y = from[1];
                if (there > 2) v[i].z = from[2];
            }
        }
#pragma unroll
        for (int i = 0; i < kInFlight; ++i) {
            const int r = r0 + i * kRowsPerIter;
            if (r < rows) *reinterpret_cast<float4*>(xs + r * kTileBatch + 4 * q) = v[i];
        }
    }
}

// xs[n][b] = src[(b0 + b) * ld + n] for b < 32 (zero beyond `rows`), n < ld: four columns of four rows per thread and step, eight
// threads side by side for the 32 rows.
template <int THREADS>
__device__ __forceinline__ void stage_columns32(float* __restrict__ xs, const float* __restrict__ src, int ld, int rows, int b0) {
    const int c = threadIdx.x & 7;
#pragma unroll 1
    for (int n = (threadIdx.x >> 3) * 4; n < ld; n += THREADS / 2) {
        float v[4][4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int b = b0 + 4 * c + i;
            const float* from = src + (size_t)min(b, rows - 1) * ld + n;
            if (n + 4 <= ld) {
                const f32x4_unaligned q = *reinterpret_cast<const f32x4_unaligned*>(from);
                v[i][0] = q.x; v[i][1] = q.y; v[i][2] = q.z; v[i][3] = q.w;
            } else {
#pragma unroll
                for (int k = 0; k < 4; ++k) v[i][k] = from[min(k, ld - 1 - n)];
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) v[i][k] = b < rows ? v[i][k] : 0.f;
        }
#pragma unroll
        for (int k = 0; k < 4; ++k)
            if (n + k < ld) *reinterpret_cast<float4*>(xs + (size_t)(n + k) * kTileBatch + 4 * c) = make_float4(v[0][k], v[1][k], v[2][k], v[3][k]);
    }
}

// Raw buffer resource over `bytes` bytes at p (gfx9 family: 32-bit data format word).  Loads
// through it take a per-lane byte offset plus a wave-uniform (scalar) byte offset, and reads
// beyond `bytes` return zero instead of faulting.
using buffer_rsrc = __amdgpu_buffer_rsrc_t;
__device__ __forceinline__ buffer_rsrc make_rsrc(const void* p, size_t bytes) {
    const unsigned n = bytes > 0xfffffffeull ? 0xfffffffeu : (unsigned)bytes;
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, n, 0x00020000);
}
__device__ __forceinline__ float buffer_load_f32(buffer_rsrc r, unsigned lane_off, unsigned wave_off) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, lane_off, wave_off, 0));
}

// v[b] = m[(b0+b)*ld + col] for b < 32 (zero beyond `rows`); rows of m are reached through the
// scalar offset, `col` is the only per-lane address register.  m + b0*ld is rebased in 64 bits,
// the remaining offsets (< 32*ld*4) must fit 32 bits: callers guarantee ld < 2^25.
__device__ __forceinline__ void load_rows32(const float* __restrict__ m, int ld, int b0, int rows, unsigned col,
                                            float (&v)[32]) {
    const float* base = m + (size_t)b0 * (size_t)ld;
    const int nrows = min(32, rows - b0);
    const buffer_rsrc r = make_rsrc(base, (size_t)nrows * (size_t)ld * sizeof(float));
    const unsigned lane_off = col * 4u;
    const unsigned stride = (unsigned)ld * 4u;
#pragma unroll
    for (int b = 0; b < 32; ++b) v[b] = buffer_load_f32(r, lane_off, (unsigned)b * stride);
}

// ---- lane-per-row gathers -------------------------------------------------------------------------
// Every lane reads its OWN 128-byte row (row ids unrelated between lanes).  Bank conflicts are
// kept low by skewing the order in which a lane walks the eight 16-byte chunks of its row: at step
// c lane l reads chunk c ^ (l & 7).  Rows are 128-byte aligned, so inside one half of the banks
// the bank group depends on the chunk number only, and any eight consecutive lanes hit eight
// different bank groups (4.3x faster than the unskewed order, 1.4x faster than padded rows).
// Consequence: register group c of lane l holds batch entries 4*(c ^ (l&7)) .. +3.
// A 128-byte row covers half of the 64 banks (even rows one half, odd rows the other).  The LDS
// serves a ds_read_b128 at 16 lanes per clock (256 bytes) only when eight of those lanes read each
// half; measured with this access pattern: 4 clocks per wavefront read when the lanes with bit 3 of
// their id clear read even rows and the others odd rows, 8 clocks when row parities are random or
// all equal.  Kernels whose row order is theirs to choose (the input gradient, through its plan)
// arrange that; the forward pass and the weight gradient take rows in the order of the lookup
// matrix and run at the 8-clock rate.

__device__ __forceinline__ void cond_swap(bool p, float& a, float& b) {
    const float t = p ? b : a;
    b = p ? a : b;
    a = t;
}

// v[4c+i] <-> v[4(c ^ r)+i] for r in [0,8): its own inverse; three stages of conditional swaps.
__device__ __forceinline__ void xor_permute_groups(float (&v)[32], int r) {
    const bool b4 = r & 4, b2 = r & 2, b1 = r & 1;
#pragma unroll
    for (int e = 0; e < 32; ++e)
        if (!(e & 16)) cond_swap(b4, v[e], v[e + 16]);
#pragma unroll
    for (int e = 0; e < 32; ++e)
        if (!(e & 8)) cond_swap(b2, v[e], v[e + 8]);
#pragma unroll
    for (int e = 0; e < 32; ++e)
        if (!(e & 4)) cond_swap(b1, v[e], v[e + 4]);
}

// The same permutation applied to the 32 bits of a mask (bit e <-> bit e ^ 4r): halves, bytes, nibbles.
__device__ __forceinline__ unsigned xor_permute_bits(unsigned m, int r) {
    if (r & 4) m = (m >> 16) | (m << 16);
    if (r & 2) m = ((m & 0xff00ff00u) >> 8) | ((m & 0x00ff00ffu) << 8);
    if (r & 1) m = ((m & 0xf0f0f0f0u) >> 4) | ((m & 0x0f0f0f0fu) << 4);
    return m;
}

// Byte address (inside the tile) of the chunk read at step C, given base = row*128 | (lane&7)*16.
template <int C>
__device__ __forceinline__ unsigned skew_addr(unsigned base) { return C == 0 ? base : (base ^ (unsigned)(C * 16)); }

// The eight 16-byte reads of one row, all issued before the first use ...
// `base` = LDS address of the row + (lane & 7) * 16 (rows are 128-byte aligned, so the chunk bits can
// be flipped with XOR).
typedef float lds_v4f __attribute__((ext_vector_type(4)));
typedef const lds_v4f __attribute__((address_space(3)))* lds_v4f_ptr;
template <int C>
__device__ __forceinline__ float4 row_chunk(unsigned base) {
    const lds_v4f t = *(lds_v4f_ptr)(size_t)(skew_addr<C>(base));
    return make_float4(t.x, t.y, t.z, t.w);
}
__device__ __forceinline__ void read_row(unsigned base, float4 (&v)[8]) {
    v[0] = row_chunk<0>(base); v[1] = row_chunk<1>(base);
    v[2] = row_chunk<2>(base); v[3] = row_chunk<3>(base);
    v[4] = row_chunk<4>(base); v[5] = row_chunk<5>(base);
    v[6] = row_chunk<6>(base); v[7] = row_chunk<7>(base);
}
// ... and their dot product with the (equally skewed) out_grad values.
__device__ __forceinline__ float row_dot(const float4 (&v)[8], const float (&gb)[32], float acc) {
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        acc = fmaf(v[c].x, gb[4 * c + 0], acc);
        acc = fmaf(v[c].y, gb[4 * c + 1], acc);
        acc = fmaf(v[c].z, gb[4 * c + 2], acc);
        acc = fmaf(v[c].w, gb[4 * c + 3], acc);
    }
    return acc;
}

// ... or the 32 multiply-adds of the row by one weight.
__device__ __forceinline__ void row_fmas(const float4 (&v)[8], float wv, float (&acc)[32]) {
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        acc[4 * c + 0] = fmaf(wv, v[c].x, acc[4 * c + 0]);
        acc[4 * c + 1] = fmaf(wv, v[c].y, acc[4 * c + 1]);
        acc[4 * c + 2] = fmaf(wv, v[c].z, acc[4 * c + 2]);
        acc[4 * c + 3] = fmaf(wv, v[c].w, acc[4 * c + 3]);
    }
}

// f(integral_constant<int, 0>) ... f(integral_constant<int, N - 1>): a loop whose index is a constant expression
template <class F, int... Is>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, Is...>) { (f(std::integral_constant<int, Is>{}), ...); }
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) { static_for_impl(f, std::make_integer_sequence<int, N>{}); }

// The rows of ROWS connections as one stream of 16-byte reads, DEPTH of them in flight from the first to the last: `row(k)`
// is the base address of connection k's row (as above), of which CHUNKS reads are taken, `use(k, c, v)` what becomes of
// read c.  The order is pinned: GROUP reads, whose registers were used just before, then the next GROUP uses.
template <int ROWS, int CHUNKS, int DEPTH, int GROUP, class Row, class Use>
__device__ __forceinline__ void stream_rows(Row&& row, Use&& use) {
    static_assert(DEPTH % GROUP == 0 && CHUNKS % GROUP == 0, "whole groups");
    constexpr int kReads = ROWS * CHUNKS, kFirst = DEPTH < kReads ? DEPTH : kReads;
    lds_v4f v[kFirst];
    unsigned at = 0;
    auto read = [&](auto sc) {
        constexpr int s = decltype(sc)::value;
        if constexpr (s % CHUNKS == 0) at = row(std::integral_constant<int, s / CHUNKS>{});
        v[s % kFirst] = *(lds_v4f_ptr)(size_t)(at ^ (unsigned)(s % CHUNKS * 16));
    };
    static_for<kFirst>(read);
    __builtin_amdgcn_sched_barrier(0);
    static_for<kReads / GROUP>([&](auto gc) {
        constexpr int g = decltype(gc)::value * GROUP;
        static_for<GROUP>([&](auto i) {
            constexpr int s = g + decltype(i)::value;
            use(std::integral_constant<int, s / CHUNKS>{}, std::integral_constant<int, s % CHUNKS>{}, v[s % kFirst]);
        });
        if constexpr (GROUP > 1) __builtin_amdgcn_sched_barrier(0);
        if constexpr (g + kFirst < kReads) static_for<GROUP>([&](auto i) { read(std::integral_constant<int, g + kFirst + decltype(i)::value>{}); });
        __builtin_amdgcn_sched_barrier(0);
    });
}

#endif  // __HIPCC__

}  // namespace ffi

#endif  // FFI_LDS_TILE_H
