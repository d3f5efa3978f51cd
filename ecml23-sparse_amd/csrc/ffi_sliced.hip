// Forward pass for inputs whose tile does not fit in LDS (more than 1,216 columns), fp32 and bf16: gathers from
// sample-sliced tables that stay in an XCD's L2 (ffi_sliced.h).
#include "ffi_sliced.h"
#include "ffi_lds_tile.h"

#include <algorithm>
#include <cmath>

namespace ffi {
namespace {

constexpr int kSlThreads = 256;
constexpr int kSlInflight = 8;            // gathers a lane has in flight

// ---- slice tables -------------------------------------------------------------------------------------------------
// [B, rows] -> [slice][row][sl]: 64 x 64 tiles through LDS, four elements per load and store (of rows at any alignment: the
// memory system serves them), a tile's loads all in flight together.  One element at a time moved 3.0 TB/s.
template <typename T> struct Quad { T v[4]; };

template <typename T>
__global__ __launch_bounds__(256) void slices_from_batch_major_kernel(const T* __restrict__ src, T* __restrict__ dst, int rows, int B,
                                                                      int sl) {
    __shared__ T tile[64][65];                            // [row][sample]
    const int r0 = blockIdx.x * 64, b0 = blockIdx.y * 64;
    const int r4 = (threadIdx.x & 15) * 4, ty = threadIdx.x >> 4;
    Quad<T> q[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int b = b0 + ty + 16 * i, r = r0 + r4;
#pragma unroll
        for (int e = 0; e < 4; ++e) q[i].v[e] = (T)0;
        if (b < B) {
            if (r + 4 <= rows) q[i] = *reinterpret_cast<const Quad<T>*>(src + (size_t)b * rows + r);
            else
                for (int e = 0; e < 4; ++e)
                    if (r + e < rows) q[i].v[e] = src[(size_t)b * rows + r + e];
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) tile[r4 + e][ty + 16 * i] = q[i].v[e];
    __syncthreads();
    const int padded = (B + sl - 1) / sl * sl, width = sl < 64 ? sl : 64, quads = width / 4;      // (a slice inside the tile)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        // consecutive threads run over a slice's samples, then its rows, then the slices
        const int e = (int)threadIdx.x + 256 * i;
        const int in = e % quads * 4, r = e / quads % 64, t = e / (quads * 64) * width + in;
        const int b = b0 + t;
        if (r0 + r < rows && b < padded) {
            Quad<T> o;
#pragma unroll
            for (int c = 0; c < 4; ++c) o.v[c] = tile[r][t + c];
            *reinterpret_cast<Quad<T>*>(dst + ((size_t)(b / sl) * rows + r0 + r) * sl + b % sl) = o;
        }
    }
}

// [rows, B] -> [slice][row][sl]: one thread per element of a padded row, consecutive threads along it
template <typename T>
__global__ __launch_bounds__(256) void slices_from_rows_kernel(const T* __restrict__ src, T* __restrict__ dst, int rows, int B, int sl,
                                                               int padded) {
    const size_t t = (size_t)blockIdx.x * 256 + threadIdx.x;
    const size_t r = t / (unsigned)padded;
    const int b = (int)(t - r * (unsigned)padded);
    if (r >= (size_t)rows) return;
    dst[((size_t)(b / sl) * rows + r) * sl + b % sl] = b < B ? src[r * B + b] : (T)0;
}

template <typename T>
int launch_slices(const T* src, T* dst, int rows, int B, int sl, bool tp, hipStream_t s) {
    const int padded = (B + sl - 1) / sl * sl;
    if (tp) {
        const size_t total = (size_t)rows * padded;
        const size_t blocks = (total + 255) / 256;
        if (blocks > 0x7fffffffu) return FFI_ERR_TOO_LARGE;
        hipLaunchKernelGGL(slices_from_rows_kernel<T>, dim3((unsigned)blocks), dim3(256), 0, s, src, dst, rows, B, sl, padded);
    } else {
        const dim3 grid((unsigned)((rows + 63) / 64), (unsigned)((B + 63) / 64));
        if (grid.y > 65535u) return FFI_ERR_TOO_LARGE;
        hipLaunchKernelGGL(slices_from_batch_major_kernel<T>, grid, dim3(256), 0, s, src, dst, rows, B, sl);
    }
    FFI_HIP_TRY(hipGetLastError());
    return FFI_OK;
}

// ---- forward ------------------------------------------------------------------------------------------------------
// GL lanes of 16 bytes hold a row of a slice; a wavefront works on 64 / GL labels at a time, one per lane group.  Chunk by
// chunk the wavefront writes (byte offset of the row, weight) of its labels' connections into a list of its own in LDS and
// walks it, eight gathers in flight; the ids and weights of the next chunk travel meanwhile.  Entries behind the end of a
// list hold an offset beyond the table: the load returns zero without touching memory.  The lists serve SLICES slices one
// after the other where the tables of that many fit the L2 together: ids and weights are then read that many times less.
//
// QUADS: rows are made of quads on 16-byte boundaries.
//
// What bounds it: delivery from L2 while the tables fit there, ids and weights through the fabric beside it.
template <int GL> struct SlicedShape {
    static constexpr int kGroups = 64 / GL;                       // labels a wavefront works on at a time
    static constexpr int kRound = kGroups * (kSlThreads / 64);    // ... and the workgroup
    static constexpr int kRounds = GL == 8 ? 2 : 1;
    static constexpr int kLabels = kRound * kRounds;              // labels per workgroup: 64, 64, 128, 256
    static constexpr int kChunk = GL == 8 ? 64 : GL == 4 ? 32 : 16;   // connections per label and chunk, at most
    static constexpr int kQuads = kGroups * kChunk / 256;         // quads of connections per lane and chunk
};
// list stride for chunks of a multiple of eight: the lane groups' 16-byte reads fall into different banks
__host__ __device__ constexpr int list_stride(int chunk) { return chunk + 2; }
constexpr unsigned kNoRow = 0xffffff00u;

template <bool BF16> struct LaneAcc;
template <> struct LaneAcc<false> {
    static constexpr int kSamples = 4;
    float a[4];
    __device__ __forceinline__ void add(uint4 x, unsigned w) {
        const float wv = __uint_as_float(w);
        a[0] = fmaf(wv, __uint_as_float(x.x), a[0]); a[1] = fmaf(wv, __uint_as_float(x.y), a[1]);
        a[2] = fmaf(wv, __uint_as_float(x.z), a[2]); a[3] = fmaf(wv, __uint_as_float(x.w), a[3]);
    }
};
template <> struct LaneAcc<true> {
    static constexpr int kSamples = 8;
    float a[8];
    __device__ __forceinline__ void add(uint4 x, unsigned w) {
        const float wv = __uint_as_float(w);
        const unsigned v[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            a[2 * i] = fmaf(wv, __uint_as_float(v[i] << 16), a[2 * i]);
            a[2 * i + 1] = fmaf(wv, __uint_as_float(v[i] & 0xffff0000u), a[2 * i + 1]);
        }
    }
};

template <int GL, bool BF16, int SLICES, bool QUADS>
__global__ __launch_bounds__(kSlThreads) void fwd_sliced_kernel(const void* __restrict__ table, const int32_t* __restrict__ idx,
                                                                const void* __restrict__ w, const float* __restrict__ bias,
                                                                float* __restrict__ out, int B, int N, int L, int K, int slices, int chunk,
                                                                int label_blocks, int units, int add_to_out) {
    using S = SlicedShape<GL>;
    constexpr int kPer = LaneAcc<BF16>::kSamples, kSl = GL * kPer;
    constexpr unsigned kRow = GL * 16u;
    extern __shared__ __align__(16) unsigned char smem[];
    float* tile = reinterpret_cast<float*>(smem);                              // [kSl][kLabels + 1]
    constexpr size_t kTileBytes = (size_t)kSl * (S::kLabels + 1) * sizeof(float) / 16 * 16 + 16;
    const int stride = list_stride(chunk);
    const int u = xcd_unit(blockIdx.x, units);
    if (u < 0) return;
    const int slice0 = u / label_blocks * SLICES, j0 = (u % label_blocks) * S::kLabels;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int sub = lane & (GL - 1), grp = lane / GL;
    uint2* list = reinterpret_cast<uint2*>(smem + kTileBytes) + wave * S::kGroups * stride;
    const size_t slice_bytes = (size_t)N * kRow;
    buffer_rsrc rsrc[SLICES];
#pragma unroll
    for (int p = 0; p < SLICES; ++p)
        rsrc[p] = make_rsrc((const char*)table + (size_t)min(slice0 + p, slices - 1) * slice_bytes, slice_bytes);
    const unsigned lane_off = (unsigned)sub * 16u;
    const unsigned* w32 = reinterpret_cast<const unsigned*>(w);
    const unsigned short* w16 = reinterpret_cast<const unsigned short*>(w);

    LaneAcc<BF16> acc[S::kRounds][SLICES];
    uint4 ids[S::kQuads], ws[S::kQuads];                 // the chunk on its way
    auto first_label = [&](int q) { return j0 + q * S::kRound + wave * S::kGroups; };
    // Chunk k0 of the wavefront's labels.  Lane and quad v (or, without QUADS, element 4 v + e) number the connections of the
    // chunk through: label f / n, connection f % n.  Addresses behind the last label are pulled back to it, not branched
    // around: the loads go out together.
    auto place = [&](unsigned f, int n, int& l, int& k) {
        l = (int)((f * (65536u / (unsigned)n + 1u)) >> 16);       // f / n for f < 1,024 and n <= 64
        k = (int)f - l * n;
    };
    auto fetch = [&](int q, int k0) {
        const int kc = min(chunk, K - k0);
        const size_t last = (size_t)(L - 1);
#pragma unroll
        for (int v = 0; v < S::kQuads; ++v) {
            int l, k;
            if (QUADS) {
                place((unsigned)(64 * v + lane), kc / 4, l, k);
                const size_t at = min((size_t)(first_label(q) + min(l, S::kGroups - 1)), last) * K + k0 + 4 * k;
                ids[v] = *reinterpret_cast<const uint4*>(idx + at);
                if (BF16) {
                    const uint2 h = *reinterpret_cast<const uint2*>(w16 + at);
                    ws[v] = make_uint4(h.x << 16, h.x & 0xffff0000u, h.y << 16, h.y & 0xffff0000u);
                } else {
                    ws[v] = *reinterpret_cast<const uint4*>(w32 + at);
                }
            } else {
                unsigned* id4 = &ids[v].x;
                unsigned* w4 = &ws[v].x;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    place((unsigned)(64 * (4 * v + e) + lane), kc, l, k);
                    const size_t at = min((size_t)(first_label(q) + min(l, S::kGroups - 1)), last) * K + k0 + k;
                    id4[e] = (unsigned)idx[at];
                    w4[e] = BF16 ? (unsigned)w16[at] << 16 : w32[at];
                }
            }
        }
    };
    auto put = [&](int q, int k0) {
        const int kc = min(chunk, K - k0);
#pragma unroll
        for (int v = 0; v < S::kQuads; ++v) {
            int l, k;
            if (QUADS) {
                place((unsigned)(64 * v + lane), kc / 4, l, k);
                if (l < S::kGroups) {
                    const bool on = first_label(q) + l < L;
                    uint4* p = reinterpret_cast<uint4*>(list + l * stride + 4 * k);
                    p[0] = on ? make_uint4(ids[v].x * kRow, ws[v].x, ids[v].y * kRow, ws[v].y) : make_uint4(kNoRow, 0u, kNoRow, 0u);
                    p[1] = on ? make_uint4(ids[v].z * kRow, ws[v].z, ids[v].w * kRow, ws[v].w) : make_uint4(kNoRow, 0u, kNoRow, 0u);
                }
            } else {
                const unsigned id4[4] = {ids[v].x, ids[v].y, ids[v].z, ids[v].w}, w4[4] = {ws[v].x, ws[v].y, ws[v].z, ws[v].w};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    place((unsigned)(64 * (4 * v + e) + lane), kc, l, k);
                    const bool on = first_label(q) + l < L;
                    if (l < S::kGroups) list[l * stride + k] = make_uint2(on ? id4[e] * kRow : kNoRow, on ? w4[e] : 0u);
                }
            }
        }
        // the walk takes eight at a time
        if ((kc & 7) != 0 && lane < S::kGroups)
            for (int k = kc; k < (kc + 7) / 8 * 8; ++k) list[lane * stride + k] = make_uint2(kNoRow, 0u);
    };

    fetch(0, 0);
#pragma unroll
    for (int q = 0; q < S::kRounds; ++q) {
#pragma unroll
        for (int p = 0; p < SLICES; ++p)
#pragma unroll
            for (int i = 0; i < kPer; ++i) acc[q][p].a[i] = 0.f;
        int k0 = 0;
        while (true) {
            __builtin_amdgcn_wave_barrier();             // (the list is the wavefront's own, and LDS serves it in order)
            put(q, k0);
            const int n = min(chunk, K - k0);
            const bool last = k0 + chunk >= K;
            if (!last) fetch(q, k0 + chunk);
            else if (q + 1 < S::kRounds) fetch(q + 1, 0);
            __builtin_amdgcn_wave_barrier();
            const uint4* mylist = reinterpret_cast<const uint4*>(list + grp * stride);
#pragma unroll
            for (int p = 0; p < SLICES; ++p) {
#pragma unroll 1
                for (int i = 0; i < n; i += kSlInflight) {
                    uint4 e[kSlInflight / 2], x[kSlInflight];
#pragma unroll
                    for (int v = 0; v < kSlInflight / 2; ++v) e[v] = mylist[i / 2 + v];
#pragma unroll
                    for (int v = 0; v < kSlInflight; ++v)
                        x[v] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rsrc[p], ((v & 1) ? e[v / 2].z : e[v / 2].x) + lane_off, 0, 0));
#pragma unroll
                    for (int v = 0; v < kSlInflight; ++v) acc[q][p].add(x[v], (v & 1) ? e[v / 2].w : e[v / 2].y);
                }
            }
            if (last) break;
            k0 += chunk;
        }
    }
#pragma unroll
    for (int p = 0; p < SLICES; ++p) {
        if (slice0 + p >= slices) break;
        if (p > 0) __syncthreads();
#pragma unroll
        for (int q = 0; q < S::kRounds; ++q)
#pragma unroll
            for (int i = 0; i < kPer; ++i)
                tile[(sub * kPer + i) * (S::kLabels + 1) + q * S::kRound + wave * S::kGroups + grp] = acc[q][p].a[i];
        __syncthreads();
        // rows of out, 64 labels (256 bytes) per wavefront and step
        const int b0 = (slice0 + p) * kSl, nb = min(kSl, B - b0);
        constexpr int kCols = S::kLabels / 64;
        for (int e = wave; e < nb * kCols; e += kSlThreads / 64) {
            const int bb = e / kCols, jl = (e - bb * kCols) * 64 + lane, j = j0 + jl;
            if (j < L) {
                const size_t at = (size_t)(b0 + bb) * L + j;
                float v = tile[bb * (S::kLabels + 1) + jl];
                if (add_to_out) v += out[at];
                else if (bias != nullptr) v += bias[j];
                __builtin_nontemporal_store(v, out + at);     // (past the L2, which the tables need: 435 -> 371 us at 128 x 4,096 x 670,000 x 32)
            }
        }
    }
}

// ---- rows put in order of column range ----------------------------------------------------------------------------
// Every row's connections in the order of `ranges` equal column ranges, positions ascending inside a range, padded to whole
// quads with connections that name no column (the gather of one returns zero without touching memory).  The row is then
// cut into `ranges` parts of equal length, quads [Q r / ranges, Q (r + 1) / ranges) of its Q, and part r of all rows is
// stored in one piece.  Equal parts and not the ranges themselves: the lists of the lane groups stay equally long, and the
// few connections that a row has too many or too few (5 % at fan-in 72 and two ranges) merely miss the L2.
// A lane holds four entries, a row a group of Q neighbouring lanes: Q <= 64.  Both sides go through the wavefront's part
// of LDS, so that memory is read and written in whole lines.
constexpr int kMaxRanges = 4;
constexpr int kMaxRangedFanIn = 256;
__host__ __device__ constexpr int part_begin(int quads, int ranges, int r) { return quads * r / ranges; }

template <bool BF16>
__global__ __launch_bounds__(256) void rows_by_range_kernel(const int32_t* __restrict__ idx, const void* __restrict__ w,
                                                            unsigned* __restrict__ idx_out, void* __restrict__ w_out,
                                                            int L, int K, unsigned range_cols, int ranges) {
    __shared__ __align__(16) unsigned mem[4][2][256];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    unsigned* sid = mem[wave][0];
    unsigned* sw = mem[wave][1];
    const int gs = (K + 3) / 4, rows = 64 / gs;                          // lanes per row, rows per wavefront
    const long long row0 = ((long long)blockIdx.x * 4 + wave) * rows;
    const int nrows = (int)min((long long)rows, (long long)L - row0);    // (may be <= 0)
    const int total = nrows * K;
    for (int f = lane; f < total; f += 64) {
        const size_t at = (size_t)row0 * K + f;
        sid[f] = (unsigned)idx[at];
        sw[f] = BF16 ? (unsigned)reinterpret_cast<const unsigned short*>(w)[at] : reinterpret_cast<const unsigned*>(w)[at];
    }
    __builtin_amdgcn_wave_barrier();
    const int r = lane / gs, sub = lane - r * gs;
    const bool in_row = r < nrows;
    unsigned id[4], wv[4], range[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int k = 4 * sub + e;
        const bool on = in_row && k < K;
        id[e] = on ? sid[r * K + k] : 0u;
        wv[e] = on ? sw[r * K + k] : 0u;
        range[e] = on ? min(id[e] / range_cols, (unsigned)ranges - 1u) : 0xffu;
    }
    const unsigned long long group = (gs == 64 ? ~0ull : (1ull << gs) - 1ull) << (r * gs);
    const unsigned long long before = ((1ull << lane) - 1ull) & group;
    int to[4] = {0, 0, 0, 0}, begin = 0;
    for (unsigned q = 0; q < (unsigned)ranges; ++q) {
        int mine = begin;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const unsigned long long m = __ballot(range[e] == q);
            mine += __popcll(m & before);
            begin += __popcll(m & group);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (range[e] == q) to[e] = mine++;
    }
    __builtin_amdgcn_wave_barrier();
    reinterpret_cast<uint4*>(sid)[lane] = make_uint4(~0u, ~0u, ~0u, ~0u);        // (rows * gs <= 64 quads)
    reinterpret_cast<uint4*>(sw)[lane] = make_uint4(0u, 0u, 0u, 0u);
    __builtin_amdgcn_wave_barrier();
    if (in_row) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (range[e] != 0xffu) { sid[4 * r * gs + to[e]] = id[e]; sw[4 * r * gs + to[e]] = wv[e]; }
    }
    __builtin_amdgcn_wave_barrier();
    for (int q = 0; q < ranges; ++q) {
        const int begin_q = part_begin(gs, ranges, q), n = part_begin(gs, ranges, q + 1) - begin_q;
        if (n == 0) continue;
        const size_t base = (size_t)begin_q * L + (size_t)row0 * n;      // (in quads)
        for (int f = lane; f < nrows * n; f += 64) {
            const int fr = f / n, from = fr * gs + begin_q + f - fr * n;
            reinterpret_cast<uint4*>(idx_out)[base + f] = reinterpret_cast<const uint4*>(sid)[from];
            const uint4 v = reinterpret_cast<const uint4*>(sw)[from];
            if (BF16) reinterpret_cast<uint2*>(w_out)[base + f] = make_uint2(v.x | v.y << 16, v.z | v.w << 16);
            else reinterpret_cast<uint4*>(w_out)[base + f] = v;
        }
    }
}

struct FwdSliced {
    const void* table;
    const int32_t* idx;
    const void* w;
    const float* bias;
    float* out;
    int slices, per_group;         // slices; how many of them a workgroup serves with one list
    int K;                         // connections per row
    bool quads, add_to_out;
};

template <int GL, bool BF16, int SLICES>
int launch_fwd_sliced(const FwdSliced& a, const Dims& d, hipStream_t s) {
    using S = SlicedShape<GL>;
    const int label_blocks = (d.L + S::kLabels - 1) / S::kLabels, groups = (a.slices + SLICES - 1) / SLICES;
    if ((long long)label_blocks * groups > (1ll << 28)) return FFI_ERR_TOO_LARGE;
    const int units = label_blocks * groups;
    const int chunks = (a.K + S::kChunk - 1) / S::kChunk;
    const int chunk = ((a.K + chunks - 1) / chunks + 7) / 8 * 8;
    const size_t lds = (size_t)GL * LaneAcc<BF16>::kSamples * (S::kLabels + 1) * sizeof(float) / 16 * 16 + 16 +
                       (size_t)S::kRound * list_stride(chunk) * sizeof(uint2);
    const dim3 grid(xcd_grid(units)), block(kSlThreads);
    if (a.quads)
        hipLaunchKernelGGL((fwd_sliced_kernel<GL, BF16, SLICES, true>), grid, block, lds, s, a.table, a.idx, a.w, a.bias, a.out, d.B, d.N, d.L,
                           a.K, a.slices, chunk, label_blocks, units, a.add_to_out ? 1 : 0);
    else
        hipLaunchKernelGGL((fwd_sliced_kernel<GL, BF16, SLICES, false>), grid, block, lds, s, a.table, a.idx, a.w, a.bias, a.out, d.B, d.N, d.L,
                           a.K, a.slices, chunk, label_blocks, units, a.add_to_out ? 1 : 0);
    FFI_HIP_TRY(hipGetLastError());
    return FFI_OK;
}

template <int GL, bool BF16>
int launch_fwd_sliced_any(const FwdSliced& a, const Dims& d, hipStream_t s) {
    if constexpr (GL == 8) {
        if (a.per_group >= 4) return launch_fwd_sliced<GL, BF16, 4>(a, d, s);
        if (a.per_group >= 2) return launch_fwd_sliced<GL, BF16, 2>(a, d, s);
    }
    return launch_fwd_sliced<GL, BF16, 1>(a, d, s);
}

template <bool BF16>
int launch_fwd_sliced_lanes(int gl, const FwdSliced& a, const Dims& d, hipStream_t s) {
    switch (gl) {
        case 1: return launch_fwd_sliced_any<1, BF16>(a, d, s);
        case 2: return launch_fwd_sliced_any<2, BF16>(a, d, s);
        case 4: return launch_fwd_sliced_any<4, BF16>(a, d, s);
        default: return launch_fwd_sliced_any<8, BF16>(a, d, s);
    }
}

// `rows`: [ids][weights], each 4 L quads long
template <bool BF16>
int launch_rows_by_range(const int32_t* idx, const void* w, unsigned* rows, int L, int K, int N, int ranges, hipStream_t s) {
    const int quads = (K + 3) / 4, rows_per_block = 4 * (64 / quads);
    const unsigned range_cols = (unsigned)((N + ranges - 1) / ranges);
    hipLaunchKernelGGL((rows_by_range_kernel<BF16>), dim3((unsigned)((L + rows_per_block - 1) / rows_per_block)), dim3(256), 0, s, idx, w, rows,
                       rows + (size_t)L * quads * 4, L, K, range_cols, ranges);
    FFI_HIP_TRY(hipGetLastError());
    return FFI_OK;
}

}  // namespace

int launch_slices_f32(const float* src, float* dst, int rows, int B, int sl, bool tp, hipStream_t s) {
    return launch_slices(src, dst, rows, B, sl, tp, s);
}
int launch_slices_bf16(const unsigned short* src, unsigned short* dst, int rows, int B, int sl, bool tp, hipStream_t s) {
    return launch_slices(src, dst, rows, B, sl, tp, s);
}

// Passes over the columns, each over a range whose part of the slice fits an XCD's L2: they save what the gathers lose
// outside L2, and cost the rows put in order first and, from the second pass on, a read and a write of the scores.  Per
// label, in time of 1 TB/s; the rates are what the kernels reach at 300,000 to 670,091 labels: gathers 20 inside L2 (17 in
// several passes), 5.8 over the share that misses it, ordering 3.6, scores 5.5.  128 samples, 65,536 columns, fan-in 72:
// 2.26 ms in one pass, 1.73 in two; 32 samples and fan-in 32 there: 250 us in one, 320 in two.
static int sliced_ranges(size_t slice_bytes, int B, int K, int value_bytes) {
    if (K > kMaxRangedFanIn) return 1;
    if (g_options.wide_ranges > 0) return g_options.wide_ranges;
    int best = 1;
    double best_cost = 1e30;
    for (int r = 1; r <= kMaxRanges; ++r) {
        const double part = (double)slice_bytes / r, miss = std::max(0.0, 1.0 - (double)kXcdL2Bytes / part);
        const double inside = r > 1 ? 17.0 : 20.0, rate = miss > 0.0 ? std::min(inside, 5.8 / miss) : inside;
        const double cost = (double)B * K * value_bytes / rate + (r > 1 ? (double)K * 2 * (4 + value_bytes) / 3.6 + 8.0 * B * (r - 1) / 5.5 : 0.0);
        if (cost < best_cost) { best_cost = cost; best = r; }
    }
    return best;
}

int launch_forward_wide(const float* x, const int32_t* idx, const float* w, const float* bias, float* out, const Dims& d,
                        hipStream_t s) {
    const int gl = slice_lanes(d.B, 4), sl = gl * 4, slices = (d.B + sl - 1) / sl;
    const size_t slice_bytes = (size_t)d.N * sl * sizeof(float);
    if (slice_bytes >= 0xffffff00ull) return FFI_ERR_TOO_LARGE;
    float* table = nullptr;
    FFI_TRY(workspace_get(s, kWsFeaturesT, slice_bytes * slices, (void**)&table));
    FFI_TRY(launch_slices_f32(x, table, d.N, d.B, sl, d.tp, s));
    const bool quads = d.K % 4 == 0 && (((uintptr_t)idx | (uintptr_t)w) & 15) == 0;
    const int per_group = (int)std::min<size_t>((size_t)slices, kXcdL2Bytes / slice_bytes);
    const int ranges = sliced_ranges(slice_bytes, d.B, d.K, 4);
    FwdSliced a{table, idx, w, bias, out, slices, per_group, d.K, quads, false};
    if (ranges == 1) return launch_fwd_sliced_lanes<false>(gl, a, d, s);
    const int row_quads = (d.K + 3) / 4;
    unsigned* rows = nullptr;
    FFI_TRY(workspace_get(s, kWsRows, (size_t)d.L * row_quads * 32, (void**)&rows));
    FFI_TRY(launch_rows_by_range<false>(idx, w, rows, d.L, d.K, d.N, ranges, s));
    a.quads = true;
    for (int r = 0; r < ranges; ++r) {
        const int begin = part_begin(row_quads, ranges, r);
        a.K = 4 * (part_begin(row_quads, ranges, r + 1) - begin);
        if (a.K == 0) continue;
        a.idx = (const int32_t*)rows + (size_t)begin * 4 * d.L;
        a.w = rows + ((size_t)row_quads + begin) * 4 * d.L;
        FFI_TRY(launch_fwd_sliced_lanes<false>(gl, a, d, s));
        a.add_to_out = true;
    }
    return FFI_OK;
}

}  // namespace ffi
