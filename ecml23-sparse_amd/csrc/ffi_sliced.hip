// Forward pass over slices of the samples, fp32 and bf16: gathers from tables that an XCD's L2 holds (ffi_sliced.h), in phases
// where it does not hold them, or from the slice in LDS (narrow inputs in bf16 or with few samples); and the top-k of its scores
// without the score matrix.
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

typedef __bf16 bf16_pair __attribute__((ext_vector_type(2)));

template <bool BF16> struct LaneAcc;
template <> struct LaneAcc<false> {
    using Element = float;
    static constexpr int kSamples = 4;
    float a[4];
    __device__ __forceinline__ void add2(uint4 x, uint4 y, unsigned wx, unsigned wy) { add(x, wx); add(y, wy); }
    __device__ __forceinline__ void add_pair(uint4 x, uint4 y, const unsigned* w) { add(x, w[0]); add(y, w[1]); }
    __device__ __forceinline__ void add(uint4 x, unsigned w) {
        const float wv = __uint_as_float(w);
        a[0] = fmaf(wv, __uint_as_float(x.x), a[0]); a[1] = fmaf(wv, __uint_as_float(x.y), a[1]);
        a[2] = fmaf(wv, __uint_as_float(x.z), a[2]); a[3] = fmaf(wv, __uint_as_float(x.w), a[3]);
    }
};
template <> struct LaneAcc<true> {
    using Element = unsigned short;
    static constexpr int kSamples = 8;
    float a[8];
    // two connections at a time: their values of a sample side by side, one dot product with both weights (two instructions
    // per multiply-add where unpacking to fp32 takes four; the products are exact either way)
    __device__ __forceinline__ void add2(uint4 x, uint4 y, unsigned wx, unsigned wy) {
        const unsigned w = __builtin_amdgcn_perm(wy, wx, 0x07060302u);
        add_pair(x, y, &w);
    }
    __device__ __forceinline__ void add_pair(uint4 x, uint4 y, const unsigned* w) {
        const bf16_pair wv = __builtin_bit_cast(bf16_pair, *w);
        const unsigned u[4] = {x.x, x.y, x.z, x.w}, v[4] = {y.x, y.y, y.z, y.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            a[2 * i] = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16_pair, __builtin_amdgcn_perm(v[i], u[i], 0x05040100u)), wv, a[2 * i], false);
            a[2 * i + 1] = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16_pair, __builtin_amdgcn_perm(v[i], u[i], 0x07060302u)), wv, a[2 * i + 1], false);
        }
    }
};

// Where a forward kernel that keeps no scores puts those at or above their sample's threshold.
struct TopkSink {
    const float* tau;              // [B]; null: the kernel stores scores
    int* tie;                      // [B] see TopkCandidates
    int* count;                    // [B] entries appended
    float* val;                    // [B][cap]
    int* idx;
    int cap;
};

// The lane's scores of label j for samples b0 ... b0 + n - 1: few reach their threshold, so each takes its place with an atomic.
// n bounds the samples, not a threshold that no score reaches: +inf reaches every threshold.
template <int PER>
__device__ __forceinline__ void topk_append(const TopkSink& sink, const float (&a)[PER], const float (&tau)[PER], int* tie, int b0, int n, int j, bool valid) {
    bool hit = false;
#pragma unroll
    for (int i = 0; i < PER; ++i) hit |= a[i] >= tau[i];
    if (!valid || !hit) return;
    asm volatile("" : "+v"(b0));              // keeps the samples' addresses from being formed ahead of the label loop (48 registers in bf16: spilled, 5 x 22 x 60,520 x 5 took 15 us, now 8)
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        if (i < n && a[i] >= tau[i]) {
            const int slot = topk_slot(a[i], j, tau[i], tie[i], &sink.tie[b0 + i], &sink.count[(size_t)(b0 + i) * kTopkCountStep], sink.cap);
            if (slot < sink.cap) {
                sink.val[(size_t)(b0 + i) * sink.cap + slot] = a[i];
                sink.idx[(size_t)(b0 + i) * sink.cap + slot] = j;
            }
        }
    }
}
// The thresholds of the samples from b0 on, four per load; nothing is done with them here, so that nobody waits for them.
// (Behind the batch's end: of samples that are not there, see topk_candidates_at.)
template <int PER>
__device__ __forceinline__ void topk_thresholds(const TopkSink& sink, int b0, float (&tau)[PER], int (&tie)[PER]) {
#pragma unroll
    for (int i = 0; i < PER; i += 4) {
        const float4 t = *reinterpret_cast<const float4*>(sink.tau + b0 + i);
        const int4 e = *reinterpret_cast<const int4*>(sink.tie + b0 + i);
        tau[i] = t.x; tau[i + 1] = t.y; tau[i + 2] = t.z; tau[i + 3] = t.w;
        tie[i] = e.x; tie[i + 1] = e.y; tie[i + 2] = e.z; tie[i + 3] = e.w;
    }
}

template <int GL, bool BF16, int SLICES, bool QUADS>
__global__ __launch_bounds__(kSlThreads) void fwd_sliced_kernel(const void* __restrict__ table, const int32_t* __restrict__ idx,
                                                                const void* __restrict__ w, const float* __restrict__ bias,
                                                                float* __restrict__ out, int B, int N, int L, int K, int slices, int chunk,
                                                                int label_blocks, int units, const TopkSink sink) {
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
                    for (int v = 0; v < kSlInflight / 2; ++v) acc[q][p].add2(x[2 * v], x[2 * v + 1], e[v].y, e[v].w);
                }
            }
            if (last) break;
            k0 += chunk;
        }
    }
    if (sink.tau != nullptr) {
#pragma unroll
        for (int p = 0; p < SLICES; ++p) {
            if (slice0 + p >= slices) break;                               // (a workgroup's surplus slices repeat the last one)
            const int b0 = (slice0 + p) * kSl + sub * kPer;
            float tau[kPer];
            int tie[kPer];
            topk_thresholds(sink, b0, tau, tie);
#pragma unroll
            for (int q = 0; q < S::kRounds; ++q) {
                const int j = first_label(q) + grp;
                if (bias != nullptr) {
                    const float bj = bias[min(j, L - 1)];
#pragma unroll
                    for (int i = 0; i < kPer; ++i) acc[q][p].a[i] += bj;
                }
                topk_append(sink, acc[q][p].a, tau, tie, b0, B - b0, j, j < L);
            }
        }
        return;
    }
#pragma unroll
    for (int p = 0; p < SLICES; ++p) {
        if (p > 0) __syncthreads();
#pragma unroll
        for (int q = 0; q < S::kRounds; ++q)
#pragma unroll
            for (int i = 0; i < kPer; ++i)
                tile[(sub * kPer + i) * (S::kLabels + 1) + q * S::kRound + wave * S::kGroups + grp] = acc[q][p].a[i];
        __syncthreads();
        // rows of out, 64 labels (256 bytes) per wavefront and step
        const int b0 = (slice0 + p) * kSl, nb = min(kSl, B - b0);         // (<= 0 beyond the last slice)
        constexpr int kCols = S::kLabels / 64;
        for (int e = wave; e < nb * kCols; e += kSlThreads / 64) {
            const int bb = e / kCols, jl = (e - bb * kCols) * 64 + lane, j = j0 + jl;
            if (j < L) {
                const size_t at = (size_t)(b0 + bb) * L + j;
                float v = tile[bb * (S::kLabels + 1) + jl];
                if (bias != nullptr) v += bias[j];
                __builtin_nontemporal_store(v, out + at);     // (past the L2, which the tables need: 435 -> 371 us at 128 x 4,096 x 670,000 x 32)
            }
        }
    }
}

// ---- forward, slice in LDS ----------------------------------------------------------------------------------------
// For slices that fit in LDS beside the lists: narrow inputs with few samples or in bf16.  The workgroup brings its slice, then
// its wavefronts take rounds of consecutive labels (every row_step-th row of the layer), a lane group per label, the rows of the
// slice read from LDS.
//
// What bounds it: for one to four samples the stream of ids and weights from memory; from there on LDS delivery (a row of
// 16 GL bytes per connection and lane group, and the lists) and the instructions around it.
//   Scores leave from the registers: the lanes' low bits change places with the rounds (exchange_bit), which makes pieces of 32
// labels without the tile in LDS that took them through it twice more; pieces of 32 bytes cost 140 us at 128 x 768 x 300,000 x 32
// in bf16, the tile 112, these 84.  What a lane fetches is the same place of every chunk, so its divisions are done once.
//   A wavefront takes 32 labels at a time, the last ones in even shares; with fewer labels than that for all, the workgroups are
// as many as give each wavefront one round (64 x 768 x 8,192 x 32 in bf16: 28.7 us with 32 labels each, 18.0 so).
//   The slice comes in with four columns of a lane's four samples per step, lanes side by side holding a row of the slice: with
// a column per lane, 32 lanes wrote to one pair of banks (the same shape: 18.0 -> 14.4 us, a first list already in flight).
// COLUMNS: [B,N] of eight samples comes in by a column's samples per lane all the same, one way or the other and not both in one
// kernel, whose first instructions are some of its 7 us.  From more than 512 columns on: top-k of 5 x 768 x 30,000 x 16 27.2 us by four
// columns, 26.8 so; 400 columns 26.7 and 27.0, 300 and fewer the same.
//   At 100 x 500 x 131,073 x 24 in bf16, all of it together: 45.6 -> 36.4 us.
typedef unsigned lds_v4u __attribute__((ext_vector_type(4)));
constexpr int kLdThreads = 1024;
constexpr size_t kLdThresholdBytes = 512;       // (behind the rest: thresholds of up to 64 samples, which would take 16 registers through the label loop)
constexpr size_t kLdBudget = 160 * 1024 - kLdThresholdBytes;

template <int GL, bool BF16> struct LdsShape {
    static constexpr int kGroups = 64 / GL;
    static constexpr int kRounds = GL / 2;                                // whose scores leave together: of 32 labels
    static constexpr int kChunk = GL == 8 ? 32 : 16;
    static constexpr int kQuads = (kGroups * kChunk + 255) / 256;
    // a label's list, in words: (row offset, weight) pairs; in bf16 the offsets, and in an array of their own the weights as they are,
    // two to a word
    static constexpr int kPitch = BF16 ? kChunk + 4 : 2 * kChunk + 4, kWeightPitch = BF16 ? kChunk / 2 + 2 : 0;
    static constexpr int kWaveBytes = kGroups * (kPitch + kWeightPitch) * 4;
};
template <int GL, bool BF16> inline size_t lds_kernel_bytes(int N) { return (size_t)(N + 1) * GL * 16 + (size_t)(kLdThreads / 64) * LdsShape<GL, BF16>::kWaveBytes; }

// Lanes whose bit is clear and set (DPP step CTRL pairs them): the pair's a to the former in place of (a, b), its b to the latter.
template <int CTRL> __device__ __forceinline__ void exchange_bit(bool bit, float& a, float& b) {
    const int send = __float_as_int(bit ? a : b);
    const float other = __int_as_float(__builtin_amdgcn_update_dpp(send, send, CTRL, 0xf, 0xf, false));
    a = bit ? other : a;
    b = bit ? b : other;
}

typedef unsigned u32x4_unaligned __attribute__((ext_vector_type(4), aligned(4)));
typedef unsigned u32x2_unaligned __attribute__((ext_vector_type(2), aligned(2)));

// How ids and weights are read: one by one; by quads, of rows of whole quads on 16-byte boundaries; by quads of any rows, the quad that a row
// ends in being its last four connections.  300,000 labels of 8 samples x 768 by ones and by quads: fan-in 7 17.1 and 12.0 us, 10 15.5 and 13.1, 22 23.0
// and 20.2, 33 34.8 and 32.2, 34 35.6 and 34.0, but 38 38.8 and 42.6, 46 46.8 and 58.5, 47 48.6 and 59.5 (16 samples 34 and 32, bf16 64 and 58), 62 60 and
// 76, 65 69 and 88 (44 and 42, 78 and 72), 126 108 and 135; with cold caches, one sample x 670,091 and four samples x 300,000 the line is the same.
enum LdsRows { kOneByOne = 0, kQuads = 1, kAnyQuads = 2 };
template <int GL> constexpr bool any_quads_pay(int K) { return K >= 4 && (GL >= 4 || K <= 33); }

template <int GL, bool BF16, int ROWS, bool COLUMNS = false>
__global__ __launch_bounds__(kLdThreads) void fwd_lds_kernel(const void* __restrict__ features, const int32_t* __restrict__ idx,
                                                             const void* __restrict__ w, const float* __restrict__ bias,
                                                             float* __restrict__ out, int B, int N, int L, int K, int tp, int row_step,
                                                             int slices, int streams, int chunk, const TopkSink sink) {
    using S = LdsShape<GL, BF16>;
    constexpr bool QUADS = ROWS != kOneByOne;
    constexpr int kPer = LaneAcc<BF16>::kSamples, kSl = GL * kPer, kWaves = kLdThreads / 64;
    constexpr unsigned kRow = GL * 16u;
    extern __shared__ __align__(16) unsigned char smem[];
    const int u = xcd_contiguous_block(blockIdx.x, gridDim.x);            // (the slices of a stream share ids and weights in an L2)
    const int slice = u % slices, stream = u / slices;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int sub = lane & (GL - 1), grp = lane / GL;
    auto stage = [&]() {
        // four samples of a column from a row of [N,B], or of four columns from four rows of [B,N]; lanes side by side hold a
        // column's samples, and write its row of the slice together
        using T = typename LaneAcc<BF16>::Element;
        const T* x = static_cast<const T*>(features);
        Quad<T>* dst = reinterpret_cast<Quad<T>*>(smem);
        constexpr int kQ = kSl / 4;
        const int width = tp ? B : N;                                     // of a row of the features
        auto read4 = [&](int row, int at) {
            const T* from = x + (size_t)row * width;
            Quad<T> q;
            if (at + 4 <= width) {
                q = *reinterpret_cast<const Quad<T>*>(from + at);         // (at any alignment)
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) q.v[i] = from[min(at + i, width - 1)];
            }
            return q;
        };
        if (tp) {
#pragma unroll 4
            for (int e = threadIdx.x; e < N * kQ; e += kLdThreads) {
                const int n = e / kQ, c = e % kQ, b = slice * kSl + 4 * c;
                Quad<T> q = read4(n, b);
#pragma unroll
                for (int i = 0; i < 4; ++i) q.v[i] = b + i < B ? q.v[i] : (T)0;
                dst[n * kQ + c] = q;
            }
        } else if constexpr (COLUMNS) {
#pragma unroll 4
            for (int e = threadIdx.x; e < N * kQ; e += kLdThreads) {
                const int n = e % N, c = e / N, b = slice * kSl + 4 * c;
                Quad<T> q;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const T v = x[(size_t)min(b + i, B - 1) * N + n];
                    q.v[i] = b + i < B ? v : (T)0;
                }
                dst[n * kQ + c] = q;
            }
        } else {
#pragma unroll 2
            for (int e = threadIdx.x; e < (N + 3) / 4 * kQ; e += kLdThreads) {
                const int n = e / kQ * 4, c = e % kQ, b = slice * kSl + 4 * c;
                Quad<T> rows[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) rows[i] = read4(min(b + i, B - 1), n);
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    Quad<T> q;
#pragma unroll
                    for (int i = 0; i < 4; ++i) q.v[i] = b + i < B ? rows[i].v[v] : (T)0;
                    if (n + v < N) dst[(n + v) * kQ + c] = q;
                }
            }
        }
        if (threadIdx.x < GL) reinterpret_cast<uint4*>(smem)[N * GL + threadIdx.x] = make_uint4(0u, 0u, 0u, 0u);    // what entries behind a list's end name
    };
    float* const slice_tau = reinterpret_cast<float*>(smem + (size_t)(N + 1) * kRow + (size_t)kWaves * S::kWaveBytes);
    int* const slice_tie = reinterpret_cast<int*>(slice_tau + kSl);
    unsigned char* const mine = smem + (size_t)(N + 1) * kRow + (size_t)wave * S::kWaveBytes;
    unsigned* const list = reinterpret_cast<unsigned*>(mine);
    unsigned* const list_w = list + S::kGroups * S::kPitch;               // (bf16)
    // (raw LDS addresses: what a column id beyond the slice names is outside the LDS and reads as zero, or some of the LDS)
    const unsigned rows = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)smem + (unsigned)sub * 16u;
    const unsigned no_row = (unsigned)N * kRow;
    const unsigned* w32 = reinterpret_cast<const unsigned*>(w);
    const unsigned short* w16 = reinterpret_cast<const unsigned short*>(w);
    const int b0 = slice * kSl, nb = min(kSl, B - b0);
    const int mine0 = b0 + sub * kPer;                                    // first sample of this lane

    // Lane and quad v (or, without QUADS, element 4 v + e) number the connections of a chunk of kGroups labels through: label f / n,
    // connection f % n, the same for every chunk.  What lies behind the row, or the last label, is read in place of something else.
    uint4 ids[S::kQuads], ws[S::kQuads];
    auto place = [&](unsigned f, int n, int& l, int& k) {
        l = (int)((f * (65536u / (unsigned)n + 1u)) >> 16);               // f / n for f < 1,024 and n <= 32
        k = (int)f - l * n;
    };
    const unsigned row_pitch = (unsigned)row_step * (unsigned)K;          // (labels * row_step * K < 2^31)
    const int per = min(chunk, K);                                        // connections of a chunk (a multiple of four where there are several)
    auto fetch = [&](int q, int k0) {
        const int kc = min(chunk, K - k0), j = q * S::kGroups;
#pragma unroll
        for (int v = 0; v < S::kQuads; ++v) {
            int l, k;
            if (QUADS) {
                place((unsigned)(64 * v + lane), chunk / 4, l, k);
                const int row = min(j + min(l, S::kGroups - 1), L - 1), off = 4 * k < kc ? 4 * k : 0;
                if constexpr (ROWS == kAnyQuads) {
                    const unsigned at = (unsigned)row * row_pitch + (unsigned)(k0 + min(off, kc - 4));
                    const u32x4_unaligned id = *reinterpret_cast<const u32x4_unaligned*>(idx + at);
                    ids[v] = make_uint4(id.x, id.y, id.z, id.w);
                    if (BF16) {
                        const u32x2_unaligned h = *reinterpret_cast<const u32x2_unaligned*>(w16 + at);
                        ws[v].x = h.x; ws[v].y = h.y;
                    } else {
                        const u32x4_unaligned f = *reinterpret_cast<const u32x4_unaligned*>(w32 + at);
                        ws[v] = make_uint4(f.x, f.y, f.z, f.w);
                    }
                } else {
                    const unsigned at = (unsigned)row * row_pitch + (unsigned)(k0 + off);
                    ids[v] = *reinterpret_cast<const uint4*>(idx + at);
                    if (BF16) {
                        const uint2 h = *reinterpret_cast<const uint2*>(w16 + at);
                        ws[v].x = h.x; ws[v].y = h.y;
                    } else {
                        ws[v] = *reinterpret_cast<const uint4*>(w32 + at);
                    }
                }
            } else {
                unsigned* id4 = &ids[v].x;
                unsigned* w4 = &ws[v].x;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    place((unsigned)(64 * (4 * v + e) + lane), per, l, k);
                    const unsigned at = (unsigned)min(j + min(l, S::kGroups - 1), L - 1) * row_pitch + (unsigned)(k0 + (k < kc ? k : 0));
                    id4[e] = (unsigned)idx[at];
                    w4[e] = BF16 ? (unsigned)w16[at] : w32[at];
                }
            }
        }
    };
    auto put = [&](int k0) {
        const int kc = min(chunk, K - k0);
#pragma unroll
        for (int v = 0; v < S::kQuads; ++v) {
            int l, k;
            if (QUADS) {
                place((unsigned)(64 * v + lane), chunk / 4, l, k);
                if (l < S::kGroups && 4 * k < kc) {
                    if (ROWS == kAnyQuads && (kc & 3)) {                  // (of the quad that the row ends in, the quad before holds the first)
                        const int seen = 4 * k + 4 - kc;
                        const uint4 was = ids[v], wt = ws[v];
                        ids[v].x = seen > 0 ? (unsigned)N : was.x; ids[v].y = seen > 1 ? (unsigned)N : was.y; ids[v].z = seen > 2 ? (unsigned)N : was.z;
                        if (BF16) {
                            ws[v].x = seen > 1 ? 0u : seen > 0 ? wt.x & 0xffff0000u : wt.x;
                            ws[v].y = seen > 2 ? wt.y & 0xffff0000u : wt.y;
                        } else {
                            ws[v].x = seen > 0 ? 0u : wt.x; ws[v].y = seen > 1 ? 0u : wt.y; ws[v].z = seen > 2 ? 0u : wt.z;
                        }
                    }
                    if (BF16) {
                        *reinterpret_cast<uint4*>(list + l * S::kPitch + 4 * k) = make_uint4(ids[v].x * kRow, ids[v].y * kRow, ids[v].z * kRow, ids[v].w * kRow);
                        *reinterpret_cast<uint2*>(list_w + l * S::kWeightPitch + 2 * k) = make_uint2(ws[v].x, ws[v].y);
                    } else {
                        uint4* p = reinterpret_cast<uint4*>(list + l * S::kPitch + 8 * k);
                        p[0] = make_uint4(ids[v].x * kRow, ws[v].x, ids[v].y * kRow, ws[v].y);
                        p[1] = make_uint4(ids[v].z * kRow, ws[v].z, ids[v].w * kRow, ws[v].w);
                    }
                }
            } else {
                const unsigned id4[4] = {ids[v].x, ids[v].y, ids[v].z, ids[v].w}, w4[4] = {ws[v].x, ws[v].y, ws[v].z, ws[v].w};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    place((unsigned)(64 * (4 * v + e) + lane), per, l, k);
                    if (l >= S::kGroups) continue;
                    const unsigned row = k < kc ? id4[e] * kRow : no_row, wv = k < kc ? w4[e] : 0u;       // (the walk takes four at a time)
                    if (BF16) {
                        list[l * S::kPitch + k] = row;
                        reinterpret_cast<unsigned short*>(list_w + l * S::kWeightPitch)[k] = (unsigned short)wv;
                    } else {
                        *reinterpret_cast<uint2*>(list + l * S::kPitch + 2 * k) = make_uint2(row, wv);
                    }
                }
            }
        }
    };
    if (!QUADS)                                                           // (the walk takes four at a time: what no chunk of a short fan-in writes)
        for (int k = per; k < (per + 3) / 4 * 4; ++k)
            for (int l = lane; l < S::kGroups; l += 64) {
                if (BF16) {
                    list[l * S::kPitch + k] = no_row;
                    reinterpret_cast<unsigned short*>(list_w + l * S::kWeightPitch)[k] = 0;
                } else {
                    *reinterpret_cast<uint2*>(list + l * S::kPitch + 2 * k) = make_uint2(no_row, 0u);
                }
            }
    const unsigned* const mylist = list + grp * S::kPitch;
    const unsigned* const my_w = list_w + grp * S::kWeightPitch;
    // Rounds of kGroups consecutive labels.  The wavefronts take kRounds at a time, side by side, as long as all have some to take, then
    // an even share of what is left.
    const int rounds = (L + S::kGroups - 1) / S::kGroups, all = streams * kWaves, me = stream * kWaves + wave;
    const int full = rounds / (all * S::kRounds), tail = rounds - full * all * S::kRounds, share = (tail + all - 1) / all;
    auto begin_of = [&](int t) { return t < full ? (t * all + me) * S::kRounds : min(full * all * S::kRounds + me * share, rounds); };
    fetch(begin_of(0), 0);                                                // (in flight beside the slice)
    stage();
    if (sink.tau != nullptr && threadIdx.x < kSl) {
        slice_tau[threadIdx.x] = sink.tau[slice * kSl + threadIdx.x];
        slice_tie[threadIdx.x] = sink.tie[slice * kSl + threadIdx.x];
    }
    __syncthreads();
    if (full == 0 && begin_of(0) >= rounds) return;
    const int lane_row = (sub & ~(S::kRounds - 1)) * kPer;                // first of the rows of out that this lane stores
    for (int t = 0; t <= full; ++t) {
        const int q = begin_of(t), q_end = t < full ? q + S::kRounds : min(q + share, rounds), after = min(begin_of(min(t + 1, full)), rounds - 1);
        LaneAcc<BF16> acc[S::kRounds];
#pragma unroll
        for (int r = 0; r < S::kRounds; ++r) {
#pragma unroll
            for (int i = 0; i < kPer; ++i) acc[r].a[i] = 0.f;
            if (q + r >= q_end) continue;                                 // (wave-uniform)
            for (int k0 = 0; k0 < K; k0 += chunk) {
                __builtin_amdgcn_wave_barrier();                          // (the list is the wavefront's own, and LDS serves it in order)
                put(k0);
                if (k0 + chunk < K) fetch(q + r, k0 + chunk);
                else fetch(q + r + 1 < q_end ? q + r + 1 : after, 0);
                __builtin_amdgcn_wave_barrier();
                const int n = min(chunk, K - k0);
#pragma unroll 2
                for (int i = 0; i < n; i += 4) {
                    uint4 x[4];
                    unsigned at[4], wv[4];
                    if (BF16) {
                        const uint4 e = *reinterpret_cast<const uint4*>(mylist + i);
                        const uint2 f = *reinterpret_cast<const uint2*>(my_w + i / 2);
                        at[0] = e.x; at[1] = e.y; at[2] = e.z; at[3] = e.w;
                        wv[0] = f.x; wv[1] = f.y;
                    } else {
#pragma unroll
                        for (int v = 0; v < 2; ++v) {
                            const uint4 e = *reinterpret_cast<const uint4*>(mylist + 2 * i + 4 * v);
                            at[2 * v] = e.x; at[2 * v + 1] = e.z;
                            wv[2 * v] = e.y; wv[2 * v + 1] = e.w;
                        }
                    }
#pragma unroll
                    for (int v = 0; v < 4; ++v) x[v] = __builtin_bit_cast(uint4, *(const lds_v4u __attribute__((address_space(3)))*)(size_t)(rows + at[v]));
#pragma unroll
                    for (int v = 0; v < 2; ++v) acc[r].add_pair(x[2 * v], x[2 * v + 1], wv + v * (BF16 ? 1 : 2));
                }
            }
            const int j = (q + r) * S::kGroups + grp;
            if (bias != nullptr) {
                const float bj = bias[(size_t)min(j, L - 1) * row_step];
#pragma unroll
                for (int i = 0; i < kPer; ++i) acc[r].a[i] += bj;
            }
            if (sink.tau != nullptr) {
                float tau[kPer];
#pragma unroll
                for (int i = 0; i < kPer; ++i) tau[i] = slice_tau[sub * kPer + i];
                topk_append(sink, acc[r].a, tau, slice_tie + sub * kPer, mine0, B - mine0, j, j < L);
            }
        }
        if (sink.tau != nullptr) continue;
        // Rows of out leave in pieces of 32 labels: the lanes' low bits, which number samples, change places with the rounds.
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            if constexpr (S::kRounds >= 2) {
#pragma unroll
                for (int r = 0; r < S::kRounds; r += 2) exchange_bit<0xb1>((sub & 1) != 0, acc[r].a[i], acc[r + 1].a[i]);
            }
            if constexpr (S::kRounds == 4) {
#pragma unroll
                for (int r = 0; r < 2; ++r) exchange_bit<0x4e>((sub & 2) != 0, acc[r].a[i], acc[r + 2].a[i]);
            }
        }
        const int j = (q + (sub & (S::kRounds - 1))) * S::kGroups + grp;
        const bool have = j < min(L, q_end * S::kGroups);
        float* to = out + (size_t)(b0 + lane_row) * L + min(j, L - 1);
        if (nb == kSl) {
            if (have) {
#pragma unroll
                for (int r = 0; r < S::kRounds; ++r)
#pragma unroll
                    for (int i = 0; i < kPer; ++i) to[(size_t)(r * kPer + i) * L] = acc[r].a[i];
            }
        } else {
            const int mine_nb = have ? nb : 0;
#pragma unroll
            for (int r = 0; r < S::kRounds; ++r)
#pragma unroll
                for (int i = 0; i < kPer; ++i)
                    if (lane_row + r * kPer + i < mine_nb) to[(size_t)(r * kPer + i) * L] = acc[r].a[i];
        }
    }
}

// ---- rows put in order of column range ----------------------------------------------------------------------------
// Every row's connections in the order of `ranges` equal column ranges, positions ascending inside a range, padded to whole
// octs with connections that name no column (the gather of one returns zero without touching memory).  Oct r of all rows --
// part r -- is stored in one piece.  Octs of the ordered row and not the ranges themselves: the lists of the lane groups are
// equally long, and the columns of a part still lie close together.
// Eight lanes have a row, each an eighth of it, one connection after the other: a counter per range in a byte of a register
// says where the next connection of that range goes.  Both sides pass through the wavefront's part of LDS, so that memory is
// read and written in whole lines.
//
// What bounds it: memory.  (With the places from ballots, range by range, 3.9 instructions of a wavefront per connection and
// bound by them: 300 us for 670,091 x 72 in fp32, 210 for x 64 in bf16.)
constexpr int kMaxRanges = 16;
constexpr int kMaxRangedFanIn = 256;
constexpr int kRbrRows = 8;                                       // rows per wavefront
// connections per lane: odd, so that the lanes' words fall into different banks
__host__ __device__ constexpr int ranged_share(int K) { return (K + 7) / 8 | 1; }
inline size_t rows_by_range_lds(int K) { return (size_t)4 * kRbrRows * (8 * ranged_share(K) + (K + 7) / 8 * 8) * 2 * sizeof(unsigned); }

template <bool BF16, bool MANY>
__global__ __launch_bounds__(256) void rows_by_range_kernel(const int32_t* __restrict__ idx, const void* __restrict__ w,
                                                            unsigned* __restrict__ idx_out, void* __restrict__ w_out,
                                                            int L, int K, unsigned magic, int ranges) {
    extern __shared__ __align__(16) unsigned rbr_mem[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int share = ranged_share(K), pitch = 8 * share, octs = (K + 7) / 8, out_pitch = octs * 8;
    unsigned* const in_id = rbr_mem + wave * (kRbrRows * (pitch + out_pitch) * 2);
    unsigned* const in_w = in_id + kRbrRows * pitch;
    unsigned* const out_id = in_w + kRbrRows * pitch;
    unsigned* const out_w = out_id + kRbrRows * out_pitch;
    const long long row0 = ((long long)blockIdx.x * 4 + wave) * kRbrRows;
    const int nrows = (int)min((long long)kRbrRows, (long long)L - row0);    // (may be <= 0)
    const int total = nrows * K;
    const unsigned per_row = (1u << 21) / (unsigned)K + 1u;                  // f / K = f * per_row >> 21 for f < 2,560 and K <= 256
    constexpr int kTogether = 8;                                             // loads in flight
    for (int f0 = lane; f0 < total; f0 += 64 * kTogether) {
        unsigned id[kTogether], wv[kTogether];
#pragma unroll
        for (int i = 0; i < kTogether; ++i) {
            const size_t at = (size_t)row0 * K + min(f0 + 64 * i, total - 1);
            id[i] = (unsigned)idx[at];
            wv[i] = BF16 ? (unsigned)reinterpret_cast<const unsigned short*>(w)[at] : reinterpret_cast<const unsigned*>(w)[at];
        }
#pragma unroll
        for (int i = 0; i < kTogether; ++i) {
            const int f = f0 + 64 * i, r = (int)((unsigned)f * per_row >> 21), to = r * pitch + (f - r * K);
            if (f < total) { in_id[to] = id[i]; in_w[to] = wv[i]; }
        }
    }
    __builtin_amdgcn_wave_barrier();                                         // (the memory is the wavefront's own, and LDS serves it in order)
    const int r = lane >> 3, sub = lane & 7;
    const int first = sub * share, n = r < nrows ? min(share, K - first) : 0;
    const unsigned* my_id = in_id + r * pitch + first;
    const unsigned* my_w = in_w + r * pitch + first;
    // any function of the id that never falls would do: this one is the column's range, give or take rounding
    auto range_of = [&](unsigned id) { return min(__umulhi(id, magic), (unsigned)ranges - 1u); };
    // a byte per range: the lane's connections, those of the lanes before it, all of the row's.  (A count of 256 runs over into
    // bytes of ranges that are then empty.)
    unsigned long long lo = 0, hi = 0;
    for (int i = 0; i < n; ++i) {
        const unsigned q = range_of(my_id[i]);
        const unsigned long long one = 1ull << (8 * (q & 7));
        if (MANY && q >= 8) hi += one;
        else lo += one;
    }
    auto before = [&](unsigned long long mine, unsigned long long& row) {
        unsigned long long sum = mine;
#pragma unroll
        for (int d = 1; d < 8; d *= 2) {
            const unsigned long long other = __shfl_up(sum, d, 8);
            if (sub >= d) sum += other;
        }
        row = __shfl(sum, 7, 8);
        return sum - mine;
    };
    unsigned long long lo_row, hi_row = 0;
    const unsigned long long lo_before = before(lo, lo_row), hi_before = MANY ? before(hi, hi_row) : 0;
    constexpr unsigned long long kOnes = 0x0101010101010101ull;
    const unsigned long long lo_upto = lo_row * kOnes;                       // byte q: the row's connections of ranges up to q
    unsigned long long lo_next = (lo_upto << 8) + lo_before;
    unsigned long long hi_next = MANY ? ((hi_row * kOnes) << 8) + (lo_upto >> 56) * kOnes + hi_before : 0;
    for (int i = 0; i < n; ++i) {
        const unsigned id = my_id[i], wv = my_w[i], q = range_of(id), shift = 8 * (q & 7);
        const bool up = MANY && q >= 8;
        const unsigned to = (unsigned)((up ? hi_next : lo_next) >> shift) & 255u;
        if (up) hi_next += 1ull << shift;
        else lo_next += 1ull << shift;
        out_id[r * out_pitch + to] = id;
        out_w[r * out_pitch + to] = wv;
    }
    if (K + sub < out_pitch) {
        out_id[r * out_pitch + K + sub] = ~0u;
        out_w[r * out_pitch + K + sub] = 0u;
    }
    __builtin_amdgcn_wave_barrier();
    for (int f = lane; f < octs * 2 * kRbrRows; f += 64) {
        const int q = f / (2 * kRbrRows), e = f % (2 * kRbrRows);            // oct; quad e & 1 of row e / 2
        if (e >= 2 * nrows) continue;
        const size_t to = (size_t)q * 2 * L + (size_t)row0 * 2 + e;          // (in quads)
        const int from = (e >> 1) * out_pitch + q * 8 + (e & 1) * 4;
        *(reinterpret_cast<uint4*>(idx_out) + to) = *reinterpret_cast<const uint4*>(out_id + from);
        const uint4 v = *reinterpret_cast<const uint4*>(out_w + from);
        if (BF16) reinterpret_cast<uint2*>(w_out)[to] = make_uint2(v.x | v.y << 16, v.z | v.w << 16);
        else reinterpret_cast<uint4*>(w_out)[to] = v;
    }
}

// ---- forward in phases --------------------------------------------------------------------------------------------
// For slices that do not fit an XCD's L2: a workgroup takes 88 M labels -- their sums stay in registers -- and goes through the
// parts of their rows (above: one oct of connections per label and part) in order, the first quads of all labels and then the second, a
// barrier behind either.  All workgroups of
// an XCD begin at the same time and do the same work, so the gathers of a phase hit the few MB of the slice that its part of
// the rows names.
//
// One wavefront brings the lists of all others, two parts ahead and past the registers; the others have nothing but gathers in
// flight.  Loads return in order, and lists that each wavefront asked for itself held its gathers up for the time of the fabric
// once a phase (with their lines marked for one use, which takes longer, the pass went from 2.1 to 2.9 ms).  The gathers of a
// step (sixteen labels, a quad each) are issued before the sums of the step before them, so that a wavefront always has eight in
// flight.  Twelve wavefronts and not sixteen: with 168 registers the sums of 704 labels fit a workgroup, and a slice is gone
// through less often (misses of L2 77 -> 60 M lines in bf16).
//
// A phase of quads, of rows ordered by twice as many ranges as they have octs, names a narrower part of the slice than one of octs
// and one range an oct, and L2 holds more of it: top-5 of 512 samples, 100,000 columns, 670,091 labels of fan-in 64 in bf16 2,258 -> 2,227 us,
// scores of 64 samples, 131,072 columns, 300,000 labels of fan-in 40 166 -> 159, of 190, 60,791, 157,519 and 20 154 -> 153.
//
// What bounds it: the L1, whose address side is busy 89 % of the time in bf16 and 92 in fp32, its data side 96.  670,091 labels,
// against sixteen wavefronts that bring their own lists, 512 labels: 128 samples, 65,536 columns, fan-in 72 in fp32 1,215 -> 1,145 us
// (21.6 TB/s); 512 samples, 100,000 columns, fan-in 64 in bf16 2,112 -> 2,000 us.
constexpr int kPhWaves = 11, kPhThreads = (kPhWaves + 1) * 64;    // wavefronts that walk, and one that brings their lists

// `bytes` (a multiple of 1,024) from the resource's begin on into LDS, past the registers, by one wavefront
__device__ __forceinline__ void bring_to_lds(buffer_rsrc from, unsigned char* to, int bytes, int lane) {
#pragma unroll 4
    for (int t = 0; t < bytes; t += 1024)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(from, (__attribute__((address_space(3))) unsigned char*)to + t, 16, lane * 16 + t, 0, 0, 0);
}

template <bool BF16, int M> struct PhasedShape {                  // M: labels per lane group
    static constexpr int kWaveLabels = 8 * M;
    static constexpr int kLabels = kWaveLabels * kPhWaves;
    static constexpr int kIdBytes = kLabels * 32, kWeightBytes = (kLabels * (BF16 ? 16 : 32) + 1023) / 1024 * 1024;
    static constexpr int kPartBytes = kIdBytes + kWeightBytes;    // a part of the rows: ids, then weights
    static constexpr int kBuffers = 3;
    static constexpr size_t kLdsBytes = (size_t)kBuffers * kPartBytes;
    static_assert(kIdBytes % 1024 == 0, "whole loads of a wavefront");
};

template <bool BF16, int M>
__global__ __launch_bounds__(kPhThreads) void fwd_phased_kernel(const void* __restrict__ table, const unsigned* __restrict__ idx,
                                                                const void* __restrict__ w, const float* __restrict__ bias,
                                                                float* __restrict__ out, int B, int N, int L, int octs, int label_blocks,
                                                                int units, const TopkSink sink) {
    using S = PhasedShape<BF16, M>;
    constexpr int GL = 8, kPer = LaneAcc<BF16>::kSamples, kSl = GL * kPer;
    constexpr unsigned kRow = 128u;
    extern __shared__ __align__(16) unsigned char smem[];
    const int u = xcd_unit(blockIdx.x, units);
    if (u < 0) return;
    const int slice = u / label_blocks;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int sub = lane & (GL - 1), grp = lane / GL;
    const int j0 = (u % label_blocks) * S::kLabels;                                     // first label of the workgroup
    // a barrier that leaves the gathers in flight alone
    auto pace = [] { asm volatile("" ::: "memory"); __builtin_amdgcn_s_barrier(); asm volatile("" ::: "memory"); };
    if (wave == kPhWaves) {
        // Part r of the workgroup's rows into its buffer, past the registers.  Behind the last label nothing is read (the
        // buffers' ends are the resources').
        const size_t left = (size_t)min(S::kLabels, L - j0);
        auto bring = [&](int r) {
            const size_t base = ((size_t)r * L + j0) * 8;
            const buffer_rsrc ri = make_rsrc(idx + base, left * 32), rw = make_rsrc((const char*)w + base * (BF16 ? 2 : 4), left * (BF16 ? 16 : 32));
            unsigned char* to = smem + (size_t)(r % S::kBuffers) * S::kPartBytes;
            bring_to_lds(ri, to, S::kIdBytes, lane);
            bring_to_lds(rw, to + S::kIdBytes, S::kWeightBytes, lane);
        };
        bring(0);
        if (octs > 1) bring(1);
        __builtin_amdgcn_s_waitcnt(0x0f70);                                             // vmcnt(0)
        pace();
        for (int r = 0; r < octs; ++r) {
            if (r + 2 < octs) bring(r + 2);
            pace();                                                                     // (behind the first quads)
            __builtin_amdgcn_s_waitcnt(0x0f70);
            pace();
        }
        __syncthreads();
        return;
    }
    const int jw = j0 + wave * S::kWaveLabels;                                          // first label of this wavefront
    const size_t slice_bytes = (size_t)N * kRow;
    const buffer_rsrc rows = make_rsrc((const char*)table + (size_t)slice * slice_bytes, slice_bytes);
    const unsigned lane_off = (unsigned)sub * 16u;
    LaneAcc<BF16> acc[M];
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
        for (int i = 0; i < kPer; ++i) acc[m].a[i] = 0.f;
    uint4 x[2][8];
    constexpr int kWt = BF16 ? 4 : 8;
    unsigned wt[2][kWt];
    // (entries of no connection hold ~0: behind the slice's end, where a load returns zero without touching memory)
    auto gather = [&](int r, int m, uint4 (&xs)[8], unsigned (&wv)[kWt]) {
        const unsigned char* part = smem + (size_t)(r % S::kBuffers) * S::kPartBytes;
        const int label = wave * S::kWaveLabels + 2 * (m % (M / 2)) * 8 + grp, half = m / (M / 2);
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            const uint4* ids = reinterpret_cast<const uint4*>(part + (label + 8 * p) * 32);
            const unsigned char* ws = part + S::kIdBytes + (label + 8 * p) * (kWt * 4);
            if (BF16) {
                const uint2 e = reinterpret_cast<const uint2*>(ws)[half];
                wv[2 * p] = e.x; wv[2 * p + 1] = e.y;
            } else {
                const uint4 e = reinterpret_cast<const uint4*>(ws)[half];
                wv[kWt / 2 * p] = e.x; wv[kWt / 2 * p + 1] = e.y; wv[kWt / 2 * p + 2] = e.z; wv[kWt / 2 * p + 3] = e.w;
            }
            const uint4 a = ids[half];
            const unsigned at[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
            for (int v = 0; v < 4; ++v)
                xs[4 * p + v] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rows, at[v] * kRow + lane_off, 0, 0));
        }
    };
    pace();
    gather(0, 0, x[0], wt[0]);
    for (int r = 0; r < octs; ++r) {
#pragma unroll
        for (int m = 0; m < M; ++m) {
            if (m + 1 < M) gather(r, m + 1, x[(m + 1) & 1], wt[(m + 1) & 1]);
            else gather(min(r + 1, octs - 1), 0, x[(m + 1) & 1], wt[(m + 1) & 1]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[2 * (m % (M / 2)) + v / 2].add_pair(x[m & 1][2 * v], x[m & 1][2 * v + 1], &wt[m & 1][v * (kWt / 4)]);
            __builtin_amdgcn_sched_barrier(0);
            if (m == M / 2 - 1) pace();
        }
        pace();
    }
    __syncthreads();
    const int b0 = slice * kSl;
    if (sink.tau != nullptr) {
        const int mine0 = b0 + sub * kPer;               // first sample of this lane
        float tau[kPer];
        int tie[kPer];
        topk_thresholds(sink, mine0, tau, tie);
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const int j = jw + m * 8 + grp;
            if (bias != nullptr) {
                const float bj = bias[min(j, L - 1)];
#pragma unroll
                for (int i = 0; i < kPer; ++i) acc[m].a[i] += bj;
            }
            topk_append(sink, acc[m].a, tau, tie, mine0, B - mine0, j, j < L);
        }
        return;
    }
    // a wavefront's labels are consecutive: rows of out leave in pieces of 8 M labels, through the wavefront's part of LDS
    constexpr int kPitch = S::kWaveLabels + 1, kTake = 16;                                     // samples at a time
    float* tile = reinterpret_cast<float*>(smem) + wave * (kTake * kPitch);
    const int nb = min(kSl, B - b0);
    static_assert((size_t)kPhWaves * kTake * kPitch * sizeof(float) <= S::kLdsBytes && kSl % kTake == 0, "the tiles lie in the lists' place");
    for (int s0 = 0; s0 < nb; s0 += kTake) {
        __builtin_amdgcn_wave_barrier();
        if (sub * kPer >= s0 && sub * kPer < s0 + kTake) {
#pragma unroll
            for (int m = 0; m < M; ++m)
#pragma unroll
                for (int i = 0; i < kPer; ++i) tile[(sub * kPer + i - s0) * kPitch + m * 8 + grp] = acc[m].a[i];
        }
        __builtin_amdgcn_wave_barrier();
        const int count = min(kTake, nb - s0) * S::kWaveLabels;
        for (int f = lane; f < count; f += 64) {
            const int e = f / S::kWaveLabels, jl = f - e * S::kWaveLabels, j = jw + jl;
            if (j < L) __builtin_nontemporal_store(bias != nullptr ? tile[e * kPitch + jl] + bias[j] : tile[e * kPitch + jl], out + (size_t)(b0 + s0 + e) * L + j);
        }
    }
}

struct FwdSliced {
    const void* table;             // the slices; the caller's features where the kernel makes them in LDS
    const int32_t* idx;
    const void* w;
    const float* bias;
    float* out;
    int slices, per_group;         // slices; how many of them a workgroup serves with one list
    int row_step;                  // (kernel with the slice in LDS only) row of label j: j * row_step
    bool quads;
    TopkSink sink;
};

template <int GL, bool BF16, int SLICES>
int launch_fwd_sliced(const FwdSliced& a, const Dims& d, hipStream_t s) {
    using S = SlicedShape<GL>;
    const int label_blocks = (d.L + S::kLabels - 1) / S::kLabels, groups = (a.slices + SLICES - 1) / SLICES;
    if ((long long)label_blocks * groups > (1ll << 28)) return FFI_ERR_TOO_LARGE;
    const int units = label_blocks * groups;
    const int chunks = (d.K + S::kChunk - 1) / S::kChunk;
    const int chunk = ((d.K + chunks - 1) / chunks + 7) / 8 * 8;
    const size_t lds = (size_t)GL * LaneAcc<BF16>::kSamples * (S::kLabels + 1) * sizeof(float) / 16 * 16 + 16 +
                       (size_t)S::kRound * list_stride(chunk) * sizeof(uint2);
    const dim3 grid(xcd_grid(units)), block(kSlThreads);
    if (a.quads)
        hipLaunchKernelGGL((fwd_sliced_kernel<GL, BF16, SLICES, true>), grid, block, lds, s, a.table, a.idx, a.w, a.bias, a.out, d.B, d.N, d.L,
                           d.K, a.slices, chunk, label_blocks, units, a.sink);
    else
        hipLaunchKernelGGL((fwd_sliced_kernel<GL, BF16, SLICES, false>), grid, block, lds, s, a.table, a.idx, a.w, a.bias, a.out, d.B, d.N, d.L,
                           d.K, a.slices, chunk, label_blocks, units, a.sink);
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

template <int GL, bool BF16>
int launch_fwd_lds(const FwdSliced& a, const Dims& d, hipStream_t s) {
    using S = LdsShape<GL, BF16>;
    const int chunks = (d.K + S::kChunk - 1) / S::kChunk, chunk = ((d.K + chunks - 1) / chunks + 3) / 4 * 4;
    const int waves = kLdThreads / 64, rounds = (d.L + S::kGroups - 1) / S::kGroups;
    const int streams = std::max(1, std::min((rounds + waves - 1) / waves, device_cu_count() / a.slices));
    const size_t lds = lds_kernel_bytes<GL, BF16>(d.N) + (a.sink.tau != nullptr ? kLdThresholdBytes : 0);
    static_assert(2 * GL * LaneAcc<BF16>::kSamples * 4 <= kLdThresholdBytes, "thresholds of a slice");
    const dim3 grid((unsigned)(streams * a.slices)), block(kLdThreads);
    const int how = a.quads ? kQuads : any_quads_pay<GL>(d.K) ? kAnyQuads : kOneByOne;
    auto go = [&](auto kernel) -> int {
        FFI_HIP_TRY(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        hipLaunchKernelGGL(kernel, grid, block, lds, s, a.table, a.idx, a.w, a.bias, a.out, d.B, d.N, d.L, d.K, d.tp ? 1 : 0, a.row_step, a.slices,
                           streams, chunk, a.sink);
        FFI_HIP_TRY(hipGetLastError());
        return FFI_OK;
    };
    if constexpr (GL == 2 && !BF16)
        if (!d.tp && d.N > 512)
            return how == kQuads ? go(fwd_lds_kernel<GL, BF16, kQuads, true>) : how == kAnyQuads ? go(fwd_lds_kernel<GL, BF16, kAnyQuads, true>) :
                                   go(fwd_lds_kernel<GL, BF16, kOneByOne, true>);
    return how == kQuads ? go(fwd_lds_kernel<GL, BF16, kQuads>) : how == kAnyQuads ? go(fwd_lds_kernel<GL, BF16, kAnyQuads>) :
                           go(fwd_lds_kernel<GL, BF16, kOneByOne>);
}

// the ordered copy of the layer: [ids][weights], part by part
template <bool BF16> size_t phased_rows_bytes(int L, int K) { return (size_t)L * ((K + 7) / 8) * 8 * (4 + sizeof(typename LaneAcc<BF16>::Element)); }

template <bool BF16, int M>
int launch_phased_walk(const FwdSliced& a, const unsigned* rows, const void* row_w, const Dims& d, hipStream_t s) {
    using S = PhasedShape<BF16, M>;
    const int label_blocks = (d.L + S::kLabels - 1) / S::kLabels, units = label_blocks * a.slices;
    FFI_HIP_TRY(hipFuncSetAttribute((const void*)fwd_phased_kernel<BF16, M>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)S::kLdsBytes));
    hipLaunchKernelGGL((fwd_phased_kernel<BF16, M>), dim3(xcd_grid(units)), dim3(kPhThreads), S::kLdsBytes, s, a.table, rows, row_w, a.bias, a.out,
                       d.B, d.N, d.L, (d.K + 7) / 8, label_blocks, units, a.sink);
    FFI_HIP_TRY(hipGetLastError());
    return FFI_OK;
}

int phased_labels(int L, int slices);

template <bool BF16>
int launch_fwd_phased(const FwdSliced& a, const Dims& d, hipStream_t s) {
    const int octs = (d.K + 7) / 8, ranges = std::min(kMaxRanges, 2 * octs);
    unsigned* rows = nullptr;
    FFI_TRY(workspace_get(s, kWsRows, phased_rows_bytes<BF16>(d.L, d.K), (void**)&rows));
    void* row_w = rows + (size_t)d.L * octs * 8;
    const size_t rbr_lds = rows_by_range_lds(d.K);
    const auto rbr = ranges > 8 ? rows_by_range_kernel<BF16, true> : rows_by_range_kernel<BF16, false>;
    FFI_HIP_TRY(hipFuncSetAttribute((const void*)rbr, hipFuncAttributeMaxDynamicSharedMemorySize, (int)rbr_lds));
    hipLaunchKernelGGL(rbr, dim3((unsigned)((d.L + 4 * kRbrRows - 1) / (4 * kRbrRows))), dim3(256), rbr_lds, s, a.idx, a.w, rows, row_w, d.L, d.K,
                       (unsigned)(((unsigned long long)ranges << 32) / (unsigned long long)d.N), ranges);
    FFI_HIP_TRY(hipGetLastError());
    return phased_labels(d.L, a.slices) == 8 ? launch_phased_walk<BF16, 8>(a, rows, row_w, d, s)
                                             : launch_phased_walk<BF16, 4>(a, rows, row_w, d, s);
}

// Rounds of workgroups, one per CU and each with its XCD's share of the work, times the labels of a lane group.
long long phased_cost(int L, int slices, int m) {
    const long long units = ((long long)L + 8 * m * kPhWaves - 1) / (8 * m * kPhWaves) * slices;
    const long long per_xcd = (units + kXcds - 1) / kXcds, cus = std::max(1, device_cu_count() / kXcds);
    return (per_xcd + cus - 1) / cus * m;
}
// As many labels per lane group as the registers hold sums of -- a slice is gone through once a round -- or fewer where that
// leaves CUs idle.
int phased_labels(int L, int slices) { return phased_cost(L, slices, 8) <= phased_cost(L, slices, 4) ? 8 : 4; }

// The phased kernel or the plain one, for slices of 128-byte rows.  In bytes of a gather per 1 TB/s; the rates are what the
// kernels reach at 20,000 to 670,091 labels: plain 20 inside L2 and 5.8 over the share that misses it; in phases 21.5 for rounds
// that fill the CUs, as far as L2 holds what the rows of a phase name -- a part of the slice and some two
// spreads of a row's connection of that number --, ordering the rows 5, two launches.  us, plain and in phases: fp32, 128 samples,
// 65,536 columns, 670,091 labels, fan-in 72: 2,180 and 1,300; 32 samples there 554 and 498, at fan-in 32 243 and 244; 128
// samples, 8,000 labels, fan-in 64 38 and 56; bf16, 64 samples, 65,536 columns, 300,000 labels, fan-in 64 211 and 189; 131,072
// columns, 500,000 labels, fan-in 16 150 and 171; 512 samples, 34,000 columns, 100,000 labels, fan-in 32 178 and 218.
bool takes_phases(size_t slice_bytes, int gl, int slices, int L, int K, int value_bytes) {
    if (gl != 8 || K > kMaxRangedFanIn) return false;
    if (g_options.wide_phases != 0) return g_options.wide_phases > 0;
    if (K <= 8) return false;
    auto rate = [](double peak, double bytes) {
        const double miss = std::max(0.0, 1.0 - (double)kXcdL2Bytes / bytes);
        return miss > 0.0 ? std::min(peak, 5.8 / miss) : peak;
    };
    const double live = (double)slice_bytes * std::min(1.0, 8.0 / K + 0.9 / std::sqrt((double)K));
    const double rounds = (double)phased_cost(L, slices, phased_labels(L, slices)) * 8 * kPhWaves * device_cu_count();     // labels
    const double plain = 128.0 * slices * K * L / rate(20.0, (double)slice_bytes);
    return 128.0 * K * rounds / rate(21.5, live) + 2.0 * K * (4 + value_bytes) * L / 5.0 + 8e6 < plain;
}

// How a forward pass over slices runs: lanes per row, number of slices, and whether a slice lies in LDS (then with as many
// lanes per row as fit; eight otherwise for more than 16 (fp32) or 32 (bf16) samples).
struct SlicedForm {
    int gl, sl, slices;
    bool in_lds;
};
template <bool BF16>
SlicedForm sliced_form(int B, int N) {
    constexpr int kPer = LaneAcc<BF16>::kSamples;
    SlicedForm f;
    f.gl = slice_lanes(B, kPer);
    // (two lanes per row at least: with one the lists of a wavefront are as long as its ids are short of a line; one sample,
    // 670,091 labels: 98 us against 51)
    auto fits = [&](int gl) { return (gl == 8 ? lds_kernel_bytes<8, BF16>(N) : gl == 4 ? lds_kernel_bytes<4, BF16>(N) : lds_kernel_bytes<2, BF16>(N)) <= kLdBudget; };
    f.in_lds = fits(std::max(f.gl, 2));
    if (f.in_lds) f.gl = std::max(f.gl, 2);
    else if (f.gl == 8 && fits(4)) { f.gl = 4; f.in_lds = true; }
    f.sl = f.gl * kPer;
    f.slices = (B + f.sl - 1) / f.sl;
    return f;
}

// the features in slices, in the stream's workspace
template <bool BF16>
int make_table(const void* x, const Dims& d, hipStream_t s, const void** table) {
    const SlicedForm f = sliced_form<BF16>(d.B, d.N);
    if (f.in_lds) { *table = x; return FFI_OK; }
    const size_t slice_bytes = (size_t)d.N * f.gl * 16;
    if (slice_bytes >= 0xffffff00ull) return FFI_ERR_TOO_LARGE;
    void* ws = nullptr;
    FFI_TRY(workspace_get(s, kWsFeaturesT, slice_bytes * f.slices, &ws));
    *table = ws;
    if (BF16) return launch_slices((const unsigned short*)x, (unsigned short*)ws, d.N, d.B, f.sl, d.tp, s);
    return launch_slices((const float*)x, (float*)ws, d.N, d.B, f.sl, d.tp, s);
}

// (`like`, where not 0: the number of labels whose kernel is taken -- a label's score is then the same number)
template <bool BF16>
int forward_wide(const void* table, const int32_t* idx, const void* w, const float* bias, float* out, const TopkSink& sink, const Dims& d,
                 hipStream_t s, int row_step = 1, int like = 0) {
    const SlicedForm f = sliced_form<BF16>(d.B, d.N);
    const size_t slice_bytes = (size_t)d.N * f.gl * 16;
    const bool quads = d.K % 4 == 0 && ((uintptr_t)idx & 15) == 0 && ((uintptr_t)w & (BF16 ? 7 : 15)) == 0;
    const int per_group = (int)std::min<size_t>((size_t)f.slices, kXcdL2Bytes / slice_bytes);
    const FwdSliced a{table, idx, w, bias, out, f.slices, per_group, row_step, quads, sink};
    if (f.in_lds) {
        switch (f.gl) {
            case 2: return launch_fwd_lds<2, BF16>(a, d, s);
            case 4: return launch_fwd_lds<4, BF16>(a, d, s);
            default: return launch_fwd_lds<8, BF16>(a, d, s);
        }
    }
    if (takes_phases(slice_bytes, f.gl, f.slices, like > 0 ? like : d.L, d.K, BF16 ? 2 : 4)) return launch_fwd_phased<BF16>(a, d, s);
    return launch_fwd_sliced_lanes<BF16>(f.gl, a, d, s);
}

}  // namespace

int launch_slices_f32(const float* src, float* dst, int rows, int B, int sl, bool tp, hipStream_t s) {
    return launch_slices(src, dst, rows, B, sl, tp, s);
}

int launch_forward_wide(const float* x, const int32_t* idx, const float* w, const float* bias, float* out, const Dims& d,
                        hipStream_t s) {
    const void* table = nullptr;
    FFI_TRY(make_table<false>(x, d, s, &table));
    return forward_wide<false>(table, idx, w, bias, out, TopkSink{}, d, s);
}

int launch_forward_bf16(const unsigned short* x, const int32_t* idx, const unsigned short* w, float* out, const Dims& d, hipStream_t s) {
    const void* table = nullptr;
    FFI_TRY(make_table<true>(x, d, s, &table));
    return forward_wide<true>(table, idx, w, nullptr, out, TopkSink{}, d, s);
}

void forward_wide_workspaces(const Dims& d, size_t* features, size_t* rows) {
    const SlicedForm f = sliced_form<false>(d.B, d.N);
    const size_t slice_bytes = (size_t)d.N * f.gl * 16;
    *features = f.in_lds ? 0 : slice_bytes * f.slices;
    *rows = !f.in_lds && takes_phases(slice_bytes, f.gl, f.slices, d.L, d.K, 4) ? phased_rows_bytes<false>(d.L, d.K) : 0;
}

// Narrow inputs, fp32: up to 16 samples half or more of a 32-sample tile would be computed for nothing (768 x 670,091 x 32, one to
// 16 samples: 58 -> 50 us, with top-k 110 -> 75; 100 x 500,000 x 17: 36 -> 28; 20 samples and more: no faster than the tile).
bool few_samples(const Dims& d) { return d.B <= 16; }

// ---- top-k without the scores -------------------------------------------------------------------------------------
namespace {

// Every step-th label is in the sample: a sixteenth, whose threshold some 16 k labels reach, but some 2,000 labels at least and 16,384 at
// most.  (16,384 labels of every layer and so, us for the pass: 200 x 30,000 x 30,000 x 30 fp32 128 and 86, 512 x 700 x 20,000 x 30 bf16 86 and 69,
// 8 x 48,006 x 80,864 x 76 fp32 76 and 72.)
constexpr int kTopkSampleMost = 16384, kTopkSampleLeast = 2048, kTopkSampleStep = 16;

// the rows of every step-th label
template <typename T>
__global__ __launch_bounds__(256) void sample_rows_kernel(const int32_t* __restrict__ idx, const T* __restrict__ w, const float* __restrict__ bias,
                                                          int32_t* __restrict__ idx_out, T* __restrict__ w_out, float* __restrict__ bias_out,
                                                          int step, int K, int S) {
    const size_t t = (size_t)blockIdx.x * 256 + threadIdx.x;
    const size_t i = t / (unsigned)K;
    if (i >= (size_t)S) return;
    const size_t j = i * step, at = j * K + (t - i * K);
    idx_out[t] = idx[at];
    w_out[t] = w[at];
    if (bias != nullptr && t == i * K) bias_out[i] = bias[j];
}

// Few scores in short rows: written out and scanned.  The threshold costs the sample's pass, its own launch and a list of candidates
// that many labels of a short row reach; the scan reads each score once (10 MB at most, out of the caches) in two launches.  us for the
// pass by threshold and by scan: 1 x 40,000 x 10,000 x 90 fp32 65 and 36, 16 x 2,000 x 10,000 x 90 bf16 57 and 35, 128 x 2,000 x 10,000 x 90
// fp32 97 and 54, 40 x 2,000 x 65,000 x 40 bf16 50 and 43.  From some four million scores on, or in longer rows, which launch_topk_f32 itself
// takes by a threshold, the scores' way through memory costs more: 128 x 30,000 labels bf16 up to 17 % slower, 12 x 300,000 x 6 32 and 38.
constexpr long long kTopkFewScores = 5LL << 19;

inline bool topk_scans_scores(const Dims& d) {
    return d.L <= kTopkShortRow && (long long)d.B * d.L <= kTopkFewScores && d.B <= 65535;      // (a row of the scan's grid for every sample)
}

// The k-th best of a sample of the labels is a threshold that k labels reach; the same kernel scores the sample and all
// labels, so that a label's score is the same number in both.
template <bool BF16>
int forward_topk_sliced(const void* x, const int32_t* idx, const void* w, const float* bias, const TopkArgs& tk, const Dims& d, hipStream_t s) {
    if (topk_scans_scores(d)) {
        float* scores = nullptr;
        const void* table = nullptr;
        FFI_TRY(workspace_get(s, kWsTopk, (size_t)d.B * d.L * sizeof(float), (void**)&scores));
        FFI_TRY(make_table<BF16>(x, d, s, &table));
        FFI_TRY(forward_wide<BF16>(table, idx, w, bias, scores, TopkSink{}, d, s));
        return launch_topk_f32(scores, d.B, d.L, tk.k, tk.values, tk.indices, s);      // (its lists lie in a slot of their own)
    }
    using T = typename LaneAcc<BF16>::Element;
    const int step = std::max({1, d.L / kTopkSampleMost, std::min(kTopkSampleStep, d.L / kTopkSampleLeast)}), S = std::min(d.L, (d.L + step - 1) / step);
    const size_t rows = (size_t)S * d.K, rows_bytes = (rows * (4 + sizeof(T)) + (size_t)S * 4 + 32) / 16 * 16;
    const bool in_lds = sliced_form<BF16>(d.B, d.N).in_lds;
    unsigned char* ws = nullptr;
    FFI_TRY(workspace_get(s, kWsTopk, topk_candidate_bytes(d.B, S) + 16 + (in_lds ? 0 : rows_bytes), (void**)&ws));
    const TopkCandidates c = topk_candidates_at(ws, d.B, S);
    const void* table = nullptr;
    FFI_TRY(make_table<BF16>(x, d, s, &table));
    Dims ds = d;
    ds.L = S;
    if (in_lds) {
        FFI_TRY(forward_wide<BF16>(table, idx, w, bias, c.sample, TopkSink{}, ds, s, step, d.L));
    } else {
        int32_t* sample_idx = reinterpret_cast<int32_t*>(ws + (topk_candidate_bytes(d.B, S) + 15) / 16 * 16);
        T* sample_w = reinterpret_cast<T*>(sample_idx + (rows + 3) / 4 * 4);
        float* sample_bias = reinterpret_cast<float*>(sample_w + (rows + 3) / 4 * 4);
        hipLaunchKernelGGL(sample_rows_kernel<T>, dim3((unsigned)((rows + 255) / 256)), dim3(256), 0, s, idx, (const T*)w, bias, sample_idx,
                           sample_w, sample_bias, step, d.K, S);
        FFI_HIP_TRY(hipGetLastError());
        FFI_TRY(forward_wide<BF16>(table, sample_idx, sample_w, bias ? sample_bias : nullptr, c.sample, TopkSink{}, ds, s, 1, d.L));
    }
    FFI_TRY(launch_topk_threshold(c.sample, (size_t)S, 1, S, TopkSampleLabels{step, 0}, tk.k, c, d.B, s));
    FFI_TRY(forward_wide<BF16>(table, idx, w, bias, nullptr, TopkSink{c.tau, c.tie, c.count, c.val, c.idx, kTopkCap}, d, s));
    TopkRowSource src;
    src.x = x; src.tp = d.tp; src.bf16 = BF16; src.idx = idx; src.w = w; src.bias = bias; src.N = d.N; src.L = d.L; src.K = d.K;
    return launch_topk_select(c, d.B, tk, src, s);
}

}  // namespace

int launch_forward_topk_sliced(const void* x, const int32_t* idx, const void* w, const float* bias, bool bf16, const TopkArgs& tk, const Dims& d,
                               hipStream_t s) {
    if (takes_topk_direct(d)) return launch_topk_direct(x, idx, w, bias, bf16, tk, d, s);
    return bf16 ? forward_topk_sliced<true>(x, idx, w, bias, tk, d, s) : forward_topk_sliced<false>(x, idx, w, bias, tk, d, s);
}

}  // namespace ffi
