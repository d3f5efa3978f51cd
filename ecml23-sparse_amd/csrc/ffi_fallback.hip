// Kernels that recompute both gradients straight from the lookup matrix, without any preprocessed view of it.
// They are enqueued behind the plan-driven kernels of the stateless backward entry points and run only when the
// device-side check of the lookup (ffi_check.h) found that the cached plan is outdated -- the one call after an
// in-place rewiring (sparse/custom_layer.py:32-43) -- and return at once otherwise.  Semantics:
// tfsparse/cc/kernels/backward.cpp:8-36 (weight gradient) and :39-73 (input gradient).  Ids outside [0, num_features) are
// skipped.  Narrow inputs take one kernel for both gradients and so do wide ones; few samples of many columns, and fan-ins beyond the LDS, plain
// ones whose input gradient scatters with float atomics, as the reference's GPU kernels do (backward.cu.h:119,139,161,182).
#include "ffi_internal.h"
#include "ffi_lds_tile.h"

#include <algorithm>

namespace ffi {
namespace {

constexpr int kFbBlock = 256;

__global__ __launch_bounds__(kFbBlock) void fallback_zero_kernel(const unsigned long long* __restrict__ verdict, float* __restrict__ p,
                                                                 size_t count) {
    if (*verdict != 0) return;
    for (size_t i = (size_t)blockIdx.x * kFbBlock + threadIdx.x; i < count; i += (size_t)gridDim.x * kFbBlock) p[i] = 0.f;
}

// one thread per connection (j,k): gw[j,k] = sum_b x[b, id] * g[b, j], b ascending; gx[b, id] += w[j,k] * g[b, j]
template <bool TP>
__global__ __launch_bounds__(kFbBlock) void fallback_backward_kernel(const unsigned long long* __restrict__ verdict,
                                                                     const float* __restrict__ x, const int32_t* __restrict__ idx,
                                                                     const float* __restrict__ w, const float* __restrict__ g,
                                                                     float* __restrict__ gx, float* __restrict__ gw,
                                                                     float* __restrict__ bias_grad, int B, int N, int L, int K) {
    if (*verdict != 0) return;
    const size_t total = (size_t)L * K;
    for (size_t p = (size_t)blockIdx.x * kFbBlock + threadIdx.x; p < total; p += (size_t)gridDim.x * kFbBlock) {
        const int j = (int)(p / K), k = (int)(p - (size_t)j * K);
        const unsigned id = (unsigned)idx[p];
        const bool ok = id < (unsigned)N;
        const float wv = w[p];
        float acc = 0.f, gsum = 0.f;
        for (int b = 0; b < B; ++b) {
            const float gv = g[(size_t)b * L + j];
            gsum += gv;
            if (ok) {
                const size_t xi = TP ? (size_t)id * B + b : (size_t)b * N + id;
                if (gw != nullptr) acc = fmaf(x[xi], gv, acc);
                if (gx != nullptr) atomicAdd(&gx[xi], wv * gv);
            }
        }
        if (gw != nullptr) gw[p] = acc;
        if (bias_grad != nullptr && k == 0) bias_grad[j] = gsum;
    }
}

// ---- narrow inputs: both gradients in one kernel -------------------------------------------------------------------
// What is launched behind every backward pass and exits at once counts its launches: one of 256 workgroups, where a kernel per
// gradient (and zeros by a third) took 3.8 us each.
//
// Weight gradient: the rows of one batch tile in LDS, a unit of (label, 16 connections) per thread, its sums in registers across
// all batch tiles (ffi_weight_grad.hip).  (32 connections: 54 spilled registers.)
//
// Input gradient: a workgroup takes a stream of label tiles for one batch tile and a window of the columns, a thread per column,
// and sorts each tile's connections by column itself: counts per column (integer LDS atomics), an exclusive scan, then every
// connection takes the next free place of its column's bucket.  Thread t then walks the bucket of column col_lo + t, gathering
// rows of the tile's out_grad from LDS.  No slot balancing (rows lie in label order, so row parities are random and the reads
// run at the 8-clock rate; a wavefront walks as long as its longest bucket), and the order inside a bucket and of the streams is
// whatever the atomics gave: sums are not reproducible bit for bit.  (670,091 labels x fan-in 32 over 768 columns, batch 128: float
// atomics into an LDS tile of gx -- ds_add_f32 retires a third of a lane per clock and CU here, integer atomics seven lanes -- took
// 14.3 ms.)
//
// What bounds it: a CU holds one workgroup, so each of its phases has to have its loads in flight together -- ids and weights eight at
// a time (one: 1,640 us for the pass behind an edit of that layer, 1,450 so), features of [B,N] by four columns of four samples (element
// by element, all to one pair of LDS banks: 2,050) -- and the streams' sums must not wait for each other: atomics on memory with the
// columns side by side (32 x 768 x 131,072 x 32 in [B,N] 184 us; partial sums that the last workgroup of 16 and then the last of all added up,
// each behind a device-scope fence, 400; in 32 bits 170; and with the columns 32 samples apart, in [N,B], 430).
// LDS: gs[tile_labels][32] | ws[tile_labels * K] | lst[tile_labels * K] | cursor[threads] | wave sums[16].
constexpr int kRedoThreads = 1024;
constexpr int kRedoInFlight = 8;      // loads of a thread, in loops that hand each value to LDS
constexpr int kRedoChunk = 16;        // connections per unit of the weight gradient

struct RedoShape {
    int nbt, windows, lower;              // batch tiles; windows of the columns, the first one's size
    int tile_labels, tiles, tiles_per_stream, streams;
    size_t lds;
};
struct RedoArgs {
    const unsigned long long* verdict;
    const float *x, *w, *g;
    const int32_t* idx;
    float *gx, *gw, *bias_grad;           // gx or gw may be null
    double* sums;                         // [window][batch tile][32][lower], zero between launches
    unsigned* tickets;                    // [window][batch tile], zero between launches
    int B, N, L, K;
    RedoShape s;
};

template <bool TP>
__device__ __forceinline__ void redo_weight_grad(const RedoArgs& a, float* xs) {
    const int lane = threadIdx.x & 63, K = a.K, nchunks = (K + kRedoChunk - 1) / kRedoChunk;
    const long long units = (long long)a.L * nchunks;
    for (long long u0 = (long long)blockIdx.x * kRedoThreads; u0 < units; u0 += (long long)gridDim.x * kRedoThreads) {
        const bool mine = u0 + threadIdx.x < units;
        const long long u = min(u0 + (long long)threadIdx.x, units - 1);
        const int j = (int)(u / nchunks), k0 = (int)(u - (long long)j * nchunks) * kRedoChunk;
        const int32_t* irow = a.idx + (size_t)j * K + k0;
        // two 16-bit ids per register; row a.N - 1 in place of ids out of range, whose sums are not kept
        unsigned ids[kRedoChunk / 2], out_of_range = 0;
#pragma unroll
        for (int k = 0; k < kRedoChunk; ++k) {
            const unsigned id = k0 + k < K ? (unsigned)irow[k] : 0u, row = min(id, (unsigned)a.N - 1u);
            ids[k / 2] = (k & 1) ? ids[k / 2] | row << 16 : row;
            out_of_range |= (id >= (unsigned)a.N ? 1u : 0u) << k;
        }
        float res[kRedoChunk], gsum = 0.f;
#pragma unroll
        for (int k = 0; k < kRedoChunk; ++k) res[k] = 0.f;
        for (int bt = 0; bt < a.s.nbt; ++bt) {
            const int b0 = bt * kTileBatch;
            __syncthreads();                                   // everyone is done with the previous tile
            if (TP) {
                stage_rows32<kRedoThreads>(xs, a.x, a.N, a.B, b0);
            } else {
                stage_columns32<kRedoThreads>(xs, a.x, a.N, a.B, b0);
            }
            __syncthreads();
            unsigned skew = (unsigned)(size_t)(__attribute__((address_space(3))) float*)xs + (unsigned)(lane & 7) * 16u;
            asm volatile("" : "+v"(skew));                     // keep the LDS addresses out of loop-invariant hoisting
            float gb[32];
            load_rows32(a.g, a.L, b0, a.B, (unsigned)j, gb);
            if (a.bias_grad != nullptr) {
#pragma unroll
                for (int b = 0; b < 32; ++b) gsum += gb[b];
            }
            xor_permute_groups(gb, lane & 7);                  // match the skewed chunk order of the gathers
#pragma unroll
            for (int k = 0; k < kRedoChunk; ++k) {
                // (four of the row's reads at a time: the registers hold no more)
                const unsigned base = (((k & 1) ? ids[k / 2] >> 16 : ids[k / 2] & 0xffffu) << 7) + skew;
                float sum = res[k];
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const float4 v[4] = {h ? row_chunk<4>(base) : row_chunk<0>(base), h ? row_chunk<5>(base) : row_chunk<1>(base),
                                         h ? row_chunk<6>(base) : row_chunk<2>(base), h ? row_chunk<7>(base) : row_chunk<3>(base)};
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        const float* gc = gb + 16 * h + 4 * c;
                        sum = fmaf(v[c].w, gc[3], fmaf(v[c].z, gc[2], fmaf(v[c].y, gc[1], fmaf(v[c].x, gc[0], sum))));
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
                res[k] = sum;
            }
        }
        if (mine) {
            float* grow = a.gw + (size_t)j * K + k0;
            if (a.bias_grad != nullptr && k0 == 0) a.bias_grad[j] = gsum;
#pragma unroll
            for (int k = 0; k < kRedoChunk; ++k)
                if (k0 + k < K) grow[k] = (out_of_range >> k & 1u) ? 0.f : res[k];
        }
    }
}

template <bool TP>
__device__ __forceinline__ void redo_input_grad(const RedoArgs& a, int item, float* gs) {
    const int K = a.K, L = a.L, tile_labels = a.s.tile_labels;
    const int bt = item % a.s.nbt, stream = item / a.s.nbt % a.s.streams, window = item / (a.s.nbt * a.s.streams);
    const int b0 = bt * kTileBatch, col_lo = window == 0 ? 0 : a.s.lower, ncols = window == 0 ? a.s.lower : a.N - a.s.lower;
    float* ws = gs + (size_t)tile_labels * kTileBatch;
    unsigned* lst = reinterpret_cast<unsigned*>(ws + (size_t)tile_labels * K);
    int* cursor = reinterpret_cast<int*>(lst + (size_t)tile_labels * K);
    int* wave_sum = cursor + kRedoThreads;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const unsigned skewbase = (unsigned)(size_t)(__attribute__((address_space(3))) float*)gs + (unsigned)(lane & 7) * 16u;
    char* gs_bytes = reinterpret_cast<char*>(gs);
    const int t_begin = stream * a.s.tiles_per_stream, t_end = min(t_begin + a.s.tiles_per_stream, a.s.tiles);
    float acc[32];
#pragma unroll
    for (int i = 0; i < 32; ++i) acc[i] = 0.f;
    for (int t = t_begin; t < t_end; ++t) {
        const int j0 = t * tile_labels;
        const int nl = min(tile_labels, L - j0);
        const int total = nl * K;
        const int32_t* src = a.idx + (size_t)j0 * K;
        __syncthreads();                                   // the previous tile is no longer being read
        cursor[threadIdx.x] = 0;
        for (int jl = threadIdx.x; jl < nl; jl += kRedoThreads) {
            float gb[32];
            load_rows32(a.g, L, b0, a.B, (unsigned)(j0 + jl), gb);
            const int r = jl & 7;
            xor_permute_groups(gb, r);
            char* rowp = gs_bytes + ((size_t)jl << 7);
#pragma unroll
            for (int c = 0; c < 8; ++c)
                *reinterpret_cast<float4*>(rowp + ((c ^ r) << 4)) = make_float4(gb[4 * c], gb[4 * c + 1], gb[4 * c + 2], gb[4 * c + 3]);
        }
        for (int q0 = threadIdx.x; q0 < total; q0 += kRedoInFlight * kRedoThreads) {
            float v[kRedoInFlight];
#pragma unroll
            for (int i = 0; i < kRedoInFlight; ++i) v[i] = a.w[(size_t)j0 * K + min(q0 + i * kRedoThreads, total - 1)];
#pragma unroll
            for (int i = 0; i < kRedoInFlight; ++i)
                if (q0 + i * kRedoThreads < total) ws[q0 + i * kRedoThreads] = v[i];
        }
        __syncthreads();
        // the thread's entries e0 + i * kRedoThreads: column inside the window (ids outside [0, N) or outside the window: beyond it)
        auto columns = [&](int e0, unsigned (&c)[kRedoInFlight]) {
#pragma unroll
            for (int i = 0; i < kRedoInFlight; ++i) c[i] = (unsigned)(src[min(e0 + i * kRedoThreads, total - 1)] - col_lo);
#pragma unroll
            for (int i = 0; i < kRedoInFlight; ++i) c[i] = e0 + i * kRedoThreads < total ? c[i] : ~0u;
        };
        for (int e0 = threadIdx.x; e0 < total; e0 += kRedoInFlight * kRedoThreads) {
            unsigned c[kRedoInFlight];
            columns(e0, c);
#pragma unroll
            for (int i = 0; i < kRedoInFlight; ++i)
                if (c[i] < (unsigned)ncols) atomicAdd(&cursor[c[i]], 1);
        }
        __syncthreads();
        // exclusive scan of the counts over the workgroup
        const int mine = cursor[threadIdx.x];
        int incl = mine;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int v = __shfl_up(incl, off, 64);
            if (lane >= off) incl += v;
        }
        if (lane == 63) wave_sum[wave] = incl;
        __syncthreads();
        int before = 0;
        for (int q = 0; q < wave; ++q) before += wave_sum[q];
        const int begin = before + incl - mine;
        cursor[threadIdx.x] = begin;
        __syncthreads();
        {
            // (label of entry e without a division per entry: the thread's entries are kRedoThreads apart)
            int l = (int)threadIdx.x / K, k = (int)threadIdx.x - l * K;
            const int dl = kRedoThreads / K, dk = kRedoThreads - dl * K;
            for (int e0 = threadIdx.x; e0 < total; e0 += kRedoInFlight * kRedoThreads) {
                unsigned c[kRedoInFlight];
                columns(e0, c);
#pragma unroll
                for (int i = 0; i < kRedoInFlight; ++i) {
                    if (c[i] < (unsigned)ncols) lst[atomicAdd(&cursor[c[i]], 1)] = (unsigned)(e0 + i * kRedoThreads) << 10 | (unsigned)l;
                    l += dl; k += dk;
                    if (k >= K) { k -= K; ++l; }
                }
            }
        }
        __syncthreads();
        const int len = cursor[threadIdx.x] - begin;
        int longest = len;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) longest = max(longest, __shfl_xor(longest, off, 64));
        for (int i = 0; i < longest; ++i) {
            if (i < len) {
                const unsigned entry = lst[begin + i];
                const float wv = ws[entry >> 10];
                float4 xv[8];
                read_row(((entry & 1023u) << 7) + skewbase, xv);
                row_fmas(xv, wv, acc);
            }
        }
    }
    xor_permute_groups(acc, lane & 7);
    auto column = [&](int n, int b) -> float& { return a.gx[TP ? (size_t)(col_lo + n) * a.B + b0 + b : (size_t)(b0 + b) * a.N + col_lo + n]; };
    const int nb = min(kTileBatch, a.B - b0);
    if (a.s.streams == 1) {                                    // (few labels, or so many batch tiles that one workgroup each is all)
#pragma unroll
        for (int b = 0; b < kTileBatch; ++b)
            if ((int)threadIdx.x < ncols && b < nb) column(threadIdx.x, b) = acc[b];
        return;
    }
    // The streams add their sums up in memory that is zero between launches, the columns of a sample side by side, in 64 bits (up to 256
    // streams in any order: 3.0e-7 of the result in 32, 1.4e-7 by teams of 16 and so); who adds last takes them from there.  All of that is done by atomics at device scope, which are waited for before the ticket is drawn.
    double* const sums = a.sums + (size_t)(window * a.s.nbt + bt) * ((size_t)a.s.lower * kTileBatch);
#pragma unroll
    for (int b = 0; b < kTileBatch; ++b)
        if ((int)threadIdx.x < ncols && b < nb) unsafeAtomicAdd(&sums[(size_t)b * a.s.lower + threadIdx.x], (double)acc[b]);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    unsigned* const ticket = a.tickets + window * a.s.nbt + bt;
    if (threadIdx.x == 0) wave_sum[0] = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (unsigned)a.s.streams - 1u;
    __syncthreads();
    if (wave_sum[0] == 0) return;
#pragma unroll 8
    for (int e = threadIdx.x; e < nb * ncols; e += kRedoThreads) {
        const int b = e / ncols, n = e - b * ncols;
        column(n, b) = (float)__hip_atomic_exchange(&sums[(size_t)b * a.s.lower + n], 0.0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (threadIdx.x == 0) __hip_atomic_store(ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <bool TP>
__global__ __launch_bounds__(kRedoThreads) void redo_backward_kernel(const RedoArgs a) {
    if (*a.verdict != 0) return;
    extern __shared__ __align__(16) float redo_mem[];
    if (a.gw != nullptr) redo_weight_grad<TP>(a, redo_mem);
    if (a.gx == nullptr) return;
    const int items = a.s.nbt * a.s.streams * a.s.windows;
    for (int item = blockIdx.x; item < items; item += gridDim.x) {
        __syncthreads();
        redo_input_grad<TP>(a, item, redo_mem);
    }
}

// ---- wide inputs: both gradients in one kernel ---------------------------------------------------------------------
// An item is a range of columns and a slice of the samples, whose rows of the features and of their gradient lie in LDS.  Its workgroup reads
// all ids, 32 a thread and step, keeps those of its columns in short lists, a list for every wavefront's ids, and every wavefront takes
// the connections of its own columns (every sixteenth) from all lists: the lanes are the samples, so that no add meets another one.  A
// connection's row of out_grad comes from the slices that the passes over the plan left in their slot; eight are fetched at once.
// Bound by the steps of 32,768 ids, some 15 us each: what 16 wavefronts pick out of the lists, two barriers and a round trip for rows.
// One thread a connection, its samples one by one and its input gradient by atomics in memory (the kernel above), the whole call at
// 128 x 65,536 x 670,091 x 72: 313 ms, 45 so, with 84 to 108 bytes of spills (16 ids a thread, all eight rows fetched also where fewer are left: 64; the next ids
// in registers of their own, 152 bytes of spills: 47); at 50 x 32,768 x 670,000 x 32 51 and 10.2, at 128 x 1,300 x 100,000 x 32 14.9 and 2.8.
constexpr int kOutIds = 32, kOutWaves = 16, kOutThreads = 64 * kOutWaves, kOutList = 256, kOutFetch = 8;
constexpr int kOutTile = 16384;                // floats of a tile
constexpr unsigned kOutStep = kOutIds * kOutThreads, kOutNone = ~0u;

struct OutdatedWide {
    const unsigned long long* verdict;
    const float *x, *w, *g;                    // g: slices [slice][L][sl]
    const int32_t* idx;
    float *gx, *gw;                            // gw (may be null, and x with it): zeros where the verdict is 0
    int B, N, L, K, sl, slices, cols, ranges;
    unsigned inverse_k;                        // 2^32 / K, and one more
};

template <bool TP>
__global__ __launch_bounds__(kOutThreads) void outdated_wide_kernel(const OutdatedWide a) {
    if (*a.verdict != 0) return;
    extern __shared__ __align__(16) float out_mem[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    float* const gxt = out_mem;
    float* const xt = out_mem + a.cols * a.sl;
    unsigned* const list = reinterpret_cast<unsigned*>(xt + a.cols * a.sl);
    int* const len = reinterpret_cast<int*>(list + kOutWaves * kOutList);
    const unsigned total = (unsigned)a.L * (unsigned)a.K;
    for (int item = blockIdx.x; item < a.ranges * a.slices; item += gridDim.x) {
        const int slice = item / a.ranges, c0 = (item - slice * a.ranges) * a.cols, ncols = min(a.cols, a.N - c0);
        if (ncols <= 0) continue;
        const int b0 = slice * a.sl, nb = min(a.sl, a.B - b0);
        auto cell = [&](int n, int b) { return TP ? (size_t)(c0 + n) * a.B + b0 + b : (size_t)(b0 + b) * a.N + c0 + n; };
        auto each = [&](auto f) {              // every column and sample of the item, side by side as they lie in memory
            const int inner = TP ? a.sl : ncols, count = ncols * a.sl;
            for (int e = threadIdx.x; e < count; e += kOutThreads) {
                const int outer = e / inner, in = e - outer * inner;
                f(TP ? outer : in, TP ? in : outer);
            }
        };
        __syncthreads();                       // (the item before this one)
        each([&](int n, int b) {
            gxt[n * a.sl + b] = 0.f;
            xt[n * a.sl + b] = a.gw != nullptr && b < nb ? a.x[cell(n, b)] : 0.f;
        });
        const float* const rows = a.g + (size_t)slice * a.L * a.sl + min(lane, a.sl - 1);
        int ids[kOutIds];
        auto fetch = [&](unsigned first, int (&v)[kOutIds]) {
#pragma unroll
            for (int q = 0; q < kOutIds / 4; ++q) {
                const unsigned at = first + (unsigned)wave * (64u * kOutIds) + (unsigned)q * 256u + (unsigned)lane * 4u;
                if (at + 4u <= total) {
                    const i32x4_unaligned four = *reinterpret_cast<const i32x4_unaligned*>(a.idx + at);
                    v[4 * q] = four.x; v[4 * q + 1] = four.y; v[4 * q + 2] = four.z; v[4 * q + 3] = four.w;
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i) v[4 * q + i] = at + i < total ? a.idx[at + i] : -1;
                }
            }
        };
        fetch(0, ids);
        __syncthreads();
        for (unsigned first = 0; first < total; first += kOutStep) {
            int from = 0;
            bool more;
            do {
                // a list takes the ids of four rows at least; what it has no room for goes into the next round
                int n = 0, to = from;
#pragma unroll
                for (int u = 0; u < kOutIds; ++u) {
                    if (u < from || n > kOutList - 64) continue;
                    const unsigned col = (unsigned)ids[u] - (unsigned)c0;
                    const bool hit = ids[u] >= 0 && col < (unsigned)ncols;
                    const unsigned long long hits = __ballot(hit);
                    to = u + 1;
                    if (hits == 0) continue;
                    const int at = n + __builtin_amdgcn_mbcnt_hi((unsigned)(hits >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)hits, 0));
                    if (hit) list[wave * kOutList + at] = col << 15 | (unsigned)wave << 11 | (unsigned)((u >> 2) * 256 + lane * 4 + (u & 3));
                    n += (int)__popcll(hits);
                }
                if (from < kOutIds && to == kOutIds && first + kOutStep < total) fetch(first + kOutStep, ids);      // (on their way through the rest of the step)
                from = to;
                if (lane == 0) len[wave] = n;
                more = __syncthreads_or(from < kOutIds) != 0;
                // sixteen entries of every list at a time
                for (int t = 0;; t += 16) {
                    unsigned e[4];
                    unsigned long long mine[4];
                    bool left = false;
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int l = i * 4 + (lane >> 4), at = t + (lane & 15), entries = len[l];
                        e[i] = at < entries ? list[l * kOutList + at] : kOutNone;
                        mine[i] = __ballot(e[i] != kOutNone && (int)((e[i] >> 15) & (kOutWaves - 1)) == wave);
                        left |= entries > t + 16;
                    }
                    while ((mine[0] | mine[1] | mine[2] | mine[3]) != 0) {
                        unsigned at[kOutFetch], p[kOutFetch];
                        float gv[kOutFetch], wv[kOutFetch];
#pragma unroll
                        for (int h = 0; h < kOutFetch; ++h) {
                            unsigned v = kOutNone;
#pragma unroll
                            for (int i = 3; i >= 0; --i)
                                if (mine[i] != 0) v = (unsigned)__builtin_amdgcn_readlane((int)e[i], (int)__builtin_ctzll(mine[i]));
                            bool taken = false;
#pragma unroll
                            for (int i = 0; i < 4; ++i) {
                                if (!taken && mine[i] != 0) {
                                    mine[i] &= mine[i] - 1;
                                    taken = true;
                                }
                            }
                            p[h] = kOutNone;
                            if (v == kOutNone) continue;
                            p[h] = first + (v & 32767u);
                            at[h] = (v >> 15) * (unsigned)a.sl;
                            unsigned label = a.K > 1 ? __umulhi(p[h], a.inverse_k) : p[h];         // p / K, or one more
                            label -= label * (unsigned)a.K > p[h] ? 1u : 0u;
                            gv[h] = rows[(size_t)label * a.sl];
                            wv[h] = a.w[p[h]];
                        }
                        float dot = 0.f;
                        unsigned where = kOutNone;
#pragma unroll
                        for (int h = 0; h < kOutFetch; ++h) {
                            if (p[h] == kOutNone) continue;
                            float d = 0.f;
                            if (lane < a.sl) {
                                const unsigned o = at[h] + (unsigned)lane;
                                gxt[o] = fmaf(wv[h], gv[h], gxt[o]);
                                d = xt[o] * gv[h];
                            }
                            if (a.gw == nullptr) continue;
#pragma unroll
                            for (int off = 32; off > 0; off >>= 1) d += __shfl_xor(d, off, 64);
                            if (lane == h) { dot = d; where = p[h]; }
                        }
                        if (where != kOutNone) unsafeAtomicAdd(a.gw + where, dot);      // (the other slices' sums)
                    }
                    if (!__any(left)) break;
                }
                __syncthreads();
            } while (more);
        }
        if (a.gx != nullptr)
            each([&](int n, int b) {
                if (b < nb) a.gx[cell(n, b)] = gxt[n * a.sl + b];
            });
    }
}

// Items so that the rounds of all CUs are full, a tile's room permitting.  Every item reads all ids, whatever the samples: few samples
// of many columns keep the kernel above.  ms for the call by that and by this one, of one round: 4 x 131,072 x 300,000 x 40 2.7 and 5.8,
// 8 of them 5.0 and 5.9, 32 x 131,072 x 100,000 x 30 4.8 and 1.5; 512 x 100,000 x 4,000 x 30, thirteen rounds, 3.6 and 1.3.
bool outdated_wide_shape(const ffi_plan* p, const Dims& d, OutdatedWide* a) {
    a->sl = 256 / p->members;
    a->slices = (d.B + a->sl - 1) / a->sl;
    const int cus = device_cu_count(), most = kOutTile / a->sl;
    const long long rounds = ((long long)((d.N + most - 1) / most) * a->slices + cus - 1) / cus;
    a->ranges = (int)std::min<long long>(d.N, std::max<long long>((d.N + most - 1) / most, rounds * cus / a->slices));
    a->cols = (d.N + a->ranges - 1) / a->ranges;
    return (long long)a->ranges * a->slices < (1ll << 31) && 12 * rounds <= d.B;
}

size_t redo_lds_bytes(int tile_labels, int K) {
    return (size_t)tile_labels * (kTileBatch * sizeof(float) + 8u * (size_t)K) + (size_t)kRedoThreads * 4u + 64u;
}

// Whether the kernel above takes the shape -- inputs that fit the LDS tile, fan-ins whose tile of one label fits beside it -- and how.
bool redo_shape(const Dims& d, RedoShape* s) {
    s->nbt = (d.B + kTileBatch - 1) / kTileBatch;
    s->windows = d.N > kRedoThreads ? 2 : 1;
    s->lower = s->windows == 1 ? d.N : ((d.N + 1) / 2 + 63) / 64 * 64;
    if (!tile_path_fits(d.N) || d.N > 2 * kRedoThreads || d.L >= (1 << 25) || redo_lds_bytes(1, d.K) > kPlanLdsBudget)
        return false;
    // as many labels per tile as the LDS holds (entries keep the label in 10 bits), then evened out so that every
    // workgroup of a batch tile gets the same number of tiles
    const size_t per_label = kTileBatch * sizeof(float) + 8u * (size_t)d.K;
    int tl = (int)std::min<size_t>(1023, (kPlanLdsBudget - redo_lds_bytes(0, d.K)) / per_label);
    const int streams0 = std::max(1, device_cu_count() / std::max(1, s->nbt));
    const int tiles0 = (d.L + tl - 1) / tl;
    s->tiles_per_stream = (tiles0 + streams0 - 1) / streams0;
    if (tiles0 > streams0) tl = std::min(tl, (int)(((long long)d.L + (long long)s->tiles_per_stream * streams0 - 1) / ((long long)s->tiles_per_stream * streams0)));
    s->tile_labels = tl;
    s->tiles = (d.L + tl - 1) / tl;
    s->streams = (s->tiles + s->tiles_per_stream - 1) / s->tiles_per_stream;
    s->lds = std::max(redo_lds_bytes(tl, d.K), tile_lds_bytes(d.N));
    return s->streams == 1 || (long long)s->nbt * s->windows <= kTicketCount;
}

}  // namespace

size_t backward_if_outdated_workspace(const Dims& d) {
    RedoShape s;
    return redo_shape(d, &s) && s.streams > 1 ? (size_t)s.windows * s.nbt * s.lower * kTileBatch * sizeof(double) : 0;
}

int backward_if_outdated_prepare(const Dims& d, hipStream_t s) {
    void* ws = nullptr;
    const size_t bytes = backward_if_outdated_workspace(d);
    if (bytes == 0) return FFI_OK;
    FFI_TRY(zeroed_get(s, kWsSums, bytes, &ws));
    return tickets_get(s, &ws);
}

bool takes_outdated_wide(const ffi_plan* p, const Dims& d) {
    OutdatedWide a;
    RedoShape r;
    return !p->tiled && !redo_shape(d, &r) && outdated_wide_shape(p, d, &a);
}

int launch_outdated_wide(const ffi_plan* p, const float* x, const int32_t* idx, const float* w, const float* g_slices, float* gx, float* gw,
                         const Dims& d, hipStream_t s) {
    OutdatedWide a{};
    if (!outdated_wide_shape(p, d, &a)) return FFI_ERR_BAD_ARGUMENT;
    a.verdict = p->d_guard + kGuardVerdict;
    a.x = x; a.w = w; a.g = g_slices; a.idx = idx; a.gx = gx; a.gw = x != nullptr ? gw : nullptr;
    a.B = d.B; a.N = d.N; a.L = d.L; a.K = d.K;
    a.inverse_k = d.K > 1 ? (unsigned)((1ull << 32) / (unsigned)d.K) + 1u : 0u;
    const size_t lds = ((size_t)2 * a.cols * a.sl + kOutWaves * kOutList + kOutWaves) * sizeof(float);
    const auto kernel = d.tp ? outdated_wide_kernel<true> : outdated_wide_kernel<false>;
    FFI_HIP_TRY(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(kernel, dim3((unsigned)std::min(device_cu_count(), a.ranges * a.slices)), dim3(kOutThreads), lds, s, a);
    FFI_HIP_TRY(hipGetLastError());
    return FFI_OK;
}

int launch_backward_if_outdated(const unsigned long long* verdict, const float* features, const int32_t* lookup,
                                const float* weights, const float* out_grad, float* feature_grad, float* weight_grad,
                                float* bias_grad, const Dims& d, bool zeroed, hipStream_t s) {
    const int cus = device_cu_count();
    float* gw = features != nullptr ? weight_grad : nullptr;
    float* gb = features != nullptr ? bias_grad : nullptr;
    RedoArgs a{};
    if (redo_shape(d, &a.s)) {
        a.verdict = verdict;
        a.x = features; a.w = weights; a.g = out_grad; a.idx = lookup;
        a.gx = feature_grad; a.gw = gw; a.bias_grad = gb;
        a.B = d.B; a.N = d.N; a.L = d.L; a.K = d.K;
        if (a.s.streams > 1) {
            FFI_TRY(zeroed_get(s, kWsSums, backward_if_outdated_workspace(d), (void**)&a.sums));
            FFI_TRY(tickets_get(s, (void**)&a.tickets));
        }
        const auto kernel = d.tp ? redo_backward_kernel<true> : redo_backward_kernel<false>;
        FFI_HIP_TRY(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)a.s.lds));
        const int items = std::min(a.s.nbt * a.s.streams * a.s.windows, 4 * cus);
        hipLaunchKernelGGL(kernel, dim3((unsigned)std::max(cus, items)), dim3(kRedoThreads), a.s.lds, s, a);
        FFI_HIP_TRY(hipGetLastError());
        return FFI_OK;
    }
    if (feature_grad != nullptr && !zeroed) {
        hipLaunchKernelGGL(fallback_zero_kernel, dim3(cus), dim3(kFbBlock), 0, s, verdict, feature_grad, (size_t)d.B * d.N);
        FFI_HIP_TRY(hipGetLastError());
    }
    if (d.tp)
        hipLaunchKernelGGL(fallback_backward_kernel<true>, dim3(cus * 2), dim3(kFbBlock), 0, s, verdict, features, lookup, weights,
                           out_grad, feature_grad, gw, gb, d.B, d.N, d.L, d.K);
    else
        hipLaunchKernelGGL(fallback_backward_kernel<false>, dim3(cus * 2), dim3(kFbBlock), 0, s, verdict, features, lookup, weights,
                           out_grad, feature_grad, gw, gb, d.B, d.N, d.L, d.K);
    FFI_HIP_TRY(hipGetLastError());
    return FFI_OK;
}

}  // namespace ffi
