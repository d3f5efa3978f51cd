// Backward pass for inputs whose tile does not fit in LDS (more than 1,216 columns), and for any other shape whose plan has the
// global form: both gradients in one walk over the plan's lists, out_grad gathered from slices that an XCD's L2 holds a block of
// labels of at a time (ffi_sliced.h); and the weight gradient alone, straight from the lookup, whose gathers of whole rows of the
// batch-major features come through the cache hierarchy.
#include "ffi_internal.h"
#include "ffi_lds_tile.h"
#include "ffi_sliced.h"

#include <algorithm>

namespace ffi {
namespace {

constexpr int kWideThreads = 256;   // 4 wavefronts per workgroup
constexpr int kWideLabels = 64;     // labels per workgroup: 16 per wavefront
constexpr int kWideBatch = 128;     // batch entries per pass: each lane owns b and b+64
constexpr int kWideInflight = 8;      // connections whose gathers a wavefront has in flight
constexpr int kWideStride = kWideBatch + 1;   // LDS row stride in floats (odd: conflict-free both ways)

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    return v;
}

// ---- weight gradient ----------------------------------------------------------------------------
// grid (label blocks).  Per batch pass the workgroup brings g[b, j0..j0+63] into LDS (coalesced
// along labels), then every wavefront handles 16 labels: per connection one 512-byte piece of the
// xT row times the label's out_grad, summed over the lanes, accumulated over the batch passes in
// LDS by a single lane (fixed order: reproducible).
template <bool TWO>
__global__ __launch_bounds__(kWideThreads) void wgrad_wide_kernel(const float* __restrict__ xT,
                                                                  const int32_t* __restrict__ idx,
                                                                  const float* __restrict__ g, float* __restrict__ gw,
                                                                  float* __restrict__ bias_grad, int B, int N, int L,
                                                                  int K, int ldb) {
    extern __shared__ float smem[];
    float* gt = smem;                                   // [64 labels][129]
    float* res = smem + kWideLabels * kWideStride;      // [64 labels][K]
    float* bres = res + kWideLabels * K;                // [64 labels] column sums of out_grad
    if (threadIdx.x < kWideLabels) bres[threadIdx.x] = 0.f;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int j0 = blockIdx.x * kWideLabels;
    const buffer_rsrc xr = make_rsrc(xT, (size_t)N * (size_t)ldb * sizeof(float));
    const unsigned row_bytes = (unsigned)ldb * 4u;
    for (int t = threadIdx.x; t < kWideLabels * K; t += kWideThreads) res[t] = 0.f;
    for (int bc0 = 0; bc0 < B; bc0 += kWideBatch) {
        __syncthreads();
        {
            const int jl = threadIdx.x & 63;
            const bool in = j0 + jl < L;
            for (int bb = threadIdx.x >> 6; bb < (TWO ? kWideBatch : kWideBatch / 2); bb += kWideThreads / 64) {
                const int b = bc0 + bb;
                gt[jl * kWideStride + bb] = (in && b < B) ? g[(size_t)b * L + j0 + jl] : 0.f;
            }
        }
        __syncthreads();
        const unsigned lane_off0 = (unsigned)(bc0 + lane) * 4u, lane_off1 = lane_off0 + 256u;
        // lanes past the end of the batch would read the next row of xT: their out_grad is zero, but
        // keep their x operand finite too
        const bool in0 = bc0 + lane < B, in1 = bc0 + 64 + lane < B;
        for (int q = 0; q < kWideLabels / 4; ++q) {
            const int jl = wave * (kWideLabels / 4) + q;
            const int j = j0 + jl;
            if (j >= L) break;                                  // wave-uniform
            const float g0 = gt[jl * kWideStride + lane], g1 = TWO ? gt[jl * kWideStride + 64 + lane] : 0.f;
            if (bias_grad != nullptr) {                         // wave-uniform
                const float gs = wave_sum(g0 + g1);
                if (lane == 0) bres[jl] += gs;
            }
            const int32_t* irow = idx + (size_t)j * K;
            for (int k0 = 0; k0 < K; k0 += 64) {
                const int kn = min(64, K - k0);
                const unsigned iv = (lane < kn) ? (unsigned)irow[k0 + lane] : 0u;
                float mine = 0.f;                               // lane k collects connection k0+k
                int k = 0;
                for (; k + kWideInflight <= kn; k += kWideInflight) {
                    float x0[kWideInflight], x1[kWideInflight];
#pragma unroll
                    for (int u = 0; u < kWideInflight; ++u) {
                        const unsigned n = (unsigned)__builtin_amdgcn_readlane((int)iv, k + u);
                        x0[u] = buffer_load_f32(xr, lane_off0, n * row_bytes);
                        x1[u] = TWO ? buffer_load_f32(xr, lane_off1, n * row_bytes) : 0.f;
                    }
#pragma unroll
                    for (int u = 0; u < kWideInflight; ++u) {
                        const float p = TWO ? fmaf(in1 ? x1[u] : 0.f, g1, (in0 ? x0[u] : 0.f) * g0) : (in0 ? x0[u] : 0.f) * g0;
                        const float s = wave_sum(p);
                        if (lane == k + u) mine = s;
                    }
                }
                if (k < kn) {
                    // (the last, partly filled group: gathers in flight together, the connections behind the end repeat
                    // the last one and are not kept)
                    float x0[kWideInflight], x1[kWideInflight];
#pragma unroll
                    for (int u = 0; u < kWideInflight; ++u) {
                        const unsigned n = (unsigned)__builtin_amdgcn_readlane((int)iv, min(k + u, kn - 1));
                        x0[u] = buffer_load_f32(xr, lane_off0, n * row_bytes);
                        x1[u] = TWO ? buffer_load_f32(xr, lane_off1, n * row_bytes) : 0.f;
                    }
#pragma unroll
                    for (int u = 0; u < kWideInflight; ++u) {
                        if (k + u < kn) {                       // wave-uniform
                            const float p = TWO ? fmaf(in1 ? x1[u] : 0.f, g1, (in0 ? x0[u] : 0.f) * g0) : (in0 ? x0[u] : 0.f) * g0;
                            const float s = wave_sum(p);
                            if (lane == k + u) mine = s;
                        }
                    }
                }
                if (lane < kn) res[jl * K + k0 + lane] += mine;
            }
        }
    }
    __syncthreads();
    for (int t = threadIdx.x; t < kWideLabels * K; t += kWideThreads) {
        const int jl = t / K;
        if (j0 + jl < L) gw[(size_t)j0 * K + t] = res[t];
    }
    if (bias_grad != nullptr && threadIdx.x < kWideLabels && j0 + (int)threadIdx.x < L) bias_grad[j0 + threadIdx.x] = bres[threadIdx.x];
}

// ---- input gradient and weight gradient over the plan's global form ------------------------------------------------
// Column n's gradient sums w * g[label] over its connections; the weight gradient of a connection is the dot product of
// x[n] and g[label].  Both need row `label` of out_grad, so one walk over the lists of the plan gathers it once: GL lanes of
// 16 bytes hold a row of a slice of out_grad (ffi_sliced.h), a wavefront owns M x (64 / GL) columns -- their sums stay in
// LDS -- and goes through the label blocks of its stream in order.  All workgroups of an XCD do so
// at the same pace, so the block's rows of out_grad (a few MB) are what the L2 holds.
//
// A lane group copies its list through LDS, a window of a few octs of slots at a time, the next window on its way while it
// walks.  Weight gradients leave in the order of the plan's slots
// (weight_grads_in_place_kernel moves them).
//
// What bounds it: L2 delivery of the gathered rows (31 TB/s at most) and, with DOT, the instructions beside it (per oct and
// lane 64 multiply-adds, 21 for the sums over the lanes, 8 gathers).
constexpr int kWalkThreads = kWalkColumns * 8;
constexpr int kWalkMaxM = 4;
// octs per window of a lane group, quads of it that a lane brings, and the window's place in LDS (16-byte words, one more
// than it holds: the groups read from different banks)
constexpr int walk_octs(int gl) { return gl >= 4 ? 4 : gl; }
constexpr int walk_quads(int gl) { return walk_octs(gl) * 2 / gl; }
constexpr int walk_stride(int gl) { return walk_octs(gl) * 4 + 1; }

// v + (v of the lane that CTRL pairs with this one)
template <int CTRL> __device__ __forceinline__ float dpp_add(float keep, float send) {
    return keep + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, send), CTRL, 0xf, 0xf, true));
}

// Sums eight values over the GL lanes of a group; lane `sub` is left with values sub * (8 / GL) ... of them, in p[0 ... 8 / GL).
template <int GL> __device__ __forceinline__ void group_sums(float (&p)[8], int sub) {
    constexpr int kHalfMirror = 0x141, kQuadMirror = 0x1b, kQuadSwap = 0xb1;    // lanes i <-> 7 - i, 3 - i, i ^ 1
    if constexpr (GL == 8) {
        const bool up = (sub & 4) != 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) p[i] = dpp_add<kHalfMirror>(up ? p[i + 4] : p[i], up ? p[i] : p[i + 4]);
    }
    if constexpr (GL >= 4) {
        constexpr int n = GL == 8 ? 2 : 4;
        const bool up = (sub & 2) != 0;
#pragma unroll
        for (int i = 0; i < n; ++i) p[i] = dpp_add<kQuadMirror>(up ? p[i + n] : p[i], up ? p[i] : p[i + n]);
    }
    if constexpr (GL >= 2) {
        constexpr int n = GL == 8 ? 1 : GL == 4 ? 2 : 4;
        const bool up = (sub & 1) != 0;
#pragma unroll
        for (int i = 0; i < n; ++i) p[i] = dpp_add<kQuadSwap>(up ? p[i + n] : p[i], up ? p[i] : p[i + n]);
    }
}

template <int GL, bool DOT>
__global__ __launch_bounds__(kWalkThreads) void walk_columns_kernel(const float* __restrict__ gtab, const float* __restrict__ xtab,
                                                                    const unsigned* __restrict__ oct_ptr,
                                                                    const unsigned short* __restrict__ slot_lab,
                                                                    const float* __restrict__ slot_w, float* __restrict__ gx_part,
                                                                    float* __restrict__ gw_slots, int add_gw, size_t slots, int N, int L,
                                                                    int nblocks, int block_labels, int blocks_per_stream, int col_chunks,
                                                                    int units, int M) {
    constexpr int kGroups = 64 / GL;
    constexpr unsigned kRow = GL * 16u;
    constexpr unsigned kNoRow = 0xffffff00u;
    constexpr int kOcts = walk_octs(GL), kQuads = walk_quads(GL);
    // per wavefront: its groups' windows of (row offset, weight) pairs, two per entry, and the sums of its M x 64 lanes
    extern __shared__ __align__(16) uint4 walk_mem[];
    const int u = xcd_unit(blockIdx.x, units);
    if (u < 0) return;
    const int chunk = u % col_chunks, stream = u / col_chunks;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int sub = lane & (GL - 1), grp = lane / GL;
    const int n0 = (chunk * (kWalkThreads / 64) + wave) * M * kGroups;     // first column of this wavefront
    if (n0 >= N) return;                                                    // (the barriers below count the wavefronts that are left)
    uint4* const wave_mem = walk_mem + wave * (kGroups * walk_stride(GL) + 64 * M);
    uint4* list = wave_mem + grp * walk_stride(GL);
    float4* sums = reinterpret_cast<float4*>(wave_mem + kGroups * walk_stride(GL)) + lane;
    const unsigned lane_off = (unsigned)sub * 16u;
    for (int m = 0; m < M; ++m) sums[64 * m] = make_float4(0.f, 0.f, 0.f, 0.f);
    const int blk_end = min((stream + 1) * blocks_per_stream, nblocks);
    int blk = stream * blocks_per_stream;
    // octs of this lane group's list of (blk, m), and its column's row of x (fetched anew for every block: held for all m
    // it would cost a wavefront per SIMD); columns behind the last have no octs
    auto list_of = [&](int b, int m, unsigned& begin, unsigned& end, float4& x) {
        const size_t at = (size_t)b * N;
        const int n = n0 + m * kGroups + grp;
        begin = oct_ptr[at + min(n, N)];
        end = oct_ptr[at + min(n + 1, N)];
        if (DOT) x = *reinterpret_cast<const float4*>(xtab + (size_t)min(n, N - 1) * (GL * 4) + sub * 4);
    };
    uint4 next_w[kQuads];
    uint2 next_lab[kQuads];
    auto fetch = [&](unsigned oct) {                                        // (behind the plan's end: its last quad)
#pragma unroll
        for (int v = 0; v < kQuads; ++v) {
            const size_t at = min((size_t)oct * 8 + 4 * (v * GL + sub), slots - 4);
            next_w[v] = *reinterpret_cast<const uint4*>(slot_w + at);
            next_lab[v] = *reinterpret_cast<const uint2*>(slot_lab + at);
        }
    };
    unsigned begin = 0, end = 0;
    float4 xv = make_float4(0.f, 0.f, 0.f, 0.f);
    if (blk < blk_end) {
        list_of(blk, 0, begin, end, xv);
        fetch(begin);
    }
    for (; blk < blk_end; ++blk) {
        __syncthreads();
        const int label0 = blk * block_labels;
        const buffer_rsrc rsrc = make_rsrc(gtab + (size_t)label0 * (GL * 4), (size_t)min(block_labels, L - label0) * kRow);
#pragma unroll 1
        for (int m = 0; m < M; ++m) {
            float4 acc = sums[64 * m];
            int longest = (int)(end - begin);
#pragma unroll
            for (int off = 32; off >= GL; off >>= 1) longest = max(longest, __shfl_xor(longest, off));
            longest = __builtin_amdgcn_readfirstlane(longest);
            unsigned after_begin = 0, after_end = 0;                        // the lists that follow
            float4 after_x = make_float4(0.f, 0.f, 0.f, 0.f);
            if (m + 1 < M) list_of(blk, m + 1, after_begin, after_end, after_x);
            else if (blk + 1 < blk_end) list_of(blk + 1, 0, after_begin, after_end, after_x);
            for (int w0 = 0; w0 < longest || w0 == 0; w0 += kOcts) {
                __builtin_amdgcn_wave_barrier();                            // (the windows are the wavefront's own: LDS serves it in order)
                const unsigned at = begin + (unsigned)w0;
                const int here = min(kOcts, (int)(end - at));               // octs of this group's list in this window (<= 0: none)
                float4 gw_old[DOT ? kQuads : 1];
#pragma unroll
                for (int v = 0; v < kQuads; ++v) {
                    const int q = v * GL + sub;
                    const uint2 lab = next_lab[v];
                    const unsigned l0 = lab.x & 0xffffu, l1 = lab.x >> 16, l2 = lab.y & 0xffffu, l3 = lab.y >> 16;
                    list[2 * q] = make_uint4(l0 == kNoLabel ? kNoRow : l0 * kRow, next_w[v].x, l1 == kNoLabel ? kNoRow : l1 * kRow, next_w[v].y);
                    list[2 * q + 1] = make_uint4(l2 == kNoLabel ? kNoRow : l2 * kRow, next_w[v].z, l3 == kNoLabel ? kNoRow : l3 * kRow, next_w[v].w);
                    if (DOT) {
                        gw_old[v] = make_float4(0.f, 0.f, 0.f, 0.f);
                        if (add_gw && q < 2 * here) gw_old[v] = *reinterpret_cast<const float4*>(gw_slots + (size_t)at * 8 + 4 * q);
                    }
                }
                fetch(w0 + kOcts < longest ? at + kOcts : after_begin);
                __builtin_amdgcn_wave_barrier();
                const int steps = min(kOcts, longest - w0);
#pragma unroll 1
                for (int i = 0; i < steps; ++i) {
                    if (i < here) {
                        uint4 e[4], x[8];
#pragma unroll
                        for (int v = 0; v < 4; ++v) e[v] = list[4 * i + v];
#pragma unroll
                        for (int v = 0; v < 8; ++v)
                            x[v] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, ((v & 1) ? e[v / 2].z : e[v / 2].x) + lane_off, 0, 0));
                        float p[8];
#pragma unroll
                        for (int v = 0; v < 8; ++v) {
                            const float wv = __uint_as_float((v & 1) ? e[v / 2].w : e[v / 2].y);
                            const float r0 = __uint_as_float(x[v].x), r1 = __uint_as_float(x[v].y), r2 = __uint_as_float(x[v].z), r3 = __uint_as_float(x[v].w);
                            acc.x = fmaf(wv, r0, acc.x); acc.y = fmaf(wv, r1, acc.y);
                            acc.z = fmaf(wv, r2, acc.z); acc.w = fmaf(wv, r3, acc.w);
                            if (DOT) p[v] = fmaf(xv.w, r3, fmaf(xv.z, r2, fmaf(xv.y, r1, xv.x * r0)));
                        }
                        if (DOT) {
                            group_sums<GL>(p, sub);
#pragma unroll
                            for (int v = 0; v < 8 / GL; ++v) reinterpret_cast<float*>(list + 4 * i)[sub * (8 / GL) + v] = p[v];   // (in place of the oct)
                        }
                    }
                }
                if (DOT) {
                    __builtin_amdgcn_wave_barrier();
#pragma unroll
                    for (int v = 0; v < kQuads; ++v) {
                        const int q = v * GL + sub;
                        if (q < 2 * here) {
                            const float4 d = *reinterpret_cast<const float4*>(list + 4 * (q >> 1) + (q & 1));
                            *reinterpret_cast<float4*>(gw_slots + (size_t)at * 8 + 4 * q) =
                                make_float4(gw_old[v].x + d.x, gw_old[v].y + d.y, gw_old[v].z + d.z, gw_old[v].w + d.w);
                        }
                    }
                }
            }
            sums[64 * m] = acc;
            begin = after_begin; end = after_end; xv = after_x;
        }
    }
    for (int m = 0; m < M; ++m) {
        const int n = n0 + m * kGroups + grp;
        if (n < N)
            *reinterpret_cast<float4*>(gx_part + ((size_t)stream * N + n) * (GL * 4) + sub * 4) = sums[64 * m];
    }
}

typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

// slot_w[slot] = the weight of the slot's connection (0 in padding).  Slots are dealt to the XCDs in eight consecutive
// ranges: an XCD reads the weights of one label block after the other, which its L2 holds.
__global__ __launch_bounds__(256) void slot_weights_kernel(const float* __restrict__ w, const int32_t* __restrict__ slot_pos,
                                                           float* __restrict__ slot_w, size_t slots, int units) {
    const int u = xcd_unit(blockIdx.x, units);
    if (u < 0) return;
    const size_t q = (size_t)u * 256 + threadIdx.x;
    if (q * 4 >= slots) return;
    // (what is touched once goes past the L2, which the gathered array needs: 395 -> 369 us at 670,091 labels x fan-in 72)
    const v4i at = __builtin_nontemporal_load(reinterpret_cast<const v4i*>(slot_pos) + q);
    v4f v;
    v.x = w[max(at.x, 0)]; v.y = w[max(at.y, 0)]; v.z = w[max(at.z, 0)]; v.w = w[max(at.w, 0)];
    if (at.x < 0) v.x = 0.f;
    if (at.y < 0) v.y = 0.f;
    if (at.z < 0) v.z = 0.f;
    if (at.w < 0) v.w = 0.f;
    __builtin_nontemporal_store(v, reinterpret_cast<v4f*>(slot_w) + q);
}

// gw[pos] = gw_slots[pos_slot[pos]]; positions are dealt to the XCDs like the slots above.  (Reads at random places: the same
// permutation as scattered writes, from the slots' side, took twice as long.)
__global__ __launch_bounds__(256) void weight_grads_in_place_kernel(const float* __restrict__ gw_slots, const unsigned* __restrict__ pos_slot,
                                                                    float* __restrict__ gw, size_t count, int units) {
    const int u = xcd_unit(blockIdx.x, units);
    if (u < 0) return;
    const size_t p0 = ((size_t)u * 256 + threadIdx.x / 64 * 64) * 4 + (threadIdx.x & 63);
    float v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = gw_slots[__builtin_nontemporal_load(pos_slot + min(p0 + 64 * i, count - 1))];
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (p0 + 64 * i < count) __builtin_nontemporal_store(v[i], gw + p0 + 64 * i);
}

// gx ([N,B] or [B,N]) = sum over the streams of part[slice][stream][n][sl], ascending; 32 columns x 32 samples per workgroup
template <bool TP>
__global__ __launch_bounds__(256) void gather_gx_kernel(const float* __restrict__ part, float* __restrict__ gx, int N, int B, int sl,
                                                        int streams) {
    __shared__ float tile[32][33];
    const int n0 = blockIdx.x * 32, b0 = blockIdx.y * 32;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    for (int i = ty; i < 32; i += 8) {
        const int n = n0 + i, b = b0 + tx;
        float v = 0.f;
        if (n < N && b < B)
            for (int t = 0; t < streams; ++t) v += part[(((size_t)(b / sl) * streams + t) * N + n) * sl + b % sl];
        if (TP) {
            if (n < N && b < B) gx[(size_t)n * B + b] = v;
        } else {
            tile[i][tx] = v;
        }
    }
    if (TP) return;
    __syncthreads();
    for (int i = ty; i < 32; i += 8) {
        const int n = n0 + tx, b = b0 + i;
        if (n < N && b < B) gx[(size_t)b * N + n] = tile[tx][i];
    }
}

// bias_grad[j] = sum over the samples of g[b, j]: 64 labels per workgroup, four partial sums added in order
__global__ __launch_bounds__(256) void column_sums_kernel(const float* __restrict__ g, float* __restrict__ bias_grad, int B, int L) {
    __shared__ float part[4][64];
    const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
    const int j = blockIdx.x * 64 + tx;
    float v = 0.f;
    if (j < L)
        for (int b = ty; b < B; b += 4) v += g[(size_t)b * L + j];
    part[ty][tx] = v;
    __syncthreads();
    if (ty == 0 && j < L) bias_grad[j] = ((part[0][tx] + part[1][tx]) + part[2][tx]) + part[3][tx];
}

struct WalkArgs {
    const float *gtab, *xtab, *slot_w;
    float *gx_part, *gw_slots;
    bool add_gw;
    int streams, blocks_per_stream;
};

template <int GL, bool DOT>
int launch_walk(int m, const ffi_plan* p, const WalkArgs& a, hipStream_t s) {
    const int wg_cols = kWalkThreads / 64 * m * (64 / GL), col_chunks = (p->N + wg_cols - 1) / wg_cols;
    const int units = col_chunks * a.streams;
    const size_t lds = (size_t)(kWalkThreads / 64) * (64 / GL * walk_stride(GL) + 64 * m) * sizeof(uint4);
    FFI_HIP_TRY(hipFuncSetAttribute((const void*)walk_columns_kernel<GL, DOT>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL((walk_columns_kernel<GL, DOT>), dim3(xcd_grid(units)), dim3(kWalkThreads), lds, s, a.gtab, a.xtab, p->oct_ptr,
                       p->slot_lab, a.slot_w, a.gx_part, a.gw_slots, a.add_gw ? 1 : 0, (size_t)p->slots, p->N, p->L, p->nblocks,
                       p->block_labels, a.blocks_per_stream, col_chunks, units, m);
    FFI_HIP_TRY(hipGetLastError());
    return FFI_OK;
}

template <bool DOT>
int launch_walk_gl(int gl, int m, const ffi_plan* p, const WalkArgs& a, hipStream_t s) {
    if (gl == 1) return launch_walk<1, DOT>(m, p, a, s);
    if (gl == 2) return launch_walk<2, DOT>(m, p, a, s);
    if (gl == 4) return launch_walk<4, DOT>(m, p, a, s);
    return launch_walk<8, DOT>(m, p, a, s);
}

}  // namespace

// Row stride (in floats) of the library's own [rows][batch] copies: a multiple of 32, so that rows start on 128-byte
// lines and a gathered row piece touches as few lines as it can.
int wide_row_stride(int B) { return (B + 31) / 32 * 32; }

bool wide_offsets_fit(long long rows, long long B) { return rows * wide_row_stride((int)B) * 4 < (1ll << 32); }

namespace {

// xT[N][ldb] for the wide kernels: the caller's [N,B] buffer itself when its rows are aligned already, else a copy.
int wide_features(const float* x, const Dims& d, hipStream_t s, const float** xT, int* ldb) {
    const int ld = wide_row_stride(d.B);
    if (d.tp && ld == d.B) { *xT = x; *ldb = d.B; return FFI_OK; }
    float* ws = nullptr;
    FFI_TRY(workspace_get(s, kWsFeaturesT, (size_t)d.N * ld * sizeof(float), (void**)&ws));
    if (d.tp) {
        FFI_HIP_TRY(hipMemcpy2DAsync(ws, (size_t)ld * sizeof(float), x, (size_t)d.B * sizeof(float), (size_t)d.B * sizeof(float),
                                     (size_t)d.N, hipMemcpyDeviceToDevice, s));
    } else {
        FFI_TRY(launch_transpose(x, ws, d.B, d.N, s, d.N, ld));     // [B,N] -> [N,ld]
    }
    *xT = ws;
    *ldb = ld;
    return FFI_OK;
}

}  // namespace

int launch_weight_grad_wide(const float* x, const int32_t* idx, const float* g, float* gw, float* bias_grad, const Dims& d,
                            hipStream_t s) {
    if (!wide_offsets_fit(d.N, d.B)) return FFI_ERR_TOO_LARGE;
    const size_t lds = ((size_t)kWideLabels * kWideStride + (size_t)kWideLabels * d.K + kWideLabels) * sizeof(float);
    if (lds > 150 * 1024) return FFI_ERR_TOO_LARGE;               // fan-in beyond ~450
    const float* xT = nullptr;
    int ldb = 0;
    FFI_TRY(wide_features(x, d, s, &xT, &ldb));
    const dim3 grid((d.L + kWideLabels - 1) / kWideLabels);
    if (d.B > 64) {
        FFI_HIP_TRY(hipFuncSetAttribute((const void*)wgrad_wide_kernel<true>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        hipLaunchKernelGGL(wgrad_wide_kernel<true>, grid, dim3(kWideThreads), lds, s, xT, idx, g, gw, bias_grad, d.B, d.N, d.L, d.K, ldb);
    } else {
        FFI_HIP_TRY(hipFuncSetAttribute((const void*)wgrad_wide_kernel<false>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        hipLaunchKernelGGL(wgrad_wide_kernel<false>, grid, dim3(kWideThreads), lds, s, xT, idx, g, gw, bias_grad, d.B, d.N, d.L, d.K, ldb);
    }
    FFI_HIP_TRY(hipGetLastError());
    return FFI_OK;
}

// How the walk is cut: columns per lane group (m) and streams of label blocks, so that about 16 wavefronts per CU are in
// flight: as many columns per group as that allows (a walk of all blocks each), else several streams whose sums are added.
void walk_shape(int N, int B, int L, int nblocks, int* gl, int* slices, int* m, int* streams, int* blocks_per_stream) {
    *gl = slice_lanes(B, 4);
    *slices = (B + *gl * 4 - 1) / (*gl * 4);
    const long long target = device_cu_count();                             // workgroups
    const int group_cols = kWalkThreads / *gl;                              // columns per workgroup and m
    *m = kWalkMaxM;
    while (*m > 1 && (long long)(N + group_cols * *m - 1) / (group_cols * *m) < target) *m /= 2;
    const long long wgs = (N + group_cols * *m - 1) / (group_cols * *m);
    const int want = (int)std::min<long long>(nblocks, std::max<long long>(1, target / wgs));
    *blocks_per_stream = (nblocks + want - 1) / want;
    *streams = (nblocks + *blocks_per_stream - 1) / *blocks_per_stream;
}

int launch_backward_wide(const ffi_plan* p, const float* x, const float* w, const float* g, float* gx, float* gw, float* bias_grad, int B,
                         bool tp, hipStream_t s) {
    if (!p->oct_ptr || !p->slot_pos || !p->slot_lab) return FFI_ERR_BAD_ARGUMENT;
    // (before anything is enqueued: a refused call leaves its outputs alone)
    const dim3 gx_grid((unsigned)((p->N + 31) / 32), (unsigned)(((long long)B + 31) / 32));
    if (gx_grid.y > 65535u) return FFI_ERR_TOO_LARGE;
    const bool dot = gw != nullptr;
    int gl, slices, m;
    WalkArgs a{};
    walk_shape(p->N, B, p->L, p->nblocks, &gl, &slices, &m, &a.streams, &a.blocks_per_stream);
    const int sl = gl * 4;
    const size_t slots = (size_t)p->slots, count = (size_t)p->L * p->K, gslice = (size_t)p->L * sl, part = (size_t)p->N * sl * a.streams;
    float* ws = nullptr;
    FFI_TRY(workspace_get(s, kWsPartials, (gslice + part) * slices * sizeof(float), (void**)&ws));
    float* slot_w = nullptr;
    FFI_TRY(workspace_get(s, kWsSlots, slots * sizeof(float), (void**)&slot_w));
    FFI_TRY(launch_slices_f32(g, ws, p->L, B, sl, false, s));
    float* const parts = ws + gslice * slices;
    float* xtab = nullptr;
    if (dot) {
        FFI_TRY(workspace_get(s, kWsFeaturesT, (size_t)p->N * sl * slices * sizeof(float), (void**)&xtab));
        FFI_TRY(launch_slices_f32(x, xtab, p->N, B, sl, tp, s));
        FFI_TRY(workspace_get(s, kWsWeightParts, slots * sizeof(float), (void**)&a.gw_slots));
    }
    const int slot_units = (int)((slots / 4 + 255) / 256);
    hipLaunchKernelGGL(slot_weights_kernel, dim3(xcd_grid(slot_units)), dim3(256), 0, s, w, p->slot_pos, slot_w, slots, slot_units);
    FFI_HIP_TRY(hipGetLastError());
    // one slice after the other: their weight gradients add up in place
    a.slot_w = slot_w;
    for (int q = 0; q < slices; ++q) {
        a.gtab = ws + gslice * q; a.gx_part = parts + part * q; a.add_gw = q > 0;
        a.xtab = dot ? xtab + (size_t)p->N * sl * q : nullptr;
        FFI_TRY(dot ? launch_walk_gl<true>(gl, m, p, a, s) : launch_walk_gl<false>(gl, m, p, a, s));
    }
    if (dot) {
        const int units = (int)((count + 1023) / 1024);
        hipLaunchKernelGGL(weight_grads_in_place_kernel, dim3(xcd_grid(units)), dim3(256), 0, s, a.gw_slots, p->pos_slot, gw, count, units);
        FFI_HIP_TRY(hipGetLastError());
    }
    if (bias_grad != nullptr) {
        hipLaunchKernelGGL(column_sums_kernel, dim3((unsigned)((p->L + 63) / 64)), dim3(256), 0, s, g, bias_grad, B, p->L);
        FFI_HIP_TRY(hipGetLastError());
    }
    if (tp) hipLaunchKernelGGL(gather_gx_kernel<true>, gx_grid, dim3(256), 0, s, parts, gx, p->N, B, sl, a.streams);
    else hipLaunchKernelGGL(gather_gx_kernel<false>, gx_grid, dim3(256), 0, s, parts, gx, p->N, B, sl, a.streams);
    FFI_HIP_TRY(hipGetLastError());
    return FFI_OK;
}

}  // namespace ffi
