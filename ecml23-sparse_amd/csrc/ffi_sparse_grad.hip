// Backward pass for an out_grad that is mostly exact zeros (a hinge loss late in training: every
// satisfied margin has gradient 0).  The reference's GPU kernels skip such entries one by one
// (`if(out == 0) continue`, tfsparse/cc/kernels/backward.cu.h:73,94,131,151); here the zero pattern is
// made explicit once, as bit masks, and the kernels walk the set bits only:
//
//   words[t][j]      bit i set  <=>  out_grad[32 t + i, j] may be non-zero          (per label: weight gradient)
//   bits[b][j / 64]  bit j % 64 set  <=>  the same for sample b                      (per sample: input gradient)
//
//   nz_scan_kernel          words from out_grad
//   nz_count_kernel, nz_count_finish_kernel   the number of set bits (two steps, no atomics)
//   nz_transpose_kernel     bits from words
//   wgrad_adam_kernel       wgrad_sparse_kernel and the Adam step on all rows, those without a set bit included
//   wgrad_sparse_kernel     a wavefront lists the labels of its block that have a set bit, then lane <-> listed
//                           label: every lane walks the set bits of its own label and keeps 32 sums (one chunk of
//                           connections) in registers; labels with many set bits are done by the whole wavefront
//                           afterwards, lane <-> connection; rows of labels without a set bit come out as zeros
//   igrad_sparse_kernel     one workgroup per (sample, label segment): a wavefront lists the set bits of a chunk of
//                           the sample's bit row, every lane takes listed labels and adds g * w of the label's
//                           connections into per-wavefront accumulators gx[n] in LDS (LDS float adds issued in a
//                           fixed order)
//   igrad_sparse_reduce_kernel  sums the segments in ascending order into feature_grad
#include "ffi_adam.h"
#include "ffi_internal.h"
#include "ffi_lds_tile.h"

#include <algorithm>
#include <mutex>
#include <vector>

namespace ffi {
namespace {

constexpr int kScanThreads = 256;
constexpr int kCountBlocks = 1024;

__global__ __launch_bounds__(kScanThreads) void nz_scan_kernel(const float* __restrict__ g, unsigned* __restrict__ words,
                                                               int B, int L) {
    // two labels per thread (j and j + kScanThreads): 64 independent loads in flight
    const int j0 = blockIdx.x * (2 * kScanThreads) + threadIdx.x;
    const int t = blockIdx.y;
    const int rows = min(32, B - 32 * t);
    const float* tile = g + (size_t)(32 * t) * L;
    float v[2][32];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int j = min(j0 + h * kScanThreads, L - 1);
#pragma unroll
        for (int i = 0; i < 32; ++i) v[h][i] = i < rows ? tile[(size_t)i * L + j] : 0.f;
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int j = j0 + h * kScanThreads;
        unsigned m = 0;
#pragma unroll
        for (int i = 0; i < 32; ++i) m |= (v[h][i] != 0.f ? 1u : 0u) << i;
        if (j < L) words[(size_t)t * L + j] = m;
    }
}

// g[32 t + i, j] = 0 wherever bit i of words[t][j] is clear (thread <-> label, rows written 256 bytes per wavefront).
__global__ __launch_bounds__(kScanThreads) void nz_zero_unmasked_kernel(float* __restrict__ g, const unsigned* __restrict__ words,
                                                                        int B, int L) {
    const int j = blockIdx.x * kScanThreads + threadIdx.x;
    const int t = blockIdx.y;
    if (j >= L) return;
    const int rows = min(32, B - 32 * t);
    const unsigned m = words[(size_t)t * L + j];
    float* col = g + (size_t)(32 * t) * L + j;
#pragma unroll
    for (int i = 0; i < 32; ++i)
        if (i < rows && !((m >> i) & 1u)) col[(size_t)i * L] = 0.f;
}

__global__ __launch_bounds__(kScanThreads) void nz_count_kernel(const unsigned* __restrict__ words, size_t n,
                                                                unsigned long long* __restrict__ block_counts) {
    __shared__ unsigned red[kScanThreads / 64];
    unsigned c = 0;
    const size_t stride = (size_t)gridDim.x * kScanThreads;
    size_t i = (size_t)blockIdx.x * kScanThreads + threadIdx.x;
    for (; i + 3 * stride < n; i += 4 * stride) {       // four loads in flight
        const unsigned a0 = words[i], a1 = words[i + stride], a2 = words[i + 2 * stride], a3 = words[i + 3 * stride];
        c += __popc(a0) + __popc(a1) + __popc(a2) + __popc(a3);
    }
    for (; i < n; i += stride) c += __popc(words[i]);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) c += __shfl_xor(c, off, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long t = 0;
        for (int i = 0; i < kScanThreads / 64; ++i) t += red[i];
        block_counts[blockIdx.x] = t;
    }
}

__global__ __launch_bounds__(kCountBlocks) void nz_count_finish_kernel(const unsigned long long* __restrict__ block_counts, int n,
                                                                       unsigned long long* __restrict__ host_count) {
    __shared__ unsigned long long red[kCountBlocks / 64];
    unsigned long long t = (int)threadIdx.x < n ? block_counts[threadIdx.x] : 0ull;       // n <= kCountBlocks
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) t += __shfl_xor(t, off, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = t;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long all = 0;
        for (int i = 0; i < kCountBlocks / 64; ++i) all += red[i];
        *host_count = all;                              // pinned host memory: the host reads it after the stream has drained
    }
}

// One wavefront per (batch tile t, kTransposeBlocks blocks of 64 labels): bits[32 t + i][blk] = bit i of the block's 64
// words.  Each half of the wavefront transposes its 32 x 32 bit matrix in five exchange steps between lanes (blocks of
// 16, 8, 4, 2, 1 swapped across the diagonal); lane i < 32 then holds sample i's bits of labels 0..31 and lane 32 + i those
// of labels 32..63.  The words of all blocks are requested before the first is used.
constexpr int kTransposeBlocks = 16;
__global__ __launch_bounds__(kScanThreads) void nz_transpose_kernel(const unsigned* __restrict__ words,
                                                                    unsigned long long* __restrict__ bits, int B, int L,
                                                                    int nwords) {
    __shared__ unsigned long long staged[kScanThreads / 64][32][kTransposeBlocks + 1];   // per wavefront: [sample][block]
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int blk0 = (blockIdx.x * (kScanThreads / 64) + wv) * kTransposeBlocks;
    const int t = blockIdx.y;
    if (blk0 >= nwords) return;
    unsigned m[kTransposeBlocks];
#pragma unroll
    for (int q = 0; q < kTransposeBlocks; ++q) {
        const int j = (blk0 + q) * 64 + lane;
        m[q] = words[(size_t)t * L + min(j, L - 1)];
        if (j >= L) m[q] = 0u;
    }
#pragma unroll
    for (int q = 0; q < kTransposeBlocks; ++q) {
        unsigned v = m[q];
#pragma unroll
        for (int step = 0; step < 5; ++step) {
            const int sh = 16 >> step;
            const unsigned low = step == 0 ? 0x0000ffffu : step == 1 ? 0x00ff00ffu : step == 2 ? 0x0f0f0f0fu
                               : step == 3 ? 0x33333333u : 0x55555555u;
            const unsigned other = (unsigned)__shfl_xor((int)v, sh, 64);
            v = (lane & sh) ? ((v & ~low) | ((other & ~low) >> sh)) : ((v & low) | ((other & low) << sh));
        }
        const unsigned upper = (unsigned)__shfl_xor((int)v, 32, 64);
        if (lane < 32) staged[wv][lane][q] = (unsigned long long)v | ((unsigned long long)upper << 32);
    }
    __builtin_amdgcn_wave_barrier();            // (LDS operations of a wavefront complete in order)
    // a sample's kTransposeBlocks words are neighbours in its bit row: 128-byte pieces, four samples per store
    const int q = lane & (kTransposeBlocks - 1);
#pragma unroll
    for (int r = 0; r < 32 / (64 / kTransposeBlocks); ++r) {
        const int i = r * (64 / kTransposeBlocks) + lane / kTransposeBlocks;
        const int b = 32 * t + i;
        if (b < B && blk0 + q < nwords) bits[(size_t)b * nwords + blk0 + q] = staged[wv][i][q];
    }
}

constexpr int kHeavyBits = 12;     // labels with more set bits than this are left to the whole wavefront

// x is addressed as x[b * xsb + n * xsn] (either layout; byte strides), through a buffer resource with 32-bit
// offsets: batch * num_features * 4 < 2^32, checked by the launcher.
// ZERO_FILL == true: rows of labels without a set bit (and their bias gradients) are written as zeros.
// ZERO_FILL == false: they are left alone.
// `done(labels listed, how many, first label of the block)` comes behind each block of kWsBlock labels.  Returns the set bits that
// the lane's labels had.
constexpr int kWsLabelsPerLane = 4;                  // at most
constexpr int kWsBlock = 64 * kWsLabelsPerLane;      // labels a wavefront looks at in one go

struct SparseRows {
    const float* x;
    unsigned xsb, xsn;
    const int32_t* idx;
    const float* g;
    const unsigned* words;
    float* gw;
    float* bias_grad;
    int B, N, L, K, nbt;
    int per_lane;                  // labels of a lane: 1, 2 or kWsLabelsPerLane
};

template <bool VEC4, bool ZERO_FILL, class Done>
__device__ __forceinline__ unsigned sparse_rows(const SparseRows& r, int block, int nblocks, Done done) {
    const float* __restrict__ x = r.x;
    const int32_t* __restrict__ idx = r.idx;
    const float* __restrict__ g = r.g;
    const unsigned* __restrict__ words = r.words;
    float* gw = r.gw;
    float* bias_grad = r.bias_grad;
    const unsigned xsb = r.xsb, xsn = r.xsn;
    const int B = r.B, N = r.N, L = r.L, K = r.K, nbt = r.nbt;
    // per wavefront: the labels of its block that have a set bit, as (set bits << 8) | offset in the block.  Most labels
    // have none when the gradient is sparse; the lanes then work on the compacted list, not on 64 neighbouring labels of
    // which a few are busy.
    __shared__ unsigned active_list[4][kWsBlock];
    unsigned set_bits = 0;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int wave = block * 4 + wv;
    const int nwaves = nblocks * 4;
    const int block_labels = 64 * r.per_lane, nblk = (L + block_labels - 1) / block_labels;
    const unsigned tail = (B & 31) ? (1u << (B & 31)) - 1u : 0xffffffffu;   // bits past the batch are ignored
    const buffer_rsrc xr = make_rsrc(x, (size_t)B * (size_t)N * sizeof(float));
    unsigned* mylist = active_list[wv];
    for (int blk = wave; blk < nblk; blk += nwaves) {
        const int block_base = blk * block_labels;
        int cnts[kWsLabelsPerLane];
#pragma unroll
        for (int q = 0; q < kWsLabelsPerLane; ++q) cnts[q] = 0;
        for (int t = 0; t < nbt; ++t) {
#pragma unroll
            for (int q = 0; q < kWsLabelsPerLane; ++q) {
                if (q >= r.per_lane) break;                             // (uniform)
                unsigned m = words[(size_t)t * L + min(block_base + q * 64 + lane, L - 1)];
                if (t == nbt - 1) m &= tail;
                cnts[q] += __popc(m);
            }
        }
        int total = 0;
#pragma unroll
        for (int q = 0; q < kWsLabelsPerLane; ++q) {
            const int base = block_base + q * 64;
            if (base >= L || q >= r.per_lane) break;                // wave-uniform
            const int rows = min(64, L - base);
            const bool mine = lane < rows;
            const int cnt = cnts[q];
            if (ZERO_FILL) {
                // rows of labels without a set bit: zeros, written by the whole wavefront (the rows of 64 neighbouring
                // labels are contiguous in gw).  The row of 16-byte element e is e / (K/4), formed in floating point
                // (exact here: e + 0.5 is at least 0.5 / (K/4) away from a multiple).
                const unsigned long long zero_rows = __ballot(mine && cnt == 0);
                float* blockrows = gw + (size_t)base * K;
                if (VEC4) {
                    const int k4 = K / 4;
                    const float inv_k4 = 1.f / (float)k4;
                    for (int e = lane; e < rows * k4; e += 64)
                        if ((zero_rows >> (int)(((float)e + 0.5f) * inv_k4)) & 1ull)
                            reinterpret_cast<float4*>(blockrows)[e] = make_float4(0.f, 0.f, 0.f, 0.f);
                } else {
                    for (int e = lane; e < rows * K; e += 64)
                        if ((zero_rows >> (e / K)) & 1ull) blockrows[e] = 0.f;
                }
                if (bias_grad != nullptr && mine && cnt == 0) bias_grad[base + lane] = 0.f;
            }
            if (mine) set_bits += (unsigned)cnt;
            const bool busy = mine && cnt > 0;
            const unsigned long long bal = __ballot(busy);
            if (busy) mylist[total + __popcll(bal & ((1ull << lane) - 1ull))] = ((unsigned)cnt << 8) | (unsigned)(q * 64 + lane);
            total += __popcll(bal);
        }
        __builtin_amdgcn_wave_barrier();        // (LDS operations of a wavefront complete in order)
        for (int e0 = 0; e0 < total; e0 += 64) {
        const bool mine = e0 + lane < total;
        const unsigned entry = mylist[min(e0 + lane, total - 1)];
        const int j = block_base + (int)(entry & 255u);
        const int cnt = (int)(entry >> 8);
        const bool heavy = cnt > kHeavyBits;
        const bool light = mine && !heavy;
        // ---- every lane its own label ----
        float gsum = 0.f;
        for (int k0 = 0; k0 < K; k0 += 32) {
            unsigned ids[32];
            if (light) {
                if (VEC4 && k0 + 32 <= K) {
#pragma unroll
                    for (int q = 0; q < 8; ++q) {
                        const int4 v = *reinterpret_cast<const int4*>(idx + (size_t)j * K + k0 + 4 * q);
                        ids[4 * q] = (unsigned)v.x; ids[4 * q + 1] = (unsigned)v.y; ids[4 * q + 2] = (unsigned)v.z; ids[4 * q + 3] = (unsigned)v.w;
                    }
                } else {
#pragma unroll
                    for (int k = 0; k < 32; ++k) ids[k] = k0 + k < K ? (unsigned)idx[(size_t)j * K + k0 + k] : 0u;
                }
                // column ids -> byte offsets of the columns in x
#pragma unroll
                for (int k = 0; k < 32; ++k) ids[k] = (ids[k] < (unsigned)N ? ids[k] : 0u) * xsn;
            } else {
#pragma unroll
                for (int k = 0; k < 32; ++k) ids[k] = 0u;
            }
            float acc[32];
#pragma unroll
            for (int k = 0; k < 32; ++k) acc[k] = 0.f;
            // the label's mask words, eight batch tiles at a time in registers; every step each lane takes the
            // next set bit of its own label (g and the 32 gathered x values are requested together)
            for (int tb = 0; tb < nbt; tb += 8) {
                unsigned mw[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const int t = tb + u;
                    mw[u] = (light && t < nbt) ? words[(size_t)t * L + j] : 0u;
                    if (t == nbt - 1) mw[u] &= tail;
                }
                for (;;) {
                    int usel = -1;
                    unsigned msel = 0;
#pragma unroll
                    for (int u = 7; u >= 0; --u)
                        if (mw[u]) { usel = u; msel = mw[u]; }
                    if (!__ballot(usel >= 0)) break;
                    if (usel >= 0) {
                        const int b = 32 * (tb + usel) + __ffs((int)msel) - 1;
#pragma unroll
                        for (int u = 0; u < 8; ++u)
                            if (u == usel) mw[u] = msel & (msel - 1);
                        const float gv = g[(size_t)b * L + j];
                        const unsigned xrow = (unsigned)b * xsb;
                        // 16 gathers in flight at a time
#pragma unroll
                        for (int h = 0; h < 2; ++h) {
                            float xv[16];
#pragma unroll
                            for (int k = 0; k < 16; ++k) xv[k] = buffer_load_f32(xr, ids[16 * h + k] + xrow, 0);
#pragma unroll
                            for (int k = 0; k < 16; ++k) acc[16 * h + k] = fmaf(gv, xv[k], acc[16 * h + k]);
                        }
                        if (k0 == 0) gsum += gv;
                    }
                }
            }
            if (light) {
                float* orow = gw + (size_t)j * K + k0;
                if (VEC4 && k0 + 32 <= K) {
#pragma unroll
                    for (int q = 0; q < 8; ++q)
                        *reinterpret_cast<float4*>(orow + 4 * q) = make_float4(acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]);
                } else {
#pragma unroll
                    for (int k = 0; k < 32; ++k)
                        if (k0 + k < K) orow[k] = acc[k];
                }
            }
        }
        if (bias_grad != nullptr && light) bias_grad[j] = gsum;
        // ---- labels with many set bits: the whole wavefront on one label, lane <-> connection ----
        unsigned long long todo = __ballot(mine && heavy);
        while (todo) {
            const int r = __builtin_amdgcn_readfirstlane(__ffsll((long long)todo) - 1);
            todo &= todo - 1;
            const int jh = __builtin_amdgcn_readlane(j, r);
            float hsum = 0.f;
            for (int k0 = 0; k0 < K; k0 += 64) {
                const int k = k0 + lane;
                const unsigned id = k < K ? (unsigned)idx[(size_t)jh * K + k] : 0u;
                const unsigned xcol = (id < (unsigned)N ? id : 0u) * xsn;
                float acc = 0.f;
                hsum = 0.f;
                for (int t = 0; t < nbt; ++t) {
                    unsigned m = __builtin_amdgcn_readfirstlane(words[(size_t)t * L + jh]);
                    if (t == nbt - 1) m &= tail;
                    // up to four set bits per step, their loads in flight together
                    while (m) {
                        int bb[4];
                        float gv[4], xv[4];
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            bb[u] = m ? 32 * t + __ffs((int)m) - 1 : -1;
                            m &= m ? m - 1 : 0u;
                        }
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            const int b = bb[u] < 0 ? 0 : bb[u];
                            gv[u] = bb[u] < 0 ? 0.f : g[(size_t)b * L + jh];
                            xv[u] = buffer_load_f32(xr, xcol, (unsigned)b * xsb);
                        }
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            acc = fmaf(gv[u], xv[u], acc);
                            hsum += gv[u];
                        }
                    }
                }
                if (k < K) gw[(size_t)jh * K + k] = acc;
            }
            if (bias_grad != nullptr && lane == 0) bias_grad[jh] = hsum;
        }
        }
        done(mylist, total, block_base);
    }
    return set_bits;
}

template <bool VEC4>
__global__ __launch_bounds__(256, 4) void wgrad_sparse_kernel(const SparseRows rows) {
    sparse_rows<VEC4, true>(rows, blockIdx.x, gridDim.x, [](const unsigned*, int, int) {});
}

// The same gradients and the Adam step on weights and bias in one launch: labels without a set bit take the step of a zero gradient,
// which nothing but the moments and variables is read for, labels with one take theirs from the rows that their own wavefront has
// just formed.  The former are bound by memory and the latter by the latency of their gathers: the latter's workgroups come first, the
// others take the room that they leave.  (Alternating, 174 us for the step below: under the others' loads every gather waits longer.)
// They also count the set bits, which the next call decides from (host_count; totals: a sum and a count of workgroups, zero between
// launches).
// (32 x 768 x 670,091 x 32, 0.2 % of the gradients not zero, late in training: two launches that count 9.6 us, the gradient 22, the
// step on the weights 72 and on the bias 5.8; 92 so.  The whole step with its forward pass 183 -> 170.)
//   A wavefront that steps looks at the masks of its labels first and leaves out the rows with a gradient, by accesses that the end of
// a buffer keeps from memory: no branch parts the loads.  (All rows read beside the masks, 168 us for the whole step above, and this
// 168; loads under branches 172.  What rows of other lengths share sixteen bytes of is read element by element, three a lane at most.)
__device__ __forceinline__ f32x4_unaligned& four_at(float* p) { return *reinterpret_cast<f32x4_unaligned*>(p); }
__device__ __forceinline__ void adam_element(f32x4_unaligned& w, f32x4_unaligned& m, f32x4_unaligned& v, int q, float g, const AdamCoefficients& a) {
    float wq = w[q], mq = m[q], vq = v[q];
    adam_one(wq, mq, vq, g, a);
    w[q] = wq; m[q] = mq; v[q] = vq;
}
struct AdamRows {
    float *var, *m, *v, *bias, *bias_m, *bias_v;
    AdamCoefficients a;
    unsigned long long* totals;
    unsigned long long* host_count;
    int gradient_blocks;
};

typedef unsigned four_words __attribute__((ext_vector_type(4)));

template <bool VEC4>
__global__ __launch_bounds__(256, 4) void wgrad_adam_kernel(const SparseRows r, const AdamRows o) {
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if ((int)blockIdx.x < o.gradient_blocks) {
        const unsigned bits = sparse_rows<VEC4, false>(r, blockIdx.x, o.gradient_blocks, [&](const unsigned* list, int total, int base) {
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");        // (rows and list are the wavefront's own)
            __builtin_amdgcn_wave_barrier();
            const int len = (r.K + 3) / 4;
            for (int e = lane; e < total * len; e += 64) {
                const int i = e / len, k = 4 * (e - i * len), n = min(4, r.K - k);
                const size_t at = (size_t)(base + (int)(list[i] & 255u)) * r.K + (size_t)k;
                if (n == 4) {
                    f32x4_unaligned w4 = four_at(o.var + at), m4 = four_at(o.m + at), v4 = four_at(o.v + at);
                    const f32x4_unaligned g4 = four_at(r.gw + at);
#pragma unroll
                    for (int q = 0; q < 4; ++q) adam_element(w4, m4, v4, q, g4[q], o.a);
                    four_at(o.var + at) = w4;
                    four_at(o.m + at) = m4;
                    four_at(o.v + at) = v4;
                } else {
                    for (int q = 0; q < n; ++q) adam_one(o.var[at + q], o.m[at + q], o.v[at + q], r.gw[at + q], o.a);
                }
            }
            if (o.bias != nullptr)
                for (int i = lane; i < total; i += 64) {
                    const int j = base + (int)(list[i] & 255u);
                    adam_one(o.bias[j], o.bias_m[j], o.bias_v[j], r.bias_grad[j], o.a);
                }
            __builtin_amdgcn_wave_barrier();
        });
        unsigned long long n = bits;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) n += __shfl_xor(n, off, 64);
        __shared__ unsigned long long of_wave[4];
        if (lane == 0) of_wave[wv] = n;
        __syncthreads();
        if (threadIdx.x == 0) {
            n = (of_wave[0] + of_wave[1]) + (of_wave[2] + of_wave[3]);
            // the ticket is drawn once the sum is known to have this workgroup's bits
            const unsigned long long before = __hip_atomic_fetch_add(o.totals, n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const unsigned long long one = before == ~0ull ? 0ull : 1ull;
            if (__hip_atomic_fetch_add(o.totals + 1, one, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (unsigned long long)o.gradient_blocks - 1ull) {
                *o.host_count = __hip_atomic_exchange(o.totals, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);      // pinned host memory
                __hip_atomic_store(o.totals + 1, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        return;
    }
    // 64 labels per wavefront and step, sixteen bytes of their rows at a time, where those end and begin does not matter.  Rows with a set bit
    // belong to another wavefront, which may be writing them: nothing of them is read (buffer accesses beyond the end do not touch memory).
    const int stepper = (int)blockIdx.x - o.gradient_blocks, steppers = gridDim.x - o.gradient_blocks;
    const unsigned tail = (r.B & 31) ? (1u << (r.B & 31)) - 1u : 0xffffffffu;
    const float inv_len = 1.f / (float)r.K;
    constexpr unsigned kNowhere = 0x80000000u;
    for (long long first = (stepper * 4 + wv) * 64ll; first < r.L; first += steppers * 256ll) {
        const int base = (int)first, rows = min(64, r.L - base);
        unsigned set = 0u;
        for (int t = 0; t < r.nbt; ++t) {
            const unsigned m = r.words[(size_t)t * r.L + base + min(lane, rows - 1)];
            set |= t == r.nbt - 1 ? m & tail : m;
        }
        const bool idle_row = lane < rows && set == 0u;
        const unsigned long long idle = __ballot(idle_row);
        const int all_quads = !VEC4 && r.K < 4 ? 0 : rows * r.K / 4;        // (rows of three and fewer go element by element)
        const size_t at = (size_t)base * r.K;
        auto row_of = [&](int e) {                                        // e / K, once it is set right
            const int row = min((int)((float)e * inv_len), rows - 1);
            return row + (e >= (row + 1) * r.K ? 1 : e < row * r.K ? -1 : 0);
        };
        auto load = [&](buffer_rsrc from, unsigned off) { return __builtin_bit_cast(f32x4_unaligned, __builtin_amdgcn_raw_buffer_load_b128(from, off, 0, 0)); };
        auto store = [&](buffer_rsrc to, unsigned off, f32x4_unaligned q) { __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(four_words, q), to, off, 0, 0); };
        // The lane's row ends in a quad that holds the first elements of the next one: where one of the two has a set bit, or the next
        // is not there, the other's elements go one by one.  All elements of rows of three and fewer do.
        int edge = 0;
        size_t edge_at = at + (size_t)lane * r.K;
        if (!VEC4 && lane < rows) {
            const bool next = lane < 63 && (idle >> (lane + 1) & 1ull) != 0ull;
            const int mine = (lane + 1) * r.K & 3;
            if (r.K < 4) {
                edge = idle_row ? r.K : 0;
            } else if (mine != 0 && idle_row != next) {
                edge = idle_row ? mine : 4 - mine;
                edge_at += (size_t)(idle_row ? r.K - mine : r.K);
            }
        }
        float ew[3], em[3], ev[3];
        if (!VEC4) {
#pragma unroll
            for (int i = 0; i < 3; ++i)
                if (i < edge) { ew[i] = o.var[edge_at + i]; em[i] = o.m[edge_at + i]; ev[i] = o.v[edge_at + i]; }
        }
        constexpr int kAtOnce = 4;
        for (int from = 0; from < all_quads; from += 64 * kAtOnce) {
            const int quads = min(all_quads - from, 64 * kAtOnce);
            const size_t here = at + 4 * (size_t)from;
            const buffer_rsrc wr = make_rsrc(o.var + here, quads * 16u), mr = make_rsrc(o.m + here, quads * 16u), vr = make_rsrc(o.v + here, quads * 16u);
            f32x4_unaligned w4[kAtOnce], m4[kAtOnce], v4[kAtOnce];
            unsigned off[kAtOnce];
#pragma unroll
            for (int u = 0; u < kAtOnce; ++u) {
                if (64 * u >= quads) break;                               // (uniform)
                const int q = lane + 64 * u, e = 4 * (from + min(q, quads - 1)), row = row_of(e);
                bool on = (idle >> row & 1ull) != 0ull;
                if (!VEC4 && e + 4 > (row + 1) * r.K) on = on && (idle >> (row + 1) & 1ull) != 0ull;
                off[u] = on && q < quads ? 16u * (unsigned)q : kNowhere;
                w4[u] = load(wr, off[u]); m4[u] = load(mr, off[u]); v4[u] = load(vr, off[u]);
            }
#pragma unroll
            for (int u = 0; u < kAtOnce; ++u) {
                if (64 * u >= quads) break;
#pragma unroll
                for (int q = 0; q < 4; ++q) adam_element(w4[u], m4[u], v4[u], q, 0.f, o.a);
                store(wr, off[u], w4[u]); store(mr, off[u], m4[u]); store(vr, off[u], v4[u]);
            }
        }
        if (!VEC4) {
#pragma unroll
            for (int i = 0; i < 3; ++i)
                if (i < edge) {
                    adam_one(ew[i], em[i], ev[i], 0.f, o.a);
                    o.var[edge_at + i] = ew[i]; o.m[edge_at + i] = em[i]; o.v[edge_at + i] = ev[i];
                }
        }
        if (o.bias != nullptr && idle_row) adam_one(o.bias[base + lane], o.bias_m[base + lane], o.bias_v[base + lane], 0.f, o.a);
    }
}

constexpr int kSgThreads = 512;
constexpr int kSgWaves = kSgThreads / 64;

constexpr int kSgWordsPerLane = 8;
constexpr int kSgChunk = 64 * kSgWordsPerLane;      // words of a bit row a wavefront takes in one go: 32,768 labels
constexpr int kSgList = 512;                        // set bits of a chunk that a wavefront can list

// One workgroup per (sample, label segment).  A wavefront takes its share of the sample's bit row in chunks of
// kSgChunk words, lists the labels of the chunk's set bits in LDS (when the gradient is sparse most words are empty:
// the lanes then work on the list, not each on its own word), and every lane adds g * w of its label's connections
// (a 32-connection chunk at a time) into the wavefront's own accumulators gx[n] in LDS.  A chunk with more set
// bits than the list holds is walked word by word instead.  No barriers inside the walk; the order of the adds is
// fixed by the lane assignment.  The wavefronts' accumulators are summed in ascending order at the end.
template <bool VEC4>
__global__ __launch_bounds__(kSgThreads) void igrad_sparse_kernel(const unsigned long long* __restrict__ bits, int nwords,
                                                                  const int32_t* __restrict__ idx,
                                                                  const float* __restrict__ w, const float* __restrict__ g,
                                                                  float* __restrict__ partial, int B, int N, int L, int K,
                                                                  int S, int words_per_seg) {
    extern __shared__ __align__(16) unsigned char sg_lds[];
    float* acc = reinterpret_cast<float*>(sg_lds);                                        // [kSgWaves][N]
    int* lists = reinterpret_cast<int*>(acc + (size_t)kSgWaves * N);                      // [kSgWaves][kSgList]
    const int b = blockIdx.x / S, seg = blockIdx.x % S;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    for (int i = threadIdx.x; i < kSgWaves * N; i += kSgThreads) acc[i] = 0.f;
    __syncthreads();
    const int w_begin = seg * words_per_seg;
    const int w_end = min(w_begin + words_per_seg, nwords);
    const unsigned long long* row = bits + (size_t)b * nwords;
    const float* grow = g + (size_t)b * L;
    float* myacc = acc + (size_t)wv * N;
    int* mylist = lists + wv * kSgList;
    // g[b, j] times the weights of label j, added at the label's columns
    auto add_label = [&](int j) {
        const float gv = grow[j];
        const size_t at = (size_t)j * K;
        for (int k0 = 0; k0 < K; k0 += 32) {
            unsigned n[32];
            float wk[32];
            if (VEC4 && k0 + 32 <= K) {
#pragma unroll
                for (int q = 0; q < 8; ++q) {
                    const int4 v = *reinterpret_cast<const int4*>(idx + at + k0 + 4 * q);
                    const float4 f = *reinterpret_cast<const float4*>(w + at + k0 + 4 * q);
                    n[4 * q] = (unsigned)v.x; n[4 * q + 1] = (unsigned)v.y; n[4 * q + 2] = (unsigned)v.z; n[4 * q + 3] = (unsigned)v.w;
                    wk[4 * q] = f.x; wk[4 * q + 1] = f.y; wk[4 * q + 2] = f.z; wk[4 * q + 3] = f.w;
                }
            } else {
#pragma unroll
                for (int k = 0; k < 32; ++k) {
                    const bool in = k0 + k < K;
                    n[k] = in ? (unsigned)idx[at + k0 + k] : 0xffffffffu;
                    wk[k] = in ? w[at + k0 + k] : 0.f;
                }
            }
#pragma unroll
            for (int k = 0; k < 32; ++k)
                if (n[k] < (unsigned)N) atomicAdd(&myacc[n[k]], gv * wk[k]);
        }
    };
    for (int c0 = w_begin + wv * kSgChunk; c0 < w_end; c0 += kSgWaves * kSgChunk) {
        unsigned long long m[kSgWordsPerLane];
        int mine = 0;
#pragma unroll
        for (int q = 0; q < kSgWordsPerLane; ++q) {
            const int wi = c0 + q * 64 + lane;
            m[q] = wi < w_end ? row[wi] : 0ull;
            mine += __popcll(m[q]);
        }
        int upto = mine;                                   // inclusive prefix sum over the lanes
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int t = __shfl_up(upto, off, 64);
            if (lane >= off) upto += t;
        }
        const int total = __builtin_amdgcn_readlane(upto, 63);
        if (total == 0) continue;
        if (total <= kSgList) {
            int at = upto - mine;
#pragma unroll
            for (int q = 0; q < kSgWordsPerLane; ++q) {
                unsigned long long mm = m[q];
                const int j0 = (c0 + q * 64 + lane) * 64;
                while (mm) {
                    mylist[at++] = j0 + __ffsll((long long)mm) - 1;
                    mm &= mm - 1;
                }
            }
            __builtin_amdgcn_wave_barrier();    // (LDS operations of a wavefront complete in order)
            for (int e = lane; e < total; e += 64) add_label(mylist[e]);
            __builtin_amdgcn_wave_barrier();
        } else {
#pragma unroll 1
            for (int q = 0; q < kSgWordsPerLane; ++q) {
                unsigned long long mm = m[q];
                const int j0 = (c0 + q * 64 + lane) * 64;
                while (__ballot(mm != 0)) {
                    if (mm) {
                        const int j = j0 + __ffsll((long long)mm) - 1;
                        mm &= mm - 1;
                        add_label(j);
                    }
                }
            }
        }
    }
    __syncthreads();
    float* out = partial + ((size_t)seg * B + b) * N;
    for (int n = threadIdx.x; n < N; n += kSgThreads) {
        float t = acc[n];
#pragma unroll
        for (int i = 1; i < kSgWaves; ++i) t += acc[(size_t)i * N + n];
        out[n] = t;
    }
}

__global__ __launch_bounds__(256) void igrad_sparse_reduce_kernel(const float* __restrict__ partial, int S, int B, int N,
                                                                  float* __restrict__ gx, int tp) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (size_t)B * N) return;
    float t = 0.f;
    for (int s = 0; s < S; ++s) t += partial[(size_t)s * B * N + i];
    const int b = (int)(i / N), n = (int)(i - (size_t)b * N);
    gx[tp ? (size_t)n * B + b : i] = t;
}

// Pinned words the set-bit counts are written to by the count kernel, one per (device, stream), together with
// the shape of the call that wrote it: a later call on the same stream may decide from it without waiting.
struct CountSlot {
    int device;
    hipStream_t stream;
    unsigned long long* host;    // hipHostMalloc'ed, written by nz_count_finish_kernel or wgrad_adam_kernel
    int B, L;                    // shape of the last call (0: none yet)
};
std::mutex g_count_mutex;
std::vector<CountSlot> g_count_slots;

// (under the lock; the slot stays where it is as long as that is held)
int count_slot(int dev, hipStream_t s, CountSlot** out) {
    for (CountSlot& c : g_count_slots)
        if (c.device == dev && c.stream == s) { *out = &c; return FFI_OK; }
    CountSlot c{dev, s, nullptr, 0, 0};
    if (hipHostMalloc((void**)&c.host, 64) != hipSuccess) { (void)hipGetLastError(); return FFI_ERR_OUT_OF_MEMORY; }
    *c.host = 0;
    g_count_slots.push_back(c);
    *out = &g_count_slots.back();
    return FFI_OK;
}

}  // namespace

bool nonzero_previous(int B, int L, hipStream_t s, unsigned long long* count_out) {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess) return false;
    std::lock_guard<std::mutex> lock(g_count_mutex);
    for (const CountSlot& c : g_count_slots) {
        if (c.device != dev || c.stream != s || c.B != B || c.L != L) continue;
        *count_out = *reinterpret_cast<volatile unsigned long long*>(c.host);
        return true;
    }
    return false;
}

int launch_nonzero_scan(const float* g, unsigned* words, int B, int L, hipStream_t s) {
    const int nbt = (B + 31) / 32;
    hipLaunchKernelGGL(nz_scan_kernel, dim3((L + 2 * kScanThreads - 1) / (2 * kScanThreads), nbt), dim3(kScanThreads), 0, s, g, words, B, L);
    FFI_HIP_TRY(hipGetLastError());
    return FFI_OK;
}

int launch_zero_unmasked(float* g, const unsigned* words, int B, int L, hipStream_t s) {
    const int nbt = (B + 31) / 32;
    hipLaunchKernelGGL(nz_zero_unmasked_kernel, dim3((L + kScanThreads - 1) / kScanThreads, nbt), dim3(kScanThreads), 0, s, g, words,
                       B, L);
    FFI_HIP_TRY(hipGetLastError());
    return FFI_OK;
}

int nonzero_count(const float* g, const unsigned* given_words, int B, int L, hipStream_t s, bool lagged,
                  const unsigned** words_out, unsigned long long* count_out) {
    const int nbt = (B + 31) / 32;
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess) return FFI_ERR_NO_DEVICE;
    const size_t head = (size_t)kCountBlocks * sizeof(unsigned long long);           // block counts
    const size_t words_bytes = (size_t)nbt * L * sizeof(unsigned);
    unsigned char* ws = nullptr;
    FFI_TRY(workspace_get(s, kWsNonzero, head + (given_words ? 0 : words_bytes), (void**)&ws));
    unsigned long long* block_counts = reinterpret_cast<unsigned long long*>(ws);
    const unsigned* words = given_words;
    if (!given_words) {
        unsigned* scanned = reinterpret_cast<unsigned*>(ws + head);
        FFI_TRY(launch_nonzero_scan(g, scanned, B, L, s));
        words = scanned;
    }
    *words_out = words;
    std::lock_guard<std::mutex> lock(g_count_mutex);
    CountSlot* slot = nullptr;
    FFI_TRY(count_slot(dev, s, &slot));
    // the count of an earlier call of the same shape on this stream, read before this call's kernels can overwrite it
    const bool use_previous = lagged && slot->B == B && slot->L == L;
    const unsigned long long previous = *reinterpret_cast<volatile unsigned long long*>(slot->host);
    hipLaunchKernelGGL(nz_count_kernel, dim3(kCountBlocks), dim3(kScanThreads), 0, s, words, (size_t)nbt * L, block_counts);
    hipLaunchKernelGGL(nz_count_finish_kernel, dim3(1), dim3(kCountBlocks), 0, s, block_counts, kCountBlocks, slot->host);
    FFI_HIP_TRY(hipGetLastError());
    if (use_previous) {
        *count_out = previous;
        return FFI_OK;
    }
    FFI_HIP_TRY(hipStreamSynchronize(s));
    *count_out = *reinterpret_cast<volatile unsigned long long*>(slot->host);
    slot->B = B;
    slot->L = L;
    return FFI_OK;
}

void nonzero_count_forget(int device) {
    std::lock_guard<std::mutex> lock(g_count_mutex);
    for (CountSlot& c : g_count_slots)
        if (c.device == device) { c.B = 0; c.L = 0; }
}

namespace {
// Labels of a lane: as many as leave a workgroup for every second CU.  (Batch 166 x 43 x 18,691 x 55, a step of which 28 % of the labels
// have a gradient: the whole step 128 us with four each, 97 with one; 41 x 4,096 x 245,894 x 5: 116 with four, 122 with two, 131 with one.)
int sparse_per_lane(const Dims& d) {
    int per = kWsLabelsPerLane;
    while (per > 1 && (d.L + 256 * per - 1) / (256 * per) < device_cu_count() / 2) per /= 2;
    return per;
}
SparseRows sparse_rows_of(const float* x, const int32_t* idx, const float* g, const unsigned* words, float* gw, float* bias_grad, const Dims& d) {
    // byte strides of x along the batch and along the features
    return SparseRows{x, (d.tp ? 1u : (unsigned)d.N) * 4u, (d.tp ? (unsigned)d.B : 1u) * 4u, idx, g, words, gw, bias_grad, d.B, d.N, d.L, d.K, (d.B + 31) / 32,
                      sparse_per_lane(d)};
}
int sparse_rows_blocks(const Dims& d) {
    const int labels = 256 * sparse_per_lane(d);
    return std::max(1, std::min((d.L + labels - 1) / labels, device_cu_count() * 8));
}
}  // namespace

int launch_weight_grad_sparse(const float* x, const int32_t* idx, const float* g, const unsigned* words, float* gw,
                              float* bias_grad, const Dims& d, hipStream_t s) {
    const bool vec4 = (d.K % 4 == 0) && (((uintptr_t)gw | (uintptr_t)idx) % 16 == 0);
    hipLaunchKernelGGL((vec4 ? wgrad_sparse_kernel<true> : wgrad_sparse_kernel<false>), dim3(sparse_rows_blocks(d)), dim3(256), 0, s,
                       sparse_rows_of(x, idx, g, words, gw, bias_grad, d));
    FFI_HIP_TRY(hipGetLastError());
    return FFI_OK;
}

int launch_weight_grad_adam_sparse(const float* x, const int32_t* idx, const float* g, const unsigned* words, float* gw, float* bias_grad,
                                   const AdamVariables& v, float lr, float beta_1, float beta_2, float eps, long long step, const Dims& d,
                                   unsigned long long set_bits, hipStream_t s) {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess) return FFI_ERR_NO_DEVICE;
    unsigned* tickets = nullptr;
    FFI_TRY(tickets_get(s, (void**)&tickets));
    std::lock_guard<std::mutex> lock(g_count_mutex);
    CountSlot* slot = nullptr;
    FFI_TRY(count_slot(dev, s, &slot));
    // A CU holds four of the workgroups.  On layers of so many labels that the gradients' would take all these places first, and the steps
    // begin when they end, they are fewer where few labels have a gradient: 8 x 400 x 1,000,000 x 5 with 1.6 % of the labels 95 us so many,
    // 85 so; 32 x 400 x 1,000,000 and 6.4 %, fan-in 5 96 and 87, 32 263 and 259.  (64 samples, 13 % and fan-in 16: 193 and 200.  Little
    // more than the limit is no good either, two rounds where there was one: 32 x 400 x 800,000 x 8 83 and 86.)
    int gradient_blocks = sparse_rows_blocks(d);
    const int cus = device_cu_count(), steps = (int)(((long long)d.L + 255) / 256);
    if (4 * gradient_blocks >= 13 * cus && set_bits < (unsigned long long)d.L / 10) gradient_blocks = 11 * cus / 4;
    const bool vec4 = (d.K % 4 == 0) && (((uintptr_t)gw | (uintptr_t)idx | (uintptr_t)v.weights | (uintptr_t)v.weight_m | (uintptr_t)v.weight_v) % 16 == 0);
    const AdamRows o{v.weights, v.weight_m, v.weight_v, v.bias, v.bias_m, v.bias_v, adam_coefficients(lr, beta_1, beta_2, eps, step),
                     reinterpret_cast<unsigned long long*>(tickets), slot->host, gradient_blocks};
    const int steppers = std::min(steps, 16 * cus);
    hipLaunchKernelGGL((vec4 ? wgrad_adam_kernel<true> : wgrad_adam_kernel<false>), dim3(gradient_blocks + steppers), dim3(256), 0, s,
                       sparse_rows_of(x, idx, g, words, gw, bias_grad, d), o);
    FFI_HIP_TRY(hipGetLastError());
    return FFI_OK;
}

bool sparse_weight_grad_fits(int B, int N) { return (unsigned long long)B * (unsigned long long)N < (1ull << 30); }

bool sparse_input_grad_fits(int N, int K) { return N <= kSparseMaxFeatures && K <= 65535; }

int launch_input_grad_sparse(const int32_t* idx, const float* w, const float* g, const unsigned* words, float* gx,
                             const Dims& d, hipStream_t s) {
    const int nbt = (d.B + 31) / 32;
    const int nwords = (d.L + 63) / 64;
    // label segments per sample: a chunk of words for every wavefront of a workgroup, more segments only as far as
    // the GPU would otherwise not be filled (a segment costs a set of LDS accumulators to clear and to sum)
    const int chunks = (nwords + kSgChunk - 1) / kSgChunk;
    const int s_full = (chunks + kSgWaves - 1) / kSgWaves;
    const int s_fill = (2 * device_cu_count() + d.B - 1) / d.B;
    int S = std::max(1, std::max(s_full, std::min(s_fill, chunks)));
    const int words_per_seg = (nwords + S - 1) / S;
    S = (nwords + words_per_seg - 1) / words_per_seg;
    const size_t bits_bytes = (size_t)d.B * nwords * sizeof(unsigned long long);
    const size_t partial_bytes = (size_t)S * d.B * d.N * sizeof(float);
    unsigned char* ws = nullptr;
    FFI_TRY(workspace_get(s, kWsPartials, bits_bytes + partial_bytes, (void**)&ws));
    unsigned long long* bits = reinterpret_cast<unsigned long long*>(ws);
    float* partial = reinterpret_cast<float*>(ws + bits_bytes);
    hipLaunchKernelGGL(nz_transpose_kernel, dim3((nwords + 4 * kTransposeBlocks - 1) / (4 * kTransposeBlocks), nbt), dim3(kScanThreads), 0, s, words, bits, d.B, d.L, nwords);
    FFI_HIP_TRY(hipGetLastError());
    const size_t lds = (size_t)kSgWaves * d.N * sizeof(float) + (size_t)kSgWaves * kSgList * sizeof(int);
    const bool vec4 = (d.K % 4 == 0) && (((uintptr_t)w | (uintptr_t)idx) % 16 == 0);
    if (vec4) {
        FFI_HIP_TRY(hipFuncSetAttribute((const void*)igrad_sparse_kernel<true>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        hipLaunchKernelGGL(igrad_sparse_kernel<true>, dim3(d.B * S), dim3(kSgThreads), lds, s, bits, nwords, idx, w, g, partial, d.B,
                           d.N, d.L, d.K, S, words_per_seg);
    } else {
        FFI_HIP_TRY(hipFuncSetAttribute((const void*)igrad_sparse_kernel<false>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        hipLaunchKernelGGL(igrad_sparse_kernel<false>, dim3(d.B * S), dim3(kSgThreads), lds, s, bits, nwords, idx, w, g, partial, d.B,
                           d.N, d.L, d.K, S, words_per_seg);
    }
    FFI_HIP_TRY(hipGetLastError());
    const size_t total = (size_t)d.B * d.N;
    hipLaunchKernelGGL(igrad_sparse_reduce_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, partial, S, d.B, d.N,
                       gx, d.tp ? 1 : 0);
    FFI_HIP_TRY(hipGetLastError());
    return FFI_OK;
}

}  // namespace ffi
