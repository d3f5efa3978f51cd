// Column-ordered view ("plan") of a lookup matrix, built on the device.
//
// The input gradient sums, for every input column n, over all connections (j,k) with
// lookup[j,k] == n.  The plan lists those connections column by column so that they can be walked
// sequentially, without atomics, in an order that never changes from run to run.
#include "ffi_internal.h"
#include "ffi_check.h"
#include "ffi_scan.h"
#include "ffi_lds_tile.h"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <functional>

#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/types/double_buffer.hpp>

namespace ffi {
namespace {

constexpr int kBlock = 256;
constexpr int kFingerprintBlocks = 1024;                 // workgroups of the fingerprint kernel (at most)
constexpr int kScratchWords = 8 + 2 * kFingerprintBlocks;  // plan scratch: 8 words for the build, then fingerprint partial sums

// Order-independent 64-bit content fingerprint: sum over positions p of mix(id_p + p * odd), plus
// the number of ids outside [0,N).  Every workgroup writes its own pair of partial sums (no atomics:
// thousands of adds to one address serialise); the host adds them up.  Four ids per load when the
// array allows it.
__global__ __launch_bounds__(kBlock) void fingerprint_kernel(const int32_t* __restrict__ idx,
                                                              size_t total, unsigned N,
                                                              unsigned long long* __restrict__ out) {
    unsigned long long h = 0;
    unsigned bad = 0;
    const size_t stride = (size_t)gridDim.x * kBlock;
    const size_t tid = (size_t)blockIdx.x * kBlock + threadIdx.x;
    const bool vec = ((uintptr_t)idx & 15) == 0;
    const size_t nvec = vec ? total / 4 : 0;
    const int4* idx4 = reinterpret_cast<const int4*>(idx);
#pragma unroll 4
    for (size_t q = tid; q < nvec; q += stride) {
        const int4 v = idx4[q];
        const unsigned p = (unsigned)(q * 4);
        h += mix32((unsigned)v.x + p * 0x9e3779b1u);
        h += mix32((unsigned)v.y + (p + 1) * 0x9e3779b1u);
        h += mix32((unsigned)v.z + (p + 2) * 0x9e3779b1u);
        h += mix32((unsigned)v.w + (p + 3) * 0x9e3779b1u);
        bad += ((unsigned)v.x >= N) + ((unsigned)v.y >= N) + ((unsigned)v.z >= N) + ((unsigned)v.w >= N);
    }
    for (size_t p = nvec * 4 + tid; p < total; p += stride) {
        const unsigned id = (unsigned)idx[p];
        h += mix32(id + (unsigned)p * 0x9e3779b1u);
        bad += id >= N;
    }
    unsigned long long b64 = bad;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        h += __shfl_down(h, off);
        b64 += __shfl_down(b64, off);
    }
    __shared__ unsigned long long part[2][kBlock / 64];
    if ((threadIdx.x & 63) == 0) { part[0][threadIdx.x >> 6] = h; part[1][threadIdx.x >> 6] = b64; }
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long hs = 0, bs = 0;
#pragma unroll
        for (int i = 0; i < kBlock / 64; ++i) { hs += part[0][i]; bs += part[1][i]; }
        out[2 * blockIdx.x] = hs;
        out[2 * blockIdx.x + 1] = bs;
    }
}

__global__ __launch_bounds__(64) void guard_init_kernel(unsigned long long* __restrict__ guard, unsigned long long fingerprint) {
    const int i = threadIdx.x;
    if (i < 8) guard[i] = i == 3 || i == 5 ? fingerprint : i == 4 ? 1ull : 0ull;
}

__global__ __launch_bounds__(kCheckThreads) void fingerprint_guard_kernel(const LookupCheck check) {
    __shared__ CheckShared shared;
    check_block(check, blockIdx.x, shared);
}

// ---- tiled form ---------------------------------------------------------------------------------

// Order of a column's slots inside a tile.  The kernel that walks the plan reads, per slot, the
// 128-byte LDS row of the slot's label; rows of even labels sit in one half of the LDS banks, rows
// of odd labels in the other, and the LDS serves 16 lanes per clock only if 8 of them read each
// half.  So the lanes whose id has bit 3 clear walk their column as even, odd, even, ... labels
// and the lanes with bit 3 set as odd, even, odd, ...: slot 2t holds the t-th label of the lane's
// first parity, slot 2t+1 the t-th label of the other parity, holes are padding slots that point
// at an all-zero row of the right parity.  Inside a parity class positions ascend.
__device__ __forceinline__ unsigned parity_first(unsigned thread) { return (thread >> 3) & 1u; }       // parity walked at even slots
__device__ __forceinline__ unsigned column_slots(unsigned thread, unsigned even, unsigned odd) {
    const unsigned first = parity_first(thread) ? odd : even, second = parity_first(thread) ? even : odd;
    return max(first ? 2u * first - 1u : 0u, 2u * second);
}

// The sum of v over each LANES consecutive lanes (32 or 64), in all of them.
template <int LANES> __device__ __forceinline__ int lanes_total(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0xb1, 0xf, 0xf, true);         // lane ^ 1
    v += __builtin_amdgcn_update_dpp(0, v, 0x4e, 0xf, 0xf, true);         // lane ^ 2
    v += __builtin_amdgcn_update_dpp(0, v, 0x141, 0xf, 0xf, true);        // 7 - lane within eight
    v += __builtin_amdgcn_update_dpp(0, v, 0x140, 0xf, 0xf, true);        // 15 - lane within sixteen
    const auto rows = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    v = (int)(rows[0] + rows[1]);
    if (LANES == 32) return v;
    const auto halves = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return (int)(halves[0] + halves[1]);
}

// Which LDS row of the walking kernel's tile each label is staged into (rowpos[j], inside the label's tile).
// The bank half a row lies in is the parity of its row number, and a column is walked fastest when its labels
// split evenly between the halves (see above: every hole costs a slot).  The label's own parity would split a
// column's labels like coin flips (about sqrt(n) excess); here the labels of a tile are taken in ascending order
// and each goes to the half that the columns it feeds have used less so far (weighted sum over its connections
// of even-count minus odd-count of the column), which keeps the columns that matter close to an even split.
// Rows of a half are handed out in ascending order, at most `cap` per half.  One workgroup per tile; the tile's
// column ids are staged in LDS, one wavefront then decides label after label (lane <-> connection), or two at a time where 32 lanes
// hold a fan-in; beyond a fan-in of 64 a lane has several connections.
// (`col_lo`: the plan covers the columns [col_lo, col_lo + ncols) only; connections into other columns are left out)
// (`all_columns_count`: plans that hand the columns to threads by length -- there every column is about as long as the
// longest of its slice, so every column's balance weighs the same)
template <int LANES, bool MORE>              // (MORE: fan-ins above LANES = 64)
__global__ __launch_bounds__(256) void tile_color_kernel(const int32_t* __restrict__ idx, int L, int K, int tile_labels, int cap,
                                                         int ncols, unsigned short* __restrict__ rowpos, int col_lo,
                                                         int all_columns_count, unsigned* __restrict__ counts) {
    extern __shared__ int color_lds[];
    // (entry `ncols` of both: where connections into columns outside the window go -- weight 0, so they never count)
    int* imb = color_lds;                                                        // [ncols + 1] even minus odd labels per column
    // The tile's column ids, three 10-bit ids per word, a label's ids in W = ceil(K / 3) words of its own, and the weights as
    // 16-bit numbers: with 16-bit ids and 32-bit weights a tile of 582 labels x fan-in 32 took 44 KB of LDS, three workgroups per
    // CU and two rounds for 1,152 tiles; now 30 KB, five workgroups per CU, all tiles at once (the work of a tile is one
    // wavefront's sequential loop).
    const int W = (K + 2) / 3;
    unsigned* ids3 = reinterpret_cast<unsigned*>(color_lds + ncols + 1);         // [tile_labels * W]
    unsigned short* wt = reinterpret_cast<unsigned short*>(ids3 + (size_t)tile_labels * W);   // [ncols + 1] weight of the column's balance (at most 256)
    const int t = blockIdx.x;
    const int j0 = t * tile_labels;
    const int nl = min(tile_labels, L - j0);
    const int* src = idx + (size_t)j0 * K;
    const unsigned outside = (unsigned)min(ncols, 1023);                          // (windows are at most 640 columns wide; a single window has no ids outside)
    for (int i = threadIdx.x; i <= ncols; i += 256) { imb[i] = 0; wt[i] = 0; }
    __syncthreads();
    for (int wi = threadIdx.x; wi < nl * W; wi += 256) {
        const int jl = wi / W, k0 = 3 * (wi - jl * W);
        unsigned word = 0;
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            unsigned c = outside;
            if (k0 + i < K) {
                const unsigned v = (unsigned)(src[jl * K + k0 + i] - col_lo);
                if (v < (unsigned)ncols) { c = v; atomicAdd(&imb[v], 1); }       // column lengths first (in imb: the LDS adds whole words)
            } else {
                c = (unsigned)min(ncols, 1023);                                  // (behind the label's last id: never read)
            }
            word |= c << (10 * i);
        }
        ids3[wi] = word;
    }
    __syncthreads();
    // Only the longest columns of a slice (64 columns, one wavefront of the walking kernel) set its number of slot
    // rows, so their balance counts most: weight = 256 * (length / longest of the slice)^8.
    for (int c = threadIdx.x; c < ncols; c += 256) {
        const int len = imb[c];
        imb[c] = 0;
        int longest = len;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) longest = max(longest, __shfl_xor(longest, off, 64));
        float r = longest > 0 ? (float)len / (float)longest : 0.f;
        r *= r; r *= r; r *= r;
        wt[c] = (unsigned short)(all_columns_count ? (len > 0 ? 256 : 0) : (int)(256.f * r));
    }
    __syncthreads();
    // the half a label goes to: bit 30 of its first word
    auto half_of = [&](int jl) { return (int)(ids3[jl * W] >> 30 & 1u); };
    const int lane = threadIdx.x & 63;
    auto decide_all = [&]() {
    constexpr int kAbreast = 64 / LANES;                                         // labels decided together
    const int groups = (nl + kAbreast - 1) / kAbreast, k_mine = lane & (LANES - 1), abreast = lane / LANES;
    int placed[2] = {0, 0};
    // What bounds the kernel is the chain from one step's adds to the next step's decision: an LDS round trip, the sum over the
    // lanes by DPP and lane swaps, a comparison in every lane; what it does to the counts of placed labels is beside the chain.  Of
    // two labels decided together the second does not see what the first just did: 670,091 labels x fan-in 32 over 768 columns
    // 322 -> 181 us, 200,000 x 8 over 300 143 -> 81, with slot rows per connection 1.1522 -> 1.1523, 2.0510 -> 2.0514.  (Four
    // together: 0.1 to 0.4 % more slot rows, which every walk pays for.  Two of a fan-in of 64, two connections a lane: 528 -> 455
    // us at 501,070 labels, for 0.16 % more.)
    // A lane's column is asked for two steps ahead, the column's weight one.
    auto place_of = [&](int k) { return make_int2(k / 3, 10 * (k % 3)); };
    const int2 place = place_of(min(k_mine, K - 1));
    auto label_of = [&](int g) { return g * kAbreast + abreast; };
    auto word_of = [&](int g) { return ids3[min(label_of(g), nl - 1) * W + place.x]; };
    const bool on = k_mine < K;
    int col1 = 0, w1 = 0;                                                        // the next label's
    unsigned word2 = 0;
    auto advance = [&](int g) {                                                  // to label_of(g), whose word is here
        col1 = (int)((word2 >> place.y) & 1023u);
        if (kAbreast > 1 && label_of(g) >= nl) col1 = ncols;                     // (behind the last label: weight 0)
        word2 = word_of(g + 1);
        const int w = (int)wt[col1];
        w1 = on ? w : 0;
    };
    // connections behind the first of a lane (fan-ins above 64)
    auto rest = [&](int g, auto visit) {
        if (!MORE) return;
        for (int k = lane + 64; k < K; k += 64) {
            const int2 at = place_of(k);
            visit((int)((ids3[label_of(g) * W + at.x] >> at.y) & 1023u));
        }
    };
    // the balance that a lane's label asks for, after `back` (0: nothing) is added to its columns; then `decide` says which half
    auto step = [&](int g, int had, int back, auto decide) {
        const int c = col1, w = w1;
        if (back != 0) {
            if (__builtin_expect(on, 1)) atomicAdd(&imb[c], back);
            rest(g, [&](int q) { atomicAdd(&imb[q], back); });
        }
        int sum = __mul24(w, imb[c]);
        advance(g + 1);
        rest(g, [&](int q) { sum += wt[q] * imb[q]; });
        const int color = decide(lanes_total<LANES>(sum)), delta = color ? -1 : 1;
        if (__builtin_expect(on, 1)) atomicAdd(&imb[c], delta);                                          // (a column may occur twice in a label)
        rest(g, [&](int q) { atomicAdd(&imb[q], delta); });
        if (k_mine == 0 && label_of(g) < nl && color != had) atomicXor(&ids3[label_of(g) * W], 1u << 30);
    };
    // where the labels of a step go once the halves may be full: `color` as far as there is room, else `other`
    auto settle = [&](int g, int color, int other, bool again) {
        const unsigned long long first = kAbreast == 1 ? 1ull : 1ull | 1ull << LANES;            // a label's first lane
        const unsigned long long there = first & (g * kAbreast + kAbreast > nl ? 1ull : ~0ull);
        unsigned long long to = __ballot(color != 0) & there;
        const unsigned long long was = __ballot(other != 0) & there;
        if (again) {
            placed[1] -= __popcll(was);
            placed[0] -= __popcll(there & ~was);
        }
        if (__builtin_expect(max(placed[0], placed[1]) + kAbreast > cap, 0)) {                          // (uniform)
            int room[2] = {cap - placed[0], cap - placed[1]};
            // (labels that stay keep their places: theirs first)
#pragma unroll
            for (int pass = 0; pass < 2; ++pass)
#pragma unroll
                for (int h = 0; h < kAbreast; ++h) {
                    const unsigned long long bit = 1ull << (h * LANES);
                    if (!(there & bit) || (again && ((to ^ was) & bit)) != (pass == 1)) continue;
                    if (room[(to & bit) ? 1 : 0] <= 0) to ^= bit;
                    --room[(to & bit) ? 1 : 0];
                }
            color = (int)(to >> (abreast * LANES) & 1ull);
        }
        placed[1] += __popcll(to);
        placed[0] += __popcll(there & ~to);
        return color;
    };
    word2 = word_of(0);
    advance(0);
    for (int g = 0; g < groups; ++g) {
        const int even = placed[1] < placed[0] ? 1 : 0;
        step(g, 0, 0, [&](int sum) { return settle(g, sum > 0 ? 1 : (sum < 0 ? 0 : even ^ abreast), 0, false); });
    }
    // Second sweep: every label is taken out and put back into the half its columns now ask for -- the first sweep placed
    // the early labels knowing nothing of the later ones.  (Measured on uniformly drawn ids, 586-label tiles of fan-in 32
    // over 768 columns: slot rows 1.528 -> 1.514 per connection, where columns of unconstrained order would need 1.490.)
    word2 = word_of(0);
    advance(0);
    int next_old = half_of(min(label_of(0), nl - 1));       // (written by this wavefront above, whose LDS accesses are in order)
    for (int g = 0; g < groups; ++g) {
        const int old = next_old;
        next_old = half_of(min(label_of(g + 1), nl - 1));
        step(g, old, old ? 1 : -1, [&](int sum) { return settle(g, sum > 0 ? 1 : (sum < 0 ? 0 : old), old, true); });
    }
    // rows of a half are handed out in ascending label order
    int next[2] = {0, 0};
    for (int l0 = 0; l0 < nl; l0 += 64) {
        const bool on = l0 + lane < nl, odd = on && half_of(min(l0 + lane, nl - 1)) != 0;
        const unsigned long long odds = __ballot(odd), evens = __ballot(on && !odd), before = (1ull << lane) - 1ull;
        if (on) rowpos[j0 + l0 + lane] = (unsigned short)(2 * (next[odd] + __popcll((odd ? odds : evens) & before)) + (odd ? 1 : 0));
        next[0] += __popcll(evens);
        next[1] += __popcll(odds);
    }
    };
    if (threadIdx.x < 64) decide_all();
    __syncthreads();
    // what became of the columns: labels in even rows | in odd rows << 16, for the kernels that lay the slots out
    for (int c = threadIdx.x; c <= ncols; c += 256) imb[c] = 0;
    __syncthreads();
    for (int wi = threadIdx.x; wi < nl * W; wi += 256) {
        const int jl = wi / W, k0 = 3 * (wi - jl * W);
        const unsigned word = ids3[wi];
        const int one = half_of(jl) ? 0x10000 : 1;
#pragma unroll
        for (int i = 0; i < 3; ++i)
            if (k0 + i < K) atomicAdd(&imb[(word >> (10 * i)) & 1023u], one);
    }
    __syncthreads();
    for (int c = threadIdx.x; c < ncols; c += 256) counts[(size_t)t * ncols + c] = (unsigned)imb[c];
}

// Which column each thread of the walking kernel takes in each tile (plans with `colperm`).  A wavefront walks as many
// slot rows as the longest of its 64 columns needs, so with thread t <-> column t every slice pays for its longest
// column (about 1.5 slot rows per connection for ids drawn uniformly); here the tile's columns are sorted by the slots
// they need (stable: equal columns stay in index order), cut into blocks of 64 about equally long columns, and the
// blocks dealt to the wavefronts so that the wavefronts of a SIMD (wave, wave + 4, wave + 8, ...) have about the same
// rows in total: longest block first, each to the SIMD with the least so far that still has a wavefront free.
// One workgroup per tile, one thread per column (columns up to the workgroup size exist for this purpose: the ones
// beyond the input's width have no connections).  Sorted by counting; the dealing is done by four lanes for the four SIMDs;
// the columns' lengths come from tile_color_kernel, whose ids lie in LDS.  (670,091 labels over 768 columns 157 us, 85 with four lanes
// dealing, 58 with no comparison of every column with every other, 16 with no reading of the ids -- which there costs 12.)
// Also stores the slot rows of each slice, as tile_count_kernel does for plans without the permutation.  LDS: keys [threads].
constexpr int kPermLengths = 512;            // sorted by counting up to here
__global__ void tile_perm_kernel(const unsigned* __restrict__ counts, unsigned short* __restrict__ colperm, unsigned* __restrict__ slice_len) {
    extern __shared__ __align__(16) unsigned key[];                       // [threads]
    const int t = blockIdx.x, nthreads = blockDim.x, nslices = nthreads >> 6;
    const unsigned halves = counts[(size_t)t * nthreads + threadIdx.x], even = halves & 0xffffu, odd = halves >> 16;
    __shared__ unsigned short wave_of_block[16];
    __shared__ unsigned slice_rows[16];
    __shared__ __align__(16) unsigned char of_wave[16][kPermLengths];     // columns of each length in a wavefront
    __shared__ unsigned longer[kPermLengths];                             // columns of greater length
    if (threadIdx.x < 16) slice_rows[threadIdx.x] = 0u;
    for (int i = threadIdx.x; i < nslices * kPermLengths / 16; i += nthreads) reinterpret_cast<uint4*>(of_wave)[i] = make_uint4(0u, 0u, 0u, 0u);
    // (the slots a column needs depend by one on the lane it gets; the larger of the two; columns of equal length stay in index order)
    const unsigned length = max(even, odd);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    // place among the columns in descending order of the length: the longer ones, the equal ones of the wavefronts before, the equal
    // ones of the lanes before
    unsigned place = 0;
    if (!__syncthreads_or(length >= (unsigned)kPermLengths)) {
        unsigned long long equal = ~0ull;
#pragma unroll
        for (int bit = 1; bit < kPermLengths; bit <<= 1) {
            const unsigned long long set = __ballot((length & bit) != 0u);
            equal &= (length & bit) != 0u ? set : ~set;
        }
        const unsigned below = (unsigned)__popcll(equal & ((1ull << lane) - 1ull));
        if (below == 0u) of_wave[wave][length] = (unsigned char)__popcll(equal);      // (at most 64)
        __syncthreads();
        for (int n = threadIdx.x; n < kPermLengths; n += nthreads) {
            unsigned all = 0;
            for (int v = 0; v < nslices; ++v) all += of_wave[v][n];
            longer[n] = all;
        }
        __syncthreads();
        if (wave == 0) {
            constexpr int kPer = kPermLengths / 64;
            unsigned n[kPer], sum = 0;
#pragma unroll
            for (int i = 0; i < kPer; ++i) { n[i] = longer[lane * kPer + i]; sum += n[i]; }
            unsigned from = sum;                                          // columns of this lane's lengths and of longer ones
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                const unsigned above = __shfl_down(from, off, 64);
                if (lane + off < 64) from += above;
            }
            from -= sum;
#pragma unroll
            for (int i = kPer - 1; i >= 0; --i) { longer[lane * kPer + i] = from; from += n[i]; }
        }
        __syncthreads();
        place = longer[length] + below;
        for (int v = 0; v < wave; ++v) place += of_wave[v][length];
    } else {
        // (lengths that few tiles have: every column compared with every other)
        key[threadIdx.x] = length;
        __syncthreads();
        for (int c = 0; c < nthreads; ++c) place += key[c] > length || (key[c] == length && c < (int)threadIdx.x) ? 1u : 0u;
        __syncthreads();
    }
    // key[] now by place: the first of each block of 64 is the block's longest column
    key[place] = 2u * length;
    __syncthreads();
    if (threadIdx.x < 64) {
        // (four lanes are the SIMDs: their sums so far, wavefronts handed out)
        unsigned sum = 0u;
        int used = 0;
        const int q = (int)threadIdx.x;
        for (int b = 0; b < nslices; ++b) {
            unsigned best = (q < 4 && q + 4 * used < nslices) ? sum * 4u + (unsigned)q : ~0u;       // (none left on that SIMD: not taken)
            best = min(best, (unsigned)__shfl_xor((int)best, 1, 64));
            best = min(best, (unsigned)__shfl_xor((int)best, 2, 64));
            if (q < 4 && (best & 3u) == (unsigned)q) {
                wave_of_block[b] = (unsigned short)(q + 4 * used);
                sum += (used == 0 ? 3u : 1u) * key[b * 64];              // (a SIMD's longest wavefront ends up walking alone)
                ++used;
            }
        }
    }
    __syncthreads();
    const unsigned thread = wave_of_block[place >> 6] * 64u + (place & 63u);
    colperm[(size_t)t * nthreads + thread] = (unsigned short)threadIdx.x;
    // the slot rows of each slice: those of its longest column, now that every column knows its lane
    atomicMax(&slice_rows[thread >> 6], column_slots(thread, even, odd));
    __syncthreads();
    if ((int)threadIdx.x < nslices) slice_len[(size_t)t * nslices + threadIdx.x] = slice_rows[threadIdx.x];
}

// The slot rows of each slice, those of its longest column, where thread t takes column t.  One workgroup per label tile, one
// thread per column.
__global__ void tile_count_kernel(const unsigned* __restrict__ counts, unsigned* __restrict__ slice_len) {
    const int t = blockIdx.x, nthreads = blockDim.x;
    const unsigned halves = counts[(size_t)t * nthreads + threadIdx.x];
    unsigned c = column_slots(threadIdx.x, halves & 0xffffu, halves >> 16);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) c = max(c, (unsigned)__shfl_xor((int)c, off));
    if ((threadIdx.x & 63) == 0) slice_len[(size_t)t * (nthreads >> 6) + (threadIdx.x >> 6)] = c;
}

// Exclusive prefix sum of n values into off[0..n] by one workgroup, and with `group` the largest sum of `group` consecutive ones
// from a multiple of it on, both to the host's memory (n is a few thousand; 25 us with the threads' sums added up by one of them,
// 15 with a thread's values asked for one by one, 13 so, 3 of them the largest sum).
__global__ __launch_bounds__(1024) void slice_scan_kernel(const unsigned* __restrict__ len, unsigned* __restrict__ off,
                                                           int n, int group, unsigned long long* __restrict__ total_out) {
    constexpr int kAtOnce = 16;
    const int per = (n + 1023) / 1024;
    const int b = min((int)threadIdx.x * per, n), e = min(b + per, n);
    unsigned long long sum = 0, total = 0;
    unsigned v[kAtOnce];                                                  // (the last ones asked for stay)
    auto ask = [&](int i0) {
#pragma unroll
        for (int i = 0; i < kAtOnce; ++i) v[i] = i0 + i < e ? len[i0 + i] : 0u;
    };
    for (int i0 = b; i0 < e; i0 += kAtOnce) {
        ask(i0);
#pragma unroll
        for (int i = 0; i < kAtOnce; ++i) sum += v[i];
    }
    unsigned long long run = block_sum_below<1024>(sum, &total);
    for (int i0 = b; i0 < e; i0 += kAtOnce) {
        if (per > kAtOnce) ask(i0);
#pragma unroll
        for (int i = 0; i < kAtOnce; ++i) {
            if (i0 + i < e) off[i0 + i] = (unsigned)run;
            run += v[i];
        }
    }
    if (threadIdx.x == 1023) {
        off[n] = (unsigned)total;
        *total_out = total;
    }
    if (group <= 0) return;
    __shared__ unsigned longest;
    if (threadIdx.x == 0) longest = 0u;
    __syncthreads();                                                      // (off[] as well)
    unsigned most = 0u;
    for (int t = threadIdx.x; t < n / group; t += 1024) most = max(most, off[(t + 1) * group] - off[t * group]);
    atomicMax(&longest, most);
    __syncthreads();
    if (threadIdx.x == 0) total_out[1] = longest;
}

// Slots of a tile, one workgroup per tile; its wavefronts take consecutive stretches of the tile's connections.
// Per slot: lab16 = LDS row of the label (rowpos), pos16 = position inside the tile's rows of lookup; the
// slots a column leaves empty up to the slice's length become padding: pos16 = pad_pos (kPadPos; in plans whose walking
// kernel keeps the tile's weights in LDS, tile_labels * K: the position of a zero word behind them), lab16 =
// zero_row + parity (all-zero rows).
// With `slot32` (plans whose walking kernel keeps the tile's weights in LDS) the two go into one word per slot,
// (position << 17) | (LDS row << 7): one load per slot, the row's byte offset already in place.
// Every wavefront counts its connections per column and bank half; sums over the wavefronts turn the counts into the slots that
// each wavefront's first connection of a column and half goes to (see column_slots), counted from the tile's first; then the wavefronts
// walk their stretches again, 64 connections at a time, and each takes the slot it finds and leaves the next one there.  Slots are
// in the order of flat positions: of several connections of one column and half among 64, which find what one of the others has
// already moved on, the lanes' order decides, not the LDS's.
// STAGED: the tile's positions gather in LDS and leave in whole rows; the next form, for tiles that do not fit there or whose
// slots 16 bits do not number, counts ranks and writes slots where they belong.
// Bound by the LDS's atomics and the latency of the walk.  Written where they belong one by one, slots are bound by the L2's write
// requests instead.  670,091 labels x fan-in 32 over 768 columns 216 -> 129 us, against bitmaps of labels per column with chains for
// labels that list a column twice, slots written one by one; 501,070 x 64 over 512 772 -> 171; with two workgroups on a CU, where
// both fit, the former 112; tiles that had no room for the bitmaps,
// or more such labels than the chains held, were scanned: 200,000 x 40 over 1,000 4,392 -> 76, 300,000 x 16 over 768 2,254 -> 288 (all
// of the build).
constexpr int kFillThreads = 1024;
constexpr unsigned kFillRows = 1021;         // (a slot of its last row and 128 more are below 2^16)
template <bool STAGED>
__global__ __launch_bounds__(kFillThreads) void tile_fill_kernel(const int32_t* __restrict__ idx, const unsigned short* __restrict__ rowpos, int L, int K,
                                                                 int tile_labels, int zero_row, const unsigned* __restrict__ slice_off,
                                                                 unsigned short* __restrict__ lab16, unsigned short* __restrict__ pos16, unsigned pad_pos,
                                                                 unsigned* __restrict__ slot32, int col_lo, const unsigned short* __restrict__ colperm,
                                                                 int ncols, unsigned stage_rows) {
    extern __shared__ __align__(16) unsigned fill_lds[];
    constexpr int kInflight = 8;
    constexpr unsigned kNone = 0xffffu;                                   // (no position: a tile has fewer than 2^16 - 1 connections)
    const int t = blockIdx.x, nthreads = blockDim.x, nwaves = nthreads >> 6, nslices = ncols >> 6;
    const unsigned* const offs = slice_off + (size_t)t * nslices;         // [nslices + 1]
    const unsigned tile_row0 = offs[0], tile_rows = offs[nslices] - tile_row0;
    const bool staged = tile_rows <= stage_rows;                          // (stage_rows <= kFillRows)
    if (staged != STAGED) return;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    unsigned short* const stage = reinterpret_cast<unsigned short*>(fill_lds);        // [stage_rows][64] positions
    unsigned* const base_of = fill_lds;                                   // (not staged: [ncols] a column's first slot << 1 | half that even slots hold)
    unsigned* const counts = fill_lds + (STAGED ? (size_t)stage_rows * 32 : (size_t)ncols);     // [wave][ncols] for labels in even rows | in odd rows << 16
    unsigned short* const row_of = reinterpret_cast<unsigned short*>(counts + (size_t)nwaves * ncols);          // [tile_labels]
    unsigned* const mine = counts + (size_t)wave * ncols;
    const int j0 = t * tile_labels, nl = min(tile_labels, L - j0);
    const int total = nl * K;
    const int* src = idx + (size_t)j0 * K;
    for (int i = threadIdx.x; i < nwaves * ncols; i += nthreads) counts[i] = 0u;
    for (int i = threadIdx.x; i < nl; i += nthreads) row_of[i] = rowpos[j0 + i];
    if (STAGED)
        for (unsigned i = threadIdx.x; i < tile_rows * 8u; i += nthreads) reinterpret_cast<uint4*>(stage)[i] = make_uint4(~0u, ~0u, ~0u, ~0u);
    __syncthreads();
    // this wavefront's connections, kInflight x 64 at a time: visit(column or ~0, LDS row of the label, position)
    const float per_label = 1.f / (float)K;
    auto label_at = [&](unsigned e) { return (unsigned)(((float)e + 0.5f) * per_label); };         // e / K for e < 2^16
    const int stretch = ((total + nwaves - 1) / nwaves + 63) & ~63, e_begin = min(wave * stretch, total), e_end = min(e_begin + stretch, total);
    auto walk = [&](auto visit) {
        unsigned next[kInflight];
        auto fetch = [&](int e0) {
#pragma unroll
            for (int i = 0; i < kInflight; ++i) {
                const int e = e0 + 64 * i + lane;
                next[i] = e < e_end ? (unsigned)(src[e] - col_lo) : ~0u;  // (columns outside the plan's window: no thread's)
            }
        };
        fetch(e_begin);
        for (int e0 = e_begin; e0 < e_end; e0 += 64 * kInflight) {
            unsigned c[kInflight], row[kInflight];
#pragma unroll
            for (int i = 0; i < kInflight; ++i) {
                c[i] = next[i];
                row[i] = row_of[label_at((unsigned)min(e0 + 64 * i + lane, e_end - 1))];
            }
            fetch(e0 + 64 * kInflight);
            visit(c, row, (unsigned)(e0 + lane));
        }
    };
    walk([&](const unsigned* c, const unsigned* row, unsigned) {
#pragma unroll
        for (int i = 0; i < kInflight; ++i)
            if (c[i] < (unsigned)ncols) atomicAdd(&mine[c[i]], (row[i] & 1u) ? 0x10000u : 1u);
    });
    __syncthreads();
    const size_t tile_slot0 = (size_t)tile_row0 * 64;
    auto put = [&](size_t slot, unsigned lab, unsigned pos) {
        const size_t at = tile_slot0 + slot;
        if (slot32 != nullptr) slot32[at] = (pos << 17) | (lab << 7);
        else { lab16[at] = (unsigned short)lab; pos16[at] = (unsigned short)pos; }
    };
    for (int walker = threadIdx.x; walker < ncols; walker += nthreads) {
        // (counts are kept per column; slices, lanes and slot parities belong to the threads that walk the plan)
        const unsigned col = colperm != nullptr ? colperm[(size_t)t * ncols + walker] : walker;
        const int sl = wave + (walker - (int)threadIdx.x) / 64;
        const unsigned first = parity_first(walker), base = (offs[sl] - tile_row0) * 64u + (unsigned)lane;
        unsigned run = STAGED ? (base + first * 64u) | (base + (first ^ 1u) * 64u) << 16 : 0u;
        for (int v = 0; v < nwaves; ++v) {
            const unsigned n = counts[(size_t)v * ncols + col];
            counts[(size_t)v * ncols + col] = run;
            run += STAGED ? n * 128u : n;                                 // (the next slot of a half is two rows on; both halves stay below 2^16)
        }
        if (!STAGED) {
            base_of[col] = base << 1 | first;                             // (rows < 2^24)
            const unsigned cnt[2] = {run & 0xffffu, run >> 16}, rows = offs[sl + 1] - offs[sl];
            for (unsigned r = 0; r < rows; ++r) {
                const unsigned par = (r & 1u) ^ first;                    // bank half this slot belongs to
                if ((r >> 1) >= cnt[par]) put((size_t)base + (size_t)r * 64, (unsigned)zero_row + par, pad_pos);
            }
        }
    }
    __syncthreads();
    walk([&](const unsigned* c, const unsigned* row, unsigned e) {
        constexpr unsigned kStep = STAGED ? 128u : 1u;
        unsigned before[kInflight], found[kInflight];
#pragma unroll
        for (int i = 0; i < kInflight; ++i) {
            before[i] = found[i] = 0u;
            if (c[i] < (unsigned)ncols) {
                before[i] = mine[c[i]];
                found[i] = atomicAdd(&mine[c[i]], (row[i] & 1u) ? kStep << 16 : kStep);
            }
        }
#pragma unroll
        for (int i = 0; i < kInflight; ++i) {
            const bool on = c[i] < (unsigned)ncols;
            const unsigned par = row[i] & 1u, shift = par * 16u, key = on ? c[i] * 2u + par : ~0u;
            unsigned at = before[i] >> shift & 0xffffu;
            for (unsigned long long left = __ballot(on && (found[i] >> shift & 0xffffu) != at); left != 0ull;) {
                const unsigned k = (unsigned)__builtin_amdgcn_readlane((int)key, __builtin_ctzll(left));
                const unsigned long long same = __ballot(key == k);
                if (key == k) at += kStep * (unsigned)__popcll(same & ((1ull << lane) - 1ull));
                left &= ~same;
            }
            if (on) {
                if (STAGED) {
                    stage[at] = (unsigned short)(e + 64u * i);
                } else {
                    const unsigned base = base_of[c[i]];
                    put((size_t)(base >> 1) + (size_t)(2u * at + (par ^ (base & 1u))) * 64, row[i], e + 64u * i);
                }
            }
        }
    });
    if (!STAGED) return;
    __syncthreads();
    // eight slots of a row per lane; two wavefronts take the rows of a slice
    for (int u = wave; u < 2 * nslices; u += nwaves) {
        const int sl = u >> 1;
        const unsigned begin = offs[sl] - tile_row0, len = offs[sl + 1] - offs[sl], lane8 = (unsigned)lane & 7u;
        const unsigned first = parity_first(8u * lane8);
        for (unsigned r = (unsigned)(u & 1) * 8u + ((unsigned)lane >> 3); r < len; r += 16u) {
            const uint4 q = reinterpret_cast<const uint4*>(stage)[(begin + r) * 8u + lane8];
            const unsigned w[4] = {q.x, q.y, q.z, q.w};
            unsigned lab[8], pos[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const unsigned at = w[i / 2] >> (16 * (i & 1)) & 0xffffu;
                const bool pad = at == kNone;
                lab[i] = row_of[pad ? 0u : label_at(at)];
                lab[i] = pad ? (unsigned)zero_row + ((r & 1u) ^ first) : lab[i];
                pos[i] = pad ? pad_pos : at;
            }
            const size_t to = tile_slot0 + (size_t)(begin + r) * 64 + 8u * lane8;
            if (slot32 != nullptr) {
                uint4* out = reinterpret_cast<uint4*>(slot32 + to);
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    out[h] = make_uint4(pos[4 * h] << 17 | lab[4 * h] << 7, pos[4 * h + 1] << 17 | lab[4 * h + 1] << 7,
                                        pos[4 * h + 2] << 17 | lab[4 * h + 2] << 7, pos[4 * h + 3] << 17 | lab[4 * h + 3] << 7);
            } else {
                *reinterpret_cast<uint4*>(lab16 + to) = make_uint4(lab[0] | lab[1] << 16, lab[2] | lab[3] << 16, lab[4] | lab[5] << 16, lab[6] | lab[7] << 16);
                *reinterpret_cast<uint4*>(pos16 + to) = make_uint4(pos[0] | pos[1] << 16, pos[2] | pos[3] << 16, pos[4] | pos[5] << 16, pos[6] | pos[7] << 16);
            }
        }
    }
}
// LDS of a workgroup, without its stage; the form that has none has the columns' slots in its place
inline size_t tile_fill_lds(int threads, int ncols, int tile_labels) {
    return (size_t)(threads / 64) * ncols * sizeof(unsigned) + (size_t)((tile_labels + 1) & ~1) * sizeof(unsigned short);
}

// ---- blocked global form ------------------------------------------------------------------------

// ptr[n] = first position in the sorted key array whose key is >= n (n in [0,nkeys]), and the octs that the kListsPerBlock lists
// of a workgroup take together
constexpr int kListsPerBlock = kBlock - 1;
__global__ __launch_bounds__(kBlock) void list_ptr_kernel(const unsigned* __restrict__ sorted_keys, int total, int nkeys,
                                                          int32_t* __restrict__ ptr, unsigned* __restrict__ block_octs) {
    __shared__ int begin[kBlock];
    const int n = (int)min(blockIdx.x * (unsigned)kListsPerBlock + threadIdx.x, (unsigned)nkeys);
    int lo = 0, hi = total;
    while (lo < hi) {
        const int mid = lo + ((hi - lo) >> 1);
        if (sorted_keys[mid] < (unsigned)n) lo = mid + 1; else hi = mid;
    }
    ptr[n] = lo;
    begin[threadIdx.x] = lo;
    __syncthreads();
    // (behind the last list begin and end are the same)
    const unsigned octs = threadIdx.x < kListsPerBlock ? (unsigned)(begin[threadIdx.x + 1] - lo + 7) / 8u : 0u;
    unsigned long long sum = 0;
    (void)block_sum_below<kBlock>(octs, &sum);
    if (threadIdx.x == 0) block_octs[blockIdx.x] = (unsigned)sum;
}

// oct_ptr[n] = octs of the lists before list n, from the octs before the list's workgroup of list_ptr_kernel
__global__ __launch_bounds__(kBlock) void oct_ptr_kernel(const int32_t* __restrict__ ptr, int nkeys, const unsigned* __restrict__ octs_before,
                                                         unsigned* __restrict__ oct_ptr) {
    const unsigned n = blockIdx.x * (unsigned)kListsPerBlock + threadIdx.x;
    const bool mine = threadIdx.x < kListsPerBlock && n < (unsigned)nkeys;
    const unsigned octs = mine ? (unsigned)(ptr[n + 1] - ptr[n] + 7) / 8u : 0u;
    unsigned long long sum = 0;
    const unsigned at = octs_before[blockIdx.x] + (unsigned)block_sum_below<kBlock>(octs, &sum);
    if (mine) {
        oct_ptr[n] = at;
        if (n == (unsigned)nkeys - 1u) oct_ptr[nkeys] = at + octs;
    }
}

int bits_for(unsigned max_value) {
    int b = 1;
    while (b < 32 && (max_value >> b) != 0) ++b;
    return b;
}

// Detaches the arrays from the plan.  keep == true (a rebuild follows): their buffers go to the spare list.
void free_spares(ffi_plan* p);
void free_arrays(ffi_plan* p, bool keep = false) {
    if (p->upper != nullptr) {
        // (the second column window's arrays: freed, never kept -- inputs that wide are rare and their plans small)
        free_arrays(p->upper, false);
        free_spares(p->upper);
        delete p->upper;
        p->upper = nullptr;
    }
    p->col_lo = 0; p->col_n = 0;
    for (const ffi_plan::Buffer& b : p->owned) {
        if (keep) p->spare.push_back(b);
        else (void)hipFree(b.ptr);
    }
    p->owned.clear();
    p->rowpos = nullptr;
    p->oct_ptr = nullptr; p->slot_pos = nullptr; p->slot_lab = nullptr; p->pos_slot = nullptr; p->slots = 0; p->slice_off = nullptr; p->lab16 = nullptr; p->pos16 = nullptr; p->slot32 = nullptr; p->idx16 = nullptr; p->colperm = nullptr;
    p->tiled = false; p->w_in_lds = false; p->total_rows = 0; p->bytes = 0;
}

void free_spares(ffi_plan* p) {
    for (const ffi_plan::Buffer& b : p->spare) (void)hipFree(b.ptr);
    p->spare.clear();
}

// A buffer of `count` elements for one of the plan's arrays: a spare one that fits (and is not more than half as
// large again), else a new allocation with 3 % of headroom, so that the next rebuild's slightly different sizes fit.
template <class T>
bool dev_alloc(ffi_plan* p, T** ptr, size_t count) {
    const size_t need = std::max<size_t>(count, 1) * sizeof(T);
    size_t best = p->spare.size();
    for (size_t i = 0; i < p->spare.size(); ++i)
        if (p->spare[i].bytes >= need && p->spare[i].bytes <= need + need / 2 + 4096 &&
            (best == p->spare.size() || p->spare[i].bytes < p->spare[best].bytes)) best = i;
    if (best != p->spare.size()) {
        *ptr = static_cast<T*>(p->spare[best].ptr);
        p->owned.push_back(p->spare[best]);
        p->spare.erase(p->spare.begin() + best);
        return true;
    }
    const size_t bytes = need + need / 32 + 256;
    void* raw = nullptr;
    if (hipMalloc(&raw, bytes) != hipSuccess) {
        (void)hipGetLastError();
        raw = nullptr;
        if (!p->spare.empty()) {                           // (what the last build left may be what is missing)
            free_spares(p);
            if (hipMalloc(&raw, bytes) != hipSuccess) { (void)hipGetLastError(); raw = nullptr; }
        }
    }
    if (raw == nullptr) {
        *ptr = nullptr;
        return false;
    }
    *ptr = static_cast<T*>(raw);
    p->owned.push_back({raw, bytes});
    return true;
}

// Returns a buffer obtained from dev_alloc to the spare list (temporaries of the build).
void dev_release(ffi_plan* p, void* ptr) {
    for (size_t i = 0; i < p->owned.size(); ++i)
        if (p->owned[i].ptr == ptr) {
            p->spare.push_back(p->owned[i]);
            p->owned.erase(p->owned.begin() + i);
            return;
        }
}

}  // namespace

// Labels per block of the global form: the block's rows of one slice of out_grad (128 bytes each) take five eighths of an
// XCD's L2 -- shared by as many blocks as the workgroups of that many columns leave room for at a time -- unless the
// lists of a block's columns would then hold fewer than eight connections.  Few columns (kWalkColumns to a workgroup of the walk) and
// few labels get as many blocks as the CUs have workgroups for in one go, as far as the lists keep twelve.  All passes at 126 x 1,242
// x 15,823 x 95: 449 us with three blocks, 160 with 25; 128 x 2,000 x 13,330 x 32 197 and 97, 128 x 2,500 x 131,072 x 32 351 and 328.
// (One block more, so that some CUs have two workgroups: 418 us at 128 x 1,300 x 131,072 x 32, where the former blocks took 345 and these 331.)
int plan_block_labels(int N, int K, int L) {
    const double resident = 20480.0 * std::min(1.0, (double)N / 4096.0), filled = 8.0 * (double)N / (double)K;
    const int chunks = (N + kWalkColumns - 1) / kWalkColumns, wanted = std::max(1, device_cu_count() / chunks);
    const double busy = std::max(std::max(128.0, 12.0 * N / K), std::ceil((double)L / wanted));
    const int labels = (int)std::min(65535.0, std::max(std::min(busy, 1024.0), std::max(std::min(resident, busy), filled)));
    return std::min(labels, L);
}

// Labels per tile of the tiled form, and whether the walking kernel keeps the tile's weights in LDS (then the tiles
// are smaller).
int plan_tile_labels(int N, int K, int L, int batch_hint, bool* weights_in_lds) {
    const int threads = ((N + 63) / 64) * 64;
    int TL = std::min((std::min(std::min(kPlanTileLabels, L), threads > 768 ? threads : 2 * threads) + 1) & ~1,
                      (int)((kPadPos - 1) / (unsigned)K) & ~1);
    // Tiles whose weights fit in LDS beside the tile of out_grad: the walking kernel then reads each slot's weight
    // through the slot's word, and the weights need not be brought into slot order first (no permutation kernel, no slot-ordered
    // copy of the weights in memory).
    // Measured (gx pass, 0.2-0.67 M labels, fan-in 8...128, 64...1024 columns), against permutation + walk with the
    // tiles and workgroups per CU that suit each form (tiled_workgroups_per_cu): with up to four batch tiles the form is
    // 5-60 % faster (most where the fan-in exceeds 32); with five to eight batch
    // tiles the tile's weights are staged that many times per tile: at fan-in 32 and below still -1...-8 % with 512 or 768 columns; with 576 to 768
    // columns -5...-13 % at every fan-in from 40 to 128 (one workgroup per CU either way); but +12 % at fan-in
    // 64 / 512 columns against the two-workgroup slot-ordered form, which also wins at 320-448 columns; with sixteen
    // batch tiles -7...+6 %: not taken.
    // The tile: as many labels as fit the LDS with their weights, one label per thread to stage; a thread carries
    // 8 x 16 bytes of the tile's weights in registers across the barrier, what exceeds that is copied behind it.
    // A slot's position inside the tile's weights has 15 bits (the zero word that padding slots read included).
    bool w_in_lds = false;
    const int nbt_hint = (batch_hint + 31) / 32;
    // Measured again once a tile's columns were sorted by length (which the form gets at 384 columns and more): 576 to 768
    // columns at 12 and 16 batch tiles, fan-in 32 and 64: -2...-6 % against the slot-ordered form, so workgroups of more than
    // 512 threads take the form at any batch size.  And at 256 columns and fewer, where several workgroups share a CU in
    // either form (670,091 labels): fan-in 16 -9...-20 % up to eight batch tiles; fan-in 32 -15...-36 % at one and two
    // batch tiles, equal at three, at four -21 % with 192 columns but +8 % with 256 (+16 % at fan-in 64), and +14...+30 %
    // at five to eight batch tiles (128 and 256 columns): from fan-in 32 on the slot-ordered form takes over there.
    const bool by_shape = threads > 512 ? true
                        : threads <= 256 ? (K < 32 ? nbt_hint <= 8 : (nbt_hint <= 3 || (nbt_hint == 4 && threads < 256)))
                                         : (nbt_hint <= 4 || (nbt_hint <= 8 && K <= 32 && threads == 512));
    const bool wanted = batch_hint > 0 && g_options.plan_weights_in_lds >= 0 && (g_options.plan_weights_in_lds > 0 || by_shape);   // (unknown batch size: the form for large batches)
    if (wanted && threads <= 768) {
        int tw = std::min(TL, threads & ~1);
        // (workgroups of at most 256 threads share a CU when there are batch tiles to overlap: tiled_workgroups_per_cu)
        const size_t budget = (threads <= 256 && nbt_hint >= 2) ? kPlanLdsBudget / (size_t)(768 / threads) : kPlanLdsBudget;
        while (tw >= 64 && tiled_lds_bytes(tw, K, true) > budget) tw -= 2;
        while (tw >= 64 && (long long)tw * K >= 32768) tw -= 2;
        // Tiles per workgroup come in whole numbers: the walking kernel runs cus / batch tiles label streams of
        // ceil(tiles / streams) tiles each, and the largest tile can leave the last stream nearly empty, or whole CUs
        // without a stream (670,091 labels in 618-label tiles: 1,085, of which the last of 64 streams gets 14 and the others 17).
        // The tile shrinks to what fills every stream with that same number of tiles (616 labels in that example); a
        // smaller tile pads a little more per connection, which costs less than the idle streams.  (Workgroups that share
        // a CU are left alone: there the streams outnumber the CUs.)
        if (tw >= 64 && (threads > 256 || nbt_hint < 2)) {
            const long long streams = std::max(1, device_cu_count() / std::max(1, nbt_hint));
            const long long tiles = ((long long)L + tw - 1) / tw;
            if (tiles > streams) {
                const long long per_stream = (tiles + streams - 1) / streams;
                int even = (int)(((long long)L + streams * per_stream - 1) / (streams * per_stream));
                even = (even + 1) & ~1;
                if (even >= 64 && even <= tw && even * 10 >= tw * 9) tw = even;
            }
        }
        if (tw >= 64) { TL = tw; w_in_lds = true; }
    }
    // the forms with weights in slot order, workgroups of at most 512 threads: one label per thread, so that two or more
    // workgroups share a CU (see tiled_workgroups_per_cu)
    if (!w_in_lds && threads <= 512) TL = std::min(TL, std::max(2, threads & ~1));
    *weights_in_lds = w_in_lds;
    return TL;
}

namespace {

// Builds the tiled form.  Returns FFI_OK with p->tiled == false if the padded size would exceed
// three times the connection count, lanes without a column aside (heavily skewed column usage): the caller then builds the
// global form instead.
// (`after_row_assignment`, may be empty: called once the kernel that assigns the labels' LDS rows is enqueued, and before any that relies
// on the ids' range -- it takes
// nearly all of every CU's LDS for itself, and work for another stream enqueued behind it starts when it ends instead of
// halving the number of its workgroups that fit)
int build_tiled(ffi_plan* p, const int32_t* lookup, hipStream_t s, const std::function<int()>& after_row_assignment = {}) {
    const int cols = p->col_n ? p->col_n : p->N;           // the columns this plan's tiled form covers, from col_lo on
    const int threads = ((cols + 63) / 64) * 64;
    // every thread of the kernel that walks the plan stages at most two labels of a tile (one when
    // the workgroup is larger than 768 threads and registers are scarcer)
    // (even, so that label parity inside a tile is the parity of the LDS row)
    // and small enough for the positions inside a tile to fit 16 bits
    bool w_in_lds = false;
    const int TL = plan_tile_labels(cols, p->K, p->L, p->batch_hint, &w_in_lds);
    const int slices = threads / 64;
    const int tiles = (p->L + TL - 1) / TL;
    const size_t nslices = (size_t)tiles * slices;
    // (the walking kernel hands its sums from the tile's thread to the column's own thread through LDS: built for the
    // weights-in-LDS form, whose workgroup has the registers for both sets of sums)
    // Measured (input gradient, weights-in-LDS form, sorted against thread t <-> column t): 768 columns x fan-in 32, batch 128:
    // 1.517 -> 1.150 slot rows per connection, 251 -> 239 us; batch 64: 151 -> 141; fan-in 16: 178 -> 170; fan-in 64 (300,000
    // labels): 207 -> 190; 512 columns: 261 -> 251; 640 columns, batch 256: 226 -> 215; no gain at 256 columns and fewer (few
    // slices to sort into, several workgroups per CU), and a loss where a workgroup walks a single tile (131,072 labels, batch
    // 32: 35.4 -> 36.5 us): there the order of the columns stays.
    const bool sorted_columns = plan_sorts_columns(threads, TL, p->K, w_in_lds, tiles, p->batch_hint);
    p->colperm = nullptr;
    unsigned *slice_len = nullptr, *counts = nullptr;
    if (!dev_alloc(p, &p->slice_off, nslices + 1) || !dev_alloc(p, &slice_len, nslices) || !dev_alloc(p, &counts, (size_t)tiles * threads)) return FFI_ERR_OUT_OF_MEMORY;
    // rows per bank half: half the tile plus some room for the balancing, within the LDS the walking kernel can have
    const int cap = tiled_rows_per_half(TL);
    if (!dev_alloc(p, &p->rowpos, (size_t)p->L)) return FFI_ERR_OUT_OF_MEMORY;
    {
        const size_t lds = ((size_t)threads + 1) * sizeof(int) + (size_t)TL * ((p->K + 2) / 3) * sizeof(unsigned) + ((size_t)threads + 2) * sizeof(unsigned short);
        const auto color = p->K <= 32 ? tile_color_kernel<32, false> : p->K <= 64 ? tile_color_kernel<64, false> : tile_color_kernel<64, true>;
        hipError_t ea = hipFuncSetAttribute((const void*)color, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (ea != hipSuccess) return hip_fail(ea);
        hipLaunchKernelGGL(color, dim3(tiles), dim3(256), lds, s, lookup, p->L, p->K, TL, cap, threads, p->rowpos, p->col_lo,
                           sorted_columns ? 1 : 0, counts);
    }
    if (after_row_assignment) {
        const int st = after_row_assignment();
        if (st != FFI_OK) return st;
    }
    if (sorted_columns) {
        if (!dev_alloc(p, &p->colperm, (size_t)tiles * threads)) return FFI_ERR_OUT_OF_MEMORY;
        hipLaunchKernelGGL(tile_perm_kernel, dim3(tiles), dim3(threads), threads * sizeof(unsigned), s, counts, p->colperm, slice_len);
    } else {
        hipLaunchKernelGGL(tile_count_kernel, dim3(tiles), dim3(threads), 0, s, counts, slice_len);
    }
    unsigned long long* found = nullptr;                   // (slot rows, and those of the longest tile: written where the host reads them)
    FFI_HIP_TRY(hipHostGetDevicePointer((void**)&found, p->h_scratch + 2, 0));
    hipLaunchKernelGGL(slice_scan_kernel, dim3(1), dim3(1024), 0, s, slice_len, p->slice_off, (int)nslices,
                       slices, found);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    dev_release(p, slice_len);
    dev_release(p, counts);
    if (e != hipSuccess) return hip_fail(e);
    const unsigned long long rows = p->h_scratch[2], longest_tile = p->h_scratch[3];
    const unsigned long long connections = (unsigned long long)p->L * p->K;
    // Too skewed (a window of the columns may have two slots per connection of the layer: how many of them fall into
    // it is not counted), or beyond what the walking kernel's 32-bit buffer offsets reach (256 bytes per row).  Lanes
    // that have no column do not count: they take slots, but no time that another form would save.  (With them counted,
    // inputs of fewer than some 30 columns, of 40 where tiles are small, took the global form, whose walk has too few columns
    // to fill the GPU.  Both gradients at 21 columns, tiled against global: 327 x 5,088 x 7 64 us against 391,
    // 64 x 100,000 x 16 74 / 263, 128 x 670,091 x 32 1,115 / 2,614; at 12 columns, 8 x 200,000 x 12, 201 / 237.  At 6 and 3
    // columns that last shape is the one that turns, 323 / 276 and 559 / 418; 327 x 5,088 x 7 there 80 / 1,023 and 99 / 2,020.)
    const unsigned long long allowed = p->col_n ? 2ull : 3ull;
    if (rows * 64ull * (unsigned long long)cols > (allowed * connections + 64ull * nslices) * (unsigned long long)threads || rows >= (1ull << 24)) return FFI_OK;
    if (w_in_lds) {
        if (!dev_alloc(p, &p->slot32, (size_t)rows * 64)) return FFI_ERR_OUT_OF_MEMORY;
    } else if (!dev_alloc(p, &p->lab16, (size_t)rows * 64) || !dev_alloc(p, &p->pos16, (size_t)rows * 64)) {
        return FFI_ERR_OUT_OF_MEMORY;
    }
    {
        const unsigned pad_pos = w_in_lds ? (unsigned)TL * (unsigned)p->K : kPadPos;
        // a wavefront for each eight rounds of 64 connections, fewer where two workgroups fit a CU, or one does, only then; what does not
        // fit even so is left to the other form
        const size_t cu = 160 * 1024, whole = std::min<size_t>((size_t)longest_tile, kFillRows);
        int fill_threads = std::min(kFillThreads, std::max(1, TL * p->K / 512) * 64);
        for (const size_t most : {cu / 2, cu}) {
            int fewer = fill_threads;
            while (fewer >= 512 && tile_fill_lds(fewer, threads, TL) + whole * 128 > most) fewer -= 64;
            if (fewer >= std::min(fill_threads, 512)) { fill_threads = fewer; break; }
        }
        const size_t counts = tile_fill_lds(fill_threads, threads, TL), stage_rows = std::min((cu - counts) / 128, whole);
        for (const bool staged : {true, false}) {
            if (!staged && longest_tile <= stage_rows) break;
            const auto fill = staged ? tile_fill_kernel<true> : tile_fill_kernel<false>;
            const size_t lds = counts + (staged ? stage_rows * 128 : threads * sizeof(unsigned));
            hipError_t ea = hipFuncSetAttribute((const void*)fill, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
            if (ea != hipSuccess) return hip_fail(ea);
            hipLaunchKernelGGL(fill, dim3(tiles), dim3(fill_threads), lds, s, lookup, p->rowpos, p->L, p->K, TL, 2 * cap, p->slice_off,
                               p->lab16, p->pos16, pad_pos, p->slot32, p->col_lo, p->colperm, threads, (unsigned)stage_rows);
        }
    }
    e = hipGetLastError();
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) return hip_fail(e);
    p->tiled = true;
    p->w_in_lds = w_in_lds;
    p->tile_labels = TL; p->threads = threads; p->slices = slices; p->tiles = tiles; p->zero_row = 2 * cap;
    p->total_rows = (long long)rows;
    p->bytes += (size_t)rows * 64 * 2 * sizeof(unsigned short) + (nslices + 1) * sizeof(unsigned) + (size_t)p->L * sizeof(unsigned short) +
                (p->colperm ? (size_t)tiles * threads * sizeof(unsigned short) : 0);
    return FFI_OK;
}

// key[p] = (label block of p) * N + column id of p
__global__ __launch_bounds__(kBlock) void block_key_kernel(const int32_t* __restrict__ idx, int total, int K, int N,
                                                           int block_labels, unsigned* __restrict__ key, int32_t* __restrict__ pos) {
    const int p = blockIdx.x * kBlock + threadIdx.x;
    if (p >= total) return;
    const int j = p / K;
    key[p] = (unsigned)(j / block_labels) * (unsigned)N + (unsigned)idx[p];
    pos[p] = p;
}

// All slots say that they are padding, four at a time.
__global__ __launch_bounds__(kBlock) void slot_clear_kernel(int4* __restrict__ slot_pos, uint2* __restrict__ slot_lab, size_t quads) {
    const size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= quads) return;
    slot_pos[i] = make_int4(-1, -1, -1, -1);
    slot_lab[i] = make_uint2((unsigned)kNoLabel * 0x10001u, (unsigned)kNoLabel * 0x10001u);
}

// The slots of every list's connections; what is left of its last oct is padding.  Bound by scattered stores, pos_slot's above all.
// (Build of 65,536 x 670,091 x 72, 48 M connections in 2.1 M lists: 2.41 ms with the padding written by each list's last
// connection -- 0.91 here, a few lanes of a wavefront in turn -- 2.30 by a kernel over the lists, 2.25 by a clear pass ahead: 0.05
// and 0.68 here.  32,768 x 670,000 x 32 1.07 / 1.04 / 1.04; 5,000 x 131,072 x 32 0.241 / 0.247 / 0.247.)
__global__ __launch_bounds__(kBlock) void slot_fill_kernel(const unsigned* __restrict__ sorted_keys, const int32_t* __restrict__ sorted_pos,
                                                           const int32_t* __restrict__ ptr, const unsigned* __restrict__ oct_ptr, int total,
                                                           int K, int N, int block_labels, int32_t* __restrict__ slot_pos,
                                                           unsigned short* __restrict__ slot_lab, unsigned* __restrict__ pos_slot) {
    const int e = blockIdx.x * kBlock + threadIdx.x;
    if (e >= total) return;
    const unsigned key = sorted_keys[e];
    const size_t slot = (size_t)oct_ptr[key] * 8 + (size_t)(e - ptr[key]);
    const int pos = sorted_pos[e];
    slot_pos[slot] = pos;
    pos_slot[pos] = (unsigned)slot;
    slot_lab[slot] = (unsigned short)(pos / K - (int)(key / (unsigned)N) * block_labels);
}

}  // namespace

// Slots of the global form for column ids drawn uniformly: a list's length is a Poisson count, rounded up to whole octs.
size_t plan_expected_slots(int N, int K, int L) {
    const int labels = plan_block_labels(N, K, L);
    const double lists = (double)((L + labels - 1) / labels) * N, mu = (double)L * K / lists;
    double slots = mu + 3.5;
    if (mu < 64.0) {
        double p = std::exp(-mu);
        slots = 0.0;
        for (int n = 1; n < 256; ++n) { p *= mu / n; slots += p * (double)((n + 7) / 8 * 8); }
    }
    return (size_t)(slots * lists) + 8;
}

namespace {

// The build's temporaries lie in arrays that it fills last and in the workspaces that the backward pass will ask for: nothing
// is allocated and freed again.  The plan's own arrays are allocated for the slots that uniform ids would give while the sort
// runs.  (Six buffers of the build's own, and the plan's only once the number of slots was known, held the host for 2 ms of the
// 3.6 to 4.9 of a first pass at 50 x 32,768 x 670,000 x 32, whose kernels take 2.2.)
int build_global(ffi_plan* p, const int32_t* lookup, hipStream_t s) {
    const int total = p->L * p->K;  // validated to fit int32 by the caller
    const int block_labels = plan_block_labels(p->N, p->K, p->L);
    const int nblocks = (p->L + block_labels - 1) / block_labels;
    const long long nkeys = (long long)nblocks * p->N;
    if (nkeys >= (1ll << 31) - 1) return FFI_ERR_TOO_LARGE;
    const int end_bit = bits_for((unsigned)(nkeys - 1));
    const unsigned list_blocks = (unsigned)((nkeys + kListsPerBlock - 1) / kListsPerBlock);
    size_t expected = plan_expected_slots(p->N, p->K, p->L), sort_bytes = 0;
    expected = (std::max<size_t>((size_t)total, std::min<size_t>(expected + expected / 128, (1ull << 32) - 64)) + 63) / 64 * 64;
    // (two buffers, not four: an allocation is 50 us and more; each array on a line of its own)
    auto alloc_slots = [&](size_t slots) {
        slots = (slots + 63) / 64 * 64;
        if (!dev_alloc(p, &p->slot_pos, slots + slots / 2)) return false;
        p->slot_lab = reinterpret_cast<unsigned short*>(p->slot_pos + slots);
        return true;
    };
    const size_t lists_end = ((size_t)nkeys + 1 + 63) / 64 * 64;
    if (!alloc_slots(expected) || !dev_alloc(p, &p->oct_ptr, lists_end + (size_t)total)) return FFI_ERR_OUT_OF_MEMORY;
    p->pos_slot = p->oct_ptr + lists_end;
    // stable LSD radix sort of ((block, column), flat position): positions stay ascending inside a column
    rocprim::double_buffer<unsigned> keys(reinterpret_cast<unsigned*>(p->slot_pos), nullptr);
    rocprim::double_buffer<int32_t> positions(reinterpret_cast<int32_t*>(p->pos_slot), nullptr);
    hipError_t e = rocprim::radix_sort_pairs(nullptr, sort_bytes, keys, positions, (unsigned)total, 0, end_bit, s);
    if (e != hipSuccess) return hip_fail(e);
    unsigned *key_ws = nullptr, *small_ws = nullptr;
    int32_t* pos_ws = nullptr;
    sort_bytes = (sort_bytes + 255) / 256 * 256;
    FFI_TRY(workspace_get(s, kWsSlots, expected * sizeof(unsigned), (void**)&key_ws));
    FFI_TRY(workspace_get(s, kWsWeightParts, expected * sizeof(int32_t), (void**)&pos_ws));
    FFI_TRY(workspace_get(s, kWsPartials, sort_bytes + ((size_t)nkeys + 1 + 2 * (size_t)list_blocks + 1) * sizeof(unsigned), (void**)&small_ws));
    int32_t* ptr = reinterpret_cast<int32_t*>(small_ws + sort_bytes / sizeof(unsigned));
    unsigned *block_octs = reinterpret_cast<unsigned*>(ptr) + nkeys + 1, *octs_before = block_octs + list_blocks;
    keys = rocprim::double_buffer<unsigned>(reinterpret_cast<unsigned*>(p->slot_pos), key_ws);
    positions = rocprim::double_buffer<int32_t>(reinterpret_cast<int32_t*>(p->pos_slot), pos_ws);
    auto grid = [](size_t n) { return dim3((unsigned)((n + kBlock - 1) / kBlock)); };
    hipLaunchKernelGGL(block_key_kernel, grid((size_t)total), dim3(kBlock), 0, s, lookup, total, p->K, p->N, block_labels, keys.current(),
                       positions.current());
    FFI_HIP_TRY(hipGetLastError());
    e = rocprim::radix_sort_pairs(small_ws, sort_bytes, keys, positions, (unsigned)total, 0, end_bit, s);
    if (e != hipSuccess) return hip_fail(e);
    // (after an even number of passes the result lies in the plan's arrays, which are about to be filled)
    if (keys.current() != key_ws) FFI_HIP_TRY(hipMemcpyAsync(key_ws, keys.current(), (size_t)total * sizeof(unsigned), hipMemcpyDeviceToDevice, s));
    if (positions.current() != pos_ws) FFI_HIP_TRY(hipMemcpyAsync(pos_ws, positions.current(), (size_t)total * sizeof(int32_t), hipMemcpyDeviceToDevice, s));
    unsigned long long* total_octs = nullptr;
    FFI_HIP_TRY(hipHostGetDevicePointer((void**)&total_octs, p->h_scratch, 0));
    hipLaunchKernelGGL(list_ptr_kernel, dim3(list_blocks), dim3(kBlock), 0, s, key_ws, total, (int)nkeys, ptr, block_octs);
    hipLaunchKernelGGL(slice_scan_kernel, dim3(1), dim3(1024), 0, s, block_octs, octs_before, (int)list_blocks, 0, total_octs);
    hipLaunchKernelGGL(oct_ptr_kernel, dim3(list_blocks), dim3(kBlock), 0, s, ptr, (int)nkeys, octs_before, p->oct_ptr);
    FFI_HIP_TRY(hipGetLastError());
    FFI_HIP_TRY(hipStreamSynchronize(s));
    const size_t slots = (size_t)p->h_scratch[0] * 8;
    if (slots >= (1ull << 32)) return FFI_ERR_TOO_LARGE;
    if (slots > expected || expected > slots + slots / 4 + (1u << 18)) {
        // ids that are not drawn uniformly
        dev_release(p, p->slot_pos);
        if (!alloc_slots(slots)) return FFI_ERR_OUT_OF_MEMORY;
    }
    hipLaunchKernelGGL(slot_clear_kernel, grid(slots / 4), dim3(kBlock), 0, s, reinterpret_cast<int4*>(p->slot_pos), reinterpret_cast<uint2*>(p->slot_lab), slots / 4);
    hipLaunchKernelGGL(slot_fill_kernel, grid((size_t)total), dim3(kBlock), 0, s, key_ws, pos_ws, ptr, p->oct_ptr, total, p->K, p->N,
                       block_labels, p->slot_pos, p->slot_lab, p->pos_slot);
    FFI_HIP_TRY(hipGetLastError());
    FFI_HIP_TRY(hipStreamSynchronize(s));
    p->block_labels = block_labels;
    p->nblocks = nblocks;
    p->slots = (long long)slots;
    p->bytes += slots * (sizeof(int32_t) + sizeof(unsigned short)) + ((size_t)nkeys + 1 + (size_t)total) * sizeof(unsigned);
    return FFI_OK;
}

// ---- arranged column ids for the weight gradient ------------------------------------------------
// The weight-gradient kernel reads, per connection, the 128-byte LDS row of the connection's
// column: even columns sit in one half of the LDS banks, odd columns in the other, and the LDS
// serves 16 lanes per clock only if 8 of them read each half.  Lanes l and l+8 work on labels j and
// j+8, so if the labels with bit 3 clear take their connections as even, odd, even, ... columns and
// the others as odd, even, odd, ..., the two lanes always read opposite halves (as far as a label's
// even and odd columns pair up; what is left over comes last).  One thread per (label, chunk of 32
// connections); entry i of a unit = (connection inside the chunk << 11) | column id; units are
// numbered chunk-major (u = chunk * L + label) so that consecutive lanes work on consecutive labels, and stored in
// blocks of 64 (arranged_quarter_offset).
// Half a wavefront takes a unit, a lane a connection: the connections of either role are a ballot, and a connection's place
// follows from the bits below its own.  So the ids are loaded in pieces of 128 bytes and nothing is looked at twice; a wavefront
// forms 64 consecutive units (one block of the stored layout) in LDS and stores the block's 4 KB in one piece.
// (670,091 labels x fan-in 32, beside the plan build's other kernels: a thread per unit, walking its 32 ids twice, 673 us; this 96.)

// The place of a lane's connection among the connections of its unit, which are those of `unit` (a mask of neighbouring lanes)
// with `on` set; called by whole wavefronts.
__device__ __forceinline__ unsigned arranged_place(bool on, int id, unsigned role, unsigned long long unit) {
    const bool first = ((unsigned)id & 1u) == role;               // (role: the parity taken at even places)
    const unsigned long long firsts = __ballot(on && first) & unit, seconds = __ballot(on && !first) & unit;
    const unsigned m = min((unsigned)__popcll(firsts), (unsigned)__popcll(seconds));
    const unsigned t = (unsigned)__popcll((first ? firsts : seconds) & ((1ull << (threadIdx.x & 63)) - 1ull));
    return t < m ? 2u * t + (first ? 0u : 1u) : 2u * m + (t - m);
}

__global__ __launch_bounds__(kBlock) void arrange_units_kernel(const int32_t* __restrict__ idx, int L, int K, int nchunks,
                                                                unsigned short* __restrict__ out) {
    __shared__ __align__(16) unsigned short outb[kBlock / 64][2048];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const long long total = (long long)L * nchunks;
    const long long u0 = ((long long)blockIdx.x * (kBlock / 64) + wave) * 64;
    if (u0 >= total) return;                              // (whole wavefronts; no workgroup barrier below)
    // (chunk and label of the wavefront's first unit by one division; the units behind it by stepping)
    const int c0 = (int)(u0 / L), j0 = (int)(u0 - (long long)c0 * L);
    const int k = lane & 31;
    const unsigned long long unit = 0xffffffffull << (lane & 32);
    unsigned short* ob = outb[wave];
    constexpr int kStep = 8;                              // loads in flight
    for (int r0 = 0; r0 < 32; r0 += kStep) {
        int id[kStep];
        bool on[kStep];
        unsigned role[kStep];
#pragma unroll
        for (int i = 0; i < kStep; ++i) {
            int c = c0, j = j0 + 2 * (r0 + i) + (lane >> 5);
            while (j >= L) { j -= L; ++c; }
            on[i] = c < nchunks && c * 32 + k < K;
            id[i] = on[i] ? idx[(size_t)j * K + c * 32 + k] : 0;
            role[i] = ((unsigned)j >> 3) & 1u;
        }
#pragma unroll
        for (int i = 0; i < kStep; ++i) {
            const unsigned place = arranged_place(on[i], id[i], role[i], unit);
            // a chunk the fan-in does not fill (and the units behind the last one, which pad the array to whole blocks): the
            // rest points at connection 31, which such a chunk never stores
            const unsigned pos = on[i] ? place : (unsigned)k;
            ob[(pos >> 3) * 512 + (unsigned)(2 * (r0 + i) + (lane >> 5)) * 8 + (pos & 7u)] =
                (unsigned short)(on[i] ? ((unsigned)k << kArrIdBits) | (unsigned)id[i] : 31u << kArrIdBits);
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    uint4* o4 = reinterpret_cast<uint4*>(out + (size_t)(u0 >> 6) * 2048);
    const uint4* b4 = reinterpret_cast<const uint4*>(outb[wave]);
#pragma unroll
    for (int i = 0; i < 4; ++i) o4[i * 64 + lane] = b4[i * 64 + lane];
}

// The same reordering applied in place to the lookup matrix itself and to up to four float matrices of its shape (weights,
// optimizer state): 2^lg lanes per (label, chunk of 32).  A unit whose connections are in place already is left alone: after a
// rewiring that is most of them, and then the pass is one of reading ids.  Bound by memory: all four matrices moved at 670,091
// labels x fan-in 32 are 690 MB.  (There, after one per cent of the connections was redrawn: a thread per unit with its ids and
// places in scratch memory 1,100 us; this 70.)
struct ArrangeArrays { float* a[4]; };
__global__ __launch_bounds__(kBlock) void arrange_in_place_kernel(int32_t* __restrict__ idx, ArrangeArrays arr, int L, int K,
                                                                   int nchunks, int lg) {
    const int lane = threadIdx.x & 63, width = 1 << lg, k = lane & (width - 1);
    const unsigned long long group = (lg == 5 ? 0xffffffffull : (1ull << width) - 1ull) << (lane - k);
    const long long total = (long long)L * nchunks, step = (long long)gridDim.x * kBlock >> lg;
    for (long long u = ((long long)blockIdx.x * kBlock + threadIdx.x) >> lg; u < total; u += step) {
        const int j = nchunks == 1 ? (int)u : (int)(u / nchunks), c = (int)(u - (long long)j * nchunks);
        const bool on = c * 32 + k < K;
        const size_t from = (size_t)j * K + c * 32 + k;
        const int32_t id = on ? idx[from] : 0;
        const unsigned pos = arranged_place(on, id, ((unsigned)j >> 3) & 1u, group);
        if (!on || !(__ballot(on && pos != (unsigned)k) & group)) continue;
        const size_t to = from - k + pos;
        float v[4];
#pragma unroll
        for (int a = 0; a < 4; ++a) v[a] = arr.a[a] != nullptr ? arr.a[a][from] : 0.f;
        // (every lane's loads are in before any lane stores: one wavefront, one instruction stream)
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        idx[to] = id;
#pragma unroll
        for (int a = 0; a < 4; ++a)
            if (arr.a[a] != nullptr) arr.a[a][to] = v[a];
    }
}

}  // namespace

int launch_arrange_in_place(int32_t* lookup, float* const* arrays, int n_arrays, int L, int K, hipStream_t s) {
    ArrangeArrays arr{{nullptr, nullptr, nullptr, nullptr}};
    for (int i = 0; i < n_arrays && i < 4; ++i) arr.a[i] = arrays[i];
    const int nchunks = (K + 31) / 32, lg = K <= 8 ? 3 : K <= 16 ? 4 : 5;
    const long long units = (long long)L * nchunks, blocks = ((units << lg) + kBlock - 1) / kBlock;
    hipLaunchKernelGGL(arrange_in_place_kernel, dim3((unsigned)std::min(blocks, 1ll << 20)), dim3(kBlock), 0, s, lookup, arr,
                       L, K, nchunks, lg);
    FFI_HIP_TRY(hipGetLastError());
    return FFI_OK;
}

namespace {

int build_arranged(ffi_plan* p, const int32_t* lookup, hipStream_t s) {
    const int nchunks = (p->K + 31) / 32;
    const long long units = (long long)p->L * nchunks;
    if (!dev_alloc(p, &p->idx16, arranged_words(units))) return FFI_ERR_OUT_OF_MEMORY;
    hipLaunchKernelGGL(arrange_units_kernel, dim3((unsigned)((units + kBlock - 1) / kBlock)), dim3(kBlock), 0, s, lookup,
                       p->L, p->K, nchunks, p->idx16);
    FFI_HIP_TRY(hipGetLastError());
    p->bytes += arranged_words(units) * sizeof(unsigned short);
    return FFI_OK;
}

}  // namespace

// device/pinned scratch words and the fingerprint event of a plan
int plan_scratch_alloc(ffi_plan* p) {
    const bool ok = hipMalloc(&p->d_scratch, kScratchWords * sizeof(unsigned long long)) == hipSuccess &&
                    hipHostMalloc(&p->h_scratch, kScratchWords * sizeof(unsigned long long)) == hipSuccess &&
                    hipEventCreateWithFlags(&p->fp_done, hipEventDisableTiming) == hipSuccess &&
                    hipMemset(p->d_scratch, 0, kScratchWords * sizeof(unsigned long long)) == hipSuccess &&
                    hipMalloc(&p->d_guard, kCheckWords * sizeof(unsigned long long)) == hipSuccess &&
                    hipHostMalloc(&p->h_guard, 8 * sizeof(unsigned long long)) == hipSuccess &&
                    hipMemset(p->d_guard, 0, kCheckWords * sizeof(unsigned long long)) == hipSuccess;
    if (!ok) {
        (void)hipGetLastError();
        return FFI_ERR_OUT_OF_MEMORY;
    }
    std::memset(p->h_guard, 0, 8 * sizeof(unsigned long long));      // check number 0: nothing has finished yet
    return FFI_OK;
}

void plan_reuse(ffi_plan* p, int L, int K, int N) {
    free_arrays(p, true);
    p->L = L; p->K = K; p->N = N;
    p->lookup = nullptr;
    p->fingerprint = ~0ull;
    std::memset(p->h_guard + 1, 0, 7 * sizeof(unsigned long long));      // (word 0: the number of a check, which only grows)
}

int plan_fingerprint_begin(ffi_plan* p, const int32_t* lookup, hipStream_t s) {
    const size_t total = (size_t)p->L * p->K;
    const unsigned blocks = (unsigned)std::min<size_t>((total / 4 + kBlock - 1) / kBlock + 1, kFingerprintBlocks);
    // words 0..7 of the scratch arrays belong to the plan build; the workgroups' partial sums follow
    unsigned long long* partials = p->d_scratch + 8;
    hipLaunchKernelGGL(fingerprint_kernel, dim3(blocks), dim3(kBlock), 0, s, lookup, total, (unsigned)p->N, partials);
    FFI_HIP_TRY(hipGetLastError());
    FFI_HIP_TRY(hipMemcpyAsync(p->h_scratch + 8, partials, 2 * (size_t)blocks * sizeof(unsigned long long), hipMemcpyDeviceToHost, s));
    FFI_HIP_TRY(hipEventRecord(p->fp_done, s));
    p->fp_blocks = (int)blocks;
    return FFI_OK;
}

int plan_fingerprint_end(ffi_plan* p, unsigned long long* out, unsigned long long* bad_ids) {
    FFI_HIP_TRY(hipEventSynchronize(p->fp_done));
    unsigned long long h = 0, bad = 0;
    for (int i = 0; i < p->fp_blocks; ++i) {
        h += p->h_scratch[8 + 2 * i];
        bad += p->h_scratch[8 + 2 * i + 1];
    }
    *out = h;
    *bad_ids = bad;
    return FFI_OK;
}

int plan_fingerprint(ffi_plan* p, const int32_t* lookup, hipStream_t s, unsigned long long* out,
                     unsigned long long* bad_ids) {
    FFI_TRY(plan_fingerprint_begin(p, lookup, s));
    return plan_fingerprint_end(p, out, bad_ids);
}

namespace {
int plan_build_arrays(ffi_plan* p, const int32_t* lookup, hipStream_t s, unsigned long long* fp_out);
}

// On failure the plan is left without arrays and without a lookup: it matches no cache key and
// launch_input_grad refuses it.
int plan_build(ffi_plan* p, const int32_t* lookup, hipStream_t s) {
    unsigned long long fp = 0;
    const int st = plan_build_arrays(p, lookup, s, &fp);
    if (st != FFI_OK) {
        free_arrays(p);
        p->lookup = nullptr;
        p->fingerprint = ~0ull;
        return st;
    }
    p->lookup = lookup;
    p->fingerprint = fp;
    // checks enqueued before this build (all finished: the build synchronises) are of no interest any more
    p->guard_seen = p->guard_seq;
    p->guard_stale = false;
    p->edited_by_library = false;
    return FFI_OK;
}

namespace {
int plan_build_arrays(ffi_plan* p, const int32_t* lookup, hipStream_t s, unsigned long long* fp_out) {
    // (what the host waits for first comes behind the work that is under way; the kernel below comes right behind it where there is one:
    // 1,221 us for a rewiring at 128 x 768 x 670,091 x 32, 1,235 the other way round)
    const bool wide = !tile_path_fits(p->N);
    if (wide) FFI_TRY(plan_fingerprint_begin(p, lookup, s));
    // a rebuild replaces the arrays: whatever still reads the old ones must have drained
    if (!p->owned.empty()) FFI_HIP_TRY(hipDeviceSynchronize());
    free_arrays(p, true);                      // (their buffers serve the new arrays where they fit)
    // The ids are checked, and the words that later checks compare with are set, beside the kernel that assigns the labels' rows, which
    // takes any ids: the others' LDS counters want them in range.  (A rewiring and the pass behind it at 128 x 768 x 670,091
    // x 32: 1,280 us with the host waiting before that kernel, 1,252 so.)
    if (!wide) FFI_TRY(plan_fingerprint_begin(p, lookup, s));
    bool checked = false;
    auto check_ids = [&]() -> int {
        if (checked) return FFI_OK;
        checked = true;
        unsigned long long bad = 0;
        FFI_TRY(plan_fingerprint_end(p, fp_out, &bad));
        if (bad != 0) {
            FFI_HIP_TRY(hipStreamSynchronize(s));
            return FFI_ERR_BAD_LOOKUP;
        }
        // no check of this plan is in flight, and the build waits for the stream
        hipLaunchKernelGGL(guard_init_kernel, dim3(1), dim3(64), 0, s, p->d_guard, *fp_out);
        FFI_HIP_TRY(hipGetLastError());
        return FFI_OK;
    };
    // The arranged ids of the weight gradient depend on the lookup alone: their kernel runs on a helper stream beside
    // the kernels of the tiled form (of which the longest runs one wavefront per tile and leaves the memory system idle).
    // (ids < 2^11 and an [N][32] fp32 tile in LDS: the shapes the narrow weight-gradient kernel takes)
    const bool arranged = tile_path_fits(p->N) && p->N < (1 << kArrIdBits);
    bool helper_busy = false;
    if (arranged) {
        if (p->helper_stream == nullptr) {
            if (hipStreamCreateWithFlags(&p->helper_stream, hipStreamNonBlocking) != hipSuccess ||
                hipEventCreateWithFlags(&p->helper_event, hipEventDisableTiming) != hipSuccess) {
                (void)hipGetLastError();
                if (p->helper_stream) { (void)hipStreamDestroy(p->helper_stream); p->helper_stream = nullptr; }
            }
        }
    }
    // (enqueued from inside the tiled build, behind the row-assignment kernel, where there is a tiled build)
    bool arranged_enqueued = !arranged;
    auto enqueue_arranged = [&]() -> int {
        FFI_TRY(check_ids());
        if (arranged_enqueued) return FFI_OK;
        arranged_enqueued = true;
        hipStream_t hs = p->helper_stream ? p->helper_stream : s;
        // (the host has waited for the fingerprint: the lookup is final, the helper needs no further ordering)
        if (hs != s) helper_busy = true;
        return build_arranged(p, lookup, hs);
    };
    auto join = [&]() -> int {
        if (helper_busy) { helper_busy = false; FFI_HIP_TRY(hipStreamSynchronize(p->helper_stream)); }
        return FFI_OK;
    };
    // tiled form: one thread per column (N <= 1024), tiles of at least 62 labels with positions in 16 bits
    // (and 32 rows of out_grad within 32-bit byte offsets, as the kernels' buffer loads need)
    if (p->N <= 1024 && p->K <= 1024 && p->L < (1 << 25)) {
        int st = build_tiled(p, lookup, s, enqueue_arranged);
        if (st != FFI_OK) { (void)join(); free_arrays(p); return st; }
    } else if (tile_path_fits(p->N) && p->N <= 2048 && p->K <= 1024 && p->L < (1 << 25)) {
        // 1,025 to 1,216 columns: the LDS tile of the other two passes holds them, a workgroup of one thread per column
        // does not.  Two tiled forms, one per half of the columns; each walk stages the tile's out_grad itself, which costs
        // far less than the cache-bound global form (measured at 1,216 columns, c2's other dimensions: 1.58 ms).
        const int lower = ((p->N + 1) / 2 + 63) / 64 * 64;
        p->col_lo = 0; p->col_n = lower;
        int st = build_tiled(p, lookup, s, enqueue_arranged);
        if (st == FFI_OK && p->tiled) {
            ffi_plan* u = new (std::nothrow) ffi_plan();
            if (u == nullptr) st = FFI_ERR_OUT_OF_MEMORY;
            else {
                u->device = p->device; u->L = p->L; u->K = p->K; u->N = p->N; u->batch_hint = p->batch_hint;
                u->col_lo = lower; u->col_n = p->N - lower;
                u->d_scratch = p->d_scratch; u->h_scratch = p->h_scratch;      // (borrowed for the build; never freed through `u`)
                p->upper = u;
                st = build_tiled(u, lookup, s);
                u->d_scratch = nullptr; u->h_scratch = nullptr;
                if (st == FFI_OK && u->tiled) p->bytes += u->bytes;
            }
        }
        if (st != FFI_OK) { (void)join(); free_arrays(p); return st; }
        if (!p->tiled || !p->upper || !p->upper->tiled) {
            // too skewed for the tiled form in one of the halves: both go, the global form serves all columns
            ffi_plan* u = p->upper;
            p->upper = nullptr;
            if (u) { free_arrays(u, false); free_spares(u); delete u; }
            p->tiled = false;
            p->col_lo = 0; p->col_n = 0;
        }
    }
    {
        const int st = enqueue_arranged();         // (no tiled build took place, or it ended before its row assignment)
        if (st != FFI_OK) { (void)join(); free_arrays(p); return st; }
    }
    if (!p->tiled) {
        // (the tiled form's arrays, if any were made, go back to the spare list; the arranged ids stay)
        for (void* q : {(void*)p->slice_off, (void*)p->rowpos, (void*)p->lab16, (void*)p->pos16, (void*)p->slot32, (void*)p->colperm})
            if (q) dev_release(p, q);
        p->slice_off = nullptr; p->rowpos = nullptr; p->lab16 = nullptr; p->pos16 = nullptr; p->slot32 = nullptr; p->colperm = nullptr;
        const size_t arranged_bytes = p->idx16 ? arranged_words((long long)p->L * ((p->K + 31) / 32)) * sizeof(unsigned short) : 0;
        p->bytes = 0;
        int st = build_global(p, lookup, s);
        if (st != FFI_OK) { (void)join(); free_arrays(p); return st; }
        p->bytes += arranged_bytes;
    }
    {
        const int st = join();
        if (st != FFI_OK) { free_arrays(p); return st; }
    }
    free_spares(p);                            // what this build did not reuse
    return FFI_OK;
}
}  // namespace

int plan_guard_begin(ffi_plan* p, const int32_t* lookup, hipStream_t s, LookupCheck* check) {
    // A check of this plan that may still be running on another stream shares the accumulators: the two must not
    // overlap.  The other stream's handle may be gone by now (its owner may have destroyed it), so it is not touched:
    // the host waits for the device.  Only a lookup used from two streams in turn pays this, once per switch.
    if (p->guard_seq != p->guard_seen && p->guard_stream != s) {
        FFI_HIP_TRY(hipDeviceSynchronize());
        bool seen = false, current = true;
        unsigned long long bad = 0;
        (void)plan_guard_poll(p, &seen, &current, &bad);          // (the result stays with the next check if it was bad)
        if (seen && !current) p->guard_stale = true;
    }
    const size_t total = (size_t)p->L * p->K;
    unsigned long long* mirror = nullptr;
    FFI_HIP_TRY(hipHostGetDevicePointer((void**)&mirror, p->h_guard, 0));
    *check = LookupCheck{lookup, total, (unsigned)p->N, (int)std::min<size_t>((total / 4 + kCheckThreads - 1) / kCheckThreads + 1, kCheckBlocks),
                         p->d_guard, mirror, p->guard_seq + 1};
    p->guard_seq += 1;
    p->guard_stream = s;
    return FFI_OK;
}

int plan_guard_enqueue(ffi_plan* p, const int32_t* lookup, hipStream_t s) {
    LookupCheck check;
    FFI_TRY(plan_guard_begin(p, lookup, s, &check));
    hipLaunchKernelGGL(fingerprint_guard_kernel, dim3((unsigned)check.blocks), dim3(kCheckThreads), 0, s, check);
    FFI_HIP_TRY(hipGetLastError());
    return FFI_OK;
}

int plan_guard_poll(ffi_plan* p, bool* seen, bool* current, unsigned long long* bad_ids) {
    *seen = false;
    if (p->guard_stale) {                                  // an outdated verdict met while switching streams
        p->guard_stale = false;
        *seen = true; *current = false; *bad_ids = 0;
        return FFI_OK;
    }
    if (p->guard_seq == p->guard_seen) return FFI_OK;
    // the last check that has finished (checks of a plan finish in the order they were enqueued)
    const unsigned long long word = __atomic_load_n(p->h_guard, __ATOMIC_ACQUIRE);
    const unsigned long long done = word >> 2;
    if (done <= p->guard_seen || done > p->guard_seq) return FFI_OK;        // nothing new (or a word of before the last build)
    p->guard_seen = done;
    *seen = true;
    *current = ((word >> 1) & 1ull) != 0;
    *bad_ids = word & 1ull;
    return FFI_OK;
}

void plan_free(ffi_plan* p) {
    if (!p) return;
    free_arrays(p);
    free_spares(p);
    if (p->helper_stream) { (void)hipStreamSynchronize(p->helper_stream); (void)hipStreamDestroy(p->helper_stream); p->helper_stream = nullptr; }
    if (p->helper_event) { (void)hipEventDestroy(p->helper_event); p->helper_event = nullptr; }
    if (p->d_scratch) (void)hipFree(p->d_scratch);
    if (p->h_scratch) (void)hipHostFree(p->h_scratch);
    if (p->fp_done) (void)hipEventDestroy(p->fp_done);
    if (p->d_guard) (void)hipFree(p->d_guard);
    if (p->h_guard) (void)hipHostFree(p->h_guard);
    p->d_scratch = nullptr; p->h_scratch = nullptr; p->fp_done = nullptr;
    p->d_guard = nullptr; p->h_guard = nullptr; p->guard_seq = 0; p->guard_seen = 0; p->guard_stale = false;
}

}  // namespace ffi
