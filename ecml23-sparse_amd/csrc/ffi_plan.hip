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
#include <type_traits>

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

// The sum of v over each LANES consecutive lanes (8, 32 or 64), in all of them.
template <int LANES> __device__ __forceinline__ int lanes_total(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0xb1, 0xf, 0xf, true);         // lane ^ 1
    v += __builtin_amdgcn_update_dpp(0, v, 0x4e, 0xf, 0xf, true);         // lane ^ 2
    v += __builtin_amdgcn_update_dpp(0, v, 0x141, 0xf, 0xf, true);        // 7 - lane within eight
    if (LANES == 8) return v;
    v += __builtin_amdgcn_update_dpp(0, v, 0x140, 0xf, 0xf, true);        // 15 - lane within sixteen
    const auto rows = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    v = (int)(rows[0] + rows[1]);
    if (LANES == 32) return v;
    const auto halves = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return (int)(halves[0] + halves[1]);
}

constexpr int kPastLabels = 16;         // a sweep's steps end up to seven labels behind the last one and look one step ahead
// What a sweep over a tile's labels works on, in LDS (see tile_color_kernel).
struct TileLabels {
    int* imb;                          // [ncols + 1] even minus odd labels per column
    const unsigned* ids3;              // [nl][W] column ids, three to a word
    const unsigned char* wt;           // [ncols + 1] weight of a column's balance; 0 at the end
    unsigned char* half;               // [nl + kPastLabels] the half each label goes to
    int nl, K, W, ncols, cap;
};

// One sweep, by one wavefront: 64 / LANES labels a step, PER connections of each in a lane's registers (MORE: the rest of the fan-in one by
// one).  AGAIN: every label is taken out and put back.  placed: labels in even and odd rows so far.
template <int LANES, int PER, bool MORE, bool AGAIN>
__device__ __forceinline__ void sweep_labels(const TileLabels& t, int (&placed)[2]) {
    constexpr int kAbreast = 64 / LANES;
    constexpr unsigned long long kFirst = LANES == 8 ? 0x0101010101010101ull : LANES == 32 ? 0x0000000100000001ull : 1ull;   // a label's first lane
    const int lane = threadIdx.x & 63, sub = lane & (LANES - 1), abreast = lane / LANES;
    int word_at[PER], shift[PER], col[PER], w[PER];
    unsigned word[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int k = min(sub + LANES * i, t.K - 1);
        word_at[i] = k / 3;
        shift[i] = 10 * (k % 3);
    }
    const int last = (t.nl - 1) * t.W;
    int label = abreast, row = min(abreast * t.W, last), row1 = row;       // of the step; first words of its label and of the next one asked for
    int next = abreast, next_half = 0;                                     // the label that advance() goes to
    // To `next`, whose words are here; those of the label behind it and the columns' weights are asked for.
    auto advance = [&]() {
        row1 = min(row1 + kAbreast * t.W, last);
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            // (behind the fan-in and behind the last label: the entry of weight 0)
            col[i] = sub + LANES * i < t.K && next < t.nl ? (int)((word[i] >> shift[i]) & 1023u) : t.ncols;
            word[i] = t.ids3[row1 + word_at[i]];
        }
#pragma unroll
        for (int i = 0; i < PER; ++i) w[i] = (int)t.wt[col[i]];
        if (AGAIN) next_half = t.half[next];
        next += kAbreast;
    };
    auto rest = [&](auto visit) {
        if (!MORE) return;
        for (int k = sub + LANES * PER; k < t.K; k += LANES) {
            const int c = (int)((t.ids3[row + k / 3] >> (10 * (k % 3))) & 1023u);
            visit(label < t.nl ? c : t.ncols);
        }
    };
    auto add = [&](const int (&c)[PER], int delta) {                       // (a column may occur twice in a label)
#pragma unroll
        for (int i = 0; i < PER; ++i)
            if (sub + LANES * i < t.K) atomicAdd(&t.imb[c[i]], delta);
        rest([&](int q) { atomicAdd(&t.imb[q], delta); });
    };
#pragma unroll
    for (int i = 0; i < PER; ++i) word[i] = t.ids3[row + word_at[i]];
    advance();
    const int steps = (t.nl + kAbreast - 1) / kAbreast, tie = (abreast & 1) ? -1 : 1;
    for (int g = 0; g < steps; ++g) {
        int c[PER], sum = 0;
        // (1 or -1: the half taken where the columns ask for neither -- the label's own, or the emptier one, by turns)
        const int lean = AGAIN ? (next_half ? 1 : -1) : placed[1] < placed[0] ? tie : -tie;
#pragma unroll
        for (int i = 0; i < PER; ++i) c[i] = col[i];
        if (AGAIN) add(c, lean);
#pragma unroll
        for (int i = 0; i < PER; ++i) sum += __mul24(w[i], t.imb[c[i]]);
        advance();
        rest([&](int q) { sum += t.wt[q] * t.imb[q]; });
        bool odd = 2 * lanes_total<LANES>(sum) + lean > 0;
        if (__builtin_expect(max(placed[0], placed[1]) + kAbreast > t.cap, 0)) {               // (uniform)
            // the halves may be full: where a label asks to go as far as there is room; labels that stay keep their places, theirs first
            const unsigned long long there = __ballot(label < t.nl) & kFirst, was = AGAIN ? __ballot(lean > 0) & there : 0ull;
            unsigned long long to = __ballot(odd) & there;
            const unsigned long long asked = to;
            int room[2] = {t.cap - placed[0], t.cap - placed[1]};
            if (AGAIN) {
                room[1] += __popcll(was);
                room[0] += __popcll(there & ~was);
            }
            for (int pass = 0; pass < 2; ++pass)
                for (int h = 0; h < kAbreast; ++h) {
                    const unsigned long long bit = 1ull << (h * LANES);
                    if (!(there & bit) || (AGAIN && ((asked ^ was) & bit)) != (pass == 1)) continue;
                    if (room[(to & bit) ? 1 : 0] <= 0) to ^= bit;
                    --room[(to & bit) ? 1 : 0];
                }
            placed[0] = t.cap - room[0];
            placed[1] = t.cap - room[1];
            odd = (to >> (abreast * LANES) & 1ull) != 0;
        } else if (AGAIN) {
            // (what is not there, behind the last label, stays as it was)
            const int more = ((int)__popcll(__ballot(odd)) - (int)__popcll(__ballot(lean > 0))) / LANES;
            placed[1] += more;
            placed[0] -= more;
        } else {
            const unsigned long long there = __ballot(label < t.nl) & kFirst;
            const int more = (int)__popcll(__ballot(odd) & there);
            placed[1] += more;
            placed[0] += (int)__popcll(there) - more;
        }
        add(c, odd ? -1 : 1);
        t.half[label] = odd ? 1 : 0;                                       // (all lanes of a label, one value)
        label += kAbreast;
        row = min(row + kAbreast * t.W, last);
    }
}

// Which LDS row of the walking kernel's tile each label is staged into (rowpos[j], inside the label's tile).
// The bank half a row lies in is the parity of its row number, and a column is walked fastest when its labels
// split evenly between the halves (see above: every hole costs a slot).  The label's own parity would split a
// column's labels like coin flips (about sqrt(n) excess); here the labels of a tile are taken in ascending order
// and each goes to the half that the columns it feeds have used less so far (weighted sum over its connections
// of even-count minus odd-count of the column), which keeps the columns that matter close to an even split.
// Rows of a half are handed out in ascending order, at most `cap` per half.  One workgroup per tile; the tile's
// column ids are staged in LDS, one wavefront then decides a few labels at a time (sweep_labels).
// (`col_lo`: the plan covers the columns [col_lo, col_lo + ncols) only; connections into other columns are left out)
// (`all_columns_count`: plans that hand the columns to threads by length -- there every column is about as long as the
// longest of its slice, so every column's balance weighs the same)
template <int LANES, int PER, bool MORE>     // of the second sweep: lanes per label, connections per lane (MORE: fan-ins beyond them)
__global__ __launch_bounds__(256) void tile_color_kernel(const int32_t* __restrict__ idx, int L, int K, int tile_labels, int cap,
                                                         int ncols, unsigned short* __restrict__ rowpos, int col_lo,
                                                         int all_columns_count, unsigned* __restrict__ counts) {
    extern __shared__ int color_lds[];
    // (entry `ncols` of both: where connections into columns outside the window go -- weight 0, so they never count)
    int* imb = color_lds;                                                        // [ncols + 1] even minus odd labels per column
    // The tile's column ids, three 10-bit ids per word, a label's ids in W = ceil(K / 3) words of its own, and the weights
    // and the halves in bytes: with 16-bit ids and 32-bit weights a tile of 582 labels x fan-in 32 took 44 KB of LDS, three workgroups per
    // CU and two rounds for 1,152 tiles; now 30 KB, five workgroups per CU, all tiles at once (the work of a tile is one
    // wavefront's sequential loop; 32,000 bytes are the most of which five fit, a tile of 616 labels takes 31.6 KB).
    const int W = (K + 2) / 3;
    unsigned* ids3 = reinterpret_cast<unsigned*>(color_lds + ncols + 1);         // [tile_labels * W]
    unsigned char* wt = reinterpret_cast<unsigned char*>(ids3 + (size_t)tile_labels * W);   // [ncols + 1] weight of the column's balance
    unsigned char* half = wt + ncols + 1;                                        // [tile_labels + kPastLabels] the half each label goes to
    const int t = blockIdx.x;
    const int j0 = t * tile_labels;
    const int nl = min(tile_labels, L - j0);
    const int* src = idx + (size_t)j0 * K;
    const unsigned outside = (unsigned)min(ncols, 1023);                          // (windows are at most 640 columns wide; a single window has no ids outside)
    for (int i = threadIdx.x; i <= ncols; i += 256) { imb[i] = 0; wt[i] = 0; }
    __syncthreads();
    constexpr int kTogether = 4;                                                 // words whose ids are asked for together
    for (int w0 = threadIdx.x; w0 < nl * W; w0 += 256 * kTogether) {
        unsigned v[kTogether][3];
        int k0[kTogether];
#pragma unroll
        for (int u = 0; u < kTogether; ++u) {
            const int wi = min(w0 + 256 * u, nl * W - 1), jl = wi / W;
            k0[u] = 3 * (wi - jl * W);
#pragma unroll
            for (int i = 0; i < 3; ++i) v[u][i] = (unsigned)(src[jl * K + min(k0[u] + i, K - 1)] - col_lo);
        }
#pragma unroll
        for (int u = 0; u < kTogether; ++u) {
            if (w0 + 256 * u >= nl * W) break;
            unsigned word = 0;
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                unsigned c = outside;                                            // (also behind the label's last id, where it is never read)
                if (k0[u] + i < K && v[u][i] < (unsigned)ncols) {
                    c = v[u][i];
                    atomicAdd(&imb[c], 1);                                       // column lengths first (in imb: the LDS adds whole words)
                }
                word |= c << (10 * i);
            }
            ids3[w0 + 256 * u] = word;
        }
    }
    __syncthreads();
    // Only the longest columns of a slice (64 columns, one wavefront of the walking kernel) set its number of slot
    // rows, so their balance counts most: weight = 255 * (length / longest of the slice)^8.
    for (int c = threadIdx.x; c < ncols; c += 256) {
        const int len = imb[c];
        imb[c] = 0;
        int longest = len;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) longest = max(longest, __shfl_xor(longest, off, 64));
        float r = longest > 0 ? (float)len / (float)longest : 0.f;
        r *= r; r *= r; r *= r;
        wt[c] = (unsigned char)(all_columns_count ? (len > 0 ? 1 : 0) : (int)(255.f * r));
    }
    __syncthreads();
    const int lane = threadIdx.x & 63;
    auto decide_all = [&]() {
    // What bounds the kernel is the chain from one step's adds to the next step's decision: an LDS round trip, the sum over the
    // lanes by DPP and lane swaps, a comparison in every lane, some 60 instructions of one wavefront.  Labels decided together do not see
    // what the others of the step just did.  In the first sweep that is mended by the second: eight a step.  In the second it stays: two
    // (one beyond a fan-in of 64).  Slot rows per connection, 582-label tiles of fan-in 32 over 768 columns: 1.5267 with two in both, 1.5279 so,
    // 1.5309 with four in the second; sorted columns 1.1542, 1.1549, 1.1559.  670,091 labels of fan-in 32 196 -> 126 us,
    // 14 of them ids asked for twelve at a time; 131,072 labels a whole build 248 -> 195, 50,000 of fan-in 100 897 -> 517.  Fan-ins of 33 to 64, two against one in the second: 1.3290
    // and 1.3269 (512 labels of 64 over 512 columns), 1.1888 and 1.1888 (567 of 38 over 584, sorted); builds at 501,070 x 64 and
    // 181,536 x 38 609 -> 503 us and 187 -> 125.  (The first sweep by
    // four wavefronts, a quarter of the labels each, and their sums put together: 1.5347, 1.1586.)
    int placed[2] = {0, 0};
    const TileLabels labels{imb, ids3, wt, half, nl, K, W, ncols, cap};
    sweep_labels<8, LANES / 8 * PER, MORE, false>(labels, placed);
    // Second sweep: every label is taken out and put back into the half its columns now ask for -- the first sweep placed
    // the early labels knowing nothing of the later ones.  (Measured on uniformly drawn ids, 586-label tiles of fan-in 32
    // over 768 columns: slot rows 1.528 -> 1.514 per connection, where columns of unconstrained order would need 1.490.)
    sweep_labels<LANES, PER, MORE, true>(labels, placed);
    // rows of a half are handed out in ascending label order
    int next[2] = {0, 0};
    for (int l0 = 0; l0 < nl; l0 += 64) {
        const bool on = l0 + lane < nl, odd = on && half[min(l0 + lane, nl - 1)] != 0;
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
        const int one = half[jl] ? 0x10000 : 1;
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
    unsigned long long total = 0;
    if (per <= kAtOnce) {
        const int b = min((int)threadIdx.x * per, n), e = min(b + per, n);
        unsigned long long sum = 0;
        unsigned v[kAtOnce];
#pragma unroll
        for (int i = 0; i < kAtOnce; ++i) {
            v[i] = b + i < e ? len[b + i] : 0u;
            sum += v[i];
        }
        unsigned long long run = block_sum_below<1024>(sum, &total);
#pragma unroll
        for (int i = 0; i < kAtOnce; ++i) {
            if (b + i < e) off[b + i] = (unsigned)run;
            run += v[i];
        }
    } else {
        // (very many columns: a stretch at a time, whose values come and go by whole lines)
        constexpr int kEach = 8, kStretch = 1024 * kEach;
        __shared__ unsigned stage[kStretch + kStretch / kEach];
        auto place = [](int i) { return i + i / kEach; };
        for (int n0 = 0; n0 < n; n0 += kStretch) {
#pragma unroll
            for (int i = 0; i < kEach; ++i) {
                const int at = i * 1024 + (int)threadIdx.x;
                stage[place(at)] = n0 + at < n ? len[n0 + at] : 0u;
            }
            __syncthreads();
            unsigned long long sum = 0, all = 0;
            unsigned v[kEach];
#pragma unroll
            for (int i = 0; i < kEach; ++i) {
                v[i] = stage[place((int)threadIdx.x * kEach + i)];
                sum += v[i];
            }
            unsigned long long run = total + block_sum_below<1024>(sum, &all);
#pragma unroll
            for (int i = 0; i < kEach; ++i) {
                stage[place((int)threadIdx.x * kEach + i)] = (unsigned)run;
                run += v[i];
            }
            total += all;
            __syncthreads();
#pragma unroll
            for (int i = 0; i < kEach; ++i) {
                const int at = i * 1024 + (int)threadIdx.x;
                if (n0 + at < n) off[n0 + at] = stage[place(at)];
            }
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

// ---- global form --------------------------------------------------------------------------------

// A position's stream: one per segment of labels and group of columns.
struct StreamOf {
    int K, seg_labels, segments, groups;
    __device__ __forceinline__ unsigned operator()(unsigned id, unsigned pos) const {
        const unsigned group = id / kGroupColumns;
        return segments == 1 ? group : pos / (unsigned)K / (unsigned)seg_labels * (unsigned)groups + group;
    }
};

// counts[t][u] = connections of stream u in tile t (or row of tiles: `tile_bits` is theirs), a workgroup per tile; so many streams at a time as the LDS has counters
constexpr int kTileThreads = 1024, kCountWindow = 16384;
__global__ __launch_bounds__(kTileThreads) void tile_streams_kernel(const int32_t* __restrict__ idx, int total, int tile_bits, int units,
                                                                    const StreamOf stream_of, unsigned* __restrict__ counts) {
    extern __shared__ __align__(16) unsigned tile_counts[];
    constexpr int kInflight = 8;
    const unsigned p0 = blockIdx.x << tile_bits, end = min(p0 + (1u << tile_bits), (unsigned)total);
    for (int u0 = 0; u0 < units; u0 += kCountWindow) {
        const int n = min(kCountWindow, units - u0);
        for (int i = threadIdx.x; i < n; i += kTileThreads) tile_counts[i] = 0u;
        __syncthreads();
        for (unsigned p = p0 + threadIdx.x; p < end; p += kTileThreads * kInflight) {
            unsigned id[kInflight];
#pragma unroll
            for (int i = 0; i < kInflight; ++i) id[i] = (unsigned)idx[min(p + i * kTileThreads, end - 1)];
#pragma unroll
            for (int i = 0; i < kInflight; ++i) {
                const unsigned at = p + i * kTileThreads, u = stream_of(id[i], at) - (unsigned)u0;
                if (at < end && u < (unsigned)n) atomicAdd(&tile_counts[u], 1u);
            }
        }
        __syncthreads();
        for (int i = threadIdx.x; i < n; i += kTileThreads) counts[(size_t)blockIdx.x * units + u0 + i] = tile_counts[i];
        __syncthreads();
    }
}

// counts[t][u] -> connections of stream u in the tiles before t; and of all tiles, and the chunks that the stream is given: its steps
// are at most one for every `members` connections and a partly filled one per column, and no more than its connections.
// 64 streams per workgroup, each wavefront a stretch of the tiles.
__global__ __launch_bounds__(kTileThreads) void stream_counts_kernel(unsigned* __restrict__ counts, int tiles, int units, int members,
                                                                     unsigned* __restrict__ of_stream, unsigned* __restrict__ chunks) {
    constexpr int kParts = kTileThreads / 64;
    __shared__ unsigned sums[kParts][64];
    const int lane = threadIdx.x & 63, part = threadIdx.x >> 6, u = blockIdx.x * 64 + lane;
    const int per = (tiles + kParts - 1) / kParts, from = min(part * per, tiles), to = min(from + per, tiles);
    unsigned sum = 0;
    if (u < units) {
#pragma unroll 8
        for (int t = from; t < to; ++t) sum += counts[(size_t)t * units + u];
    }
    sums[part][lane] = sum;
    __syncthreads();
    if (u >= units) return;
    unsigned run = 0, all = 0;
#pragma unroll
    for (int i = 0; i < kParts; ++i) {
        run += i < part ? sums[i][lane] : 0u;
        all += sums[i][lane];
    }
    for (int t0 = from; t0 < to; t0 += 8) {
        unsigned n[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) n[i] = counts[(size_t)min(t0 + i, to - 1) * units + u];
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (t0 + i < to) {
                counts[(size_t)(t0 + i) * units + u] = run;
                run += n[i];
            }
    }
    if (part == 0) {
        const unsigned entries = (unsigned)(kChunkSteps * members);
        of_stream[u] = all;
        chunks[u] = min((all + (unsigned)(kGroupColumns * (members - 1)) + entries - 1u) / entries, (all + kChunkSteps - 1u) / kChunkSteps);
    }
}

// A tile's connections by stream, in the order of the lookup inside a stream: tile_pos, and into the streams' lists (label inside the
// segment << 8 | column inside the group); place_of = where in the lists.  One workgroup per tile, whose wavefronts take consecutive
// stretches of it: they count their connections per stream, sums over streams and wavefronts turn the counts into places, and the
// stretches are gone through again, 64 connections at a time, each of which takes the place it finds and leaves the next one there (of
// several of one stream among the 64 the lanes' order decides, not the LDS's).  Places gather in LDS and leave by whole runs.
// As many wavefronts walk as the counters of 16 bits leave room for; the others help with the counters and the runs, which are all
// there is to do where a tile has fewer connections than there are streams.  A workgroup takes the tiles of a row of `before` in turn and moves
// the row on (one tile, unless the rows of single tiles would take too much memory).
constexpr size_t kTileCounterBytes = 61440;
__global__ __launch_bounds__(kTileThreads) void tile_sort_kernel(const int32_t* __restrict__ idx, int total, int tile_bits, int row_tiles, int units, const StreamOf stream_of,
                                                                 unsigned* __restrict__ before, const unsigned* __restrict__ begin,
                                                                 unsigned short* __restrict__ tile_pos, unsigned* __restrict__ place_of,
                                                                 unsigned* __restrict__ list, int window, int walkers) {
    extern __shared__ __align__(16) unsigned tile_lds[];
    __shared__ unsigned wave_sums[kTileThreads / 64];
    constexpr int kInflight = 8;
    constexpr int nthreads = kTileThreads;
    const int nwaves = walkers, lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const unsigned tile = 1u << tile_bits;
    unsigned short* const stage_pos = reinterpret_cast<unsigned short*>(tile_lds);                       // [tile]
    unsigned char* const stage_col = reinterpret_cast<unsigned char*>(tile_lds) + 2 * (size_t)tile;      // [tile]
    unsigned* const counters = tile_lds + 3 * (size_t)tile / 4;                                          // [wave][window / 2] two streams a word
    const int words = window / 2;
    unsigned* const mine = counters + (size_t)wave * words;
    before += (size_t)blockIdx.x * units;
    for (int t = 0; t < row_tiles; ++t) {
        const unsigned p0 = (blockIdx.x * (unsigned)row_tiles + t) << tile_bits;
        if (p0 >= (unsigned)total) break;
        const unsigned n = min(tile, (unsigned)total - p0), stretch = ((n + nwaves - 1) / nwaves + 63) & ~63u;
        const unsigned from = wave < nwaves ? min(wave * stretch, n) : n, to = min(from + stretch, n);
        unsigned placed = 0;                                                                                 // connections of the streams before the window
        for (int u0 = 0; u0 < units; u0 += window) {
            const unsigned streams = (unsigned)min(window, units - u0);
            for (int i = threadIdx.x; i < nwaves * words; i += nthreads) counters[i] = 0u;
            __syncthreads();
            auto walk = [&](auto visit) {
                if (from >= to) return;
                unsigned next[kInflight];
                auto fetch = [&](unsigned e0) {
#pragma unroll
                    for (int i = 0; i < kInflight; ++i) next[i] = (unsigned)idx[p0 + min(e0 + 64 * i + lane, n - 1)];
                };
                fetch(from);
                for (unsigned e0 = from; e0 < to; e0 += 64 * kInflight) {
                    unsigned id[kInflight], u[kInflight];
#pragma unroll
                    for (int i = 0; i < kInflight; ++i) {
                        const unsigned e = e0 + 64 * i + lane;
                        id[i] = next[i];
                        u[i] = stream_of(id[i], p0 + e) - (unsigned)u0;
                        if (e >= to || u[i] >= streams) u[i] = ~0u;
                    }
                    fetch(e0 + 64 * kInflight);
                    visit(id, u, e0 + lane);
                }
            };
            walk([&](const unsigned*, const unsigned* u, unsigned) {
#pragma unroll
                for (int i = 0; i < kInflight; ++i)
                    if (u[i] != ~0u) atomicAdd(&mine[u[i] >> 1], 1u << (16 * (u[i] & 1)));
            });
            __syncthreads();
            // each thread takes consecutive pairs of streams: their connections, those of the threads before it, and the places
            const int per = (words + nthreads - 1) / nthreads, w0 = min((int)threadIdx.x * per, words), w1 = min(w0 + per, words);
            unsigned sum = 0;
            for (int w = w0; w < w1; ++w)
                for (int v = 0; v < nwaves; ++v) {
                    const unsigned c = counters[(size_t)v * words + w];
                    sum += (c & 0xffffu) + (c >> 16);
                }
            unsigned upto = sum;
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                const unsigned below = __shfl_up(upto, off, 64);
                if (lane >= off) upto += below;
            }
            if (lane == 63) wave_sums[wave] = upto;
            __syncthreads();
            unsigned run = placed + upto - sum, all = 0;
#pragma unroll
            for (int v = 0; v < nthreads / 64; ++v) {
                run += v < wave ? wave_sums[v] : 0u;
                all += wave_sums[v];
            }
            for (int w = w0; w < w1; ++w) {
                unsigned even = run, odd = 0;
                for (int v = 0; v < nwaves; ++v) odd += counters[(size_t)v * words + w] & 0xffffu;
                odd += run;
                for (int v = 0; v < nwaves; ++v) {
                    const unsigned c = counters[(size_t)v * words + w];
                    counters[(size_t)v * words + w] = (even & 0xffffu) | odd << 16;
                    even += c & 0xffffu;
                    odd += c >> 16;
                }
                run = odd;
            }
            __syncthreads();
            walk([&](const unsigned* id, const unsigned* u, unsigned e) {
                unsigned found[kInflight], there[kInflight];
#pragma unroll
                for (int i = 0; i < kInflight; ++i) {
                    there[i] = found[i] = 0u;
                    if (u[i] != ~0u) {
                        there[i] = mine[u[i] >> 1];
                        found[i] = atomicAdd(&mine[u[i] >> 1], 1u << (16 * (u[i] & 1)));
                    }
                }
#pragma unroll
                for (int i = 0; i < kInflight; ++i) {
                    const unsigned shift = 16 * (u[i] & 1);
                    unsigned at = there[i] >> shift & 0xffffu;
                    for (unsigned long long left = __ballot(u[i] != ~0u && (found[i] >> shift & 0xffffu) != at); left != 0ull;) {
                        const unsigned k = (unsigned)__builtin_amdgcn_readlane((int)u[i], __builtin_ctzll(left));
                        const unsigned long long same = __ballot(u[i] == k);
                        if (u[i] == k) at += (unsigned)__popcll(same & ((1ull << lane) - 1ull));
                        left &= ~same;
                    }
                    if (u[i] != ~0u) {
                        stage_pos[at] = (unsigned short)(e + 64 * i);
                        stage_col[at] = (unsigned char)(id[i] % kGroupColumns);
                    }
                }
            });
            __syncthreads();
            // eight lanes to a run, or one, whose places are asked for four runs at a time; behind the walk the last wavefront's counter of a stream is
            // the end of its run
            const unsigned* const last = counters + (size_t)(nwaves - 1) * words;
            auto end_of = [&](unsigned u) { return last[u >> 1] >> (16 * (u & 1)) & 0xffffu; };
            auto leave = [&](auto lanes) {
                constexpr int kRuns = 4, kLanes = decltype(lanes)::value;
                for (unsigned u = threadIdx.x / kLanes; u < streams; u += kRuns * nthreads / kLanes) {
                    unsigned start[kRuns], end[kRuns], there[kRuns], first[kRuns];
#pragma unroll
                    for (int i = 0; i < kRuns; ++i) {
                        const unsigned v = u + i * (nthreads / kLanes);
                        start[i] = end[i] = there[i] = first[i] = 0u;
                        if (v < streams) {
                            start[i] = v > 0 ? end_of(v - 1) : placed;
                            end[i] = end_of(v);
                        }
                        if (start[i] != end[i]) {
                            there[i] = before[(unsigned)u0 + v];
                            first[i] = begin[(unsigned)u0 + v];
                        }
                    }
#pragma unroll
                    for (int i = 0; i < kRuns; ++i) {
                        if (start[i] == end[i]) continue;
                        const unsigned stream = (unsigned)u0 + u + i * (nthreads / kLanes), base = first[i] + there[i] - start[i];
                        const int label0 = (int)(stream / (unsigned)stream_of.groups) * stream_of.seg_labels;
                        for (unsigned q = start[i] + threadIdx.x % kLanes; q < end[i]; q += kLanes) {
                            const unsigned pos = stage_pos[q];
                            tile_pos[p0 + q] = (unsigned short)pos;
                            place_of[p0 + q] = base + q;
                            list[base + q] = (unsigned)((int)((p0 + pos) / (unsigned)stream_of.K) - label0) << 8 | stage_col[q];
                        }
                        if (row_tiles > 1 && threadIdx.x % kLanes == 0) before[stream] = there[i] + end[i] - start[i];
                    }
                }
            };
            // (short runs: a lane to each)
            if (n < (unsigned)units) leave(std::integral_constant<int, 1>{});
            else leave(std::integral_constant<int, 8>{});
            placed += all;
            __syncthreads();
        }
    }
}

// The steps of a stream, one wavefront per stream, 64 connections at a time in the order of the lookup: the connection of rank r
// among its column's is member r % MEMBERS of that column's step r / MEMBERS, and steps are numbered as their first members come.
// Writes the stream's entries, and for each connection of the list its slot.
// Bound by the latency of a turn (ballots for the ranks, a round trip to LDS for the number of a step), four turns' loads in flight.
constexpr int kStepWaves = 4, kStepRing = 32;            // (a turn opens at most 64 / MEMBERS steps of a column)
template <int MEMBERS>
__global__ __launch_bounds__(kStepWaves * 64) void stream_steps_kernel(const unsigned* __restrict__ list, const unsigned* __restrict__ begin,
                                                                       const unsigned* __restrict__ chunk_ptr, int units, unsigned* __restrict__ entries,
                                                                       unsigned* __restrict__ slot_at, unsigned* __restrict__ chunk_count) {
    constexpr int kEntries = kChunkSteps * MEMBERS, kAhead = 4;
    __shared__ unsigned opened[kStepWaves][kGroupColumns][kStepRing], counts[kStepWaves][kGroupColumns];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int u = blockIdx.x * kStepWaves + wave;
    if (u >= units) return;
    unsigned (*const open)[kStepRing] = opened[wave];
    unsigned* const count = counts[wave];
    if (lane < kGroupColumns) count[lane] = 0u;
    const unsigned from = begin[u], end = begin[u + 1];
    const size_t slot0 = (size_t)chunk_ptr[u] * kEntries;
    const unsigned long long below = (1ull << lane) - 1ull;
    auto slot_of = [&](unsigned step, unsigned m) { return slot0 + (size_t)(step / kChunkSteps) * kEntries + entry_in_chunk(MEMBERS, (int)(step % kChunkSteps), (int)m); };
    unsigned steps = 0;
    unsigned next[kAhead];
    auto fetch = [&](int i, unsigned at) { next[i] = list[min(at + lane, end - 1u)]; };
    if (from < end) {
#pragma unroll
        for (int i = 0; i < kAhead; ++i) fetch(i, from + 64 * i);
    }
    for (unsigned e0 = from; e0 < end; e0 += 64 * kAhead) {
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
            const unsigned e = e0 + 64 * i + lane, entry = next[i], col = entry % kGroupColumns;
            const bool on = e < end;
            fetch(i, e0 + 64 * (i + kAhead));
            unsigned long long same = __ballot(on);
#pragma unroll
            for (int bit = 0; bit < 5; ++bit) {
                const unsigned long long set = __ballot((col >> bit & 1u) != 0u);
                same &= (col >> bit & 1u) ? set : ~set;
            }
            const unsigned rank = count[col] + (unsigned)__popcll(same & below), m = rank % MEMBERS, place = rank / MEMBERS % kStepRing;
            const unsigned long long firsts = __ballot(on && m == 0u);
            if (on && m == 0u) open[col][place] = steps + (unsigned)__popcll(firsts & below);
            if (on && (same & ~below & ~(1ull << lane)) == 0ull) count[col] = rank + 1u;       // (the column's last of this turn)
            __builtin_amdgcn_wave_barrier();
            if (on) {
                const size_t slot = slot_of(open[col][place], m);
                entries[slot] = entry;
                slot_at[e] = (unsigned)slot;
            }
            steps += (unsigned)__popcll(firsts);
            __builtin_amdgcn_wave_barrier();
        }
    }
    // what is left of the columns' last steps, and of the last chunk
    if (lane < kGroupColumns && count[lane] % MEMBERS != 0u) {
        const unsigned step = open[lane][count[lane] / MEMBERS % kStepRing];
        for (unsigned m = count[lane] % MEMBERS; m < MEMBERS; ++m) entries[slot_of(step, m)] = kPadEntry | (unsigned)lane;
    }
    const unsigned chunks = (steps + kChunkSteps - 1u) / kChunkSteps, rest = chunks * kChunkSteps - steps;
    if ((unsigned)lane < rest)
        for (unsigned m = 0; m < MEMBERS; ++m) entries[slot_of(steps + (unsigned)lane, m)] = kPadEntry;
    if (lane == 0) chunk_count[u] = chunks;
}

// places in the streams' lists -> slots
__global__ __launch_bounds__(kBlock) void slots_of_places_kernel(const unsigned* __restrict__ slot_at, unsigned* __restrict__ slot_of, int total) {
    constexpr int kInflight = 4;
    const int i0 = blockIdx.x * (kBlock * kInflight) + threadIdx.x;
    unsigned v[kInflight];
#pragma unroll
    for (int i = 0; i < kInflight; ++i) v[i] = slot_of[min(i0 + i * kBlock, total - 1)];
#pragma unroll
    for (int i = 0; i < kInflight; ++i) v[i] = slot_at[v[i]];
#pragma unroll
    for (int i = 0; i < kInflight; ++i)
        if (i0 + i * kBlock < total) slot_of[i0 + i * kBlock] = v[i];
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
    p->chunk_ptr = nullptr; p->chunk_count = nullptr; p->entries = nullptr; p->slot_of = nullptr; p->tile_pos = nullptr; p->slots = 0; p->slice_off = nullptr; p->lab16 = nullptr; p->pos16 = nullptr; p->slot32 = nullptr; p->idx16 = nullptr; p->colperm = nullptr;
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

// Steps of four connections where a row of 64 samples is gathered by sixteen lanes, of eight where 32 samples are enough (the
// walking kernel takes 0.67 ms for 64 samples and 0.40 for 32 at 65,536 columns x 670,091 labels x 72).  Segments: as many as make the
// walk shortest, in steps of a wavefront -- its share of the connections, half a step per column that the last connections do not
// fill, and some forty for its beginning and end -- times the rounds that the CUs, eight wavefronts each, need for all streams and
// slices.  128 samples and more, 1,300 to 2,500 columns want a segment on every CU; 2 samples, 22,133 columns, 200,058 labels, fan-in 8
// two of them (walk 31 us; 40 with eight, whose three rounds are a little less of the connections).
// Labels and rows of a segment stay within the entries and 32-bit offsets.
// Counts per tile and stream: at most kMostCounts of them, 1 GB, and rows of several tiles where that is not enough.
constexpr long long kMostCounts = 1ll << 28;
GlobalShape global_shape(int N, int K, int L, int batch) {
    GlobalShape f{};
    f.members = batch > 0 && batch <= 32 ? 8 : 4;
    f.groups = (N + kGroupColumns - 1) / kGroupColumns;
    const double total = (double)L * K, waves = 8.0 * device_cu_count();
    const int slices = batch > 0 ? (batch + 256 / f.members - 1) / (256 / f.members) : 1, least = (int)(((long long)L + 15999999) / 16000000);
    double best = 0.0;
    f.segments = least;
    for (int s = least; s == least || (s <= 2048 && s <= L && (double)s * f.groups <= 4.0 * waves); ++s) {
        const double units = (double)s * f.groups, launches = std::ceil((double)slices / walk_slices((long long)units, slices));
        const double steps = launches * std::max(1.0, std::ceil(units / waves)) * (total / units / f.members + kGroupColumns / 2 + 40.0);
        if (s == least || steps < 0.98 * best) { best = steps; f.segments = s; }
    }
    f.seg_labels = (L + f.segments - 1) / f.segments;
    f.segments = (L + f.seg_labels - 1) / f.seg_labels;
    f.tile_bits = 10;
    while (f.tile_bits < 15 && total / (2 << f.tile_bits) >= 2.0 * device_cu_count()) ++f.tile_bits;
    // (many streams: their counts, four bytes for every tile and stream, are written once and read three times)
    while (f.tile_bits < 15 && total / (2 << f.tile_bits) >= device_cu_count() && total / (1 << f.tile_bits) * f.segments * f.groups > (double)(1 << 26)) ++f.tile_bits;
    f.row_bits = f.tile_bits;
    while (std::ceil(total / std::ldexp(1.0, f.row_bits)) * f.segments * f.groups > (double)kMostCounts && f.row_bits < 31) ++f.row_bits;
    const double streams = std::min((double)f.segments * f.groups, total);
    const int entries = kChunkSteps * f.members;
    f.max_slots = ((size_t)((total + streams * (kGroupColumns * (f.members - 1) + entries - 1)) / entries) + 1) * entries;
    return f;
}

// counts per row of tiles and stream, per stream, and the two sums over the streams
size_t global_build_words(const GlobalShape& f, long long total) { return ((size_t)((total + (1ll << f.row_bits) - 1) >> f.row_bits) + 3) * f.segments * f.groups + 1; }

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
    // (the walking kernel hands its sums from the tile's thread to the column's own thread, or to its next, through LDS)
    // Measured (input gradient, weights-in-LDS form, sorted against thread t <-> column t): 768 columns x fan-in 32, batch 128:
    // 1.517 -> 1.150 slot rows per connection, 251 -> 239 us; batch 64: 151 -> 141; fan-in 16: 178 -> 170; fan-in 64 (300,000
    // labels): 207 -> 190; 512 columns: 261 -> 251; 640 columns, batch 256: 226 -> 215; no gain at 256 columns and fewer (few
    // slices to sort into, several workgroups per CU), and a loss where a workgroup walks a single tile (131,072 labels, batch
    // 32: 35.4 -> 36.5 us): there the order of the columns stays.
    const bool sorted_columns = plan_sorts_columns(threads, TL, p->K, w_in_lds, tiles, p->batch_hint);
    p->colperm = nullptr;
    unsigned *slice_len = nullptr, *counts = nullptr;
    if (!dev_alloc(p, &p->slice_off, nslices + 1)) return FFI_ERR_OUT_OF_MEMORY;
    FFI_TRY(workspace_get(s, kWsPartials, ((size_t)tiles * threads + nslices) * sizeof(unsigned), (void**)&counts));       // (which the passes ask for too)
    slice_len = counts + (size_t)tiles * threads;
    // rows per bank half: half the tile plus some room for the balancing, within the LDS the walking kernel can have
    const int cap = tiled_rows_per_half(TL);
    if (!dev_alloc(p, &p->rowpos, (size_t)p->L)) return FFI_ERR_OUT_OF_MEMORY;
    {
        const size_t lds = ((size_t)threads + 1) * sizeof(int) + (size_t)TL * ((p->K + 2) / 3) * sizeof(unsigned) + (size_t)threads + 1 + (size_t)TL + kPastLabels;
        const auto color = p->K <= 32 ? tile_color_kernel<32, 1, false> : p->K <= 64 ? tile_color_kernel<32, 2, false>
                                    : p->K <= 128 ? tile_color_kernel<64, 2, false> : tile_color_kernel<64, 2, true>;
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
    FFI_HIP_TRY(hipGetLastError());
    p->tiled = true;
    p->w_in_lds = w_in_lds;
    p->tile_labels = TL; p->threads = threads; p->slices = slices; p->tiles = tiles; p->zero_row = 2 * cap;
    p->total_rows = (long long)rows;
    p->bytes += (size_t)rows * 64 * 2 * sizeof(unsigned short) + (nslices + 1) * sizeof(unsigned) + (size_t)p->L * sizeof(unsigned short) +
                (p->colperm ? (size_t)tiles * threads * sizeof(unsigned short) : 0);
    return FFI_OK;
}

// The build's temporaries lie in the workspaces that the backward pass will ask for: nothing is allocated and freed again, and the
// host does not wait.
int build_global(ffi_plan* p, const int32_t* lookup, hipStream_t s) {
    const int total = p->L * p->K;  // validated to fit int32 by the caller
    const GlobalShape f = global_shape(p->N, p->K, p->L, p->batch_hint);
    const long long units = (long long)f.segments * f.groups;
    if (units >= (1ll << 31) - 64 || f.max_slots >= (1ull << 32)) return FFI_ERR_TOO_LARGE;
    // (two buffers: an allocation is 50 us and more; each array on a line of its own)
    const size_t places = ((size_t)total + 63) / 64 * 64;
    if (!dev_alloc(p, &p->entries, f.max_slots + 2 * (size_t)units + 1) || !dev_alloc(p, &p->slot_of, places + (places + 1) / 2)) return FFI_ERR_OUT_OF_MEMORY;
    p->chunk_ptr = p->entries + f.max_slots;
    p->chunk_count = p->chunk_ptr + units + 1;
    p->tile_pos = reinterpret_cast<unsigned short*>(p->slot_of + places);
    const int rows = (int)(((long long)total + (1ll << f.row_bits) - 1) >> f.row_bits);
    unsigned *list = nullptr, *slot_at = nullptr, *counts = nullptr;
    FFI_TRY(workspace_get(s, kWsSlots, f.max_slots * sizeof(unsigned), (void**)&list));
    FFI_TRY(workspace_get(s, kWsWeightParts, f.max_slots * sizeof(unsigned), (void**)&slot_at));
    FFI_TRY(workspace_get(s, kWsPartials, global_build_words(f, total) * sizeof(unsigned), (void**)&counts));
    unsigned* const of_stream = counts + (size_t)rows * units;
    unsigned *const begin = of_stream + units, *const chunks = begin + units + 1;
    const StreamOf stream_of{p->K, f.seg_labels, f.segments, f.groups};
    unsigned long long* total_out = nullptr;
    FFI_HIP_TRY(hipHostGetDevicePointer((void**)&total_out, p->h_scratch, 0));
    const size_t count_lds = (size_t)std::min<long long>(units, kCountWindow) * sizeof(unsigned);
    hipLaunchKernelGGL(tile_streams_kernel, dim3((unsigned)rows), dim3(kTileThreads), count_lds, s, lookup, total, f.row_bits, (int)units, stream_of, counts);
    hipLaunchKernelGGL(stream_counts_kernel, dim3((unsigned)((units + 63) / 64)), dim3(kTileThreads), 0, s, counts, rows, (int)units, f.members,
                       of_stream, chunks);
    hipLaunchKernelGGL(slice_scan_kernel, dim3(1), dim3(1024), 0, s, of_stream, begin, (int)units, 0, total_out);
    hipLaunchKernelGGL(slice_scan_kernel, dim3(1), dim3(1024), 0, s, chunks, p->chunk_ptr, (int)units, 0, total_out);
    const int window = (int)std::min<long long>((units + 1) / 2 * 2, (long long)kTileCounterBytes / 2);
    const int waves = (int)std::max<size_t>(1, std::min<size_t>(kTileThreads / 64, kTileCounterBytes / (2 * (size_t)window)));
    const size_t sort_lds = ((size_t)3 << f.tile_bits) + (size_t)waves * window * 2;
    FFI_HIP_TRY(hipFuncSetAttribute((const void*)tile_sort_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)sort_lds));
    hipLaunchKernelGGL(tile_sort_kernel, dim3((unsigned)rows), dim3(kTileThreads), sort_lds, s, lookup, total, f.tile_bits, 1 << (f.row_bits - f.tile_bits), (int)units, stream_of,
                       counts, begin, p->tile_pos, p->slot_of, list, window, waves);
    const auto stream_steps = f.members == 4 ? stream_steps_kernel<4> : stream_steps_kernel<8>;
    hipLaunchKernelGGL(stream_steps, dim3((unsigned)((units + kStepWaves - 1) / kStepWaves)), dim3(kStepWaves * 64), 0, s, list, begin, p->chunk_ptr,
                       (int)units, p->entries, slot_at, p->chunk_count);
    hipLaunchKernelGGL(slots_of_places_kernel, dim3((unsigned)((total + 4 * kBlock - 1ll) / (4 * kBlock))), dim3(kBlock), 0, s, slot_at, p->slot_of, total);
    FFI_HIP_TRY(hipGetLastError());
    p->members = f.members;
    p->groups = f.groups;
    p->segments = f.segments;
    p->seg_labels = f.seg_labels;
    p->tile_bits = f.tile_bits;
    p->slots = (long long)f.max_slots;
    p->bytes += (f.max_slots + 2 * (size_t)units + 1 + places + places / 2) * sizeof(unsigned);
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
                    hipEventCreateWithFlags(&p->built, hipEventDisableTiming) == hipSuccess &&
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
    // checks enqueued before this build (all finished: a build that takes the place of another waits for the device) are of no interest any more
    p->guard_seen = p->guard_seq;
    p->guard_stale = false;
    p->edited_by_library = false;
    p->ids_only = false;
    return FFI_OK;
}

// Takes the place of a build for passes that read the lookup itself: finds every id in range, waiting for `s`, and lays nothing
// out.  What an earlier build laid out is of no content that counts any more; it goes when the next build replaces it.
int plan_check_ids(ffi_plan* p, const int32_t* lookup, hipStream_t s) {
    unsigned long long fp = 0, bad = 0;
    p->ids_only = true;
    free_spares(p);                            // (those of a plan that made room for this one)
    FFI_TRY(plan_fingerprint(p, lookup, s, &fp, &bad));
    if (bad != 0) return FFI_ERR_BAD_LOOKUP;
    p->lookup = lookup;
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
        // no check of this plan is in flight
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
    // (where the build fails: the helper's arrays go)
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
    // Whoever uses the plan waits for this on the device (plan_wait_built); what follows on `s` does so by itself.  The host goes on: a
    // rewiring and the pass behind it at 128 x 768 x 670,091 x 32 took 1,121 us with the host waiting here and freeing two
    // temporaries, 1,093 so; at 119 x 32,219 x 117,739 x 8 356 and 330.
    auto finish = [&]() -> int {
        if (helper_busy) {
            FFI_HIP_TRY(hipEventRecord(p->helper_event, p->helper_stream));
            FFI_HIP_TRY(hipStreamWaitEvent(s, p->helper_event, 0));
        }
        FFI_HIP_TRY(hipEventRecord(p->built, s));
        p->built_pending = true;
        return FFI_OK;
    };
    {
        const int st = finish();
        if (st != FFI_OK) { (void)hipStreamSynchronize(s); (void)join(); free_arrays(p); return st; }
    }
    free_spares(p);                            // what this build did not reuse
    return FFI_OK;
}
}  // namespace

namespace {
// The calls below may be made while this thread or another one captures a stream: none of them has to do with a capture.
class UncapturedCalls {
public:
    UncapturedCalls() { known_ = hipThreadExchangeStreamCaptureMode(&mode_) == hipSuccess; }
    ~UncapturedCalls() { if (known_) (void)hipThreadExchangeStreamCaptureMode(&mode_); }
private:
    hipStreamCaptureMode mode_ = hipStreamCaptureModeRelaxed;
    bool known_;
};
}  // namespace

int plan_wait_built(const ffi_plan* p, hipStream_t s) {
    if (!p->built_pending.load(std::memory_order_acquire)) return FFI_OK;
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    FFI_HIP_TRY(hipStreamIsCapturing(s, &capture));
    // (a graph cannot wait for an event of before its capture, and may be replayed at once and on any stream: there the host waits)
    const bool captured = capture != hipStreamCaptureStatusNone;
    hipError_t e;
    {
        const UncapturedCalls calls;
        e = captured ? hipEventSynchronize(p->built) : hipEventQuery(p->built);
    }
    if (e == hipSuccess) {
        p->built_pending.store(false, std::memory_order_release);
        return FFI_OK;
    }
    if (captured || e != hipErrorNotReady) return hip_fail(e);
    (void)hipGetLastError();
    FFI_HIP_TRY(hipStreamWaitEvent(s, p->built, 0));
    return FFI_OK;
}

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
    if (p->built) (void)hipEventDestroy(p->built);
    if (p->d_guard) (void)hipFree(p->d_guard);
    if (p->h_guard) (void)hipHostFree(p->h_guard);
    p->d_scratch = nullptr; p->h_scratch = nullptr; p->fp_done = nullptr; p->built = nullptr;
    p->d_guard = nullptr; p->h_guard = nullptr; p->guard_seq = 0; p->guard_seen = 0; p->guard_stale = false;
}

}  // namespace ffi
