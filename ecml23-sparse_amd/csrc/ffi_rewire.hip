// Rewiring support (sparse/layer.py:60-86, sparse/custom_layer.py:20-43): pick the connections whose
// magnitude is below a threshold, give them new random sources, clear optimizer state there.
//
//   threshold selection  the k-th smallest |w| (FixedFractionSelector: tf.nn.top_k(-|w|, k), last value) by a
//                        three-pass radix select over the 31-bit patterns of |w| (11 + 11 + 9 bits): each pass
//                        histograms one digit of the values that match the digits found so far, and its last
//                        workgroup picks the bin that holds the k-th value (select_pass_kernel).  Integer atomics only:
//                        the result does not depend on their order.
//   rewire_kernel        every position p with |w[p]| < threshold: lookup[p] = a source drawn uniformly from
//                        [0, num_features) by a counter-based generator keyed on (seed, p); arrays[i][p] = 0.
#include "ffi_internal.h"
#include "ffi_scan.h"

#include <algorithm>

namespace ffi {
namespace {

constexpr int kSelThreads = 1024;
constexpr int kSelBins = 2048;

// Read-modify-writes of one address take turns, some 10 ns each where their results are waited for: 512 workgroups that draw from
// one counter are 5 us.  So they draw from one of eight, each on a line of its own, and who draws last there draws from the last.
// Zero between launches.
constexpr int kDrawWays = 8;
struct Draw {
    struct __attribute__((aligned(64))) Way { unsigned long long n; } way[kDrawWays + 1];
};
// Adds `v`, below 2^40, of a workgroup (of the `parts` that call this, one thread each) to the others'; true in the one that comes last,
// which has the sum, and all that the others' had waited for before is done then.
__device__ __forceinline__ bool draw_last(Draw* d, unsigned parts, unsigned long long v, unsigned long long* sum) {
    constexpr unsigned long long one = 1ull << 40;
    const unsigned way = blockIdx.x % kDrawWays, of_way = (parts - way + kDrawWays - 1) / kDrawWays;
    unsigned long long all = __hip_atomic_fetch_add(&d->way[way].n, v + one, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + v + one;
    if (all >> 40 != of_way) return false;
    __hip_atomic_store(&d->way[way].n, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    v = all & (one - 1ull);
    all = __hip_atomic_fetch_add(&d->way[kDrawWays].n, v + one, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + v + one;
    if (all >> 40 != min(parts, (unsigned)kDrawWays)) return false;
    __hip_atomic_store(&d->way[kDrawWays].n, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *sum = all & (one - 1ull);
    return true;
}

// `prefix` and `k` are what each pass leaves for the next.
struct SelectState {
    Draw draw;
    unsigned prefix;              // digits found so far (the high bits of the answer)
    unsigned long long k;         // rank still to find among the values matching the prefix (1-based)
};

__device__ __forceinline__ unsigned magnitude_bits(float v) { return __float_as_uint(v) & 0x7fffffffu; }

// Workgroup-local bins are hist[bin] += number of values whose bits above (shift + nbits) equal the prefix and whose digit is bin.
// Weights have few exponents, so in the first pass a wavefront's lanes meet in some twenty bins: its lanes count in four copies of
// the histogram, side by side in the banks, and the workgroups add to kHistTotals totals.  (21 M normal values: 58 us in one
// copy, 31 in four or eight that all go to one total, 25 so; the second pass, which few values match, 18, what it takes to
// read them.)
// The second pass also lists the values that match the first digit, a workgroup's in a piece of its own, and the third reads the lists
// instead of all values where they all fitted, which takes values that crowd within an eighth of an octave to fail.  The workgroup
// that adds its bins last picks the bin in which the cumulative count reaches k, appends it to the prefix, reduces k by the count of the bins
// below it and clears the bins: all read-modify-writes at device scope whose results are waited for before the ticket is drawn.
// (A launch for each pick and one to clear, and all values read in the third pass: 81 us in seven launches, 56 so in three; 3.5 M 29 and 32, in four launches fewer.)
constexpr int kHistThreads = 1024, kHistCopies = 4, kHistTotals = 8, kSelLocalList = 2048, kListParts = 32;
// lists: [n_lists] counts, then n_lists pieces of kSelLocalList values (n_lists: workgroups of the second pass, at most kHistThreads)
template <int PASS>
__global__ __launch_bounds__(kHistThreads) void select_pass_kernel(const float* __restrict__ w, size_t count, unsigned long long k0,
                                                                    SelectState* __restrict__ state, unsigned* __restrict__ hist,
                                                                    unsigned* __restrict__ lists, int n_lists, float* __restrict__ threshold) {
    constexpr int kShift = PASS == 0 ? 20 : PASS == 1 ? 9 : 0, kBits = PASS == 2 ? 9 : 11, kEach = kSelBins / kHistThreads;
    constexpr unsigned kMask = (1u << kBits) - 1u;
    __shared__ __align__(16) unsigned local[kSelBins * kHistCopies];
    __shared__ unsigned mine[PASS == 1 ? kSelLocalList : 1], n_mine, is_last;
    const unsigned prefix = PASS == 0 ? 0u : state->prefix, copy = threadIdx.x % kHistCopies;
    bool from_lists = false;
    if (PASS == 2) from_lists = !__syncthreads_or((int)threadIdx.x < n_lists && lists[threadIdx.x] > (unsigned)kSelLocalList);
    // (lists have work for few workgroups: the others leave, and no ticket is expected of them)
    const unsigned parts = from_lists ? min(gridDim.x, (unsigned)kListParts) : gridDim.x;
    if (blockIdx.x >= parts) return;
    for (int i = threadIdx.x; i < kSelBins * kHistCopies; i += kHistThreads) local[i] = 0;
    if (threadIdx.x == 0) n_mine = 0u;
    __syncthreads();
    auto add = [&](unsigned key) { atomicAdd(&local[((key >> kShift) & kMask) * kHistCopies + copy], 1u); };
    if (from_lists) {
        const int lane = threadIdx.x & 63;
        for (int q = blockIdx.x + (int)parts * (threadIdx.x >> 6); q < n_lists; q += (int)parts * (kHistThreads / 64)) {
            const unsigned n = lists[q];
            const unsigned* from = lists + n_lists + (size_t)q * kSelLocalList;
            for (unsigned i = lane; i < n; i += 64)
                if (from[i] >> kBits == prefix) add(from[i]);
        }
    } else {
        constexpr int kTogether = 4;                                      // values asked for together
        constexpr unsigned kNone = ~0u;                                   // (no magnitude)
        const size_t stride = (size_t)gridDim.x * kHistThreads;
        for (size_t i0 = (size_t)blockIdx.x * kHistThreads + threadIdx.x; i0 < count; i0 += kTogether * stride) {
            unsigned keys[kTogether];
#pragma unroll
            for (int u = 0; u < kTogether; ++u) {
                const size_t i = i0 + u * stride;
                const unsigned key = magnitude_bits(w[min(i, count - 1)]);
                keys[u] = i < count ? key : kNone;
            }
#pragma unroll
            for (int u = 0; u < kTogether; ++u) {
                const unsigned key = keys[u];
                const bool match = key != kNone && (PASS == 0 || (key >> (kShift + kBits)) == prefix);
                if (match) add(key);
                if (PASS == 1) {
                    const unsigned long long matches = __ballot(match);
                    if (matches != 0ull) {                                // (one add of a wavefront)
                        const int lane = threadIdx.x & 63, first = __ffsll((long long)matches) - 1;
                        unsigned at = 0;
                        if (lane == first) at = atomicAdd(&n_mine, (unsigned)__popcll(matches));
                        at = (unsigned)__builtin_amdgcn_readlane((int)at, first) + (unsigned)__popcll(matches & ((1ull << lane) - 1ull));
                        if (match && at < (unsigned)kSelLocalList) mine[at] = key;
                    }
                }
            }
        }
    }
    __syncthreads();
    if (PASS == 1) {
        if (threadIdx.x == 0) lists[blockIdx.x] = n_mine;
        unsigned* const to = lists + n_lists + (size_t)blockIdx.x * kSelLocalList;
        for (unsigned i = threadIdx.x; i < min(n_mine, (unsigned)kSelLocalList); i += kHistThreads) to[i] = mine[i];
    }
    unsigned old = 0;
    for (int i = threadIdx.x; i < kSelBins; i += kHistThreads) {
        unsigned c = 0;
#pragma unroll
        for (int q = 0; q < kHistCopies; q += 4) {
            const uint4 v = *reinterpret_cast<const uint4*>(local + i * kHistCopies + q);
            c += (v.x + v.y) + (v.z + v.w);
        }
        if (c) old |= __hip_atomic_fetch_add(&hist[(blockIdx.x % kHistTotals) * kSelBins + i], c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    asm volatile("" :: "v"(old));                                         // (the adds have returned)
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long none;
        is_last = draw_last(&state->draw, parts, 0ull, &none);
    }
    __syncthreads();
    if (!is_last) return;
    // (walked by one thread, 2,048 bins took 22 us, all of it latency)
    const int first = threadIdx.x * kEach;
    unsigned bins[kEach][kHistTotals], bin_count[kEach];
    unsigned long long sum = 0, total = 0;
#pragma unroll
    for (int i = 0; i < kEach; ++i)
#pragma unroll
        for (int t = 0; t < kHistTotals; ++t)
            bins[i][t] = __hip_atomic_exchange(&hist[t * kSelBins + first + i], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
    for (int i = 0; i < kEach; ++i) {
        bin_count[i] = 0u;                                                // (behind the last bin: nothing was added)
#pragma unroll
        for (int t = 0; t < kHistTotals; ++t) bin_count[i] += bins[i][t];
        sum += bin_count[i];
    }
    const unsigned long long k = PASS == 0 ? k0 : state->k;
    unsigned long long below = block_sum_below<kHistThreads>(sum, &total);       // (its barrier: state is read before it is written)
    int pick = -1;
    if (below < k && below + sum >= k) {
        pick = first;
#pragma unroll
        for (int i = 0; i + 1 < kEach; ++i)
            if (pick == first + i && below + bin_count[i] < k) { below += bin_count[i]; ++pick; }
    } else if (total < k && threadIdx.x == 0) {
        pick = (1 << kBits) - 1;
        below = total;
    }
    if (pick >= 0) {
        const unsigned value = (prefix << kBits) | (unsigned)pick;
        state->prefix = value;
        state->k = k - below;
        if (PASS == 2) *threshold = __uint_as_float(value);
    }
}

__global__ void select_none_kernel(float* threshold) { *threshold = 0.f; }    // nothing is below 0 in magnitude: an empty selection

// splitmix64 finaliser over (seed, position): a counter-based generator, so the draw of a position does not
// depend on how the launch is shaped
__device__ __forceinline__ unsigned long long mix64(unsigned long long z) {
    z += 0x9e3779b97f4a7c15ull;
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    return z ^ (z >> 31);
}

struct ArrayList {
    float* p[4];
};

__global__ __launch_bounds__(kSelThreads) void rewire_kernel(int32_t* __restrict__ lookup, const float* __restrict__ w,
                                                              ArrayList arrays, int n_arrays, size_t count,
                                                              unsigned num_features, const float* __restrict__ threshold,
                                                              unsigned long long seed, Draw* __restrict__ counted,
                                                              long long* __restrict__ rewired) {
    __shared__ unsigned red[kSelThreads / 64];
    const float thr = *threshold;
    unsigned changed = 0;
    for (size_t i = (size_t)blockIdx.x * kSelThreads + threadIdx.x; i < count; i += (size_t)gridDim.x * kSelThreads) {
        if (fabsf(w[i]) < thr) {
            const unsigned long long r = mix64(seed ^ mix64((unsigned long long)i));
            lookup[i] = (int32_t)__umul64hi(r, (unsigned long long)num_features);     // uniform in [0, num_features)
            for (int a = 0; a < n_arrays; ++a) arrays.p[a][i] = 0.f;
            ++changed;
        }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) changed += __shfl_xor(changed, off, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = changed;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long t = 0;
        for (int i = 0; i < kSelThreads / 64; ++i) t += red[i];
        unsigned long long all;
        if (draw_last(counted, gridDim.x, t, &all) && rewired != nullptr) *rewired = (long long)all;
    }
}

constexpr size_t kSelectHead = 1024, kSelectBytes = kSelectHead + kSelBins * kHistTotals * sizeof(unsigned);     // the state, then the bins
static_assert(sizeof(SelectState) <= kSelectHead, "the bins lie behind it");

int stream_blocks(size_t count) {
    return (int)std::max<size_t>(1, std::min<size_t>((count + kSelThreads - 1) / kSelThreads, (size_t)device_cu_count() * 2));
}

}  // namespace

int launch_select_threshold(const float* w, size_t count, unsigned long long k, float* threshold, hipStream_t s) {
    if (k == 0) {
        hipLaunchKernelGGL(select_none_kernel, dim3(1), dim3(1), 0, s, threshold);
        FFI_HIP_TRY(hipGetLastError());
        return FFI_OK;
    }
    unsigned char* ws = nullptr;
    FFI_TRY(zeroed_get(s, kWsSelect, kSelectBytes, (void**)&ws));
    SelectState* state = reinterpret_cast<SelectState*>(ws);
    unsigned* hist = reinterpret_cast<unsigned*>(ws + kSelectHead);
    const unsigned blocks = (unsigned)std::max<size_t>(1, std::min<size_t>({(count + kHistThreads - 1) / kHistThreads, (size_t)device_cu_count() * 2, (size_t)kHistThreads}));
    unsigned* lists = nullptr;
    FFI_TRY(workspace_get(s, kWsRewire, (size_t)blocks * (1 + kSelLocalList) * sizeof(unsigned), (void**)&lists));
    for (const auto pass : {select_pass_kernel<0>, select_pass_kernel<1>, select_pass_kernel<2>})
        hipLaunchKernelGGL(pass, dim3(blocks), dim3(kHistThreads), 0, s, w, count, k, state, hist, lists, (int)blocks, threshold);
    FFI_HIP_TRY(hipGetLastError());
    return FFI_OK;
}

int launch_rewire(int32_t* lookup, const float* w, float* const* arrays, int n_arrays, size_t count, unsigned num_features,
                  const float* threshold, unsigned long long seed, long long* rewired, hipStream_t s) {
    ArrayList list{};
    for (int i = 0; i < n_arrays; ++i) list.p[i] = arrays[i];
    unsigned char* ws = nullptr;
    FFI_TRY(zeroed_get(s, kWsSelect, kSelectBytes, (void**)&ws));
    hipLaunchKernelGGL(rewire_kernel, dim3(stream_blocks(count)), dim3(kSelThreads), 0, s, lookup, w, list, n_arrays, count, num_features, threshold,
                       seed, &reinterpret_cast<SelectState*>(ws)->draw, rewired);
    FFI_HIP_TRY(hipGetLastError());
    return FFI_OK;
}

}  // namespace ffi
