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

// Zero between selections but for `prefix` and `k`, which each pass leaves for the next.
struct SelectState {
    unsigned prefix;              // digits found so far (the high bits of the answer)
    unsigned ticket;
    unsigned long long k;         // rank still to find among the values matching the prefix (1-based)
    unsigned long long listed;    // values that match the first digit: those in the list, or more than it holds
    unsigned long long rewired;   // rewire_kernel: connections changed, and the workgroups that have said so << 40
};

__device__ __forceinline__ unsigned magnitude_bits(float v) { return __float_as_uint(v) & 0x7fffffffu; }

// Workgroup-local bins are hist[bin] += number of values whose bits above (shift + nbits) equal the prefix and whose digit is bin.
// Weights have few exponents, so in the first pass a wavefront's lanes meet in some twenty bins: its lanes count in four copies of
// the histogram, side by side in the banks, and the workgroups add to kHistTotals totals.  (21 M normal values: 58 us in one
// copy, 31 in four or eight that all go to one total, 25 so; the second pass, which few values match, 18, what it takes to
// read them.)
// The second pass also puts the values that match the first digit in a list, and the third reads the list instead of all values
// where they fitted into it, which takes values that crowd within an eighth of an octave to fail.  The workgroup that adds its
// bins last picks the bin in which the cumulative count reaches k, appends it to the prefix, reduces k by the count of the bins
// below it and clears the bins: all read-modify-writes at device scope whose results are waited for before the ticket is drawn.
// (A launch for each pick and one to clear, and all values read in the third pass: 81 us in seven launches, 62 so in three; 12,291 x 7: 187 us of a rewiring and its pass against 206.)
constexpr int kHistThreads = 1024, kHistCopies = 4, kHistTotals = 8, kSelLocalList = 2048;
template <int PASS>
__global__ __launch_bounds__(kHistThreads) void select_pass_kernel(const float* __restrict__ w, size_t count, unsigned long long k0,
                                                                    SelectState* __restrict__ state, unsigned* __restrict__ hist,
                                                                    unsigned* __restrict__ list, unsigned long long capacity, float* __restrict__ threshold) {
    constexpr int kShift = PASS == 0 ? 20 : PASS == 1 ? 9 : 0, kBits = PASS == 2 ? 9 : 11, kEach = kSelBins / kHistThreads;
    constexpr unsigned kMask = (1u << kBits) - 1u;
    __shared__ __align__(16) unsigned local[kSelBins * kHistCopies];
    __shared__ unsigned mine[PASS == 1 ? kSelLocalList : 1], n_mine, is_last;
    __shared__ unsigned long long list_at;
    const unsigned prefix = PASS == 0 ? 0u : state->prefix, copy = threadIdx.x % kHistCopies;
    const bool from_list = PASS == 2 && state->listed <= capacity;
    const size_t n = from_list ? (size_t)state->listed : count;
    // (a list has work for few workgroups: the others leave, and no ticket is expected of them)
    const unsigned parts = from_list ? (unsigned)min((size_t)gridDim.x, max((n + kHistThreads - 1) / kHistThreads, (size_t)1)) : gridDim.x;
    if (blockIdx.x >= parts) return;
    for (int i = threadIdx.x; i < kSelBins * kHistCopies; i += kHistThreads) local[i] = 0;
    if (threadIdx.x == 0) n_mine = 0u;
    __syncthreads();
    constexpr int kTogether = 4;                                          // values asked for together
    constexpr unsigned kNone = ~0u;                                       // (no magnitude)
    const size_t stride = (size_t)parts * kHistThreads;
    for (size_t i0 = (size_t)blockIdx.x * kHistThreads + threadIdx.x; i0 < n; i0 += kTogether * stride) {
        unsigned keys[kTogether];
#pragma unroll
        for (int u = 0; u < kTogether; ++u) {
            const size_t i = min(i0 + u * stride, n - 1);
            const unsigned key = from_list ? list[i] : magnitude_bits(w[i]);
            keys[u] = i0 + u * stride < n ? key : kNone;
        }
#pragma unroll
        for (int u = 0; u < kTogether; ++u) {
            const unsigned key = keys[u];
            const bool match = key != kNone && (PASS == 0 || (key >> (kShift + kBits)) == prefix);
            if (match) atomicAdd(&local[((key >> kShift) & kMask) * kHistCopies + copy], 1u);
            if (PASS == 1) {
                const unsigned long long matches = __ballot(match);
                if (matches != 0ull) {                                        // (one add of a wavefront)
                    const int lane = threadIdx.x & 63, first = __ffsll((long long)matches) - 1;
                    unsigned at = 0;
                    if (lane == first) at = atomicAdd(&n_mine, (unsigned)__popcll(matches));
                    at = (unsigned)__builtin_amdgcn_readlane((int)at, first) + (unsigned)__popcll(matches & ((1ull << lane) - 1ull));
                    if (match && at < (unsigned)kSelLocalList) mine[at] = key;
                }
            }
        }
    }
    __syncthreads();
    if (PASS == 1) {
        if (threadIdx.x == 0)
            list_at = n_mine ? __hip_atomic_fetch_add(&state->listed, n_mine > (unsigned)kSelLocalList ? capacity + 1ull : (unsigned long long)n_mine, __ATOMIC_RELAXED,
                                                      __HIP_MEMORY_SCOPE_AGENT) : 0ull;
        __syncthreads();
        for (unsigned i = threadIdx.x; i < min(n_mine, (unsigned)kSelLocalList); i += kHistThreads)
            if (list_at + i < capacity) list[list_at + i] = mine[i];
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
    if (threadIdx.x == 0) is_last = __hip_atomic_fetch_add(&state->ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == parts - 1u;
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
    if (threadIdx.x == 0) {
        state->ticket = 0u;
        if (PASS == 2) state->listed = 0ull;
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
                                                              unsigned long long seed, unsigned long long* __restrict__ counted,
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
        // (fewer than 2^40 connections and 2^24 workgroups; who adds last has the sum.  Adds to one address take turns: of 2,048
        // workgroups of 256 threads they were 12 us of the kernel's 49, so it has 512 of 1,024.)
        const unsigned long long one = 1ull << 40, all = __hip_atomic_fetch_add(counted, t + one, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + t + one;
        if (all >> 40 == gridDim.x) {
            if (rewired != nullptr) *rewired = (long long)(all & (one - 1ull));
            __hip_atomic_store(counted, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
}

constexpr size_t kSelectBytes = 256 + kSelBins * kHistTotals * sizeof(unsigned);     // the state, then the bins
static_assert(sizeof(SelectState) <= 256, "the bins lie behind it");

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
    const size_t capacity = std::max<size_t>(count / 32, 1024);
    unsigned* list = nullptr;
    FFI_TRY(workspace_get(s, kWsRewire, capacity * sizeof(unsigned), (void**)&list));
    SelectState* state = reinterpret_cast<SelectState*>(ws);
    unsigned* hist = reinterpret_cast<unsigned*>(ws + 256);
    const unsigned blocks = (unsigned)std::max<size_t>(1, std::min<size_t>((count + kHistThreads - 1) / kHistThreads, (size_t)device_cu_count() * 2));
    for (const auto pass : {select_pass_kernel<0>, select_pass_kernel<1>, select_pass_kernel<2>})
        hipLaunchKernelGGL(pass, dim3(blocks), dim3(kHistThreads), 0, s, w, count, k, state, hist, list, (unsigned long long)capacity, threshold);
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
                       seed, &reinterpret_cast<SelectState*>(ws)->rewired, rewired);
    FFI_HIP_TRY(hipGetLastError());
    return FFI_OK;
}

}  // namespace ffi
