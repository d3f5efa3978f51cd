// Small layers: one launch forward, one launch for all gradients, straight from the caller's arrays.
//
// At the sizes of takes_small() the other paths' preparation (a transposed or sliced copy of the features, a check of the cached
// plan, passes over it, partial sums and their reduction) costs more than the arithmetic: with B x L x K of some ten thousand to
// a million multiply-adds a launch of 2 to 4 us is what there is to pay.  So nothing is prepared, and each kernel spreads its
// sums over as many lanes as it takes for two or three memory latencies, in one of which the ids arrive and in the next the
// operands they name, to be all that is left.
// Semantics: tfsparse/cc/kernels/forward.cpp:9-44, backward.cpp:8-73 in the reference.
#include "ffi_internal.h"

#include <algorithm>

namespace ffi {
namespace {

constexpr int kSmThreads = 256;
constexpr int kSmSamples = 8;           // samples of a lane group: independent gathers per connection

// G lanes to a label and eight samples: lane <-> every G-th connection, the lanes' sums added up by a butterfly.
// 17 x 12 x 63 x 44: 14.0 us by the 32-sample tile (and a transpose of 2.3 in front), 4.4 here.
template <int G>
__global__ __launch_bounds__(kSmThreads) void fwd_small_kernel(const float* __restrict__ x, const int32_t* __restrict__ idx,
                                                               const float* __restrict__ w, const float* __restrict__ bias,
                                                               float* __restrict__ out, int B, int N, int L, int K, int tp) {
    const int l = threadIdx.x & (G - 1);
    const int j = (blockIdx.x * kSmThreads + threadIdx.x) / G;
    if (j >= L) return;
    const int b0 = blockIdx.y * kSmSamples, nb = min(kSmSamples, B - b0);
    const size_t sample = tp ? 1 : (size_t)N, column = tp ? (size_t)B : 1;
    const float* xb = x + b0 * sample;
    float acc[kSmSamples];
#pragma unroll
    for (int i = 0; i < kSmSamples; ++i) acc[i] = 0.f;
    const size_t row = (size_t)j * K;
#pragma unroll 4
    for (int k = l; k < K; k += G) {
        const unsigned id = min((unsigned)idx[row + k], (unsigned)N - 1u);
        const float wv = w[row + k];
#pragma unroll
        for (int i = 0; i < kSmSamples; ++i) acc[i] = fmaf(wv, xb[id * column + min(i, nb - 1) * sample], acc[i]);
    }
    // sample i ends up in lane i of the group (groups of four: i & 3)
#pragma unroll
    for (int off = G / 2; off > 0; off >>= 1)
#pragma unroll
        for (int i = 0; i < kSmSamples; ++i) acc[i] += __shfl_xor(acc[i], off, 64);
    const float bj = bias != nullptr ? bias[j] : 0.f;
#pragma unroll
    for (int i = 0; i < kSmSamples; ++i)
        if ((i & (G - 1)) == l && i < nb) out[(size_t)(b0 + i) * L + j] = bias != nullptr ? acc[i] + bj : acc[i];
}

// Both gradients (and the bias gradient) of a small layer.  Workgroups [0, gx_groups): one sample, `window` columns and one of
// `parts` equal shares of the connections each; every wavefront adds its connections into a copy of its own in LDS (ds_add in
// program order, so the sums repeat), and the copies are added up in order.  That is bound by the float adds in LDS, three clocks
// a lane: 0.8 G/s per CU, hence the parts, which leave their sums in `partial`; the workgroup that draws the last ticket of its
// sample and window adds them up, again in order.  The others: 1024 / splits connections each -- the labels' bias sums stand behind the
// connections, as connections to a column of ones -- with the samples spread over `splits` wavefronts.
// Ids out of range are skipped and reported in *bad (pinned host memory).
// 17 x 12 x 63 x 44: 7.0 us, where nine launches took 47.
constexpr int kSbThreads = 1024;        // (or 256)
constexpr int kSbInflight = 8;
constexpr int kSbCells = 32 * 1024;     // sums of a workgroup in LDS, over all wavefronts

__global__ __launch_bounds__(kSbThreads) void bwd_small_kernel(const float* __restrict__ x, const int32_t* __restrict__ idx,
                                                               const float* __restrict__ w, const float* __restrict__ g,
                                                               float* __restrict__ gx, float* __restrict__ gw, float* __restrict__ gb,
                                                               int B, int N, int L, int K, int tp, int gx_groups, int window, int parts, int splits,
                                                               unsigned* partial, unsigned* tickets, unsigned long long* bad) {
    extern __shared__ float lds[];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, threads = blockDim.x, waves = threads / 64;
    const int LK = L * K;
    if ((int)blockIdx.x < gx_groups) {
        const int windows = (N + window - 1) / window;
        const int unit = blockIdx.x / parts, part = blockIdx.x - unit * parts;                    // (sample and window)
        const int b = unit / windows, n0 = (unit - b * windows) * window, n = min(window, N - n0);
        const int share = (LK + parts - 1) / parts, first = part * share, last = min(first + share, LK);
        float* mine = lds + wave * window;
        for (int c = lane; c < n; c += 64) mine[c] = 0.f;
        __builtin_amdgcn_wave_barrier();
        const float* gr = g + (size_t)b * L;
        // label and place in its row, moved along with the connection; eight connections' loads in flight
        const int dj = threads / K, dk = threads - dj * K;
        int j = (first + (int)threadIdx.x) / K, k = first + (int)threadIdx.x - j * K;
        bool seen_bad = false;
        for (int p0 = first + (int)threadIdx.x; p0 < last; p0 += threads * kSbInflight) {
            unsigned id[kSbInflight];
            float v[kSbInflight], gv[kSbInflight];
#pragma unroll
            for (int u = 0; u < kSbInflight; ++u) {
                const int p = min(p0 + u * threads, last - 1);
                id[u] = (unsigned)idx[p];
                v[u] = w[p];
                gv[u] = gr[min(j, L - 1)];
                j += dj;
                k += dk;
                if (k >= K) { k -= K; ++j; }
            }
#pragma unroll
            for (int u = 0; u < kSbInflight; ++u) {
                const bool on = p0 + u * threads < last;
                const unsigned c = id[u] - (unsigned)n0;
                if (on && c < (unsigned)n) __hip_atomic_fetch_add(&mine[c], v[u] * gv[u], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                seen_bad |= on && id[u] >= (unsigned)N;
            }
        }
        if (seen_bad && unit == 0 && bad != nullptr) __hip_atomic_store(bad, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        __syncthreads();
        for (int c = threadIdx.x; c < n; c += threads) {
            float t = 0.f;
#pragma unroll 4
            for (int i = 0; i < waves; ++i) t += lds[i * window + c];
            if (parts > 1) {
                // (an exchange whose result is waited for has reached memory that all XCDs see; a fence would first write
                // back every dirty line of this XCD's L2: 150 us in place of 2)
                const unsigned old = __hip_atomic_exchange(&partial[(size_t)blockIdx.x * window + c], __float_as_uint(t), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                asm volatile("" ::"v"(old) : "memory");
            } else gx[tp ? (size_t)(n0 + c) * B + b : (size_t)b * N + n0 + c] = t;
        }
        if (parts == 1) return;
        __shared__ bool is_last;
        __syncthreads();
        if (threadIdx.x == 0) {
            is_last = __hip_atomic_fetch_add(&tickets[unit], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (unsigned)parts - 1u;
            if (is_last) tickets[unit] = 0u;               // for the next launch
        }
        __syncthreads();
        if (!is_last) return;
        const unsigned* sums = partial + (size_t)unit * parts * window;
        for (int c = threadIdx.x; c < n; c += threads) {
            // (eight running sums: one of up to 512 parts was further from the 64-bit result than the larger layers' path, 3.9e-7
            // against 2.7e-7 at 1 x 768 x 131,072 x 32)
            float t8[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            for (int i0 = 0; i0 < parts; i0 += 8) {
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const float v = __uint_as_float(__hip_atomic_load(&sums[(size_t)min(i0 + i, parts - 1) * window + c], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
                    t8[i] += i0 + i < parts ? v : 0.f;
                }
            }
            const float t = ((t8[0] + t8[1]) + (t8[2] + t8[3])) + ((t8[4] + t8[5]) + (t8[6] + t8[7]));
            gx[tp ? (size_t)(n0 + c) * B + b : (size_t)b * N + n0 + c] = t;
        }
        return;
    }
    const int total = LK + (gb != nullptr ? L : 0);
    const int p = ((blockIdx.x - gx_groups) * (waves / splits) + wave / splits) * 64 + lane, split = wave % splits;
    const bool on = p < total, ones = p >= LK;
    const int j = !on ? 0 : ones ? p - LK : p / K;
    unsigned id = on && !ones ? (unsigned)idx[p] : 0u;
    const bool out_of_range = id >= (unsigned)N;
    if (out_of_range) id = 0u;
    const size_t sample = tp ? 1 : (size_t)N;
    const float* xc = x + (tp ? (size_t)id * B : (size_t)id);
    float acc = 0.f;
    for (int b0 = split; b0 < B; b0 += splits * kSbInflight) {
        float xv[kSbInflight], gv[kSbInflight];
#pragma unroll
        for (int u = 0; u < kSbInflight; ++u) {
            const int b = min(b0 + u * splits, B - 1);
            xv[u] = xc[b * sample];
            gv[u] = g[(size_t)b * L + j];
        }
#pragma unroll
        for (int u = 0; u < kSbInflight; ++u)
            if (b0 + u * splits < B) acc = fmaf(ones ? 1.f : xv[u], gv[u], acc);
    }
    if (splits > 1) {
        lds[wave * 64 + lane] = acc;
        __syncthreads();
        if (split != 0) return;
        for (int i = 1; i < splits; ++i) acc += lds[(wave + i) * 64 + lane];
    }
    if (!on) return;
    if (ones) gb[p - LK] = acc;
    else gw[p] = out_of_range ? 0.f : acc;
}

}  // namespace

namespace {

// Workgroups of 16 wavefronts; of 4, and four times the columns each, where wide inputs meet few connections and clearing and
// adding up the copies would be all the work.
struct SmallShape { int threads, window; long long units; };
SmallShape small_shape(const Dims& d) {
    SmallShape sh;
    sh.threads = d.N > kSbCells / 16 && (long long)d.L * d.K <= 16384 ? 256 : kSbThreads;
    sh.window = std::min(d.N, kSbCells / (sh.threads / 64));
    sh.units = (long long)d.B * ((d.N + sh.window - 1) / sh.window);
    return sh;
}

}  // namespace

// Where the launches for small layers beat the paths made for large ones.  Forward: at 4 M products 14 us against 14 to 37, at 8 M
// up to 21.  Backward, whose work is a visit of every connection per sample and window: at 4 M visits 31 to 39 us against 42 to
// 320, at 8 M 48 to 75 against 44 to 205; 4 M sums of gx take 55 to 60 us against 92.
// Layers of few labels give the larger paths few workgroups, each with all batch tiles one after the other.  Up to 1,024 labels,
// backward: 128 x 1,000 x 1,000 x 64 61 us against 117, 256 x 300 x 1,024 x 40 73 against 85, 365 x 53 x 1,000 x 32 85 against 91 (12 M
// visits; at 15 to 25 M 106 to 176 against 106 to 147); up to 512 and fan-ins up to 128: 365 x 53 x 549 x 45 67 against 119, 512 x 1,000
// x 500 x 128 216 against 372 (fan-in 200 94 against 75).  Of 818 backward passes of up to 512 labels and 10 to 33 M visits the small
// path lost 30, all of more samples than CUs, where a workgroup has all connections of a sample (2.6 us a thousand), and of fan-ins of
// 65 to 96: there the large ones take 10 us a batch tile from 513 to 768 columns and 11 to 12 up to some 330 (260 x 600 x 512 x 96 90 against
// 127, 290 x 60 x 512 x 96 108 against 128; 380 x 60 x 480 x 90 118 against 114, 290 x 500 x 512 x 96 139 against 128).
// Forward up to 512 labels and from fan-in 64 on: 128 x 300 x 256 x 200 15 against 119, 365 x 100 x 500 x 64 19 against 41, 128 x 768 x 500 x 128 18 against 30 (16 M products: 33 against 31).
bool takes_small_forward(const Dims& d) {
    const long long sums = (long long)d.B * d.L * d.K;
    if (d.B > 65535 * kSmSamples) return false;            // (groups of samples are the grid's second dimension)
    if (g_options.small_path != 0) return g_options.small_path > 0 && sums < (1ll << 30);
    return sums <= (4ll << 20) || (d.L <= 512 && d.K >= 64 && sums <= 12'000'000);
}
bool takes_small_backward(const Dims& d) {
    const long long units = small_shape(d).units, visits = units * d.L * d.K, cells = (long long)d.B * d.N;
    if (g_options.small_path != 0) return g_options.small_path > 0 && visits < (1ll << 30) && cells < (1ll << 30);
    bool few_labels = (d.L <= 1024 && visits <= 12'000'000) || (d.L <= 512 && d.K <= 128 && visits <= (32ll << 20));
    const long long tiles = (d.B + 31) / 32, connections = (long long)d.L * d.K;
    if (d.K > 64 && d.K <= 96 && (d.N <= 330 || (d.N > 512 && d.N <= 768)) && connections > tiles * (d.N > 512 ? 3900 : d.N > 128 ? 4500 : 4200) &&
        units > device_cu_count())
        few_labels = false;
    return (visits <= (4ll << 20) || (few_labels && d.N <= 1216)) && cells <= (4ll << 20);
}

int launch_forward_small(const float* x, const int32_t* idx, const float* w, const float* bias, float* out, const Dims& d, hipStream_t s) {
    const unsigned groups = (unsigned)((d.B + kSmSamples - 1) / kSmSamples);
    auto grid = [&](int G) { return dim3((unsigned)(((size_t)d.L * G + kSmThreads - 1) / kSmThreads), groups); };
    if (d.K > 8) hipLaunchKernelGGL(fwd_small_kernel<16>, grid(16), dim3(kSmThreads), 0, s, x, idx, w, bias, out, d.B, d.N, d.L, d.K, d.tp);
    else hipLaunchKernelGGL(fwd_small_kernel<4>, grid(4), dim3(kSmThreads), 0, s, x, idx, w, bias, out, d.B, d.N, d.L, d.K, d.tp);
    FFI_HIP_TRY(hipGetLastError());
    return FFI_OK;
}

namespace {

// Shares of the connections with 2,048 adds each (2.5 us), or four to each sum that the share then has to exchange (25 G/s on
// the whole GPU), as long as the workgroups stay within two per CU.
int small_parts(const Dims& d, const SmallShape& sh) {
    const long long share = (long long)std::max(2048, 4 * sh.window) * ((d.N + sh.window - 1) / sh.window), LK = (long long)d.L * d.K;
    return (int)std::max(1ll, std::min((LK + share - 1) / share, 2 * device_cu_count() / std::max(1ll, sh.units)));
}

}  // namespace

size_t small_backward_workspace(const Dims& d) {
    const SmallShape sh = small_shape(d);
    const int parts = small_parts(d, sh);
    return parts > 1 ? (size_t)sh.units * parts * sh.window * sizeof(float) : 0;
}

int launch_backward_small(const float* x, const int32_t* idx, const float* w, const float* g, float* gx, float* gw, float* gb, const Dims& d,
                          hipStream_t s, unsigned long long* bad) {
    const SmallShape sh = small_shape(d);
    const int window = sh.window, units = (int)sh.units, LK = d.L * d.K, parts = small_parts(d, sh);
    const int gx_groups = gx != nullptr ? units * parts : 0;
    unsigned* partial = nullptr;
    unsigned* tickets = nullptr;
    if (gx_groups && parts > 1) {
        FFI_TRY(workspace_get(s, kWsPartials, small_backward_workspace(d), (void**)&partial));
        FFI_TRY(tickets_get(s, (void**)&tickets));
    }
    const int splits = std::min(sh.threads / 64, d.B > 64 ? 16 : d.B > 8 ? 4 : 1), total = LK + (gb != nullptr ? d.L : 0), per = sh.threads / splits;
    const int gw_groups = gw != nullptr ? (total + per - 1) / per : 0;
    const size_t lds = std::max((size_t)(gx_groups ? sh.threads / 64 * window : 0), (size_t)(splits > 1 ? sh.threads : 0)) * sizeof(float);
    if (lds > 64 * 1024) FFI_HIP_TRY(hipFuncSetAttribute((const void*)bwd_small_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(bwd_small_kernel, dim3((unsigned)(gx_groups + gw_groups)), dim3(sh.threads), lds, s, x, idx, w, g, gx, gw, gb, d.B, d.N,
                       d.L, d.K, d.tp, gx_groups, window, parts, splits, partial, tickets, bad);
    FFI_HIP_TRY(hipGetLastError());
    return FFI_OK;
}

}  // namespace ffi
