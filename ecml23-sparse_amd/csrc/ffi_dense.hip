// Few columns (at most 64): the rows of a tile of labels are written out over all columns, in LDS, and the passes are products of
// dense matrices on the matrix cores.
//
// The other paths gather one operand per multiply-add from LDS, 4 bytes each, and the input gradient walks a plan whose slots are
// few columns long and mostly holes (5.1 slots per connection at 17 columns).  With N columns and a fan-in of K the written-out
// rows cost N / K times the multiply-adds, at 256 per clock and CU on the matrix cores (fp32 operands and sums) against 32 that
// LDS has operands for, and nothing else grows with the batch: the forward pass and the backward pass then take what it takes to
// move the scores, and no plan is built.
// Semantics: tfsparse/cc/kernels/forward.cpp:9-44, backward.cpp:8-73 in the reference.  Connections of a label into one column are
// added up before they meet the operand.  A column without a connection is a zero that meets the operand all the same, so
// operands that are not finite, and sums of weights that are not, are taken out and their products formed connection by connection.
#include "ffi_internal.h"

#include <algorithm>

namespace ffi {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kDnSamples = 128;                      // samples of a launch's group: their features lie in LDS
constexpr int kDnLdsFloats = 160 * 1024 / 4;
constexpr int kDnTile = 64;                          // labels of a wavefront's tile, one per lane where rows are written
constexpr int kDnGPitch = kDnTile + 1;              // (odd, as all pitches: 32 rows fall into 32 banks)

template <int NT> struct DenseShape {                // NT: columns in blocks of 32
    static constexpr int kColumns = 32 * NT, kPitch = kColumns + 1;     // (the last entry of a row: where ids out of range go)
    static constexpr int kRows = kDnTile * kPitch;                      // floats
    static constexpr int kForwardWaves = NT == 1 ? 8 : 7;               // (what LDS holds rows of)
};
template <int NT, int NB, bool GX, bool GW> struct DenseBackwardShape : DenseShape<NT> {      // NB: samples in blocks of 32
    using S = DenseShape<NT>;
    static constexpr int kXPitch = 32 * NB + 1, kX = GW ? S::kColumns * kXPitch : 0;
    static constexpr int kG = 32 * kDnGPitch;                           // a block of out_grad
    static constexpr int kMine = GX ? S::kRows + kG : (S::kRows > kG ? S::kRows : kG);        // (without the columns' sums the products may take its place)
    static constexpr int kFit = (kDnLdsFloats - kX) / kMine, kWaves = kFit < 8 ? kFit : 8;
    static constexpr size_t kLdsBytes = (size_t)(kX + kWaves * kMine) * sizeof(float);
    static_assert(kWaves >= 4 && S::kColumns * 32 <= kMine, "a wavefront per SIMD; the wavefronts' sums lie in their rows' place");
};

// Row and column of element r of a lane's sixteen of a 32 x 32 product (v_mfma_f32_32x32x2_f32; an operand's element of a lane is of
// row or column lane % 32 and of the product's step 2 s + lane / 32).
__device__ __forceinline__ int product_row(int r, int lane) { return 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3); }

// four words at any word's address
template <class T> struct __attribute__((packed, aligned(4))) Quad { T v[4]; };

__device__ __forceinline__ bool not_finite(float v) { return (__float_as_uint(v) & 0x7f800000u) == 0x7f800000u; }

// xs[n][b]: the features of samples b0 ... b0 + nb - 1, zero behind them, up to `width`, and behind the last column.  True where one of
// a thread's is not finite.
template <int NT>
__device__ __forceinline__ bool stage_features(const float* __restrict__ x, float* xs, int B, int N, int b0, int nb, int width, int tp) {
    using S = DenseShape<NT>;
    bool odd = false;
    for (int e = threadIdx.x; e < S::kColumns * width; e += blockDim.x) {
        int n, b;
        if (tp) { n = e / width; b = e - n * width; }
        else { b = e / S::kColumns; n = e % S::kColumns; }
        const bool there = n < N && b < nb;
        const size_t at = tp ? (size_t)min(n, N - 1) * B + b0 + min(b, nb - 1) : (size_t)(b0 + min(b, nb - 1)) * N + min(n, N - 1);
        const float v = there ? x[at] : 0.f;
        odd |= not_finite(v);
        xs[n * (width + 1) + b] = v;
    }
    return odd;
}

// rows[lane][n] = the sum of the weights of label l0 + lane into column n; zero behind the last label, and where it is not finite: the
// label's connections into such a column (a bit of *apart) are taken one by one, as what meets the sum may be zero or not finite itself, or it
// is only the sum that overflows.  True where an id is out of range (CLAMP: it counts as the last column, else not at all).
// A lane reads and writes its own row, one connection after the other.  Rows come in pieces of 16 bytes: with the 64 lanes on as many
// lines, a piece costs the L1 what a word does.  (Forward 31 x 45 x 290,420 x 75: 196 us word by word, 85 so.)
template <int NT, bool CLAMP>
__device__ __forceinline__ bool write_rows(const int32_t* __restrict__ idx, const float* __restrict__ w, float* rows, int l0, int L, int N, int K, unsigned long long* apart) {
    using S = DenseShape<NT>;
    const int lane = threadIdx.x & 63;
    float* mine = rows + lane * S::kPitch;
    for (int n = 0; n < S::kColumns; ++n) mine[n] = 0.f;
    const bool there = l0 + lane < L;
    const size_t row = (size_t)min(l0 + lane, L - 1) * K;
    bool bad = false;
    float finite = 0.f;                                                   // NaN where a sum is not finite
    auto put = [&](unsigned id, float wv) {
        bad |= there && id >= (unsigned)N;
        const unsigned n = !there ? (unsigned)S::kColumns : CLAMP ? min(id, (unsigned)N - 1u) : min(id, id < (unsigned)N ? id : (unsigned)S::kColumns);
        const float sum = mine[n] + wv;
        finite = fmaf(sum, 0.f, finite);
        mine[n] = sum;
    };
    auto done = [&]() {
        *apart = 0ull;
        if (there && !(finite == 0.f))
            for (int n = 0; n < S::kColumns; ++n)
                if (not_finite(mine[n])) { mine[n] = 0.f; *apart |= 1ull << n; }
        return bad;
    };
    if (K < 4) {
        for (int k = 0; k < K; ++k) put((unsigned)idx[row + k], w[row + k]);
        return done();
    }
    constexpr int kQuads = 4;
    for (int k0 = 0; k0 < K; k0 += 4 * kQuads) {
        Quad<unsigned> id[kQuads];
        Quad<float> wv[kQuads];
#pragma unroll
        for (int i = 0; i < kQuads; ++i) {                                // (the last quad of a row ends with it)
            const int k = min(k0 + 4 * i, K - 4);
            id[i] = *reinterpret_cast<const Quad<unsigned>*>(idx + row + k);
            wv[i] = *reinterpret_cast<const Quad<float>*>(w + row + k);
        }
#pragma unroll
        for (int i = 0; i < kQuads; ++i) {
            const int again = max(k0 + 4 * i - (K - 4), 0);               // (elements of it that the quads before it had)
#pragma unroll
            for (int v = 0; v < 4; ++v)
                if (v >= again) put(id[i].v[v], wv[i].v[v]);
        }
    }
    return done();
}

__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// *to += v, unless it is an infinity or a NaN that stays what it is: where no value is finite any more, all connections would add up in
// N x B places.
__device__ __forceinline__ void add_apart(float* to, float v) {
    const float there = __hip_atomic_load(to, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (there != there || (not_finite(there) && (there == v || !not_finite(v)))) return;
    unsafeAtomicAdd(to, v);
}

// Tile t of a wavefront: workgroups side by side first, so that few tiles spread over all CUs.
// grid: (workgroups, groups of kDnSamples samples).  LDS: xs, then each wavefront's rows.
template <int NT>
__global__ __launch_bounds__(64 * DenseShape<NT>::kForwardWaves) void fwd_dense_kernel(const float* __restrict__ x, const int32_t* __restrict__ idx,
                                                                             const float* __restrict__ w, const float* __restrict__ bias,
                                                                             float* __restrict__ out, int B, int N, int L, int K, int tp, int tiles, int width) {
    using S = DenseShape<NT>;
    extern __shared__ __align__(16) float dn_mem[];
    float* const xs = dn_mem;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), half = lane >> 5, low = lane & 31;
    float* const rows = dn_mem + S::kColumns * (width + 1) + wave * S::kRows;
    const int b0 = blockIdx.y * kDnSamples, nb = min(kDnSamples, B - b0);
    const bool odd = __syncthreads_or(stage_features<NT>(x, xs, B, N, b0, nb, width, tp));
    for (int t = blockIdx.x + gridDim.x * wave; t < tiles; t += gridDim.x * S::kForwardWaves) {
        const int l0 = t * kDnTile;
        auto by_connections = [&]() {
            const int l = l0 + lane;
            for (int b = 0; b < nb; ++b) {
                float sum = 0.f;
                for (int k = 0; k < K; ++k) sum = fmaf(w[(size_t)l * K + k], xs[min((unsigned)idx[(size_t)l * K + k], (unsigned)N - 1u) * (width + 1) + b], sum);
                out[(size_t)(b0 + b) * L + l] = bias != nullptr ? sum + bias[l] : sum;
            }
        };
        if (odd) {
            if (l0 + lane < L) by_connections();
            continue;
        }
        unsigned long long apart;
        wave_lds_fence();
        (void)write_rows<NT, true>(idx, w, rows, l0, L, N, K, &apart);
        wave_lds_fence();
        const unsigned long long aparts = __ballot(apart != 0ull);
        if (apart != 0ull) by_connections();
        float bj[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) bj[h] = bias != nullptr ? bias[min(l0 + 32 * h + low, L - 1)] : 0.f;
        for (int bt = 0; bt < nb; bt += 32) {
            f32x16 acc[2] = {};
#pragma unroll 8
            for (int s = 0; s < 16 * NT; ++s) {
                const float a = xs[(2 * s + half) * (width + 1) + bt + low];
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    acc[h] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, rows[(32 * h + low) * S::kPitch + 2 * s + half], acc[h], 0, 0, 0);
            }
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int l = l0 + 32 * h + low;
                const bool stores = l < L && (aparts >> (32 * h + low) & 1ull) == 0ull;
                float* to = out + (size_t)(b0 + bt) * L + l;
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int b = product_row(r, lane);
                    if (bt + b < nb && stores) to[(size_t)b * L] = bias != nullptr ? acc[h][r] + bj[h] : acc[h][r];
                }
            }
        }
    }
}

// Gradients of a group of samples; `first`: the first group's, which stores gw and gb where the others add.
// A wavefront takes a tile of labels: writes its rows (GX), and for each 32 samples brings out_grad through LDS, where it is
// read both ways -- as labels x samples for the weights' products with the features, as samples x labels for the columns' products
// with the rows.  The columns' sums stay in registers for all tiles; at the end the workgroup adds its wavefronts' and leaves
// them in part[workgroup][n][b].  The weights' products end up in the rows' place, from where each connection picks its column's.
// A gradient that is not finite, and a label's columns whose sums are not, go to `odd_sums` [N][B] connection by connection (zero between launches).
template <int NT, int NB, bool GX, bool GW>
__global__ __launch_bounds__((64 * DenseBackwardShape<NT, NB, GX, GW>::kWaves)) void bwd_dense_kernel(const float* __restrict__ x, const int32_t* __restrict__ idx,
                                                                             const float* __restrict__ w, const float* __restrict__ g,
                                                                             float* __restrict__ gw, float* __restrict__ gb, float* __restrict__ part,
                                                                             float* __restrict__ odd_sums, int B, int N, int L, int K, int tp,
                                                                             int b0, int first, int tiles, unsigned long long* bad) {
    using S = DenseBackwardShape<NT, NB, GX, GW>;
    extern __shared__ __align__(16) float dn_mem[];
    float* const xs = dn_mem;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), half = lane >> 5, low = lane & 31;
    float* const rows = dn_mem + S::kX + wave * S::kMine;
    float* const gt = GX ? rows + S::kRows : rows;                       // [32 samples][kDnGPitch]
    const int nb = min(kDnSamples, B - b0);
    if (GW) {
        (void)stage_features<NT>(x, xs, B, N, b0, nb, 32 * NB, tp);
        __syncthreads();
    }
    f32x16 cols[NB][NT] = {};
    bool seen_bad = false;
    for (int t = blockIdx.x + gridDim.x * wave; t < tiles; t += gridDim.x * S::kWaves) {
        const int l0 = t * kDnTile, mine = min(l0 + lane, L - 1);
        const bool there = l0 + lane < L;
        f32x16 prod[2][NT] = {};
        float bias_sum = 0.f;
        float gv[32];
        auto ask = [&](int bt) {
#pragma unroll
            for (int i = 0; i < 32; ++i) gv[i] = g[(size_t)(b0 + min(bt + i, nb - 1)) * L + mine];
        };
        constexpr bool kAhead = !(NT == 2 && NB == 4 && GX && GW);         // (no registers left for it there)
        if (kAhead) ask(0);
        unsigned long long apart = 0ull;
        if (GX) {
            wave_lds_fence();
            seen_bad |= write_rows<NT, false>(idx, w, rows, l0, L, N, K, &apart);
        }
#pragma unroll
        for (int q = 0; q < NB; ++q) {
            const int bt = 32 * q;
            if (bt >= nb) break;
            if (!kAhead) ask(bt);
            float finite = 0.f;                                           // NaN where a value is not finite
            wave_lds_fence();
#pragma unroll
            for (int i = 0; i < 32; ++i) {
                const float v = there && bt + i < nb ? gv[i] : 0.f;
                finite = fmaf(v, 0.f, finite);
                bias_sum += v;
                gt[i * kDnGPitch + lane] = v;
            }
            if (kAhead && q + 1 < NB) ask(bt + 32);
            wave_lds_fence();
            if (GW) {
#pragma unroll 4
                for (int s = 0; s < 16; ++s) {
                    const float a0 = gt[(2 * s + half) * kDnGPitch + low], a1 = gt[(2 * s + half) * kDnGPitch + 32 + low];
#pragma unroll
                    for (int c = 0; c < NT; ++c) {
                        const float v = xs[(32 * c + low) * S::kXPitch + bt + 2 * s + half];
                        prod[0][c] = __builtin_amdgcn_mfma_f32_32x32x2f32(a0, v, prod[0][c], 0, 0, 0);
                        prod[1][c] = __builtin_amdgcn_mfma_f32_32x32x2f32(a1, v, prod[1][c], 0, 0, 0);
                    }
                }
            }
            if (GX) {
                if (__ballot(apart != 0ull || !(finite == 0.f)) != 0ull) {
                    wave_lds_fence();
                    for (int i = 0; i < min(32, nb - bt); ++i) {
                        const float v = gt[i * kDnGPitch + lane];
                        const bool odd = not_finite(v);
                        if (apart == 0ull && !odd) continue;
                        if (odd) gt[i * kDnGPitch + lane] = 0.f;
                        for (int k = 0; k < K; ++k) {
                            const unsigned id = (unsigned)idx[(size_t)mine * K + k];
                            if (id < (unsigned)N && (odd || (apart >> id & 1ull) != 0ull)) add_apart(&odd_sums[(size_t)id * B + b0 + bt + i], w[(size_t)mine * K + k] * v);
                        }
                    }
                    wave_lds_fence();
                }
#pragma unroll 4
                for (int s = 0; s < 32; ++s) {
                    const float v = gt[low * kDnGPitch + s + 32 * half];
#pragma unroll
                    for (int c = 0; c < NT; ++c)
                        cols[q][c] = __builtin_amdgcn_mfma_f32_32x32x2f32(rows[(s + 32 * half) * S::kPitch + 32 * c + low], v, cols[q][c], 0, 0, 0);
                }
            }
        }
        if (gb != nullptr && there) gb[mine] = first ? bias_sum : gb[mine] + bias_sum;
        if (GW) {
            wave_lds_fence();
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int c = 0; c < NT; ++c)
#pragma unroll
                    for (int r = 0; r < 16; ++r) rows[(32 * h + product_row(r, lane)) * S::kPitch + 32 * c + low] = prod[h][c][r];
            wave_lds_fence();
            const int total = min(kDnTile, L - l0) * K, dl = 64 / K, dk = 64 - dl * K;
            const size_t from = (size_t)l0 * K;
            int l = lane / K, k = lane - l * K;
            constexpr int kTogether = 8;
            for (int e = lane; e < total; e += 64 * kTogether) {
                unsigned id[kTogether];
                float old[kTogether];
#pragma unroll
                for (int i = 0; i < kTogether; ++i) {
                    const size_t at = from + min(e + 64 * i, total - 1);
                    id[i] = (unsigned)idx[at];
                    old[i] = first ? 0.f : gw[at];
                }
#pragma unroll
                for (int i = 0; i < kTogether; ++i) {
                    const float v = id[i] < (unsigned)N ? rows[min(l, kDnTile - 1) * S::kPitch + min(id[i], (unsigned)N - 1u)] : 0.f;
                    if (e + 64 * i < total) gw[from + e + 64 * i] = first ? v : old[i] + v;
                    l += dl; k += dk;
                    if (k >= K) { k -= K; ++l; }
                }
            }
        }
    }
    if (!GX) return;
    if (seen_bad && bad != nullptr) __hip_atomic_store(bad, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    // the wavefronts' sums, 32 samples at a time: [wavefront][n][32]
    float* const sums = dn_mem;
    float* const to = part + (size_t)blockIdx.x * S::kColumns * (NB * 32);
#pragma unroll
    for (int q = 0; q < NB; ++q) {
        __syncthreads();
#pragma unroll
        for (int c = 0; c < NT; ++c)
#pragma unroll
            for (int r = 0; r < 16; ++r) sums[(wave * S::kColumns + 32 * c + product_row(r, lane)) * 32 + low] = cols[q][c][r];
        __syncthreads();
        for (int e = threadIdx.x; e < S::kColumns * 32; e += 64 * S::kWaves) {
            float sum = 0.f;
#pragma unroll
            for (int v = 0; v < S::kWaves; ++v) sum += sums[v * S::kColumns * 32 + e];
            to[(e >> 5) * (NB * 32) + 32 * q + (e & 31)] = sum;
        }
    }
}

// gx of a group's samples: the workgroups' sums added up by eight lanes' worth of shares, each in order.  One workgroup per column.
constexpr int kDnReduceShares = 8;
__global__ __launch_bounds__(kDnSamples* kDnReduceShares) void dense_reduce_kernel(const float* __restrict__ part, int parts, int columns, int width,
                                                                                   float* __restrict__ odd_sums, float* __restrict__ gx, int B, int N, int b0,
                                                                                   int nb, int tp) {
    __shared__ float share[kDnReduceShares][kDnSamples];
    const int n = blockIdx.x, b = threadIdx.x % kDnSamples, q = threadIdx.x / kDnSamples;
    float sum = 0.f;
    if (b < nb) {
        const size_t step = (size_t)columns * width;
        const float* from = part + (size_t)n * width + b;
#pragma unroll 8
        for (int p = q; p < parts; p += kDnReduceShares) sum += from[p * step];
    }
    share[q][b] = sum;
    __syncthreads();
    if (q != 0 || b >= nb) return;
    sum = 0.f;
#pragma unroll
    for (int i = 0; i < kDnReduceShares; ++i) sum += share[i][b];
    const size_t odd_at = (size_t)n * B + b0 + b;
    const float odd = odd_sums[odd_at];
    if (!(odd == 0.f)) {
        odd_sums[odd_at] = 0.f;
        sum += odd;
    }
    gx[tp ? odd_at : (size_t)(b0 + b) * N + n] = sum;
}

int dense_workgroups(const Dims& d, int groups) {
    const int tiles = (d.L + kDnTile - 1) / kDnTile;
    return std::max(1, std::min(tiles, device_cu_count() / std::max(1, std::min(groups, device_cu_count()))));
}

template <int NT>
int launch_forward_dense_of(const float* x, const int32_t* idx, const float* w, const float* bias, float* out, const Dims& d, hipStream_t s) {
    using S = DenseShape<NT>;
    const int groups = (d.B + kDnSamples - 1) / kDnSamples, tiles = (d.L + kDnTile - 1) / kDnTile;
    const int width = d.B <= 32 ? 32 : d.B <= 64 ? 64 : kDnSamples;
    const size_t lds = (size_t)(S::kColumns * (width + 1) + S::kForwardWaves * S::kRows) * sizeof(float);
    FFI_HIP_TRY(hipFuncSetAttribute((const void*)fwd_dense_kernel<NT>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(fwd_dense_kernel<NT>, dim3((unsigned)dense_workgroups(d, groups), (unsigned)groups), dim3(64 * S::kForwardWaves), lds, s, x, idx, w, bias, out,
                       d.B, d.N, d.L, d.K, d.tp, tiles, width);
    FFI_HIP_TRY(hipGetLastError());
    return FFI_OK;
}

template <int NT, int NB>
int launch_backward_dense_of(const float* x, const int32_t* idx, const float* w, const float* g, float* gx, float* gw, float* gb, const Dims& d, hipStream_t s,
                             unsigned long long* bad) {
    using S = DenseShape<NT>;
    const int tiles = (d.L + kDnTile - 1) / kDnTile, workgroups = dense_workgroups(d, 1);
    float *part = nullptr, *odd_sums = nullptr;
    if (gx != nullptr) {
        FFI_TRY(workspace_get(s, kWsPartials, (size_t)workgroups * S::kColumns * NB * 32 * sizeof(float), (void**)&part));
        FFI_TRY(zeroed_get(s, kWsDense, (size_t)d.N * d.B * sizeof(float), (void**)&odd_sums));
    }
    auto go = [&](auto shape, auto kernel) -> int {
        using S = decltype(shape);
        FFI_HIP_TRY(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)S::kLdsBytes));
        for (int b0 = 0; b0 < d.B; b0 += kDnSamples) {
            hipLaunchKernelGGL(kernel, dim3((unsigned)workgroups), dim3(64 * S::kWaves), S::kLdsBytes, s, x, idx, w, g, gw, gb, part, odd_sums, d.B, d.N, d.L, d.K,
                               d.tp, b0, b0 == 0 ? 1 : 0, tiles, bad);
            if (gx != nullptr)
                hipLaunchKernelGGL(dense_reduce_kernel, dim3((unsigned)d.N), dim3(kDnSamples * kDnReduceShares), 0, s, part, workgroups, S::kColumns, NB * 32,
                                   odd_sums, gx, d.B, d.N, b0, std::min(kDnSamples, d.B - b0), d.tp);
        }
        FFI_HIP_TRY(hipGetLastError());
        return FFI_OK;
    };
    if (gx == nullptr) return go(DenseBackwardShape<NT, NB, false, true>{}, bwd_dense_kernel<NT, NB, false, true>);
    if (gw == nullptr) return go(DenseBackwardShape<NT, NB, true, false>{}, bwd_dense_kernel<NT, NB, true, false>);
    return go(DenseBackwardShape<NT, NB, true, true>{}, bwd_dense_kernel<NT, NB, true, true>);
}

template <int NT>
int launch_backward_dense_any(const float* x, const int32_t* idx, const float* w, const float* g, float* gx, float* gw, float* gb, const Dims& d, hipStream_t s,
                              unsigned long long* bad) {
    if (d.B <= 32) return launch_backward_dense_of<NT, 1>(x, idx, w, g, gx, gw, gb, d, s, bad);
    if (d.B <= 64) return launch_backward_dense_of<NT, 2>(x, idx, w, g, gx, gw, gb, d, s, bad);
    return launch_backward_dense_of<NT, 4>(x, idx, w, g, gx, gw, gb, d, s, bad);
}

}  // namespace

// Which layers take these kernels.  Their time is that of whole blocks of 32 columns and 32 samples, of a launch for every 128 samples
// backward, and of bringing and writing the rows; the others' is that of the multiply-adds, and backward of the plan's slots.  Of 360 +
// 2,037 points (1 to 500 samples, 8 to 64 columns, 2,000 to 400,000 labels, fan-ins of 4 to 128), time of the others over time of these:
//   forward, up to 32 columns, fan-in from 16 on 1.1 to 3.5; of 8 to 15 up to 128 samples 1.0 to 1.5, above 0.9 to 1.4; of 4 and 5 0.6 to 1.4.  Up to
//   16 samples the slices in LDS are faster (0.6 to 1.0).  33 to 64 columns: fan-in from 48 on 1.0 to 2.8; below, up to 64 samples 1.1 to 1.5 up to
//   60,000 labels and 0.6 to 0.95 at 250,000; more samples 0.5 to 1.2.
//   Both gradients, one group: up to 32 columns 0.9 to 15; 33 to 64 up to 32 samples 1.0 to 4.2; up to 64 1.1 to 2.2, 0.8 to 1.1 at 250,000 labels and
//   fan-ins below 16; up to 128 0.6 to 1.3 at fan-ins below 20, 1.05 to 2.7 from 28 on.
// Each group more is another launch, of no more workgroups than there are tiles, where the others take all samples in one and spread few labels'
// samples over the CUs.  Of 1,600 points more (130 to 200,000 samples, 64 to 200,000 labels):
//   Both gradients, up to 32 columns: two groups 1.0 to 3.3, but 0.87 to 0.93 below 4,000 labels at fan-ins of 20 to 29 and 0.87 at 15,000 and 5; more 0.32
//   (1,433 samples, 852 labels) to 0.8 below 8,192 labels, from there on 0.82 to 1.0 where there are fewer than 180,000 connections to a group and
//   1.03 to 3.1 where there are more; three groups from 8,192 labels and a fan-in of 30 on 1.03 to 1.7.  33 to 64 columns: two groups 1.0 to 2.3 where the fan-in is
//   50; more 0.83 to 0.96 up to 24,000 labels, 0.96 to 1.5 above.
//   Weight gradient alone, one group: 1.0 to 3.9, but 0.6 to 1.0 for fan-ins from 40 on at 5,000 labels, where a wavefront has all connections of a tile.
//   More of few labels 0.06 (171,000 samples, 378 labels: 2.3 ms and 36) to 0.7.  Up to 32 columns: two and three groups 1.1 to 1.7 from 16,384 labels
//   on, but 0.6 to 0.8 at fan-ins below 8; more 0.4 to 0.95, from 80,000 labels (four groups: 50,000) or a million connections on 0.9 to 1.9.  33 to 64 columns:
//   0.4 to 0.95, from 20,000 labels and 0.9 million (more than three groups: 2.2) connections on 0.89 to 2.2.
bool takes_dense_forward(const Dims& d) {
    if (d.N > 64 || d.L >= (1 << 25) || d.B > 65535 * kDnSamples) return false;
    if (g_options.dense_rows != 0) return g_options.dense_rows > 0;
    if (d.B <= 16) return false;
    if (d.N <= 32) return d.K >= (d.B <= kDnSamples ? 8 : 16);
    return d.K >= 48 || (d.B <= 64 && d.L <= 65536);
}
bool takes_dense_backward(const Dims& d) {
    if (d.N > 64 || d.L >= (1 << 25)) return false;
    if (g_options.dense_rows != 0) return g_options.dense_rows > 0;
    const int groups = (d.B + kDnSamples - 1) / kDnSamples;
    if (groups == 1) return d.N <= 32 || d.B <= 32 || d.K >= 24 || (d.B <= 64 && (d.K >= 16 || d.L <= 100000));
    if (d.N > 32) return d.K >= 25 * groups && d.L >= (groups == 2 ? 16384 : 24000);
    if (groups == 2) return d.L >= 32768 || d.K >= (d.L >= 16384 ? 10 : d.L >= 4096 ? 20 : 32);
    if (groups == 3 && d.L >= 8192 && d.K >= 30) return true;
    return d.L >= 16384 && d.K >= 5 * groups && (long long)d.L * d.K >= 180000ll * groups;
}
bool takes_dense_weight_grad(const Dims& d) {
    if (d.N > 64 || d.L >= (1 << 25)) return false;
    if (g_options.dense_rows != 0) return g_options.dense_rows > 0;
    const int groups = (d.B + kDnSamples - 1) / kDnSamples;
    if (groups == 1) return d.L >= 16384 || d.K <= 32;
    const long long connections = (long long)d.L * d.K;
    if (d.N > 32) return d.L >= 20000 && connections >= (groups <= 3 ? 900000 : 2200000);
    if (groups <= 3) return d.L >= 16384 && (d.K >= 8 || d.L >= 32768);
    return d.L >= (groups == 4 ? 50000 : 80000) || (d.L >= 24000 && connections >= 1000000);
}

size_t dense_backward_workspace(const Dims& d) {
    const size_t columns = d.N <= 32 ? 32 : 64, width = d.B <= 32 ? 32 : d.B <= 64 ? 64 : 128;
    return (size_t)dense_workgroups(d, 1) * columns * width * sizeof(float);
}
size_t dense_backward_zeroed(const Dims& d) { return (size_t)d.N * d.B * sizeof(float); }

int launch_forward_dense(const float* x, const int32_t* idx, const float* w, const float* bias, float* out, const Dims& d, hipStream_t s) {
    return d.N <= 32 ? launch_forward_dense_of<1>(x, idx, w, bias, out, d, s) : launch_forward_dense_of<2>(x, idx, w, bias, out, d, s);
}

int launch_backward_dense(const float* x, const int32_t* idx, const float* w, const float* g, float* gx, float* gw, float* gb, const Dims& d, hipStream_t s,
                          unsigned long long* bad) {
    return d.N <= 32 ? launch_backward_dense_any<1>(x, idx, w, g, gx, gw, gb, d, s, bad) : launch_backward_dense_any<2>(x, idx, w, g, gx, gw, gb, d, s, bad);
}

}  // namespace ffi
