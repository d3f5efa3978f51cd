// Backward pass for inputs whose tile does not fit in LDS (more than 1,216 columns), and for any other shape whose plan has the
// global form: both gradients in one walk over the plan's streams, whose wavefronts keep 32 columns' sums in registers and gather rows
// of slices of out_grad (ffi_sliced.h), all at about the same labels at a time; and the weight gradient alone, straight from the
// lookup, whose gathers of whole rows of the batch-major features come through the cache hierarchy.
#include "ffi_internal.h"
#include "ffi_check.h"
#include "ffi_lds_tile.h"
#include "ffi_sliced.h"
#include "ffi_walk.h"

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
// x[n] and g[label].  Both need row `label` of out_grad, so one walk over the plan's streams gathers it once: GL lanes of 16
// bytes hold a row of a slice of out_grad (ffi_sliced.h; rows of fewer bytes a lane come at half the rate), and one load brings the
// rows of a step, 64 / GL connections of one column.  A wavefront owns the 32 columns of a stream.  Their sums, one per lane
// group, stay in its registers and are reached by the step's column as an index into the register file (the same for all
// lanes); their rows of x lie in LDS.  Sixteen steps, a chunk, are in flight.  Every stream goes through the labels in ascending order,
// the wavefronts of a CU held together by a barrier at every chunk: then what one brings into the L2 is there for the others of the XCD.
//
// Weights come and weight gradients leave in the order of the plan's entries, whole lines at a time; the kernels below carry
// them from and to their places.
//
// Bound by the L1s' delivery (some 20 clocks for a load of 1 KB) with the instructions beside it (15 vector instructions a step) and what
// misses the L2.  65,536 columns x 670,091 labels x 72: 64 samples 0.68 ms, of which 0.55 remain with all rows in the L1s; 1.06 without
// the barrier (the older of two wavefronts on a SIMD is served first and runs away from the other).  Sums in LDS with a lane group
// per column, whose lists of a block of labels are short and of unequal lengths, took 1.07 (two slices of 32 samples), and needed the weights in a
// random order (0.37 each way, 0.1 now).  Rows of 128 samples 1.49 instead of 1.36; 16 wavefronts of 16 columns 0.70; sixteen steps in flight 0.68.
// per wavefront: its columns' rows of x, a lane's 16 bytes apart from the next multiple of 64 banks, and two chunks' lists
constexpr int walk_rows_bytes(int gl) { return kGroupColumns * (gl + 1) * 16; }
constexpr int walk_wave_bytes(int gl) { return walk_rows_bytes(gl) + 16 * kChunkSteps * 64 / gl; }
typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));
typedef float f32x32 __attribute__((ext_vector_type(32)));

// v + (v of the lane that CTRL pairs with this one)
template <int CTRL> __device__ __forceinline__ float dpp_add(float keep, float send) {
    return keep + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, send), CTRL, 0xf, 0xf, true));
}

// Pairs of lanes that differ in bit BIT (and may differ below it) add up: a in the lane that has it clear, b in the other.
template <int BIT> __device__ __forceinline__ float fold(float a, float b, int lane) {
    constexpr int kRor8 = 0x128, kHalfMirror = 0x141, kQuadHalves = 0x4e, kQuadSwap = 0xb1;
    const bool up = (lane & BIT) != 0;
    return dpp_add<BIT == 8 ? kRor8 : BIT == 4 ? kHalfMirror : BIT == 2 ? kQuadHalves : kQuadSwap>(up ? b : a, up ? a : b);
}

// Pairs of lanes that are 32 or 16 apart add up: a in the lower one, b in the other.
template <int BIT> __device__ __forceinline__ float fold_halves(float a, float b) {
    static_assert(BIT == 32 || BIT == 16);
    const unsigned ua = __builtin_bit_cast(unsigned, a), ub = __builtin_bit_cast(unsigned, b);
    unsigned u, v;                                               // (not elements of the pair: a bit cast of one takes the first's bits)
    if constexpr (BIT == 32) { const auto r = __builtin_amdgcn_permlane32_swap(ua, ub, false, false); u = r[0]; v = r[1]; }
    else { const auto r = __builtin_amdgcn_permlane16_swap(ua, ub, false, false); u = r[0]; v = r[1]; }
    return __builtin_bit_cast(float, u) + __builtin_bit_cast(float, v);
}

// sums[column of a step] += w * g, for two steps: the registers that hold component c of all columns are consecutive ones, and
// the step's column is what is added to the number of the first.  (In one piece, so that nothing else executes while registers are
// indexed.  The columns are below 32: the plan's entries hold nothing else there.)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"                  // (M0 is clobbered, and said to be)
__device__ __forceinline__ void add_steps(f32x32 (&sum)[4], unsigned col0, float w0, const float4& g0, unsigned col1, float w1, const float4& g1) {
    asm volatile("s_set_gpr_idx_on %[c0], 0xc\n"                 // (0xc: the addend's and the result's registers)
                 "v_fma_f32 v128, %[g00], %[w0], v128\n v_fma_f32 v160, %[g01], %[w0], v160\n"
                 "v_fma_f32 v192, %[g02], %[w0], v192\n v_fma_f32 v224, %[g03], %[w0], v224\n"
                 "s_set_gpr_idx_on %[c1], 0xc\n"
                 "v_fma_f32 v128, %[g10], %[w1], v128\n v_fma_f32 v160, %[g11], %[w1], v160\n"
                 "v_fma_f32 v192, %[g12], %[w1], v192\n v_fma_f32 v224, %[g13], %[w1], v224\n"
                 "s_set_gpr_idx_off"
                 : "+{v[128:159]}"(sum[0]), "+{v[160:191]}"(sum[1]), "+{v[192:223]}"(sum[2]), "+{v[224:255]}"(sum[3])
                 : [c0] "s"(col0), [c1] "s"(col1), [w0] "v"(w0), [w1] "v"(w1), [g00] "v"(g0.x), [g01] "v"(g0.y), [g02] "v"(g0.z), [g03] "v"(g0.w),
                   [g10] "v"(g1.x), [g11] "v"(g1.y), [g12] "v"(g1.z), [g13] "v"(g1.w)
                 : "m0");
}
#pragma clang diagnostic pop

struct WalkArgs {
    const float *gtab, *x, *slot_w;             // slices of out_grad (gslice apart), the features, weights in the order of the entries
    const unsigned *entries, *chunk_ptr, *chunk_count;
    float *gx, *parts, *gw_slots;               // one segment: gx itself; more: their sums, a slice's `part` apart; a slice's gradients `slots` apart
    size_t gslice, part, slots;
    int slice0, slices, add_gw, B, N, L, units, groups, segments, seg_labels;
    bool tp;
};

template <int GL, bool DOT>
__global__ __launch_bounds__(kWalkWaves * 64) void walk_columns_kernel(const WalkArgs a) {
    static_assert(GL == 16 || GL == 8);
    constexpr int kMembers = 64 / GL, kEntries = kChunkSteps * kMembers, kHeld = kEntries / 64;     // entries of a chunk, and of a lane
    constexpr unsigned kRow = GL * 16u, kNoRow = 0xffffff00u;               // (behind every table's end: reads as zero)
    __shared__ __align__(16) unsigned char mem[kWalkWaves * walk_wave_bytes(GL)];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int sub = lane & (GL - 1), member = lane / GL;
    const int all = a.units * a.slices, wg = xcd_unit(blockIdx.x, (all + kWalkWaves - 1) / kWalkWaves);
    if (wg < 0) return;
    const bool on = wg * kWalkWaves + wave < all;
    const int at = walk_place(wg, wave, all), slice = at / a.units, u = at - slice * a.units;
    float4* const xs = reinterpret_cast<float4*>(mem + wave * walk_wave_bytes(GL));
    unsigned* const offs = reinterpret_cast<unsigned*>(mem + wave * walk_wave_bytes(GL) + walk_rows_bytes(GL));
    float* const wts = reinterpret_cast<float*>(offs + 2 * kEntries);
    const int segment = u / a.groups, n0 = (u - segment * a.groups) * kGroupColumns;
    const int label0 = segment * a.seg_labels, b0 = (a.slice0 + slice) * GL * 4;
    const buffer_rsrc rows = make_rsrc(a.gtab + (a.slice0 + slice) * a.gslice + (size_t)label0 * (GL * 4), (size_t)min(a.seg_labels, a.L - label0) * kRow);
    const unsigned lane_off = (unsigned)sub * 16u;
    const unsigned count = on ? a.chunk_count[u] : 0u;
    unsigned rounds = 0;                                                    // of the workgroup, in all its wavefronts: they meet at as many barriers
#pragma unroll
    for (int i = 0; i < kWalkWaves; ++i) rounds = max(rounds, a.chunk_count[walk_stream(wg, i, a.units, all)]);
    // this lane's part of x: 16 bytes of some columns' rows, or four samples of a column several times
    constexpr int kXLoads = kGroupColumns / kMembers;
    float4 xv[DOT ? kXLoads : 1];
    if (DOT && a.tp && a.B % 4 == 0) {
        const int b = b0 + 4 * sub;
#pragma unroll
        for (int i = 0; i < kXLoads; ++i) {
            const f32x4_any q = *reinterpret_cast<const f32x4_any*>(a.x + (size_t)min(n0 + member + i * kMembers, a.N - 1) * a.B + min(b, a.B - 4));
            xv[i] = b < a.B ? make_float4(q.x, q.y, q.z, q.w) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
    } else if (DOT) {
        const int b = a.tp ? b0 + 4 * sub : b0 + 4 * (lane / kGroupColumns);
#pragma unroll
        for (int i = 0; i < kXLoads; ++i)
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const int n = min(n0 + (a.tp ? member + i * kMembers : lane & (kGroupColumns - 1)), a.N - 1), at = b + c + (a.tp ? 0 : 8 * i);
                const float t = a.x[a.tp ? (size_t)n * a.B + min(at, a.B - 1) : (size_t)min(at, a.B - 1) * a.N + n];
                reinterpret_cast<float*>(&xv[i])[c] = at < a.B ? t : 0.f;
            }
    }
    auto put_x = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kXLoads; ++i)
            xs[a.tp ? (member + i * kMembers) * (GL + 1) + sub : (lane & (kGroupColumns - 1)) * (GL + 1) + lane / kGroupColumns + 2 * i] = xv[i];
    };
    f32x32 sum[4];
#pragma unroll
    for (int i = 0; i < kGroupColumns; ++i) { sum[0][i] = 0.f; sum[1][i] = 0.f; sum[2][i] = 0.f; sum[3][i] = 0.f; }
    if (count > 0) {
        const size_t slot0 = (size_t)a.chunk_ptr[u] * kEntries + lane;
        float* const gw_slots = a.gw_slots + slice * a.slots + slot0;
        const unsigned* const entries = a.entries + slot0;
        const float* const weights = a.slot_w + slot0;
        struct Held { unsigned entry[kHeld]; float w[kHeld]; };
        auto fetch = [&](unsigned c) __attribute__((always_inline)) {
            Held h;
#pragma unroll
            for (int k = 0; k < kHeld; ++k) {
                h.entry[k] = __builtin_nontemporal_load(entries + (size_t)min(c, count - 1u) * kEntries + 64 * k);
                h.w[k] = __builtin_nontemporal_load(weights + (size_t)min(c, count - 1u) * kEntries + 64 * k);
            }
            return h;
        };
        // this lane's first entry is that of step `step` (entry_in_chunk, the other way round), a second one that of step + 8
        const int v = GL == 16 ? sub / 2 : sub, step = ((v & 1) << 2 | (v & 2) | v >> 2) + (GL == 16 ? sub % 2 * 8 : 0);
        unsigned* const my_offs = offs + member * kChunkSteps;                  // lists: member by member, in the order of the steps
        float* const my_wts = wts + member * kChunkSteps;
        auto put = [&](const Held& h, bool there, unsigned buf) {
#pragma unroll
            for (int k = 0; k < kHeld; ++k) {
                const bool pad = !there || h.entry[k] >= kPadEntry;
                my_offs[buf * kEntries + step + 8 * k] = pad ? kNoRow : (h.entry[k] >> 8) * kRow;
                my_wts[buf * kEntries + step + 8 * k] = pad ? 0.f : h.w[k];
            }
        };
        uint4 g[kChunkSteps];
        auto request = [&](unsigned buf, int i) __attribute__((always_inline)) {
            const uint2 o = *reinterpret_cast<const uint2*>(my_offs + buf * kEntries + i);
            g[i] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rows, o.x + lane_off, 0, 0));
            g[i + 1] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rows, o.y + lane_off, 0, 0));
        };
        Held now = fetch(0), next = fetch(1);
        if (DOT) put_x();
        put(now, true, 0);
        __builtin_amdgcn_wave_barrier();                                    // (the lists are the wavefront's own: LDS serves it in order)
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < kChunkSteps; i += 2) request(0, i);
        __builtin_amdgcn_sched_barrier(0);
        for (unsigned c = 0; c < rounds; ++c) {
            __builtin_amdgcn_s_barrier();
            if (c >= count) continue;
            const unsigned buf = c & 1u;
            put(next, c + 1u < count, buf ^ 1u);
            const Held after = fetch(c + 2);
            float gw_old[kHeld];
#pragma unroll
            for (int k = 0; k < kHeld; ++k) gw_old[k] = DOT && a.add_gw ? gw_slots[(size_t)c * kEntries + 64 * k] : 0.f;
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_sched_barrier(0);
            float dots[2];
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                float p[8];
#pragma unroll
                for (int i = 0; i < 8; i += 2) {
                    // steps in an order that lets the sums over the lanes fold as they come
                    const int v0 = (i & 1) << 2 | (i & 2) | i >> 2, v1 = v0 + 4, held = GL == 16 ? 0 : q;
                    const unsigned e0 = (unsigned)__builtin_amdgcn_readlane((int)now.entry[held], GL == 16 ? 2 * v0 + q : v0);
                    const unsigned e1 = (unsigned)__builtin_amdgcn_readlane((int)now.entry[held], GL == 16 ? 2 * v1 + q : v1);
                    const float2 w = *reinterpret_cast<const float2*>(my_wts + buf * kEntries + q * 8 + i);
                    float4 x0, x1;
                    if (DOT) { x0 = xs[(e0 & (kGroupColumns - 1)) * (GL + 1) + sub]; x1 = xs[(e1 & (kGroupColumns - 1)) * (GL + 1) + sub]; }
                    const float4 g0 = __builtin_bit_cast(float4, g[q * 8 + i]), g1 = __builtin_bit_cast(float4, g[q * 8 + i + 1]);
                    add_steps(sum, e0, w.x, g0, e1, w.y, g1);               // (of an entry's word the low byte is the index)
                    if (DOT) {
                        p[v0] = fmaf(x0.w, g0.w, fmaf(x0.z, g0.z, fmaf(x0.y, g0.y, x0.x * g0.x)));
                        p[v1] = fmaf(x1.w, g1.w, fmaf(x1.z, g1.z, fmaf(x1.y, g1.y, x1.x * g1.x)));
                        p[v0] = fold<GL / 2>(p[v0], p[v1], lane);
                        if (i & 2) p[v0 & 1] = fold<GL / 4>(p[v0 & 1], p[v0], lane);
                    }
                    request(buf ^ 1u, q * 8 + i);
                    __builtin_amdgcn_sched_barrier(0);
                }
                if (DOT) dots[q] = fold<GL / 8>(p[0], p[1], lane);
            }
            if (DOT) {
                if constexpr (GL == 16) dots[0] = fold<1>(dots[0], dots[1], lane);
#pragma unroll
                for (int k = 0; k < kHeld; ++k) gw_slots[(size_t)c * kEntries + 64 * k] = gw_old[k] + dots[k];
            }
            now = next;
            next = after;
            __builtin_amdgcn_wave_barrier();
        }
    } else {
        for (unsigned c = 0; c < rounds; ++c) __builtin_amdgcn_s_barrier();
    }
    if (!on) return;
    // sums over the lane groups: a group is left with some of the columns, first .. first + kKeep - 1
    constexpr int kKeep = kGroupColumns / kMembers;
    const int first = (lane >> 5 & 1) * 16 + (lane >> 4 & 1) * 8 + (GL == 8 ? (lane >> 3 & 1) * 4 : 0);
    float4 kept[kKeep];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        float t[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) t[i] = fold_halves<32>(sum[c][i], sum[c][i + 16]);
#pragma unroll
        for (int i = 0; i < 8; ++i) t[i] = fold_halves<16>(t[i], t[i + 8]);
        if constexpr (GL == 8)
#pragma unroll
            for (int i = 0; i < 4; ++i) t[i] = fold<8>(t[i], t[i + 4], lane);
#pragma unroll
        for (int i = 0; i < kKeep; ++i) reinterpret_cast<float*>(&kept[i])[c] = t[i];
    }
    if (a.segments > 1) {
        float* const to = a.parts + (a.slice0 + slice) * a.part + ((size_t)segment * a.N + n0 + first) * (GL * 4) + sub * 4;
#pragma unroll
        for (int i = 0; i < kKeep; ++i)
            if (n0 + first + i < a.N) *reinterpret_cast<float4*>(to + i * (GL * 4)) = kept[i];
    } else if (a.tp) {
        const int b = b0 + 4 * sub;
#pragma unroll
        for (int i = 0; i < kKeep; ++i) {
            const int n = n0 + first + i;
            if (n >= a.N) continue;
            float* const to = a.gx + (size_t)n * a.B + b;
            if (b + 4 <= a.B) {
                f32x4_any o;
                o.x = kept[i].x; o.y = kept[i].y; o.z = kept[i].z; o.w = kept[i].w;
                *reinterpret_cast<f32x4_any*>(to) = o;
            } else {
                if (b < a.B) to[0] = kept[i].x;
                if (b + 1 < a.B) to[1] = kept[i].y;
                if (b + 2 < a.B) to[2] = kept[i].z;
            }
        }
    } else {
        // through LDS, where x is no longer needed: lanes run over the columns
#pragma unroll
        for (int i = 0; i < kKeep; ++i) xs[(first + i) * (GL + 1) + sub] = kept[i];
        __builtin_amdgcn_wave_barrier();
        const int i = lane & (kGroupColumns - 1), n = n0 + i;
        const float* const from = reinterpret_cast<const float*>(xs + i * (GL + 1));
        for (int q = lane / kGroupColumns; q < GL * 4 && b0 + q < a.B; q += 2)
            if (n < a.N) a.gx[(size_t)(b0 + q) * a.N + n] = from[q];
    }
}

// Weights into the order of the plan's entries, and weight gradients from it: a workgroup takes a tile of consecutive flat positions
// through LDS, so that memory sees them as they lie on this side, and runs of a stream's neighbouring entries on the other.
// (Weight gradients of `slices` slices that were formed side by side are summed, in their order.)
// Consecutive tiles go to one XCD, whose L2 gathers what several of them write to a line.
//
// The first check.blocks workgroups of the one check the lookup's content against the plan instead (ffi_check.h); where that found the plan
// outdated, the other clears what the kernel that then forms the gradients anew adds up in memory: gw, or gx (takes_outdated_wide()).  (As kernels of their own the two were 9 of the 50 to 60
// us of a backward pass of few connections, and the check 40 of 3,250 at 65,536 columns x 670,091 labels x 72.)
constexpr int kTileMoveThreads = kCheckThreads, kTileMoveAhead = 8;

__global__ __launch_bounds__(kTileMoveThreads) void weights_to_slots_kernel(const float* __restrict__ w, const unsigned short* __restrict__ tile_pos,
                                                                            const unsigned* __restrict__ slot_of, float* __restrict__ slot_w,
                                                                            size_t total, int tile_bits, int tiles, const LookupCheck check) {
    extern __shared__ __align__(16) float tile_mem[];
    __shared__ CheckShared check_shared;
    const int checks = (check.blocks + kXcds - 1) / kXcds * kXcds;
    if ((int)blockIdx.x < checks) {
        if ((int)blockIdx.x < check.blocks) check_block(check, blockIdx.x, check_shared);
        return;
    }
    const int t = xcd_unit(blockIdx.x - checks, tiles);
    if (t < 0) return;
    const size_t p0 = (size_t)t << tile_bits;
    const int n = (int)min((size_t)1 << tile_bits, total - p0);
    unsigned at[kTileMoveAhead], slot[kTileMoveAhead];
    auto places = [&](int i) {
#pragma unroll
        for (int q = 0; q < kTileMoveAhead; ++q) {
            const size_t e = p0 + min(i + q * kTileMoveThreads, n - 1);
            at[q] = __builtin_nontemporal_load(tile_pos + e);
            slot[q] = __builtin_nontemporal_load(slot_of + e);
        }
    };
    places(threadIdx.x);
    for (int i = 4 * threadIdx.x; i + 4 <= n; i += 4 * kTileMoveThreads) {
        const f32x4_any q = *reinterpret_cast<const f32x4_any*>(w + p0 + i);
        *reinterpret_cast<float4*>(tile_mem + i) = make_float4(q.x, q.y, q.z, q.w);
    }
    for (int i = (n & ~3) + (int)threadIdx.x; i < n; i += kTileMoveThreads) tile_mem[i] = w[p0 + i];
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += kTileMoveThreads * kTileMoveAhead) {
#pragma unroll
        for (int q = 0; q < kTileMoveAhead; ++q)
            if (i + q * kTileMoveThreads < n) slot_w[slot[q]] = tile_mem[at[q]];
        places(i + kTileMoveThreads * kTileMoveAhead);
    }
}

__global__ __launch_bounds__(kTileMoveThreads) void weight_grads_from_slots_kernel(const float* __restrict__ gw_slots, const unsigned short* __restrict__ tile_pos,
                                                                                   const unsigned* __restrict__ slot_of, float* __restrict__ gw,
                                                                                   size_t total, int tile_bits, int tiles, int slices, size_t slots,
                                                                                   const unsigned long long* __restrict__ verdict, float* __restrict__ clear, size_t clear_count) {
    extern __shared__ __align__(16) float tile_mem[];
    const bool outdated = verdict != nullptr && *verdict == 0;
    if (outdated)
        for (size_t i = (size_t)blockIdx.x * kTileMoveThreads + threadIdx.x; i < clear_count; i += (size_t)gridDim.x * kTileMoveThreads) clear[i] = 0.f;
    if (outdated && clear == gw) return;
    const int t = xcd_unit(blockIdx.x, tiles);
    if (t < 0) return;
    const size_t p0 = (size_t)t << tile_bits;
    const int n = (int)min((size_t)1 << tile_bits, total - p0);
    for (int i = threadIdx.x; i < n; i += kTileMoveThreads * kTileMoveAhead) {
        unsigned at[kTileMoveAhead], slot[kTileMoveAhead];
        float v[kTileMoveAhead];
#pragma unroll
        for (int q = 0; q < kTileMoveAhead; ++q) {
            const size_t e = p0 + min(i + q * kTileMoveThreads, n - 1);
            at[q] = __builtin_nontemporal_load(tile_pos + e);
            slot[q] = __builtin_nontemporal_load(slot_of + e);
        }
#pragma unroll
        for (int q = 0; q < kTileMoveAhead; ++q) v[q] = gw_slots[slot[q]];
        for (int t = 1; t < slices; ++t) {
#pragma unroll
            for (int q = 0; q < kTileMoveAhead; ++q) v[q] += gw_slots[t * slots + slot[q]];
        }
#pragma unroll
        for (int q = 0; q < kTileMoveAhead; ++q) tile_mem[at[q]] = v[q];    // (behind the end: the last one once more)
    }
    __syncthreads();
    for (int i = 4 * threadIdx.x; i + 4 <= n; i += 4 * kTileMoveThreads) {
        const float4 q = *reinterpret_cast<const float4*>(tile_mem + i);
        f32x4_any o;
        o.x = q.x; o.y = q.y; o.z = q.z; o.w = q.w;
        *reinterpret_cast<f32x4_any*>(gw + p0 + i) = o;
    }
    for (int i = (n & ~3) + (int)threadIdx.x; i < n; i += kTileMoveThreads) gw[p0 + i] = tile_mem[i];
}

// gx ([N,B] or [B,N]) = sum over the segments of part[slice][segment][n][sl], in a fixed order; 32 columns x 32 samples per workgroup, one
// sum per thread (four: 22.8 us for 3,178 columns x 32 samples of 20 segments, 4.8 so)
template <bool TP>
__global__ __launch_bounds__(1024) void gather_gx_kernel(const float* __restrict__ part, float* __restrict__ gx, int N, int B, int sl,
                                                         int segments) {
    __shared__ float tile[32][33];
    const int n0 = blockIdx.x * 32, b0 = blockIdx.y * 32;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    {
        const int n = min(n0 + ty, N - 1), b = min(b0 + tx, B - 1);
        // (eight sums side by side: loads in flight, and a shorter chain of roundings)
        const float* const from = part + ((size_t)(b / sl) * segments * N + n) * sl + b % sl;
        float q[8] = {};
        for (int t = 0; t < segments; t += 8) {
            float v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = from[(size_t)min(t + e, segments - 1) * N * sl];
#pragma unroll
            for (int e = 0; e < 8; ++e) q[e] += t + e < segments ? v[e] : 0.f;
        }
        const float v = ((q[0] + q[1]) + (q[2] + q[3])) + ((q[4] + q[5]) + (q[6] + q[7]));
        if (TP) {
            if (n0 + ty < N && b0 + tx < B) gx[(size_t)n * B + b] = v;
            return;
        }
        tile[ty][tx] = v;
    }
    __syncthreads();
    const int n = n0 + tx, b = b0 + ty;
    if (n < N && b < B) gx[(size_t)b * N + n] = tile[tx][ty];
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

template <int GL, bool DOT>
int launch_walk(const WalkArgs& a, hipStream_t s) {
    const int workgroups = (a.units * a.slices + kWalkWaves - 1) / kWalkWaves;
    hipLaunchKernelGGL((walk_columns_kernel<GL, DOT>), dim3(xcd_grid(workgroups)), dim3(kWalkWaves * 64), 0, s, a);
    FFI_HIP_TRY(hipGetLastError());
    return FFI_OK;
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

// Slices that one launch walks: as many as the CUs hold wavefronts for.
int walk_slices(long long units, int slices) {
    return (int)std::max<long long>(1, std::min<long long>(slices, (long long)kWalkWaves * device_cu_count() / units));
}

int launch_backward_wide(const ffi_plan* p, const float* x, const float* w, const float* g, float* gx, float* gw, float* bias_grad, int B,
                         bool tp, hipStream_t s, const LookupCheck* check) {
    if (!p->entries || !p->slot_of || !p->tile_pos || !p->chunk_ptr) return FFI_ERR_BAD_ARGUMENT;
    // (before anything is enqueued: a refused call leaves its outputs alone)
    if ((long long)p->segments * p->groups * ((B + 31) / 32) >= (1ll << 31)) return FFI_ERR_TOO_LARGE;
    const dim3 gx_grid((unsigned)((p->N + 31) / 32), (unsigned)(((long long)B + 31) / 32));
    if (gx_grid.y > 65535u) return FFI_ERR_TOO_LARGE;
    const bool dot = gw != nullptr;
    const int sl = 256 / p->members, slices = (B + sl - 1) / sl, units = p->segments * p->groups, at_once = walk_slices(units, slices);
    const size_t slots = (size_t)p->slots, count = (size_t)p->L * p->K, gslice = (size_t)p->L * sl, part = p->segments > 1 ? (size_t)p->N * sl * p->segments : 0;
    float *ws = nullptr, *slot_w = nullptr, *gw_slots = nullptr;
    FFI_TRY(workspace_get(s, kWsPartials, (gslice + part) * slices * sizeof(float), (void**)&ws));
    FFI_TRY(workspace_get(s, kWsSlots, slots * sizeof(float), (void**)&slot_w));
    if (dot) FFI_TRY(workspace_get(s, kWsWeightParts, slots * at_once * sizeof(float), (void**)&gw_slots));
    FFI_TRY(launch_slices_f32(g, ws, p->L, B, sl, false, s));
    float* const parts = ws + gslice * slices;
    const int tiles = (int)((count + ((size_t)1 << p->tile_bits) - 1) >> p->tile_bits);
    const size_t tile_bytes = sizeof(float) << p->tile_bits;
    for (const void* k : {(const void*)weights_to_slots_kernel, (const void*)weight_grads_from_slots_kernel})
        FFI_HIP_TRY(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)tile_bytes));
    const LookupCheck with = check != nullptr ? *check : LookupCheck{};
    hipLaunchKernelGGL(weights_to_slots_kernel, dim3(xcd_grid(with.blocks) + xcd_grid(tiles)), dim3(kTileMoveThreads), tile_bytes, s, w, p->tile_pos,
                       p->slot_of, slot_w, count, p->tile_bits, tiles, with);
    FFI_HIP_TRY(hipGetLastError());
    // one launch after the other: their weight gradients add up in place
    for (int q = 0; q < slices; q += at_once) {
        const WalkArgs a{ws, x, slot_w, p->entries, p->chunk_ptr, p->chunk_count, gx, parts, gw_slots, gslice, part, slots, q, std::min(at_once, slices - q),
                         q > 0 ? 1 : 0, B, p->N, p->L, units, p->groups, p->segments, p->seg_labels, tp};
        if (p->members == 4) FFI_TRY((dot ? launch_walk<16, true>(a, s) : launch_walk<16, false>(a, s)));
        else FFI_TRY((dot ? launch_walk<8, true>(a, s) : launch_walk<8, false>(a, s)));
    }
    if (bias_grad != nullptr) {
        hipLaunchKernelGGL(column_sums_kernel, dim3((unsigned)((p->L + 63) / 64)), dim3(256), 0, s, g, bias_grad, B, p->L);
        FFI_HIP_TRY(hipGetLastError());
    }
    if (p->segments > 1) {
        const auto gather_gx = tp ? gather_gx_kernel<true> : gather_gx_kernel<false>;
        hipLaunchKernelGGL(gather_gx, gx_grid, dim3(1024), 0, s, parts, gx, p->N, B, sl, p->segments);
        FFI_HIP_TRY(hipGetLastError());
    }
    // (last: behind an outdated plan it clears what the recomputing kernel adds up in memory)
    if (dot) {
        const bool clears_gw = check != nullptr && takes_outdated_wide(p, Dims{B, p->N, p->L, p->K, tp});
        hipLaunchKernelGGL(weight_grads_from_slots_kernel, dim3(xcd_grid(tiles)), dim3(kTileMoveThreads), tile_bytes, s, gw_slots, p->tile_pos, p->slot_of,
                           gw, count, p->tile_bits, tiles, at_once, slots, check != nullptr ? check->guard + kGuardVerdict : nullptr, clears_gw ? gw : gx, clears_gw ? count : (size_t)p->N * B);
        FFI_HIP_TRY(hipGetLastError());
    }
    return FFI_OK;
}

}  // namespace ffi
