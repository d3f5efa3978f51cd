// Forward pass of the fixed-fan-in sparse layer for gfx950:
//   out[b,j] = sum_k w[j,k] * x[b, idx[j,k]]
// (semantics of tfsparse/cc/kernels/forward.cpp:9-44 in the reference).
//
//   fwd_lane32_kernel    narrow inputs (a [N][32] fp32 tile of x fits in LDS): every multiply-add
//                        takes its x operand from LDS; the LDS delivers 128 bytes per clock per CU,
//                        which bounds the kernel (4 bytes per multiply-add), so the layout is chosen
//                        to keep the gathers free of bank conflicts and the instruction count low.
//                        Scores go into a loss or a top-k as they are formed.
//   fwd_stream32_kernel  the same for plain scores; fwd_lane64_kernel by tiles of 64 samples.
// Batches of at most 16 samples and wide inputs go to the kernels of ffi_sliced.hip.
#include "ffi_internal.h"
#include "ffi_lds_tile.h"
#include "ffi_loss.h"

#include <algorithm>
#include <climits>
#include <mutex>

namespace ffi {
namespace {

// ------------------------------------------------------------------------------------------------
// Narrow-input kernel: xs[n][c] = x[b0+c, n] for the workgroup's 32 batch rows sits in LDS (one row =
// 128 bytes); thread <-> label, 32 accumulators (one per batch row of the tile), W and idx of the
// label in registers.  Workgroups that walk the same labels for different batch tiles sit on one
// XCD, so W/idx rows fetched by one are L2 hits for the others.  Each lane reads whole 128-byte rows of xs with
// the chunk order skewed by its lane id; the accumulators are brought back to natural batch order
// before the stores, which are then full 256-byte rows of out per wavefront.
// ------------------------------------------------------------------------------------------------
// A label's row of connections against a tile of W samples in LDS: the reads of a chunk of connections as one pinned stream, two in flight from its
// first to its last (left to itself the scheduler finds that order or one that waits for each read in turn, depending on code far away from
// here; 13 % slower over the whole kernel at 32 samples a tile, 19 at 64), ids and weights by quads whatever the fan-in.  LAST says what the row ends
// in: 0 whole chunks; C > 0 up to C connections behind at least one chunk, loaded as the last ones of the row, of which those that are new are
// walked; -C no whole chunk, at most C connections.  A build for each: under run-time branches the registers of the loads count as live
// throughout, and 20 to 100 of them spill.
//
// Time with the connections drained one after the other and a part-filled chunk loaded one by one -> so, us.  Plain scores at 32 x 768 x 131,072, 128 x
// 768 x 670,091 and 100 x 1,000 x 300,000: fan-in 8 12.9 -> 11.9, 156 -> 121, 37 -> 33; 13 15.5 -> 13.6, 190 -> 141, 52 -> 43; 31 32 -> 22,
// 377 -> 243, 167 -> 97; 32 20.3 -> 18.0, 193 -> 190, 81 -> 78; 40 25.2 -> 21.3, 261 -> 243, 101 -> 94; 63 44 -> 33, 588 -> 368, 239 -> 143; 64 29 -> 26,
// 339 -> 336, 143 -> 143 (those of many rounds with the pause between stores, see store_paced).  20 x 700 x 20,000, a tenth of a round of labels: 1.2 to 1.5 times as fast from fan-in 13 on.  The fused training step of 32 x
// 768 x 670,091: fan-in 8 79 -> 74, 31 263 -> 219, 32 171 -> 161, 63 529 -> 398; top-k of 200 x 300 x 100,000: 31 153 -> 95, 32 95 -> 90, 63 281 -> 142.
// ------------------------------------------------------------------------------------------------
template <int C>
struct RowChunk {
    unsigned idp[C / 2];                   // two 16-bit ids per register
    float wv[C];
    __device__ __forceinline__ unsigned id(int k) const { return (k & 1) ? (idp[k >> 1] >> 16) : (idp[k >> 1] & 0xffffu); }
    // Quad q is that from element at(q) of the row: a lane's 16 bytes are a gather of its own, which the memory system serves at any alignment.
    // The quads of a line one after the other: the lines of 16 wavefronts do not stay in the L1 between them (mixed with the weights', 9.3 million
    // requests reached the L2 at 128 samples x 670,091 labels x 32, so 6.5).
    template <class At>
    __device__ __forceinline__ void load(const int32_t* __restrict__ irow, const float* __restrict__ wrow, At&& at) {
        i32x4_unaligned v[C / 4];
        f32x4_unaligned f[C / 4];
        static_for<C / 4>([&](auto q) { v[q] = *reinterpret_cast<const i32x4_unaligned*>(irow + at(q)); __builtin_amdgcn_sched_barrier(0); });
        static_for<C / 4>([&](auto q) { f[q] = *reinterpret_cast<const f32x4_unaligned*>(wrow + at(q)); __builtin_amdgcn_sched_barrier(0); });
#pragma unroll
        for (int q = 0; q < C / 4; ++q) {
            idp[2 * q + 0] = (unsigned)v[q].x | ((unsigned)v[q].y << 16);
            idp[2 * q + 1] = (unsigned)v[q].z | ((unsigned)v[q].w << 16);
            wv[4 * q] = f[q].x; wv[4 * q + 1] = f[q].y; wv[4 * q + 2] = f[q].z; wv[4 * q + 3] = f[q].w;
        }
    }
};

// N connections from the FIRST of a chunk on: `skewbase` is the tile's address plus 16 (lane % (W / 4)).
template <int W, int FIRST, int N, int GROUP = W == 64 ? 2 : 1, int C>
__device__ __forceinline__ void walk_chunk(const RowChunk<C>& chunk, unsigned skewbase, float (&acc)[W]) {
    stream_rows<N, W / 4, 2, GROUP>([&](auto k) { return chunk.id(FIRST + k) * (unsigned)(W * 4) + skewbase; },
                                              [&](auto k, auto c, const lds_v4f& v) {
                                                  const float wv = chunk.wv[FIRST + k];
                                                  acc[4 * c + 0] = fmaf(wv, v.x, acc[4 * c + 0]);
                                                  acc[4 * c + 1] = fmaf(wv, v.y, acc[4 * c + 1]);
                                                  acc[4 * c + 2] = fmaf(wv, v.z, acc[4 * c + 2]);
                                                  acc[4 * c + 3] = fmaf(wv, v.w, acc[4 * c + 3]);
                                              });
}

template <int LAST, int GROUP = 1>
__device__ __forceinline__ void walk_row(const int32_t* __restrict__ irow, const float* __restrict__ wrow, int K, unsigned skewbase, float (&acc)[32]) {
    if constexpr (LAST < 0) {
        // (whole quads, those behind the last one read it again; then up to three connections one by one)
        RowChunk<-LAST> chunk;
        RowChunk<4> end;
        if (K >= 4) chunk.load(irow, wrow, [&](int q) { return min(4 * q, K - 4); });
        if (K & 3) {
            unsigned id[3];
#pragma unroll
            for (int e = 0; e < 3; ++e) {
                const int at = min((K & ~3) + e, K - 1);
                id[e] = (unsigned)irow[at];
                end.wv[e] = wrow[at];
            }
            end.idp[0] = id[0] | (id[1] << 16);
            end.idp[1] = id[2];
        }
        static_for<-LAST / 4>([&](auto q) {
            if (4 * q + 4 <= K) walk_chunk<32, 4 * q, 4>(chunk, skewbase, acc);
        });
        static_for<3>([&](auto e) {
            if (e < (K & 3)) walk_chunk<32, e, 1>(end, skewbase, acc);
        });
    } else {
        int k0 = 0;
        for (; k0 + 32 <= K; k0 += 32) {
            RowChunk<32> chunk;
            chunk.load(irow, wrow, [&](int q) { return k0 + 4 * q; });
            walk_chunk<32, 0, 32, GROUP>(chunk, skewbase, acc);
        }
        if constexpr (LAST == 32) {                        // (in two steps of 16: fewer registers)
            RowChunk<16> chunk;
            chunk.load(irow, wrow, [&](int q) { return k0 + 4 * q; });
            walk_chunk<32, 0, 16>(chunk, skewbase, acc);
            k0 += 16;
        }
        if constexpr (LAST > 0) {
            constexpr int kLast = LAST == 32 ? 16 : LAST;
            RowChunk<kLast> chunk;
            chunk.load(irow, wrow, [&](int q) { return K - kLast + 4 * q; });
            const int seen = kLast - (K - k0);
            static_for<kLast / 4>([&](auto q) {
                if (4 * q >= seen) walk_chunk<32, 4 * q, 4>(chunk, skewbase, acc);
                else
                    static_for<3>([&](auto i) {
                        constexpr int k = 4 * q + 1 + i;
                        if (k >= seen) walk_chunk<32, k, 1>(chunk, skewbase, acc);
                    });
            });
        }
    }
}

// What a row of K connections ends in, for walk_row: the few sizes that are worth a build.
template <class Launch>
int for_row_end(int K, Launch&& launch) {
    const int last = K % 32;
    if (K < 32) {
        if (K <= 4) return launch(std::integral_constant<int, -4>{});
        if (K <= 8) return launch(std::integral_constant<int, -8>{});
        if (K <= 16) return launch(std::integral_constant<int, -16>{});
        return launch(std::integral_constant<int, -32>{});
    }
    if (last == 0) return launch(std::integral_constant<int, 0>{});
    if (last <= 4) return launch(std::integral_constant<int, 4>{});
    if (last <= 8) return launch(std::integral_constant<int, 8>{});
    if (last <= 16) return launch(std::integral_constant<int, 16>{});
    return launch(std::integral_constant<int, 32>{});
}

// What the kernel does with a finished score s (after the bias):
//   kEpiScores       out = s
//   kEpiLossGrad     out = scale * dloss(s, 0)/ds, the loss gradient of a position that is not a listed label
//                    (listed positions are patched afterwards), and the loss(s, 0) summed per wavefront
//   kEpiLossGradAndScores  both: scores to `out`, gradients to `gout`
//   kEpiNone         nothing is stored (only the top-k candidates below are wanted)
//   kEpiLossGradSkewed  kEpiLossGrad for launches that do not store gradients that are exactly zero (nearly nothing is
//                    stored then): the accumulators stay in the lane's skewed register order (register q holds batch
//                    entry q ^ 4 (lane & 7)), the 96 conditional moves back to natural order are left out, the few stores
//                    address their rows per lane and only the mask's bits are put in order
enum FwdEpilogue { kEpiScores = 0, kEpiLossGrad = 1, kEpiLossGradAndScores = 2, kEpiNone = 3, kEpiLossGradSkewed = 4 };

constexpr int kTopkPark = 24;           // candidates per (workgroup, batch row) parked in LDS: 32 x 24 x 8 bytes = 6 KB

// Per-sample top-k without the score matrix (TOPK): tau[b] is a score that at least k labels of sample b are
// known to reach (the k-th best of a sample of the labels, found beforehand), so the k best scores are among
// those >= tau[b]; every such (label, score) is appended to the sample's candidate list, a few hundred to a
// few thousand entries out of all labels, and a small kernel selects the k best afterwards.
struct FwdTopk {
    const float* tau;     // [B]
    int* tie;             // [B] see TopkCandidates
    int* count;           // [B] candidates appended so far (may run past cap: the list is then incomplete)
    float* cand_val;      // [B][cap]
    int* cand_idx;        // [B][cap]
    int cap;
};

struct FwdLoss {
    float* gout;        // [B,L] gradients (kEpiLossGradAndScores), else unused
    double* partial;    // [gridDim.x * wavefronts per workgroup] loss sums
    unsigned* words;    // [ceil(B/32)][L] masks of the non-zero gradients to fill in, or null
    float scale;
    int kind;
    int skip_zero_stores;   // != 0: gradients that are exactly zero are not stored (needs words)
};

// Scores of one label for the 32 samples of a batch tile -> scaled loss gradients (in place), the sum of the
// losses of the first `nrows` samples, and the mask of the non-zero gradients among them.
template <int KIND>
__device__ __forceinline__ void loss_epilogue(float (&acc)[32], bool all_rows, unsigned valid_bits, float scale, float& loss,
                                              unsigned& mask) {
    // `all_rows` (workgroup-uniform): the batch tile is full; else bit q of `valid_bits` says whether register q belongs
    // to a sample of the batch (rows past it count for nothing)
    float l = 0.f;
    unsigned m = 0;
    if (all_rows) {
#pragma unroll
        for (int b = 0; b < 32; ++b) {
            float lb, gb;
            cwise_loss_and_grad(KIND, acc[b], 0.f, lb, gb);
            l += lb;
            m |= (gb != 0.f ? 1u : 0u) << b;
            acc[b] = scale * gb;
        }
    } else {
#pragma unroll
        for (int b = 0; b < 32; ++b) {
            float lb, gb;
            cwise_loss_and_grad(KIND, acc[b], 0.f, lb, gb);
            const bool in = (valid_bits >> b) & 1u;
            l += in ? lb : 0.f;
            m |= (in && gb != 0.f ? 1u : 0u) << b;
            acc[b] = scale * gb;
        }
    }
    loss = l;
    mask = m;
}

// LAST: what a row ends in, see walk_row.
template <int LAST, int EPI, bool TOPK>
__global__ __launch_bounds__(kTileThreads) void fwd_lane32_kernel(const float* __restrict__ xT,
                                                                  const int32_t* __restrict__ idx,
                                                                  const float* __restrict__ w,
                                                                  const float* __restrict__ bias,
                                                                  float* __restrict__ out, int B, int N,
                                                                  int L, int K, int nbt, int labels_per_stream,
                                                                  FwdLoss fl, FwdTopk ft) {
    extern __shared__ __align__(128) float xs[];
    __shared__ __align__(16) float tau_s[kTileBatch];
    __shared__ int local_count[kTileBatch];      // candidates parked per batch row (may run past kTopkPark)
    __shared__ int local_base[kTileBatch];
    int2* local_cand = reinterpret_cast<int2*>(xs + (size_t)N * kTileBatch);      // behind the tile (TOPK launches only)
    const int u = xcd_contiguous_block(blockIdx.x, gridDim.x);
    const int bt = u % nbt, stream = u / nbt;
    const int b0 = bt * kTileBatch;
    stage_rows32<kTileThreads, 8>(xs, xT, N, B, b0);       // (eight loads in flight per thread: the tile arrives in one round trip at 768 rows)
    if (TOPK && threadIdx.x < kTileBatch) local_count[threadIdx.x] = 0;
    if (TOPK && threadIdx.x < kTileBatch)          // (rows past the batch: a bound that few scores reach; +inf does, so the appends are bounded by nrows)
        tau_s[threadIdx.x] = b0 + (int)threadIdx.x < B ? ft.tau[b0 + threadIdx.x] : __builtin_inff();
    __syncthreads();
    const int lane = threadIdx.x & 63;
    const unsigned skewbase = (unsigned)(size_t)(__attribute__((address_space(3))) float*)xs + (unsigned)(lane & 7) * 16u;
    const int l_begin = stream * labels_per_stream;
    const int l_end = min(l_begin + labels_per_stream, L);
    // rows of out for this batch tile, reached through a scalar row offset plus the lane's label
    const int nrows = min(kTileBatch, B - b0);
    float* obase = out + (size_t)b0 * (size_t)L;
    const buffer_rsrc orsrc = make_rsrc(obase, (size_t)nrows * (size_t)L * sizeof(float));
    buffer_rsrc grsrc = orsrc;
    if (EPI == kEpiLossGradAndScores) grsrc = make_rsrc(fl.gout + (size_t)b0 * (size_t)L, (size_t)nrows * (size_t)L * sizeof(float));
    float lsum = 0.f;

    constexpr bool SKEW = EPI == kEpiLossGradSkewed;
    constexpr bool LOSS = EPI == kEpiLossGrad || EPI == kEpiLossGradAndScores || SKEW;
    static_assert(!(SKEW && TOPK), "the top-k tests need the natural order");
    // registers (in the order the epilogue sees them) that belong to samples of the batch
    const unsigned rows_valid = nrows >= kTileBatch ? 0xffffffffu : (1u << nrows) - 1u;
    const unsigned regs_valid = SKEW ? xor_permute_bits(rows_valid, lane & 7) : rows_valid;

    for (int base = l_begin; base < l_end; base += kTileThreads) {
        if (base + (int)(threadIdx.x & ~63u) >= l_end) break;     // nothing left for this wavefront
        const int j = base + (int)threadIdx.x;
        const bool valid = j < l_end;
        const int jj = valid ? j : l_end - 1;
        const int32_t* irow = idx + (size_t)jj * K;
        const float* wrow = w + (size_t)jj * K;
        float acc[32];
#pragma unroll
        for (int i = 0; i < 32; ++i) acc[i] = 0.f;
        walk_row<LAST>(irow, wrow, K, skewbase, acc);
        if (!SKEW) xor_permute_groups(acc, lane & 7);      // back to natural batch order
        if (bias != nullptr) {                             // added after the sum, as a separate bias_add would
            const float bj = bias[jj];
#pragma unroll
            for (int i = 0; i < 32; ++i) acc[i] += bj;
        }
        if (TOPK) {
            // Scores that reach their sample's threshold are rare (about one in a thousand), but a wavefront holds 2048 of
            // them: the tests are wave-uniform and hierarchical (four groups of eight batch rows, then the rows of a group
            // that has a hit), so that a row without a hit costs one compare.
            float tv[32];
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                const float4 t4 = *reinterpret_cast<const float4*>(tau_s + 4 * c);
                tv[4 * c] = t4.x; tv[4 * c + 1] = t4.y; tv[4 * c + 2] = t4.z; tv[4 * c + 3] = t4.w;
            }
#pragma unroll
            for (int grp = 0; grp < 4; ++grp) {
                bool hit = false;
#pragma unroll
                for (int b = 8 * grp; b < 8 * grp + 8; ++b) hit |= acc[b] >= tv[b];
                hit &= valid;
                if (__ballot(hit)) {
#pragma unroll
                    for (int b = 8 * grp; b < 8 * grp + 8; ++b) {
                        const bool h = valid && b < nrows && acc[b] >= tv[b];
                        if (__ballot(h)) {
                            int tie = kTopkListFull;
                            if (h) tie = ft.tie[b0 + b];
                            if (h && topk_reaches(acc[b], j, tv[b], tie)) {
                                // parked in the workgroup's LDS segment of the sample (an LDS counter answers in a few dozen
                                // clocks, a global one in microseconds); a full segment sends the entry to memory directly
                                const int lslot = atomicAdd(&local_count[b], 1);
                                if (lslot < kTopkPark) {
                                    local_cand[b * kTopkPark + lslot] = make_int2(j, __float_as_int(acc[b]));
                                } else {
                                    const int slot = topk_slot(acc[b], j, tv[b], tie, &ft.tie[b0 + b], &ft.count[(size_t)(b0 + b) * kTopkCountStep], ft.cap);
                                    if (slot < ft.cap) {
                                        ft.cand_val[(size_t)(b0 + b) * ft.cap + slot] = acc[b];
                                        ft.cand_idx[(size_t)(b0 + b) * ft.cap + slot] = j;
                                    }
                                }
                            }
                        }
                    }
                }
            }
        }
        const unsigned lane_off = (unsigned)j * 4u;
        const unsigned stride = (unsigned)L * 4u;
        if ((EPI == kEpiScores || EPI == kEpiLossGradAndScores) && valid) {
#pragma unroll
            for (int b = 0; b < 32; ++b)
                __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(int, acc[b]), orsrc, lane_off, (unsigned)b * stride, 0);
        }
        if (LOSS) {
            float l = 0.f;
            unsigned m = 0;
            const bool all_rows = nrows >= kTileBatch;
            // the loss kind is the same for the whole launch: one straight-line epilogue per kind
            if (fl.kind == FFI_LOSS_SQUARED_HINGE) loss_epilogue<FFI_LOSS_SQUARED_HINGE>(acc, all_rows, regs_valid, fl.scale, l, m);
            else if (fl.kind == FFI_LOSS_HINGE) loss_epilogue<FFI_LOSS_HINGE>(acc, all_rows, regs_valid, fl.scale, l, m);
            else loss_epilogue<FFI_LOSS_BCE>(acc, all_rows, regs_valid, fl.scale, l, m);
            if (valid) {
                lsum += l;
                if (SKEW) {
                    // register q is the gradient of batch entry q ^ r4: its row of out_grad is the lane's own
                    unsigned r4 = (unsigned)(lane & 7) << 2;
                    asm volatile("" : "+v"(r4));           // keeps the 32 row offsets from being hoisted out of the label loop
#pragma unroll
                    for (int q = 0; q < 32; ++q)
                        if ((m >> q) & 1u)
                            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(int, acc[q]), orsrc,
                                                                  lane_off + ((unsigned)q ^ r4) * stride, 0u, 0);
                    m = xor_permute_bits(m, lane & 7);
                } else if (fl.skip_zero_stores) {
#pragma unroll
                    for (int b = 0; b < 32; ++b)
                        if ((m >> b) & 1u)
                            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(int, acc[b]), EPI == kEpiLossGrad ? orsrc : grsrc, lane_off, (unsigned)b * stride, 0);
                } else {
#pragma unroll
                    for (int b = 0; b < 32; ++b)
                        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(int, acc[b]), EPI == kEpiLossGrad ? orsrc : grsrc, lane_off, (unsigned)b * stride, 0);
                }
                if (fl.words != nullptr) fl.words[(size_t)bt * L + j] = m;
            }
        }
    }
    if (TOPK) {
        // the parked candidates go to their samples' lists: one reservation per (workgroup, sample)
        __syncthreads();
        if (threadIdx.x < kTileBatch) {
            const int n = min(local_count[threadIdx.x], kTopkPark);
            local_base[threadIdx.x] = n ? atomicAdd(&ft.count[(size_t)(b0 + threadIdx.x) * kTopkCountStep], n) : 0;
        }
        __syncthreads();
        for (int e = threadIdx.x; e < kTileBatch * kTopkPark; e += kTileThreads) {
            const int b = e / kTopkPark, i = e % kTopkPark;
            if (i < min(local_count[b], kTopkPark)) {
                const int2 c = local_cand[e];
                const int slot = local_base[b] + i;
                if (slot < ft.cap) {
                    ft.cand_val[(size_t)(b0 + b) * ft.cap + slot] = __int_as_float(c.y);
                    ft.cand_idx[(size_t)(b0 + b) * ft.cap + slot] = c.x;
                }
            }
        }
    }
    if (LOSS) {
        const double t = wave_sum((double)lsum);
        if (lane == 0) fl.partial[(size_t)blockIdx.x * (kTileThreads / 64) + (threadIdx.x >> 6)] = t;
    }
}

// A lane's scores of W samples, one row of out each, through a resource of those rows.  The rows' offsets are formed one after the other (the caller
// hides the stride from the compiler: hoisted, all of them do not fit the scalar registers and come back from vector lanes).
// PAUSE: clocks between two stores.  Back to back, a wavefront's stores fill the CU's path to memory, and the wavefronts that ask for ids and
// weights wait behind them: 16 clocks pay where many rounds of labels overlap, and cost their own time and more in a launch of few.  Forward pass of
// plain scores with what the caches hold cold, back to back and with 16 clocks: 128 x 768 x 670,091 x 32, ten rounds, 212 and 200 us (in the
// passes of a benchmark step 180 and 172), x 8 126 and 115, x 31 260 and 251; 512 x 1,024 x 140,000 x 32, nine rounds, 163 and 143; 128 x 768 x 300,000 x 32, under five,
// 91 and 92, warm 82 and 88; 32 x 768 x 670,091 x 32, under three, 99 and 99, warm 56 and 57.  (Tiles of 64: 256 x 512 x 501,070 x 64 370 and
// 384, 192 x 300 x 66,001 x 32 35.5 and 36.2, but 192 x 600 x 300,000 x 16 97 and 88; without.)
template <int PAUSE, int W>
__device__ __forceinline__ void store_paced(const float (&acc)[W], const buffer_rsrc& orsrc, unsigned lane_off, unsigned stride) {
    unsigned off = 0;
#pragma unroll
    for (int b = 0; b < W; ++b) {
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(int, acc[b]), orsrc, lane_off, off, 0);
        if constexpr (PAUSE > 0) asm volatile("s_nop %0" ::"n"(PAUSE - 1));
        off += stride;
    }
}
inline __host__ __device__ bool many_rounds(int labels_per_stream) { return labels_per_stream >= 8 * kTileThreads; }

// The kernel above for plain scores, which leave as soon as they are in order: fewer registers, and a build for every way a row ends.
template <int LAST, int GROUP>
__global__ __launch_bounds__(kTileThreads) void fwd_stream32_kernel(const float* __restrict__ xT, const int32_t* __restrict__ idx,
                                                                    const float* __restrict__ w, const float* __restrict__ bias,
                                                                    float* __restrict__ out, int B, int N, int L, int K, int nbt, int labels_per_stream) {
    extern __shared__ __align__(128) float xs[];
    const int u = xcd_contiguous_block(blockIdx.x, gridDim.x);
    const int bt = u % nbt, stream = u / nbt;
    const int b0 = bt * kTileBatch;
    const int lane = threadIdx.x & 63;
    const int l_begin = stream * labels_per_stream, l_end = min(l_begin + labels_per_stream, L);
    stage_rows32<kTileThreads, 8>(xs, xT, N, B, b0);
    __syncthreads();
    const unsigned skewbase = (unsigned)(size_t)(__attribute__((address_space(3))) float*)xs + (unsigned)(lane & 7) * 16u;
    // rows of out for this batch tile, reached through a scalar row offset plus the lane's label; rows past the batch
    // lie beyond the resource's size and their stores are dropped
    const buffer_rsrc orsrc = make_rsrc(out + (size_t)b0 * (size_t)L, (size_t)min(kTileBatch, B - b0) * (size_t)L * sizeof(float));
    for (int base = l_begin; base + (int)(threadIdx.x & ~63u) < l_end; base += kTileThreads) {
        const int j = base + (int)threadIdx.x;
        const bool valid = j < l_end;
        const int32_t* irow = idx + (size_t)min(j, l_end - 1) * K;
        const float* wrow = w + (size_t)min(j, l_end - 1) * K;
        float acc[32];
#pragma unroll
        for (int i = 0; i < 32; ++i) acc[i] = 0.f;
        walk_row<LAST, GROUP>(irow, wrow, K, skewbase, acc);
        xor_permute_groups(acc, lane & 7);                 // back to natural batch order
        if (bias != nullptr) {                             // added after the sum, as a separate bias_add would
            const float bj = bias[min(j, l_end - 1)];
#pragma unroll
            for (int i = 0; i < 32; ++i) acc[i] += bj;
        }
        if (valid) {
            unsigned stride = (unsigned)L * 4u;
            asm volatile("" : "+s"(stride));               // (see store_paced)
            if (many_rounds(labels_per_stream)) store_paced<16>(acc, orsrc, (unsigned)j * 4u, stride);
            else store_paced<2>(acc, orsrc, (unsigned)j * 4u, stride);
        }
    }
}

// ------------------------------------------------------------------------------------------------
// The same kernel over batch tiles of 64 for inputs narrow enough that an [N][64] fp32 tile of x fits in LDS
// (N <= kLane64MaxN): a row is 256 bytes and covers all 64 banks, so with the chunk order skewed by (lane & 15)
// the 32 lanes the LDS serves together hit every bank exactly twice whatever rows they read (128-byte rows sit in
// one half of the banks and the random parities of the rows cost about 1.7x), and W/idx are read once per 64
// batch rows instead of once per 32.  Plain scores only.
//
// Bound by the issue of its instructions (81 to 82 for a connection's 64 multiply-adds: 289 us of them at 256 samples x 512 columns x
// 501,070 labels x 64) and by the wait for a read wherever none is in flight.  Each read waited for in turn, as the compiler ordered it,
// that layer took 394 to 435 us; a chunk's 256 reads as one pinned stream, two in flight, issued and used two at a time, 319 to 343
// (one at a time 328 to 338, four in flight 318 to 333, eight spill).
// ------------------------------------------------------------------------------------------------
constexpr int kLane64Batch = 64;
constexpr int kLane64MaxN = 608;        // 152 KB of LDS

template <int THREADS>
__device__ __forceinline__ void stage_rows64(float* __restrict__ xs, const float* __restrict__ src, int rows, int ld, int c0) {
    const bool vec = (ld % 4 == 0) && (c0 + kLane64Batch <= ld) && (((uintptr_t)src & 15) == 0);
    if (vec) {
        // thread -> (row, 16-byte chunk): 16 threads per row, all of a thread's loads before its first LDS write
        constexpr int kRowsPerIter = THREADS / 16;
        constexpr int kInFlight = 4;
        const int q = threadIdx.x & 15;
        const float* p = src + c0 + 4 * q;
        for (int r0 = threadIdx.x >> 4; r0 < rows; r0 += kRowsPerIter * kInFlight) {
            float4 v[kInFlight];
#pragma unroll
            for (int i = 0; i < kInFlight; ++i) {
                const int r = r0 + i * kRowsPerIter;
                v[i] = make_float4(0.f, 0.f, 0.f, 0.f);
                if (r < rows) v[i] = *reinterpret_cast<const float4*>(p + (size_t)r * ld);
            }
#pragma unroll
            for (int i = 0; i < kInFlight; ++i) {
                const int r = r0 + i * kRowsPerIter;
                if (r < rows) *reinterpret_cast<float4*>(xs + r * kLane64Batch + 4 * q) = v[i];
            }
        }
    } else {
        const int c = threadIdx.x & 63;
        const bool in = c0 + c < ld;
        const float* p = src + c0 + c;
        for (int r = threadIdx.x >> 6; r < rows; r += THREADS / 64)
            xs[r * kLane64Batch + c] = in ? p[(size_t)r * ld] : 0.f;
    }
}

// v[4c+i] <-> v[4(c ^ r)+i] for r in [0,16): its own inverse; four stages of conditional swaps.
__device__ __forceinline__ void xor_permute_groups64(float (&v)[64], int r) {
    const bool b8 = r & 8, b4 = r & 4, b2 = r & 2, b1 = r & 1;
#pragma unroll
    for (int e = 0; e < 64; ++e)
        if (!(e & 32)) cond_swap(b8, v[e], v[e + 32]);
#pragma unroll
    for (int e = 0; e < 64; ++e)
        if (!(e & 16)) cond_swap(b4, v[e], v[e + 16]);
#pragma unroll
    for (int e = 0; e < 64; ++e)
        if (!(e & 8)) cond_swap(b2, v[e], v[e + 8]);
#pragma unroll
    for (int e = 0; e < 64; ++e)
        if (!(e & 4)) cond_swap(b1, v[e], v[e + 4]);
}

__global__ __launch_bounds__(kTileThreads) void fwd_lane64_kernel(const float* __restrict__ xT, const int32_t* __restrict__ idx,
                                                                  const float* __restrict__ w, const float* __restrict__ bias,
                                                                  float* __restrict__ out, int B, int N, int L, int K, int nbt,
                                                                  int labels_per_stream) {
    extern __shared__ __align__(256) float xs[];
    const int u = xcd_contiguous_block(blockIdx.x, gridDim.x);
    const int bt = u % nbt, stream = u / nbt;
    const int b0 = bt * kLane64Batch;
    stage_rows64<kTileThreads>(xs, xT, N, B, b0);
    __syncthreads();
    const int lane = threadIdx.x & 63;
    const unsigned skewbase = (unsigned)(size_t)(__attribute__((address_space(3))) float*)xs + (unsigned)(lane & 15) * 16u;
    const int l_begin = stream * labels_per_stream;
    const int l_end = min(l_begin + labels_per_stream, L);
    // rows of out for this batch tile, reached through a scalar row offset plus the lane's label; rows past the batch
    // lie beyond the resource's size and their stores are dropped
    const int nrows = min(kLane64Batch, B - b0);
    const buffer_rsrc orsrc = make_rsrc(out + (size_t)b0 * (size_t)L, (size_t)nrows * (size_t)L * sizeof(float));
    for (int base = l_begin; base < l_end; base += kTileThreads) {
        if (base + (int)(threadIdx.x & ~63u) >= l_end) break;     // nothing left for this wavefront
        const int j = base + (int)threadIdx.x;
        const bool valid = j < l_end;
        const int jj = valid ? j : l_end - 1;
        const int32_t* irow = idx + (size_t)jj * K;
        const float* wrow = w + (size_t)jj * K;
        float acc[64];
#pragma unroll
        for (int i = 0; i < 64; ++i) acc[i] = 0.f;
        int k0 = 0;
        for (; k0 + 16 <= K; k0 += 16) {
            RowChunk<16> chunk;
            chunk.load(irow, wrow, [&](int q) { return k0 + 4 * q; });
            walk_chunk<64, 0, 16>(chunk, skewbase, acc);
        }
        if (k0 < K) {
            // (what is no whole chunk: the connections past the row's end load its last one again and are skipped)
            RowChunk<16> chunk;
#pragma unroll
            for (int q = 0; q < 8; ++q) chunk.idp[q] = (unsigned)irow[min(k0 + 2 * q, K - 1)] | ((unsigned)irow[min(k0 + 2 * q + 1, K - 1)] << 16);
#pragma unroll
            for (int k = 0; k < 16; ++k) chunk.wv[k] = wrow[min(k0 + k, K - 1)];
            const int kn = K - k0;
            static_for<16>([&](auto k) {
                if (k < kn) walk_chunk<64, k, 1>(chunk, skewbase, acc);
            });
        }
        xor_permute_groups64(acc, lane & 15);              // back to natural batch order
        if (bias != nullptr) {                             // added after the sum, as a separate bias_add would
            const float bj = bias[jj];
#pragma unroll
            for (int i = 0; i < 64; ++i) acc[i] += bj;
        }
        if (valid) {
            const unsigned lane_off = (unsigned)j * 4u;
            unsigned stride = (unsigned)L * 4u;
            asm volatile("" : "+s"(stride));
            store_paced<0>(acc, orsrc, lane_off, stride);
        }
    }
}

int launch_lane64(const float* xT, const int32_t* idx, const float* w, const float* bias, float* out, const Dims& d, hipStream_t s) {
    const int cus = device_cu_count();
    const int nbt = (d.B + kLane64Batch - 1) / kLane64Batch;
    int streams = std::max(1, cus / nbt);
    const int per_stream = (d.L + streams - 1) / streams;
    streams = (d.L + per_stream - 1) / per_stream;
    const size_t lds = (size_t)d.N * kLane64Batch * sizeof(float);
    FFI_HIP_TRY(hipFuncSetAttribute((const void*)fwd_lane64_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(fwd_lane64_kernel, dim3(streams * nbt), dim3(kTileThreads), lds, s, xT, idx, w, bias, out, d.B, d.N,
                       d.L, d.K, nbt, per_stream);
    FFI_HIP_TRY(hipGetLastError());
    return FFI_OK;
}

// (64 rows of out of a batch tile are reached through 32-bit byte offsets)
// Where the tile of 64 samples fits, and where it pays: it walks twice the multiply-adds per address and reads ids and weights half as often,
// and leaves half as many workgroups.  Time of the tiles of 32 over its own, 128 and 600 columns x 200,000 labels and 400 x 600,000: whole chunks of 16
// from 128 samples and fan-in 32 on 1.07...1.42, from 192 samples 1.10...1.28 at fan-in 16; fan-ins 33 and 100 1.07...1.36 from 192
// samples on, fan-in 40 (eight connections behind the last chunk, loaded one by one) 0.75...1.0; 160 samples, the last tile half empty, 0.89...1.09 at
// fan-in 32 and 1.03...1.17 from 48 on; fan-ins up to 13 0.6...1.0.  20,000 labels, 80 to 470 a workgroup: 0.4...1.0 throughout.
bool lane64_fits(const Dims& d) {
    if (d.N > kLane64MaxN || d.B <= kTileBatch || d.L >= (1 << 24) || g_options.fwd_lane64 < 0) return false;
    const int tiles = (d.B + kLane64Batch - 1) / kLane64Batch, rest = d.B % kLane64Batch, behind = d.K % 16;
    if (behind > 4 || (behind > 0 && d.K < 32) || (long long)d.L * tiles < 768ll * device_cu_count()) return false;
    if (rest != 0 && rest <= kTileBatch) return d.K >= 48 && d.B >= 2 * kLane64Batch;
    return (d.K >= 16 && d.B >= 192) || (d.K >= 32 && d.B >= 2 * kLane64Batch) || (d.K >= 48 && behind == 0);
}

}  // namespace

namespace {

constexpr int kTopkSampleBits = 12, kTopkSample = 1 << kTopkSampleBits;      // labels whose scores set the per-sample thresholds

// scores of S labels, evenly spaced, for all samples: sample_scores[b][i] (the thresholds' raw material)
__global__ __launch_bounds__(256) void fwd_sample_kernel(const float* __restrict__ xT, const int32_t* __restrict__ idx,
                                                         const float* __restrict__ w, const float* __restrict__ bias, int B, int N,
                                                         int K, int S, TopkSampleLabels labels, float* __restrict__ sample_scores) {
    const int i = blockIdx.x;
    const int j = (int)(((long long)i * labels.num) >> labels.shift);
    const int32_t* irow = idx + (size_t)j * K;
    const float* wrow = w + (size_t)j * K;
    for (int b = threadIdx.x; b < B; b += 256) {
        float acc = 0.f, mag = 0.f;
        for (int k = 0; k < K; ++k) {
            const unsigned id = (unsigned)irow[k];
            const float xv = xT[(size_t)(id < (unsigned)N ? id : 0u) * B + b];
            acc = fmaf(wrow[k], xv, acc);
            mag = fmaf(fabsf(wrow[k]), fabsf(xv), mag);
        }
        if (bias != nullptr) { acc += bias[j]; mag += fabsf(bias[j]); }
        // The main kernel sums the same products in another order; its score of this label differs from `acc` by at
        // most a few rounding errors of the largest partial sum (K * 2^-24 * mag).  The threshold must not exceed the
        // main kernel's value, so the sampled score is lowered by a bound on that difference.
        sample_scores[(size_t)b * S + i] = acc - (float)(K + 2) * 1.2e-7f * mag;
    }
}

template <int LAST, int EPI, bool TOPK>
int launch_lane32(const float* xT, const int32_t* idx, const float* w, const float* bias, float* out, const Dims& d, int nbt,
                  int per_stream, int blocks, size_t lds, const FwdLoss& fl, const FwdTopk& ft, hipStream_t s) {
    FFI_HIP_TRY(hipFuncSetAttribute((const void*)fwd_lane32_kernel<LAST, EPI, TOPK>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL((fwd_lane32_kernel<LAST, EPI, TOPK>), dim3(blocks), dim3(kTileThreads), lds, s, xT, idx, w, bias, out, d.B, d.N,
                       d.L, d.K, nbt, per_stream, fl, ft);
    FFI_HIP_TRY(hipGetLastError());
    return FFI_OK;
}

template <int LAST, int GROUP = 1>
int launch_stream32(const float* xT, const int32_t* idx, const float* w, const float* bias, float* out, const Dims& d, int nbt, int per_stream, int blocks,
                    size_t lds, hipStream_t s) {
    FFI_HIP_TRY(hipFuncSetAttribute((const void*)fwd_stream32_kernel<LAST, GROUP>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL((fwd_stream32_kernel<LAST, GROUP>), dim3(blocks), dim3(kTileThreads), lds, s, xT, idx, w, bias, out, d.B, d.N, d.L, d.K, nbt, per_stream);
    FFI_HIP_TRY(hipGetLastError());
    return FFI_OK;
}

template <int EPI>
int launch_lane32_any(bool topk, const float* xT, const int32_t* idx, const float* w, const float* bias, float* out,
                      const Dims& d, int nbt, int per_stream, int blocks, size_t lds, const FwdLoss& fl, const FwdTopk& ft,
                      hipStream_t s) {
    auto go = [&](auto top) -> int {
        constexpr bool T = decltype(top)::value;
        if (d.K < 32) return launch_lane32<-32, EPI, T>(xT, idx, w, bias, out, d, nbt, per_stream, blocks, lds, fl, ft, s);
        if (d.K % 32 == 0) return launch_lane32<0, EPI, T>(xT, idx, w, bias, out, d, nbt, per_stream, blocks, lds, fl, ft, s);
        if (d.K % 32 <= 8) return launch_lane32<8, EPI, T>(xT, idx, w, bias, out, d, nbt, per_stream, blocks, lds, fl, ft, s);
        if (d.K % 32 <= 16) return launch_lane32<16, EPI, T>(xT, idx, w, bias, out, d, nbt, per_stream, blocks, lds, fl, ft, s);
        return launch_lane32<32, EPI, T>(xT, idx, w, bias, out, d, nbt, per_stream, blocks, lds, fl, ft, s);
    };
    if constexpr (EPI != kEpiLossGradSkewed) {              // (that epilogue has no top-k form)
        if (topk) return go(std::true_type{});
    }
    if constexpr (EPI != kEpiNone && EPI != kEpiScores) return go(std::false_type{});      // (plain scores: fwd_stream32_kernel)
    else return FFI_ERR_BAD_ARGUMENT;
}

// Narrow-input forward pass with the given epilogue; `la` is needed for the loss epilogues only, `tk` (may be
// null) asks for the per-sample top-k without the score matrix.
// `xt_scratch` (may be null): room for N * B floats that takes the place of the library workspace for the
// batch-major copy of [B,N] features.
int forward_tiles(const float* x, const int32_t* idx, const float* w, const float* bias, float* out, float* gout, int epi,
                  const LossArgs* la, const TopkArgs* tk, const Dims& d, hipStream_t s, float* xt_scratch = nullptr) {
    const float* xT = x;
    if (!d.tp) {
        float* ws = xt_scratch;
        if (ws == nullptr) FFI_TRY(workspace_get(s, kWsFeaturesT, (size_t)d.N * d.B * sizeof(float), (void**)&ws));
        FFI_TRY(launch_transpose(x, ws, d.B, d.N, s));   // [B,N] -> [N,B]
        xT = ws;
    }
    const size_t lds = tile_lds_bytes(d.N);
    if (epi == kEpiScores && tk == nullptr && lane64_fits(d)) return launch_lane64(xT, idx, w, bias, out, d, s);
    const int cus = device_cu_count();
    const int nbt = (d.B + kTileBatch - 1) / kTileBatch;
    int streams = std::max(1, cus / nbt);
    const int per_stream = (d.L + streams - 1) / streams;
    streams = (d.L + per_stream - 1) / per_stream;
    const int blocks = streams * nbt;
    FwdLoss fl{gout, nullptr, nullptr, 0.f, 0, 0};
    FwdTopk ft{};
    const bool topk = tk != nullptr;
    TopkCandidates tc{};
    size_t lds_topk = lds;
    if (topk) {
        // thresholds: the k-th best score of every sample among kTopkSample evenly spaced labels
        const int S = std::min(kTopkSample, d.L);
        const TopkSampleLabels labels = d.L > S ? TopkSampleLabels{d.L, kTopkSampleBits} : TopkSampleLabels{1, 0};
        void* ws = nullptr;
        FFI_TRY(workspace_get(s, kWsTopk, topk_candidate_bytes(d.B, S), &ws));
        tc = topk_candidates_at(ws, d.B, S);
        hipLaunchKernelGGL(fwd_sample_kernel, dim3(S), dim3(256), 0, s, xT, idx, w, bias, d.B, d.N, d.K, S, labels, tc.sample);
        FFI_HIP_TRY(hipGetLastError());
        FFI_TRY(launch_topk_threshold(tc.sample, (size_t)S, 1, S, labels, tk->k, tc, d.B, s));
        // LDS behind the tile of x holds the workgroup's candidates until the end of the kernel
        ft = FwdTopk{tc.tau, tc.tie, tc.count, tc.val, tc.idx, kTopkCap};
        lds_topk = lds + (size_t)kTileBatch * kTopkPark * sizeof(int2);
    }
    // (whole chunks, and labels for many rounds: reads and their uses two at a time.  The kernel with cold caches, two and one at a time: 128 x 768 x 670,091 x 32, ten
    // rounds, 200 and 205 us, 512 x 1,024 x 140,000 x 32, nine, 143 and 151; 64 x 768 x 900,000 x 32, seven, 154 and 152, 64 x 768 x 670,091 x 32, five, 125
    // and 122; 32 x 768 x 131,072 x 32, half a round, 26 and 25)
    if (epi == kEpiScores && !topk && d.K % 32 == 0 && many_rounds(per_stream))
        return launch_stream32<0, 2>(xT, idx, w, bias, out, d, nbt, per_stream, blocks, lds, s);
    if (epi == kEpiScores && !topk)
        return for_row_end(d.K, [&](auto last) { return launch_stream32<last>(xT, idx, w, bias, out, d, nbt, per_stream, blocks, lds, s); });
    int npartial = 0;
    double* corr = nullptr;
    if (epi == kEpiLossGrad || epi == kEpiLossGradAndScores) {
        npartial = blocks * (kTileThreads / 64);
        FFI_TRY(loss_partial_buffer(s, npartial, la->nnz, &fl.partial, &corr, nullptr));
        fl.scale = la->scale;
        fl.kind = la->kind;
        fl.words = la->nz_words;
        fl.skip_zero_stores = la->skip_zero_stores ? 1 : 0;
    }
    if (epi == kEpiScores) FFI_TRY(launch_lane32_any<kEpiScores>(topk, xT, idx, w, bias, out, d, nbt, per_stream, blocks, lds_topk, fl, ft, s));
    else if (epi == kEpiLossGrad && !topk && fl.skip_zero_stores)
        FFI_TRY(launch_lane32_any<kEpiLossGradSkewed>(false, xT, idx, w, bias, out, d, nbt, per_stream, blocks, lds_topk, fl, ft, s));
    else if (epi == kEpiLossGrad) FFI_TRY(launch_lane32_any<kEpiLossGrad>(topk, xT, idx, w, bias, out, d, nbt, per_stream, blocks, lds_topk, fl, ft, s));
    else if (epi == kEpiLossGradAndScores) FFI_TRY(launch_lane32_any<kEpiLossGradAndScores>(topk, xT, idx, w, bias, out, d, nbt, per_stream, blocks, lds_topk, fl, ft, s));
    else FFI_TRY(launch_lane32_any<kEpiNone>(topk, xT, idx, w, bias, out, d, nbt, per_stream, blocks, lds_topk, fl, ft, s));
    if (topk) {
        // (a sample with more candidates than its list holds: its row once more, from the score matrix if there is one)
        TopkRowSource src;
        if (epi == kEpiScores || epi == kEpiLossGradAndScores) src.scores = out;
        src.x = xT; src.tp = true; src.idx = idx; src.w = w; src.bias = bias; src.N = d.N; src.L = d.L; src.K = d.K;
        FFI_TRY(launch_topk_select(tc, d.B, *tk, src, s));
    }
    if (epi != kEpiLossGrad && epi != kEpiLossGradAndScores) return FFI_OK;
    // the listed label positions: from the score matrix when it was written, else recomputed from x ([N,B] here)
    Dims dt = d;
    dt.tp = true;
    float* g = epi == kEpiLossGrad ? out : gout;
    return launch_loss_positives(*la, nullptr, epi == kEpiLossGrad ? nullptr : out, xT, idx, w, bias, g, dt, fl.partial, npartial,
                                 corr, s);
}

}  // namespace

int launch_forward(const float* x, const int32_t* idx, const float* w, const float* bias, float* out, const Dims& d,
                   hipStream_t s) {
    if (takes_small_forward(d)) return launch_forward_small(x, idx, w, bias, out, d, s);
    if (takes_dense_forward(d)) return launch_forward_dense(x, idx, w, bias, out, d, s);
    // (the kernel reaches the 32 rows of out of a batch tile through 32-bit byte offsets)
    if (tile_path_fits(d.N) && d.L < (1 << 25) && !few_samples(d)) return forward_tiles(x, idx, w, bias, out, nullptr, kEpiScores, nullptr, nullptr, d, s);
    return launch_forward_wide(x, idx, w, bias, out, d, s);
}

int launch_forward_loss(const float* x, const int32_t* idx, const float* w, const float* bias, const LossArgs& la,
                        float* scores, float* g, const TopkArgs* tk, const Dims& d, hipStream_t s) {
    if (tile_path_fits(d.N) && d.L < (1 << 25)) {
        if (scores == nullptr) return forward_tiles(x, idx, w, bias, g, nullptr, kEpiLossGrad, &la, tk, d, s);
        return forward_tiles(x, idx, w, bias, scores, g, kEpiLossGradAndScores, &la, tk, d, s);
    }
    // wide inputs: scores by the wide kernel (into g itself when the caller wants no scores), top-k from them, then
    // the loss gradient as a pass of its own
    float* sc = scores ? scores : g;
    FFI_TRY(launch_forward_wide(x, idx, w, bias, sc, d, s));
    if (tk != nullptr) FFI_TRY(launch_topk_f32(sc, d.B, d.L, tk->k, tk->values, tk->indices, s));
    return launch_loss_grad(la, sc, g, d.B, d.L, s);
}

int launch_forward_topk(const float* x, const int32_t* idx, const float* w, const float* bias, float* scores, const TopkArgs& tk,
                        const Dims& d, hipStream_t s) {
    if (tile_path_fits(d.N) && d.L < (1 << 25) && (scores != nullptr || !few_samples(d)))
        return forward_tiles(x, idx, w, bias, scores, nullptr, scores ? kEpiScores : kEpiNone, nullptr, &tk, d, s);
    // wide inputs: candidates as the scores are formed, or the score matrix the caller wants, then its top-k
    if (scores == nullptr) return launch_forward_topk_sliced(x, idx, w, bias, false, tk, d, s);
    FFI_TRY(launch_forward_wide(x, idx, w, bias, scores, d, s));
    return launch_topk_f32(scores, d.B, d.L, tk.k, tk.values, tk.indices, s);
}

// ---- forward pass for callers that cannot allocate ------------------------------------------------
// The only device memory the narrow forward pass needs beyond its inputs and outputs is the [N][B]
// copy of [B,N] features.  Here it lives in a fixed array inside the library's code object (one copy
// per GPU, held until the process ends) instead of a workspace from hipMalloc.
namespace {

constexpr size_t kNoAllocFloats = (size_t)1 << 20;             // 4 MiB: batch * num_features may not exceed this
static __device__ __align__(256) float scratch[kNoAllocFloats];

constexpr int kNoAllocMaxDevices = 64;
std::mutex g_scratch_mutex;
float* g_scratch_ptr[kNoAllocMaxDevices] = {nullptr};           // device address of `scratch` on each GPU

// The address of this GPU's copy of `scratch` (looked up once per device, with that device current).
int scratch_address(float** out) {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess) { (void)hipGetLastError(); return FFI_ERR_NO_DEVICE; }
    if (dev < 0 || dev >= kNoAllocMaxDevices) return FFI_ERR_NO_DEVICE;
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (g_scratch_ptr[dev] == nullptr) {
        float* ptr = nullptr;
        FFI_HIP_TRY(hipGetSymbolAddress((void**)&ptr, HIP_SYMBOL(scratch)));
        if (ptr == nullptr) return FFI_ERR_HIP;
        g_scratch_ptr[dev] = ptr;
    }
    *out = g_scratch_ptr[dev];
    return FFI_OK;
}

}  // namespace
}  // namespace ffi

extern "C" int ffi_forward_noalloc_f32(const float* features, const int32_t* lookup, const float* weights, float* result,
                                       int64_t batch, int64_t num_features, int64_t num_units, int64_t fan_in, int transposed,
                                       ffi_stream_t stream) {
    using namespace ffi;
    StreamCall call_lock((hipStream_t)stream);
    if (!features || !lookup || !weights || !result) return FFI_ERR_NULL_POINTER;
    if (batch <= 0 || num_features <= 0 || num_units <= 0 || fan_in <= 0) return FFI_ERR_BAD_SHAPE;
    if (batch >= INT32_MAX || num_features >= INT32_MAX || num_units >= INT32_MAX || fan_in >= INT32_MAX) return FFI_ERR_TOO_LARGE;
    if (num_units * fan_in >= INT32_MAX) return FFI_ERR_TOO_LARGE;
    // only the shapes of the narrow kernel, which needs nothing but the fixed array
    if (!tile_path_fits((int)num_features) || num_units >= (1 << 25)) return FFI_ERR_TOO_LARGE;
    if ((uint64_t)batch * (uint64_t)num_features > kNoAllocFloats) return FFI_ERR_TOO_LARGE;
    const Dims d{(int)batch, (int)num_features, (int)num_units, (int)fan_in, transposed != 0};
    if (takes_small_forward(d)) return launch_forward_small(features, lookup, weights, nullptr, result, d, (hipStream_t)stream);
    float* xt = nullptr;
    if (!d.tp) FFI_TRY(scratch_address(&xt));
    return forward_tiles(features, lookup, weights, nullptr, result, nullptr, kEpiScores, nullptr, nullptr, d, (hipStream_t)stream, xt);
}
