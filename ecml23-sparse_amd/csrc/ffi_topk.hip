// Per-sample top-k (k <= 8): of a score matrix, and the two ends of the forward passes that keep candidates instead of
// scores.  No counterpart in the reference, which has tf.nn.top_k inside a Keras metric (sparse/metrics.py:19); equal scores
// go to the lower label, as there.
//
// Long rows take a threshold: the k best of the maxima of disjoint groups of a sample of the labels are scores of k labels,
// so the least of them is a bound that the k best scores of the row reach.  One pass collects the few scores at or above it
// (about k L / S of L labels for a sample of S), and the k best of those are the answer.  Exact.
// Best and least are those of the order the answer is in, score and then label: of the labels whose scores equal the bound,
// only those up to the bound's own label are collected, so a row of equal scores (a sample without features) is no longer a
// list than any other.  (By score alone such a row was answered from the whole layer: one of 512 in bf16, 100,000 x 670,091 x 64,
// took 70 ms in place of 2.7.)  What can still outgrow a list -- thousands of labels above all that the sample holds -- is
// answered from the whole row by many workgroups together.
#include "ffi_internal.h"
#include "ffi_loss.h"

#include <algorithm>
#include <type_traits>

namespace ffi {
namespace {

constexpr int kTopMax = 8;                 // list length kept per thread (k <= 8)
constexpr int kNoId = 0x7fffffff;

// (score descending, label ascending) order
__device__ __forceinline__ bool better(float v, int id, float w, int wid) { return v > w || (v == w && id < wid); }

struct TopList {
    float v[kTopMax];
    int id[kTopMax];
    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int s = 0; s < kTopMax; ++s) { v[s] = -__builtin_inff(); id[s] = kNoId; }
    }
    __device__ __forceinline__ void offer(float nv, int nid) {
        if (!better(nv, nid, v[kTopMax - 1], id[kTopMax - 1])) return;
#pragma unroll
        for (int s = kTopMax - 1; s >= 0; --s) {
            const bool keep = !better(nv, nid, v[s], id[s]);                       // element s stays where it is
            const bool prev_keep = s == 0 || !better(nv, nid, v[s - (s > 0)], id[s - (s > 0)]);
            const float ov = s > 0 ? v[s - (s > 0)] : nv;
            const int oi = s > 0 ? id[s - (s > 0)] : nid;
            v[s] = keep ? v[s] : (prev_keep ? nv : ov);
            id[s] = keep ? id[s] : (prev_keep ? nid : oi);
        }
    }
    __device__ __forceinline__ void pop() {
#pragma unroll
        for (int t = 0; t + 1 < kTopMax; ++t) { v[t] = v[t + 1]; id[t] = id[t + 1]; }
        v[kTopMax - 1] = -__builtin_inff();
        id[kTopMax - 1] = kNoId;
    }
};

// The largest of the lanes' values (none of them NaN), and the smallest of their ids, in every lane: over sixteen lanes by DPP,
// whose steps cost what an addition costs, then over the four rows.
template <int CTRL> __device__ __forceinline__ int dpp_of(int v) { return __builtin_amdgcn_update_dpp(v, v, CTRL, 0xf, 0xf, false); }
template <int CTRL> __device__ __forceinline__ float dpp_of(float v) { return __int_as_float(dpp_of<CTRL>(__float_as_int(v))); }
__device__ __forceinline__ float wave_largest(float v) {
    v = fmaxf(v, dpp_of<0xb1>(v));          // lane ^ 1
    v = fmaxf(v, dpp_of<0x4e>(v));          // lane ^ 2
    v = fmaxf(v, dpp_of<0x141>(v));         // 7 - lane within eight
    v = fmaxf(v, dpp_of<0x140>(v));         // 15 - lane within sixteen
    const int i = __float_as_int(v);
    return fmaxf(fmaxf(__int_as_float(__builtin_amdgcn_readlane(i, 0)), __int_as_float(__builtin_amdgcn_readlane(i, 16))),
                 fmaxf(__int_as_float(__builtin_amdgcn_readlane(i, 32)), __int_as_float(__builtin_amdgcn_readlane(i, 48))));
}
__device__ __forceinline__ int wave_smallest(int v) {
    v = min(v, dpp_of<0xb1>(v));
    v = min(v, dpp_of<0x4e>(v));
    v = min(v, dpp_of<0x141>(v));
    v = min(v, dpp_of<0x140>(v));
    return min(min(__builtin_amdgcn_readlane(v, 0), __builtin_amdgcn_readlane(v, 16)),
               min(__builtin_amdgcn_readlane(v, 32), __builtin_amdgcn_readlane(v, 48)));
}

// The 64 lanes hold sorted lists; kTopMax rounds in which the best head is taken by lane `round` and popped by its owner.
// Afterwards lane s < 8 holds the s-th best in out_*.  (A round is a chain of twenty-odd instructions; through shuffles of score
// and label it took several times that, and the kernels below are little else: 10 -> 7 us for the thresholds of one sample.)
__device__ __forceinline__ void wave_topk(TopList& l, int rounds, float& out_v, int& out_i) {
    const int lane = threadIdx.x & 63;
    out_v = -__builtin_inff();
    out_i = kNoId;
    for (int s = 0; s < rounds; ++s) {
        const float bv = wave_largest(l.v[0]);
        const int bi = wave_smallest(l.v[0] == bv ? l.id[0] : kNoId);
        if (lane == s) { out_v = bv; out_i = bi; }
        if (bi != kNoId && l.id[0] == bi && l.v[0] == bv) l.pop();
    }
}

// The workgroup's lists down to one; afterwards lane s < rounds of wavefront 0 holds the s-th best.  One barrier.
template <int WAVES>
__device__ __forceinline__ void block_topk(TopList& l, int rounds, float& out_v, int& out_i) {
    __shared__ float lv[WAVES][kTopMax];
    __shared__ int li[WAVES][kTopMax];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    wave_topk(l, rounds, out_v, out_i);
    if (lane < kTopMax) { lv[wave][lane] = out_v; li[wave][lane] = out_i; }
    __syncthreads();
    if (wave != 0) return;
    l.clear();
    if (lane < WAVES) {
#pragma unroll
        for (int s = 0; s < kTopMax; ++s) { l.v[s] = lv[lane][s]; l.id[s] = li[lane][s]; }
    }
    wave_topk(l, rounds, out_v, out_i);
}

// Lists of a score matrix scores[B,L]: grid (splits, B); each thread scans a strided share of the split (coalesced, eight scores
// in flight), each wavefront then reduces its 64 lists to one: four lists of eight per split (label -1 = empty slot).
__global__ __launch_bounds__(256) void topk_scan_kernel(const float* __restrict__ scores, int L, int labels_per_split,
                                                        float* __restrict__ part_val, int* __restrict__ part_idx, int nlists) {
    const int b = blockIdx.y;
    const int begin = blockIdx.x * labels_per_split, end = min(begin + labels_per_split, L);
    TopList l;
    l.clear();
    const float* row = scores + (size_t)b * L;
    for (int j0 = begin + (int)threadIdx.x; j0 < end; j0 += 256 * 8) {
        float v8[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v8[u] = row[min(j0 + 256 * u, end - 1)];      // clamped, not predicated: the eight loads issue back to back
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (j0 + 256 * u < end) l.offer(v8[u], j0 + 256 * u);
    }
    float ov;
    int oi;
    wave_topk(l, kTopMax, ov, oi);
    const int lane = threadIdx.x & 63;
    if (lane < kTopMax) {
        const int list = blockIdx.x * 4 + (threadIdx.x >> 6);
        part_val[((size_t)b * nlists + list) * kTopMax + lane] = ov;
        part_idx[((size_t)b * nlists + list) * kTopMax + lane] = oi != kNoId ? oi : -1;
    }
}

// The threshold of every sample and its empty candidate list: 1,024 groups of a sample of S scores (scores[b * row + i * step],
// step > 1: straight from a score matrix), the k-th best of the groups' best.  Fewer groups than k with a score: all scores reach it.
__global__ __launch_bounds__(1024) void topk_threshold_kernel(const float* __restrict__ scores, size_t row, int step, int S, TopkSampleLabels labels,
                                                              int k, int B, float* __restrict__ tau, int* __restrict__ tie, int* __restrict__ count) {
    const int b = blockIdx.x;
    TopList l;
    l.clear();
    float best = -__builtin_inff();
    int best_i = kNoId;
    for (int i0 = threadIdx.x; i0 < S; i0 += 1024 * 8) {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = scores[(size_t)b * row + (size_t)min(i0 + 1024 * u, S - 1) * step];
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (i0 + 1024 * u < S && (v[u] > best || (v[u] == best && best_i == kNoId))) { best = v[u]; best_i = i0 + 1024 * u; }      // (ids ascend; each score in one group only)
    }
    l.v[0] = best;
    l.id[0] = best_i;
    float ov;
    int oi;
    block_topk<16>(l, k, ov, oi);
    if ((int)threadIdx.x == k - 1) {
        tau[b] = ov;
        tie[b] = oi != kNoId ? (int)(((long long)oi * labels.num) >> labels.shift) : kNoId;
    }
    if (threadIdx.x < 2) count[(size_t)b * kTopkCountStep + threadIdx.x] = 0;
    const int behind = B + (int)threadIdx.x;                                 // (a sample behind the batch's end, up to the next 64)
    if (b == 0 && behind < (B + 63) / 64 * 64) { tau[behind] = __builtin_inff(); tie[behind] = kTopkListFull; }
}

// Every score at or above its row's threshold goes to the row's candidate list.  Such scores are a tiny share of the
// row, so the scan is a plain stream: eight loads in flight per thread, one wave-wide test, the appends on the side.
__global__ __launch_bounds__(256) void topk_filter_kernel(const float* __restrict__ scores, int L, int labels_per_split,
                                                          const float* __restrict__ tau, int* tie, int* __restrict__ count,
                                                          float* __restrict__ cand_val, int* __restrict__ cand_idx, int cap) {
    constexpr int kPark = 1024;                       // hits a workgroup parks in LDS before it appends them to the row's list
    __shared__ int park_count;
    __shared__ float park_val[kPark];
    __shared__ int park_idx[kPark];
    const int b = blockIdx.y;
    const int begin = blockIdx.x * labels_per_split, end = min(begin + labels_per_split, L);
    const float t = tau[b];
    const float* row = scores + (size_t)b * L;
    if (threadIdx.x == 0) park_count = 0;
    __syncthreads();
    int last_tied = tie[b];                           // (on its way together with the scores)
    for (int j0 = begin + (int)threadIdx.x; j0 < end; j0 += 256 * 8) {
        float v8[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v8[u] = row[min(j0 + 256 * u, end - 1)];
        bool hit = false;
#pragma unroll
        for (int u = 0; u < 8; ++u) hit |= (j0 + 256 * u < end) && v8[u] >= t;
        if (__ballot(hit)) {
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int j = j0 + 256 * u;
                if (j < end && topk_reaches(v8[u], j, t, last_tied)) {
                    const int p = atomicAdd(&park_count, 1);          // an LDS counter: no round trip to memory
                    if (p < kPark) {
                        park_val[p] = v8[u];
                        park_idx[p] = j;
                    } else {
                        const int slot = topk_slot(v8[u], j, t, last_tied, &tie[b], &count[(size_t)b * kTopkCountStep], cap);
                        if (slot < cap) {
                            cand_val[(size_t)b * cap + slot] = v8[u];
                            cand_idx[(size_t)b * cap + slot] = j;
                        }
                    }
                }
            }
        }
    }
    __syncthreads();
    const int n = min(park_count, kPark);
    __shared__ int first_slot;
    if (threadIdx.x == 0) first_slot = n ? atomicAdd(&count[(size_t)b * kTopkCountStep], n) : 0;      // one reservation for the whole workgroup
    __syncthreads();
    for (int e = threadIdx.x; e < n; e += 256) {
        const int slot = first_slot + e;
        if (slot < cap) {
            cand_val[(size_t)b * cap + slot] = park_val[e];
            cand_idx[(size_t)b * cap + slot] = park_idx[e];
        }
    }
}

template <typename T> __device__ __forceinline__ float as_float(T v);
template <> __device__ __forceinline__ float as_float<float>(float v) { return v; }
template <> __device__ __forceinline__ float as_float<unsigned short>(unsigned short v) { return __uint_as_float((unsigned)v << 16); }

// The k best of a sample's candidates (workgroup b: sample b).  A sample whose candidates did not fit its list is answered from
// its whole row -- the stored scores, or scores formed anew from the layer (k ascending, bias last) -- by the first `sharers`
// workgroups: each keeps the best eight of its share in the place of the sample's candidates, the last to finish takes the best of
// those.  (One workgroup per row: 28 ms of latency for 670,091 labels of fan-in 32.)
constexpr int kTopkSharers = kTopkCap / kTopMax;        // lists of eight that fit there

template <typename T>
__global__ __launch_bounds__(256) void topk_select_kernel(float* cand_val, int* cand_idx, int* count, int cap, int k, const TopkRowSource src,
                                                          int B, int sharers, float* __restrict__ values, int* __restrict__ indices) {
    TopList l;
    float ov;
    int oi;
    auto answer = [&](int b, int n) {                                 // from n listed entries
        const float* pv = cand_val + (size_t)b * cap;
        const int* pi = cand_idx + (size_t)b * cap;
        l.clear();
        for (int c0 = threadIdx.x; c0 < n; c0 += 256 * 4) {           // four candidates per thread in flight
            float v4[4];
            int i4[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int c = min(c0 + 256 * u, n - 1);
                i4[u] = c0 + 256 * u < n ? pi[c] : -1;
                v4[u] = pv[c];
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (i4[u] >= 0) l.offer(v4[u], i4[u]);
        }
        block_topk<4>(l, k, ov, oi);
        if ((int)threadIdx.x < k) {
            values[(size_t)b * k + threadIdx.x] = ov;
            indices[(size_t)b * k + threadIdx.x] = oi != kNoId ? oi : -1;
        }
    };
    if ((int)blockIdx.x < B) {
        const int n = count != nullptr ? count[(size_t)blockIdx.x * kTopkCountStep] : cap;
        if (n <= cap) answer((int)blockIdx.x, n);
    }
    if (count == nullptr || (int)blockIdx.x >= sharers) return;
    // the samples whose lists overflowed (of 256 at a time)
    __shared__ int over[256];
    __shared__ int n_over, arrived;
    const T* x = static_cast<const T*>(src.x);
    const T* w = static_cast<const T*>(src.w);
    for (int b0 = 0; b0 < B; b0 += 256) {
        __syncthreads();
        if (threadIdx.x == 0) n_over = 0;
        __syncthreads();
        const int mine = b0 + (int)threadIdx.x;
        if (mine < B && count[(size_t)mine * kTopkCountStep] > cap) over[atomicAdd(&n_over, 1)] = mine;
        __syncthreads();
        const int todo = n_over;
        for (int t = 0; t < todo; ++t) {
            const int b = over[t];
            l.clear();
            for (int j = (int)(blockIdx.x * 256 + threadIdx.x); j < src.L; j += sharers * 256) {
                float v = 0.f;
                if (src.scores != nullptr) {
                    v = src.scores[(size_t)b * src.L + j];
                } else {
                    const size_t row = (size_t)j * src.K;
                    for (int c0 = 0; c0 < src.K; c0 += 8) {           // (eight ids, then eight operands in flight)
                        unsigned id[8];
                        float wv[8], xv[8];
#pragma unroll
                        for (int c = 0; c < 8; ++c) {
                            const size_t at = row + min(c0 + c, src.K - 1);
                            id[c] = min((unsigned)src.idx[at], (unsigned)src.N - 1u);
                            wv[c] = as_float(w[at]);
                        }
#pragma unroll
                        for (int c = 0; c < 8; ++c) xv[c] = as_float(src.tp ? x[(size_t)id[c] * B + b] : x[(size_t)b * src.N + id[c]]);
#pragma unroll
                        for (int c = 0; c < 8; ++c)
                            if (c0 + c < src.K) v = fmaf(wv[c], xv[c], v);
                    }
                    if (src.bias != nullptr) v += src.bias[j];
                }
                l.offer(v, j);
            }
            __syncthreads();                                          // (block_topk's own memory)
            block_topk<4>(l, kTopMax, ov, oi);
            if ((int)threadIdx.x < kTopMax) {
                cand_val[(size_t)b * cap + blockIdx.x * kTopMax + threadIdx.x] = ov;
                cand_idx[(size_t)b * cap + blockIdx.x * kTopMax + threadIdx.x] = oi != kNoId ? oi : -1;
            }
            __threadfence();
            __syncthreads();
            if (threadIdx.x == 0) arrived = atomicAdd(&count[(size_t)b * kTopkCountStep + 1], 1);
            __syncthreads();
            if (arrived == sharers - 1) {
                __threadfence();
                answer(b, sharers * kTopMax);
            }
        }
    }
}

// ---- few samples: scores and answer in one pass --------------------------------------------------------------------
// For up to four samples whose features fit in LDS (all of them, BP floats a column).  A group of `lanes` neighbouring lanes has a
// label, a lane four connections of it: 16 bytes of ids and of weights in whole lines, the features of a connection by one read of
// LDS, the products summed over the group by DPP.  Every lane keeps the best eight of the labels that fall to it, a workgroup the best
// of its lanes'; the workgroup that ends last takes the best of those.
//
// What bounds it: the stream of ids and weights.  One sample, 768 columns, 670,091 labels, fan-in 32: 35.6 us, 4.9 TB/s;
// a sample of the labels, a threshold, all scores and a selection took four launches and 67 us; four samples 56 against 59.
// (From eight samples on the sums over the lanes cost more than the launches.)
constexpr int kDirectThreads = 1024;
constexpr int direct_rounds(int bp) { return bp == 1 ? 4 : 2; }      // rounds of labels whose loads are in flight together
constexpr size_t kDirectLds = 144 * 1024;       // for the features
constexpr int kDirectHeld = 4;                  // labels per lane, at most

// The labels that fell to a lane.
struct FewLabels {
    float v[kDirectHeld];
    int id[kDirectHeld];
    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int s = 0; s < kDirectHeld; ++s) { v[s] = -__builtin_inff(); id[s] = kNoId; }
    }
};

// The k best of a workgroup's labels, in m.out_v and m.out_id (-inf and kNoId behind the last), for every thread to read.  The k-th best of the wavefronts' best bounds the answer from below; the few labels that reach it are listed, and
// each counts those that are better.  (By rounds that take the best of all that is left, 10 us a sample and workgroup; where
// more labels than the list holds reach the bound, that is what happens.)  k <= 16 wavefronts.
constexpr int kFewCap = 512;
struct FewShared {
    float best_v[kDirectThreads / 64], v[kFewCap], out_v[kTopMax];
    int best_id[kDirectThreads / 64], id[kFewCap], out_id[kTopMax];
    int count;
};
__device__ __forceinline__ void few_topk(const FewLabels& l, int k, FewShared& m) {
    constexpr int kWaves = kDirectThreads / 64;
    static_assert(kTopMax <= kWaves, "a bound from the wavefronts' best");
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    float bv = l.v[0];
    int bi = l.id[0];
#pragma unroll
    for (int s = 1; s < kDirectHeld; ++s)
        if (better(l.v[s], l.id[s], bv, bi)) { bv = l.v[s]; bi = l.id[s]; }
    const float wv = wave_largest(bv);
    const int wi = wave_smallest(bv == wv ? bi : kNoId);
    if (lane == 0) { m.best_v[wave] = wv; m.best_id[wave] = wi; }
    if (threadIdx.x == 0) m.count = 0;
    if (threadIdx.x < kTopMax) { m.out_v[threadIdx.x] = -__builtin_inff(); m.out_id[threadIdx.x] = kNoId; }
    __syncthreads();
    // (equal entries -- wavefronts without a label -- in the order of the wavefronts)
    const float mv = m.best_v[lane % kWaves];
    const int mi = m.best_id[lane % kWaves];
    int rank = 0;
#pragma unroll
    for (int s = 0; s < kWaves; ++s) {
        const float ov = m.best_v[s];
        const int oi = m.best_id[s];
        rank += better(ov, oi, mv, mi) || (ov == mv && oi == mi && s < lane % kWaves);
    }
    const int at = __ffsll((unsigned long long)__ballot(rank == k - 1)) - 1;
    const float tv = m.best_v[at];
    const int ti = m.best_id[at];
#pragma unroll
    for (int s = 0; s < kDirectHeld; ++s) {
        if (l.id[s] != kNoId && !better(tv, ti, l.v[s], l.id[s])) {
            const int to = atomicAdd(&m.count, 1);
            if (to < kFewCap) { m.v[to] = l.v[s]; m.id[to] = l.id[s]; }
        }
    }
    __syncthreads();
    const int n = m.count;
    if (n <= kFewCap) {
        if ((int)threadIdx.x < n) {
            const float v = m.v[threadIdx.x];
            const int id = m.id[threadIdx.x];
            int r = 0;
#pragma unroll 8
            for (int s = 0; s < n; ++s) r += better(m.v[s], m.id[s], v, id);
            if (r < k) { m.out_v[r] = v; m.out_id[r] = id; }
        }
    } else {
        TopList all;
        all.clear();
#pragma unroll
        for (int s = 0; s < kDirectHeld; ++s)
            if (l.id[s] != kNoId) all.offer(l.v[s], l.id[s]);
        float ov;
        int oi;
        block_topk<kWaves>(all, k, ov, oi);
        if ((int)threadIdx.x < k) { m.out_v[threadIdx.x] = ov; m.out_id[threadIdx.x] = oi; }
    }
    __syncthreads();
}

// the four connections of a label that begin at k0, at any alignment of their type
template <typename T> struct Four { T v[4]; };

template <bool BF16, int BP>
__global__ __launch_bounds__(kDirectThreads) void topk_direct_kernel(const void* __restrict__ features, const int32_t* __restrict__ idx,
                                                                     const void* __restrict__ weights, const float* __restrict__ bias, int B, int N,
                                                                     int L, int K, int tp, int lanes, int passes, int k, unsigned long long* part,
                                                                     unsigned* ticket, float* __restrict__ values,
                                                                     int32_t* __restrict__ indices) {
    using T = std::conditional_t<BF16, unsigned short, float>;
    const T* const x = static_cast<const T*>(features);
    const T* const w = static_cast<const T*>(weights);
    constexpr int kDirectRounds = direct_rounds(BP);
    extern __shared__ __align__(16) float direct_xs[];            // [N][BP]
    for (int e = threadIdx.x; e < N * B; e += kDirectThreads) {
        const int n = tp ? e / B : e % N, b = tp ? e % B : e / N;
        direct_xs[n * BP + b] = as_float(x[e]);
    }
    if (B < BP)
        for (int e = threadIdx.x; e < N * (BP - B); e += kDirectThreads) direct_xs[e / (BP - B) * BP + B + e % (BP - B)] = 0.f;
    __syncthreads();
    const int lane = threadIdx.x & 63, sub = lane & (lanes - 1), per_round = 64 / lanes;
    const int step = gridDim.x * (kDirectThreads / 64) * per_round * kDirectRounds;
    FewLabels list[BP];
#pragma unroll
    for (int b = 0; b < BP; ++b) list[b].clear();
    // (a round's labels from all wavefronts of the workgroup side by side: one whose few labels fell to few wavefronts had no bound from
    // the others, 52 us at 1 x 500 x 150,000 x 8 where 12 are enough)
    constexpr int kWaves = kDirectThreads / 64;
    auto label_of = [&](int j0, int u) { return j0 + u * kWaves * per_round + lane / lanes; };
    Four<int> id[kDirectRounds];
    Four<T> wt[kDirectRounds];
    auto fetch = [&](int j0, int pass) {
        const int k0 = min((pass * lanes + sub) * 4, K - 4);      // (the last quad of a row ends with it)
#pragma unroll
        for (int u = 0; u < kDirectRounds; ++u) {
            const size_t at = (size_t)min(label_of(j0, u), L - 1) * K + k0;
            id[u] = *reinterpret_cast<const Four<int>*>(idx + at);
            wt[u] = *reinterpret_cast<const Four<T>*>(w + at);
        }
    };
    int j0 = (blockIdx.x * kWaves * kDirectRounds + (threadIdx.x >> 6)) * per_round, held = 0, place = 0, mine = kNoId;
    float score[BP];
    // (NaN is no score: it takes no place)
    auto keep = [&]() {
        const float bj = bias != nullptr && mine != kNoId ? bias[mine] : 0.f;
#pragma unroll
        for (int b = 0; b < BP; ++b) {
            const float v = bias != nullptr ? score[b] + bj : score[b];
            const bool on = mine != kNoId && v == v;
#pragma unroll
            for (int t = 0; t < kDirectHeld; ++t)
                if (place == t) { list[b].v[t] = on ? v : -__builtin_inff(); list[b].id[t] = on ? mine : kNoId; }
        }
        ++place;
        held = 0;
        mine = kNoId;
    };
    if (j0 < L) fetch(j0, 0);
    for (; j0 < L; j0 += step) {
        float acc[kDirectRounds][BP];
#pragma unroll
        for (int u = 0; u < kDirectRounds; ++u)
#pragma unroll
            for (int b = 0; b < BP; ++b) acc[u][b] = 0.f;
        for (int pass = 0; pass < passes; ++pass) {
            const int first = (pass * lanes + sub) * 4;
            Four<int> at[kDirectRounds];
            Four<T> wv[kDirectRounds];
#pragma unroll
            for (int u = 0; u < kDirectRounds; ++u) { at[u] = id[u]; wv[u] = wt[u]; }
            if (pass + 1 < passes) fetch(j0, pass + 1);
            else fetch(min(j0 + step, L - 1), 0);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const bool on = min(first, K - 4) + e >= first;   // (what a pulled-back quad shares with the one before it, and quads behind the row)
#pragma unroll
                for (int u = 0; u < kDirectRounds; ++u) {
                    const float* row = direct_xs + (size_t)(unsigned)at[u].v[e] * BP;
                    const float we = on ? as_float(wv[u].v[e]) : 0.f;
                    float xv[BP];
                    if constexpr (BP == 4) { const float4 t = *reinterpret_cast<const float4*>(row); xv[0] = t.x; xv[1] = t.y; xv[2] = t.z; xv[3] = t.w; }
                    else if constexpr (BP == 2) { const float2 t = *reinterpret_cast<const float2*>(row); xv[0] = t.x; xv[1] = t.y; }
                    else xv[0] = row[0];
#pragma unroll
                    for (int b = 0; b < BP; ++b) acc[u][b] = fmaf(we, on ? xv[b] : 0.f, acc[u][b]);
                }
            }
        }
#pragma unroll
        for (int u = 0; u < kDirectRounds; ++u) {
            const int j = label_of(j0, u);
#pragma unroll
            for (int b = 0; b < BP; ++b) {
                float v = acc[u][b];
                if (lanes > 1) v += dpp_of<0xb1>(v);
                if (lanes > 2) v += dpp_of<0x4e>(v);
                if (lanes > 4) v += dpp_of<0x141>(v);
                if (lanes > 8) v += dpp_of<0x140>(v);
                if (lanes > 16) v += __shfl_xor(v, 16);
                if (lanes > 32) v += __shfl_xor(v, 32);
                if (held == sub) score[b] = v;
            }
            if (held == sub && j < L) mine = j;
            if (++held == lanes) keep();                          // every lane of the group has a label
        }
    }
    if (held > 0) keep();
    // A workgroup's answers are published by exchanges whose results are waited for, then its ticket is drawn: read-modify-writes at
    // device scope, carried out where all XCDs see them.  (A fence by all wavefronts: 94 us for the kernel, not 44.)
    __shared__ FewShared shared;
    unsigned long long seen = 0;
#pragma unroll
    for (int b = 0; b < BP; ++b) {
        if (b >= B) break;
        few_topk(list[b], k, shared);
        if ((int)threadIdx.x < k)
            seen += __hip_atomic_exchange(&part[((size_t)b * gridDim.x + blockIdx.x) * kTopMax + threadIdx.x],
                                          (unsigned long long)(unsigned)shared.out_id[threadIdx.x] << 32 | __float_as_uint(shared.out_v[threadIdx.x]),
                                          __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __shared__ bool last;
    if (threadIdx.x < 64) {
        unsigned one = 1u;
        asm volatile("" : "+v"(one) : "v"(seen));             // (of all the wavefront's lanes: they wait together)
        if (threadIdx.x == 0) last = __hip_atomic_fetch_add(ticket, one, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1;
    }
    __syncthreads();
    if (!last) return;
    // The workgroups' best before their second best, and each in all wavefronts, whose best bound the answer: with a workgroup's entries
    // in neighbouring lanes of few wavefronts the bound was none, 94 us at 4 x 500 x 10,000 x 32.  All samples' entries are on their way
    // together.
    const int entries = (int)gridDim.x * k, first = (threadIdx.x & 63) * (kDirectThreads / 64) + (threadIdx.x >> 6);
    const bool few = entries <= kDirectHeld * kDirectThreads;
    auto entry = [&](int b, int e) {
        return __hip_atomic_load(&part[((size_t)b * gridDim.x + e % (int)gridDim.x) * kTopMax + e / (int)gridDim.x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
#pragma unroll
    for (int b = 0; b < BP; ++b) {
        list[b].clear();
        if (b >= B || !few) continue;
#pragma unroll
        for (int t = 0; t < kDirectHeld; ++t) {
            const int e = first + t * kDirectThreads;
            if (e < entries) {
                const unsigned long long p = entry(b, e);
                list[b].v[t] = __uint_as_float((unsigned)p);
                list[b].id[t] = (int)(p >> 32);
            }
        }
    }
#pragma unroll
    for (int b = 0; b < BP; ++b) {
        if (b >= B) break;
        if (few) {
            few_topk(list[b], k, shared);
        } else {
            TopList more;
            more.clear();
            for (int e = threadIdx.x; e < entries; e += kDirectThreads) {
                const unsigned long long p = entry(b, e);
                if ((int)(p >> 32) != kNoId) more.offer(__uint_as_float((unsigned)p), (int)(p >> 32));
            }
            float ov;
            int oi;
            block_topk<kDirectThreads / 64>(more, k, ov, oi);
            if (threadIdx.x < kTopMax) { shared.out_v[threadIdx.x] = ov; shared.out_id[threadIdx.x] = oi; }
        }
        if ((int)threadIdx.x < k) {
            values[(size_t)b * k + threadIdx.x] = shared.out_v[threadIdx.x];
            indices[(size_t)b * k + threadIdx.x] = shared.out_id[threadIdx.x] != kNoId ? shared.out_id[threadIdx.x] : -1;
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) *ticket = 0u;
}

constexpr int kTopkRowSample = 4096;

// Label values at the k best labels of every sample, summed per rank: host[r] over all samples, and the loss of the step beside
// them.  One workgroup, the table of hits in LDS (one entry per sample and rank: the first listed position that names the pair),
// kHitSamples samples at a time; the sums are formed in double, thread by thread and then over the threads in order.
// Launch latency is all there is to it: 3 us at 32 x 5 and 160 positions, where a sort, a search and a sum of the framework
// took 22 launches for each k.
constexpr int kHitThreads = 1024;
constexpr int kHitSamples = 2048;

__global__ __launch_bounds__(kHitThreads) void topk_hits_kernel(const int32_t* __restrict__ top, int B, int top_stride, int k,
                                                                const int64_t* __restrict__ label_indices, const float* __restrict__ label_values,
                                                                int nnz, const float* __restrict__ also, double* host) {
    __shared__ unsigned first[kHitSamples * kTopMax];
    __shared__ double red[kHitThreads / 64][kTopMax];
    double sum[kTopMax];
#pragma unroll
    for (int r = 0; r < kTopMax; ++r) sum[r] = 0.0;
    for (int b0 = 0; b0 < B; b0 += kHitSamples) {
        const int nb = min(B - b0, kHitSamples);
        __syncthreads();
        for (int e = threadIdx.x; e < nb * kTopMax; e += kHitThreads) first[e] = ~0u;
        __syncthreads();
        for (int p = threadIdx.x; p < nnz; p += kHitThreads) {
            const int64_t b = label_indices[2 * (size_t)p] - b0, j = label_indices[2 * (size_t)p + 1];
            if (b < 0 || b >= nb) continue;
            const int32_t* row = top + (size_t)(b0 + b) * top_stride;
            for (int r = 0; r < k; ++r)
                if (row[r] >= 0 && row[r] == j) atomicMin(&first[b * kTopMax + r], (unsigned)p);
        }
        __syncthreads();
        for (int b = threadIdx.x; b < nb; b += kHitThreads)
#pragma unroll
            for (int r = 0; r < kTopMax; ++r) {
                const unsigned p = first[b * kTopMax + r];
                if (p != ~0u) sum[r] += label_values != nullptr ? (double)label_values[p] : 1.0;
            }
    }
#pragma unroll
    for (int r = 0; r < kTopMax; ++r) {
        const double t = wave_sum(sum[r]);
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6][r] = t;
    }
    __syncthreads();
    if ((int)threadIdx.x < kTopMax) {
        double t = 0.0;
        for (int i = 0; i < kHitThreads / 64; ++i) t += red[i][threadIdx.x];
        host[threadIdx.x] = t;
    }
    if (threadIdx.x == kTopMax && also != nullptr) host[kTopMax] = (double)*also;
}

}  // namespace

int topk_hits(const int32_t* top, int B, int top_stride, int k, const int64_t* label_indices, const float* label_values, int nnz,
              const float* also, double* result, hipStream_t s) {
    void* words = nullptr;
    FFI_TRY(host_words_get(s, &words));
    double* host = static_cast<double*>(words);
    hipLaunchKernelGGL(topk_hits_kernel, dim3(1), dim3(kHitThreads), 0, s, top, B, top_stride, k, label_indices, label_values, nnz, also, host);
    FFI_HIP_TRY(hipGetLastError());
    FFI_HIP_TRY(hipStreamSynchronize(s));
    for (int r = 0; r < k; ++r) result[r] = static_cast<volatile double*>(host)[r];
    if (also != nullptr) result[k] = static_cast<volatile double*>(host)[kTopMax];
    return FFI_OK;
}

// Thresholds, counters and candidates begin on cache lines of their own: counters that shared one with the thresholds, which
// every workgroup reads, tripled the time of a sweep (43 -> 146 us at 12 x 3,000 x 300,000 x 32).  The forward kernels read the
// thresholds a slice of up to 64 samples at a time: those of the samples behind the batch's end say that their lists are full.
static size_t line_floats(size_t n) { return (n + 31) / 32 * 32; }
static size_t padded_samples(int B) { return ((size_t)B + 63) / 64 * 64; }
size_t topk_candidate_bytes(int B, int sample) {
    return (line_floats((size_t)B * sample) + 2 * padded_samples(B) + (size_t)B * kTopkCountStep + 2 * (size_t)B * kTopkCap) * 4;
}
TopkCandidates topk_candidates_at(void* ws, int B, int sample) {
    TopkCandidates c;
    c.sample = static_cast<float*>(ws);
    c.tau = c.sample + line_floats((size_t)B * sample);
    c.tie = reinterpret_cast<int*>(c.tau + padded_samples(B));
    c.count = c.tie + padded_samples(B);
    c.val = reinterpret_cast<float*>(c.count + (size_t)B * kTopkCountStep);
    c.idx = reinterpret_cast<int*>(c.val + (size_t)B * kTopkCap);
    return c;
}

int direct_width(int B) { return B <= 1 ? 1 : B <= 2 ? 2 : 4; }
// A workgroup's k best take some 5 us a sample, which four samples have to save by the three launches and the second reading that there
// are no more: fan-ins and labels (thousands) 8 x 400 33 us against 27, 32 x 400 47 and 46, 32 x 670 56 and 59, 100 x 300 73 and 111;
// three samples 27 and 27, 40 and 45, 50 and 58, 66 and 110; one 13 and 26, 26 and 45, 35 and 58, 47 and 110.
bool takes_topk_direct(const Dims& d) {
    if (d.B == 4 && (long long)d.L * d.K < (16ll << 20)) return false;
    return d.B <= 4 && d.K >= 4 && (size_t)d.N * direct_width(d.B) * sizeof(float) <= kDirectLds;
}

int launch_topk_direct(const void* x, const int32_t* idx, const void* w, const float* bias, bool bf16, const TopkArgs& tk, const Dims& d,
                       hipStream_t s) {
    const int quads = (d.K + 3) / 4;
    int lanes = 1;
    while (lanes < 64 && lanes < quads) lanes *= 2;
    const int per_round = 64 / lanes, passes = (quads + lanes - 1) / lanes;
    const long long per_block = (long long)(kDirectThreads / 64) * per_round * direct_rounds(direct_width(d.B));     // labels per step
    const long long steps = std::max(1, kDirectHeld * lanes / direct_rounds(direct_width(d.B)));                      // of a workgroup, at most
    const long long fill = std::min<long long>(device_cu_count(), (d.L + per_block - 1) / per_block);
    const int blocks = (int)std::max(fill, (d.L + per_block * steps - 1) / (per_block * steps));
    const size_t entries = (size_t)d.B * blocks * kTopMax, lds = (size_t)d.N * direct_width(d.B) * sizeof(float);
    unsigned long long* part = nullptr;
    unsigned* ticket = nullptr;
    FFI_TRY(workspace_get(s, kWsTopk, entries * sizeof(*part), (void**)&part));
    FFI_TRY(tickets_get(s, (void**)&ticket));
    auto go = [&](auto kernel) -> int {
        FFI_HIP_TRY(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(kDirectThreads), lds, s, x, idx, w, bias, d.B, d.N, d.L, d.K, d.tp ? 1 : 0, lanes,
                           passes, tk.k, part, ticket, tk.values, tk.indices);
        FFI_HIP_TRY(hipGetLastError());
        return FFI_OK;
    };
    switch (direct_width(d.B)) {
        case 1: return bf16 ? go(topk_direct_kernel<true, 1>) : go(topk_direct_kernel<false, 1>);
        case 2: return bf16 ? go(topk_direct_kernel<true, 2>) : go(topk_direct_kernel<false, 2>);
        default: return bf16 ? go(topk_direct_kernel<true, 4>) : go(topk_direct_kernel<false, 4>);
    }
}

int launch_topk_threshold(const float* scores, size_t row, int step, int S, TopkSampleLabels labels, int k, const TopkCandidates& c, int B,
                          hipStream_t s) {
    hipLaunchKernelGGL(topk_threshold_kernel, dim3(B), dim3(1024), 0, s, scores, row, step, S, labels, k, B, c.tau, c.tie, c.count);
    FFI_HIP_TRY(hipGetLastError());
    return FFI_OK;
}

int launch_topk_select(const TopkCandidates& c, int B, const TopkArgs& tk, const TopkRowSource& src, hipStream_t s) {
    // (workgroups that find no overflowed list leave at once)
    const int sharers = std::max(1, std::min({kTopkSharers, (src.L + 255) / 256, 4 * device_cu_count()}));
    const dim3 grid((unsigned)std::max(B, sharers));
    if (src.bf16) hipLaunchKernelGGL(topk_select_kernel<unsigned short>, grid, dim3(256), 0, s, c.val, c.idx, c.count, kTopkCap, tk.k, src, B, sharers, tk.values, tk.indices);
    else hipLaunchKernelGGL(topk_select_kernel<float>, grid, dim3(256), 0, s, c.val, c.idx, c.count, kTopkCap, tk.k, src, B, sharers, tk.values, tk.indices);
    FFI_HIP_TRY(hipGetLastError());
    return FFI_OK;
}

int launch_topk_f32(const float* scores, int B, int L, int k, float* values, int32_t* indices, hipStream_t s) {
    if (k < 1 || k > kTopMax) return FFI_ERR_BAD_ARGUMENT;
    if (B > 65535) return FFI_ERR_TOO_LARGE;
    // enough workgroups to fill the GPU (8 per CU), each with at least 2048 scores to scan
    int splits = std::max(1, std::min((L + 2047) / 2048, (8 * device_cu_count() + B - 1) / std::max(1, B)));
    const int per = (L + splits - 1) / splits;
    splits = (L + per - 1) / per;
    const TopkArgs tk{k, values, indices};
    if (L <= kTopkShortRow) {
        // rows too short to be worth a threshold: every thread keeps a list, the wavefronts reduce them
        const int entries = splits * 4 * kTopMax;
        char* part = nullptr;
        const size_t list_bytes = (size_t)B * entries * 4;
        FFI_TRY(workspace_get(s, kWsPartials, 2 * list_bytes, (void**)&part));
        float* pv = (float*)part;
        int* pi = (int*)(part + list_bytes);
        hipLaunchKernelGGL(topk_scan_kernel, dim3(splits, B), dim3(256), 0, s, scores, L, per, pv, pi, splits * 4);
        hipLaunchKernelGGL(topk_select_kernel<float>, dim3(B), dim3(256), 0, s, pv, pi, (int*)nullptr, entries, k, TopkRowSource{}, B, 0, values, indices);
        FFI_HIP_TRY(hipGetLastError());
        return FFI_OK;
    }
    void* ws = nullptr;
    FFI_TRY(workspace_get(s, kWsTopk, topk_candidate_bytes(B, 0), &ws));
    const TopkCandidates c = topk_candidates_at(ws, B, 0);
    const int step = L / kTopkRowSample;
    FFI_TRY(launch_topk_threshold(scores, (size_t)L, step, kTopkRowSample, TopkSampleLabels{step, 0}, k, c, B, s));
    hipLaunchKernelGGL(topk_filter_kernel, dim3(splits, B), dim3(256), 0, s, scores, L, per, c.tau, c.tie, c.count, c.val, c.idx, kTopkCap);
    FFI_HIP_TRY(hipGetLastError());
    TopkRowSource src;
    src.scores = scores; src.L = L;
    return launch_topk_select(c, B, tk, src, s);
}

}  // namespace ffi
