// Check of a lookup's content against a plan's fingerprint, on the device, as workgroups of a kernel that has other
// work too (gfx950).
#ifndef FFI_CHECK_H
#define FFI_CHECK_H

#include "ffi_internal.h"

namespace ffi {

__device__ __forceinline__ unsigned mix32(unsigned v) {
    v ^= v >> 16; v *= 0x7feb352du;
    v ^= v >> 15; v *= 0x846ca68bu;
    v ^= v >> 16;
    return v;
}

// The same fingerprint, checked on the device.  Workgroups leave their pairs of sums in guard[8 + 2 * block ..]
// (plain stores) and take a ticket from guard[2], the only atomic: a few hundred adds to one address, not
// thousands (those serialise and were measured to triple the kernel's time).  The workgroup that draws the last
// ticket adds the pairs up (integer adds: the total does not depend on the order), compares with guard[3], leaves
// the verdict in guard[4] (1 = content unchanged and every id in range), the sums in guard[5] / guard[6], and
// clears the ticket counter for the next check.
struct CheckShared {
    unsigned long long part[2][kCheckThreads / 64];
    bool last;
};
// Workgroup `block` of check.blocks, kCheckThreads threads each.
__device__ __forceinline__ void check_block(const LookupCheck& check, int block, CheckShared& shared) {
    const int32_t* __restrict__ const idx = check.idx;
    const size_t total = check.total;
    const unsigned N = check.num_features;
    unsigned long long* __restrict__ const guard = check.guard;
    auto& part = shared.part;
    unsigned long long h = 0;
    unsigned bad = 0;
    const size_t stride = (size_t)check.blocks * kCheckThreads;
    const size_t tid = (size_t)block * kCheckThreads + threadIdx.x;
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
    if ((threadIdx.x & 63) == 0) { part[0][threadIdx.x >> 6] = h; part[1][threadIdx.x >> 6] = b64; }
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long hs = 0, bs = 0;
#pragma unroll
        for (int i = 0; i < kCheckThreads / 64; ++i) { hs += part[0][i]; bs += part[1][i]; }
        // Published with atomic exchanges whose results are waited for, then the ticket: a read-modify-write at
        // device scope is carried out where all XCDs see it, and its returned value says that it has been.  (A
        // fence here would first write back every dirty line of this XCD's L2 -- the scores the forward kernel has
        // just stored among them -- which was measured to cost a third of the kernel's time.)
        const unsigned long long o1 = __hip_atomic_exchange(&guard[8 + 2 * block], hs, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const unsigned long long o2 = __hip_atomic_exchange(&guard[9 + 2 * block], bs, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        unsigned long long one = 1ull;
        asm volatile("" : "+v"(one) : "v"(o1), "v"(o2));       // the ticket is not drawn before both exchanges have returned
        shared.last = __hip_atomic_fetch_add(&guard[2], one, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (unsigned long long)check.blocks - 1;
    }
    __syncthreads();
    if (!shared.last) return;
    // the last workgroup adds the pairs of all workgroups: one load per thread, all in flight together (a loop of
    // dependent loads per lane costs a memory round trip per step)
    static_assert(kCheckBlocks <= kCheckThreads, "one thread per pair");
    unsigned long long hs = 0, bs = 0;
    if (threadIdx.x < (unsigned)check.blocks) {
        hs = __hip_atomic_fetch_add(&guard[8 + 2 * threadIdx.x], 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        bs = __hip_atomic_fetch_add(&guard[9 + 2 * threadIdx.x], 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        hs += __shfl_down(hs, off);
        bs += __shfl_down(bs, off);
    }
    __syncthreads();                                       // (thread 0 has read part[] above)
    if ((threadIdx.x & 63) == 0) { part[0][threadIdx.x >> 6] = hs; part[1][threadIdx.x >> 6] = bs; }
    __syncthreads();
    if (threadIdx.x == 0) {
        hs = 0; bs = 0;
#pragma unroll
        for (int i = 0; i < kCheckThreads / 64; ++i) { hs += part[0][i]; bs += part[1][i]; }
        const unsigned long long verdict = (hs == guard[3] && bs == 0) ? 1ull : 0ull;
        guard[5] = hs;
        guard[6] = bs;
        guard[4] = verdict;
        guard[2] = 0;
        // For the host, one word in pinned host memory: (number of this check << 2) | (verdict << 1) | (bad ids seen).
        // The host polls that word; neither a copy command nor an event is enqueued behind the kernel (an event
        // record between two kernels was measured to open a 6-us gap in front of the second).
        __hip_atomic_store(check.host_mirror, (check.seq << 2) | (verdict << 1) | (bs != 0 ? 1ull : 0ull), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

}  // namespace ffi

#endif  // FFI_CHECK_H
