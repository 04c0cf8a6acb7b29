// fetch.h -- work distribution of the persistent traversal kernels, and the
// block-wide queue append of the kernels that fill their queues.
//
// The items [0, total) of one launch are split into kFetchParts contiguous
// partitions, each with its own fetch head; heads sit kHeadStride words (128 B)
// apart so that no two share a cache line.  A wave starts on partition wave %
// kFetchParts, claims items from its head with one atomic per refill, and moves on to the next
// partition when its own is used up.  Refills then spread their atomics over 64
// addresses instead of one, which is what lets a wave refill its idle lanes
// often.  Every item is claimed exactly once.
//
// The wave whose claim takes a partition's last item sets the partition's bit in the
// queue's used-up word, and a wave that finds its partition used up is done once
// all bits are set.  Atomics on one address are served one after the other, about
// 15 ns each: with a claim in vain on every partition, 4096 waves needed 60 us to
// find the end of a queue, however small it was, and each of those claims held up the
// rays still in flight.  Cornell box path-traced 3.76 -> 3.37 ms, a burst of
// server jobs 27.0 -> 21.2 ms, AO of 357x243 pixels 350 -> 307 us, 1920x1080
// 2.38 -> 2.39.  Going straight to a partition that is not used up is slower than the
// walk (2.43 ms): near the end all waves then claim on the same few addresses.
// Fewer items than 64 per partition: one partition, and only as many waves as these fill.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace solhip {

constexpr uint32_t kHeadStride = 32;   // words between two fetch heads
constexpr uint32_t kFetchParts = 64;
constexpr uint32_t kFetchWords = kFetchParts * kHeadStride;   // of one queue; all zero at launch
constexpr uint32_t kUsedUp = 16;       // place of its used-up word (64 bits)

// clears head k of several queues, one after the other, and what stands behind it
__device__ __forceinline__ void fetch_reset(uint32_t *heads, uint32_t k)
{
    heads[k * kHeadStride] = 0;
    heads[k * kHeadStride + kUsedUp] = 0;
    heads[k * kHeadStride + kUsedUp + 1] = 0;
}

struct PartFetch {
    uint32_t *heads;   // kFetchWords words
    uint32_t total, log2p, part, moved, lo, hi;
    bool exhausted;

    __device__ __forceinline__ void bounds()
    {
        lo = (uint32_t)(((uint64_t)total * part) >> log2p);
        hi = (uint32_t)(((uint64_t)total * (part + 1)) >> log2p);
    }

    __device__ __forceinline__ void init(uint32_t *h, uint32_t n_items)
    {
        heads = h;
        total = n_items;
        const uint32_t wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
        log2p = total >= 64u * kFetchParts ? 6u : 0u;
        part = log2p ? wave % kFetchParts : 0u;
        moved = 0;
        exhausted = (uint64_t)wave * 64u >= total;   // the waves before this one take all of a small queue
        bounds();
    }

    // Wave-uniform: claims n items of the current partition.  Returns the
    // first; items base .. min(base + n, end) - 1 are the caller's.
    __device__ __forceinline__ uint32_t claim(uint32_t n, uint32_t &end)
    {
        uint32_t base = 0;
        if ((threadIdx.x & 63u) == 0) base = atomicAdd(heads + part * kHeadStride, n);
        base = lo + __shfl(base, 0);
        end = hi;
        if (base + n >= hi) {
            // used up: on to the next one, unless all are
            unsigned long long *used = reinterpret_cast<unsigned long long *>(heads + kUsedUp);
            const uint64_t bit = 1ull << part;
            if ((threadIdx.x & 63u) == 0 && base < hi) atomicOr(used, bit);   // took the last item
            // one lane's value for the wave: bits are set meanwhile, and lanes that saw
            // different words would part here, some of them without the lane that claims
            const uint64_t word = __hip_atomic_load(used, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const uint32_t low = __builtin_amdgcn_readfirstlane((uint32_t)word);
            const uint32_t high = __builtin_amdgcn_readfirstlane((uint32_t)(word >> 32));
            exhausted = (((uint64_t)high << 32) | low | bit) == (log2p ? ~0ull : 1ull) ||
                        ++moved >= 1u << log2p;   // or this wave has seen every one used up
            if (log2p) {
                part = (part + 1) % kFetchParts;
                bounds();
            }
        }
        return base;
    }
};

// Block-wide append of one item per thread that has one: every thread of the
// block calls it with block-uniform control flow; one atomic per block (a
// producer kernel that appended once per wave put every wave of the GPU on
// one counter address, which limited it).  lds: WAVES + 1 words.
template <uint32_t WAVES>
__device__ __forceinline__ uint32_t block_append(uint32_t *counter, bool pred, uint32_t *lds)
{
    const uint64_t m = __ballot(pred);
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    if (lane == 0) lds[wave] = (uint32_t)__popcll(m);
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t total = 0;
        for (uint32_t w = 0; w < WAVES; ++w) {
            const uint32_t c = lds[w];
            lds[w] = total;
            total += c;
        }
        lds[WAVES] = total ? atomicAdd(counter, total) : 0u;
    }
    __syncthreads();
    const uint32_t base = lds[WAVES] + lds[wave];
    __syncthreads();   // lds is reused by the next call
    return base + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
}

}  // namespace solhip
