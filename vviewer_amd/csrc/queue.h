/*
 * queue.h - sharded work queues for the wavefront loop.
 *
 * Atomics on one address serialize in L2 (about 11 ns each on MI355X, against
 * about 0.3 ns when spread over separate cache lines), so every queue is split
 * into kShards shards, each with its own counter on its own 128-byte line.
 * Producers: a wave appends to the shard picked by the position of its input
 * chunk, one atomic per wave.  Consumers: persistent kernels fetch from a home
 * shard and move on to the next shard when it is drained; grid-stride kernels
 * map a global index to (shard, offset) through an LDS prefix sum.
 */
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "item_layout.h"

namespace vvpt {

constexpr uint32_t kPad = 32; /* uint32 per counter: one 128-byte line each */

struct SQueue {
    uint32_t *data;   /* kShards * cap entries */
    uint32_t *count;  /* kShards padded counters: entries appended */
    uint32_t *fetch;  /* kShards padded counters: entries handed out to persistent consumers */
    uint32_t cap;     /* entries per shard */
};

__device__ __forceinline__ uint32_t *sq_count(const SQueue &q, uint32_t s) { return q.count + s * kPad; }
__device__ __forceinline__ uint32_t *sq_fetch(const SQueue &q, uint32_t s) { return q.fetch + s * kPad; }

/* Shard of the wave whose first input index is `i0` (a multiple of 64). */
__device__ __forceinline__ uint32_t shard_of(uint32_t i0) { return (i0 >> 6) % kShards; }

/* Zero counters (and fetch counters) of a queue; call from any kKernel with >= kShards threads in block 0. */
__device__ __forceinline__ void sq_reset(const SQueue &q) {
    if (blockIdx.x == 0 && threadIdx.x < kShards) {
        q.count[threadIdx.x * kPad] = 0u;
        q.fetch[threadIdx.x * kPad] = 0u;
    }
}
__device__ __forceinline__ void sq_reset_fetch(const SQueue &q) {
    if (blockIdx.x == 0 && threadIdx.x < kShards) q.fetch[threadIdx.x * kPad] = 0u;
}

/* Wave-aggregated append of `pred` lanes to shard s.  Every lane of the wave must call it. */
__device__ __forceinline__ void sq_append(const SQueue &q, uint32_t s, bool pred, uint32_t value) {
    const unsigned long long mask = __ballot(pred);
    if (mask == 0ull) return;
    const uint32_t lane = __lane_id();
    const int leader = __ffsll((long long)mask) - 1;
    uint32_t base = 0;
    if ((int)lane == leader) base = atomicAdd(sq_count(q, s), (uint32_t)__popcll(mask));
    base = __shfl(base, leader);
    if (pred) q.data[s * q.cap + base + (uint32_t)__popcll(mask & ((1ull << lane) - 1ull))] = value;
}

/* Block-wide view of a queue's shard prefix sums (LDS), for grid-stride consumers. */
struct SQView {
    uint32_t pre[kShards + 1];
};
/* The block's first wave loads one shard counter per lane and scans them (six shuffle steps) instead of one lane
 * summing all 64 in sequence; needs blockDim.x >= 64. */
static_assert(kShards == 64, "one shard per lane of a wave");
__device__ __forceinline__ void sq_view_load(const SQueue &q, SQView &v) {
    if (threadIdx.x < kShards) {
        const uint32_t s = threadIdx.x;
        const uint32_t c = *sq_count(q, s);
        uint32_t x = c;
#pragma unroll
        for (uint32_t off = 1; off < kShards; off <<= 1) {
            const uint32_t y = __shfl_up(x, off);
            if (s >= off) x += y;
        }
        v.pre[s] = x - c;
        if (s == kShards - 1u) v.pre[kShards] = x;
    }
    __syncthreads();
}
/* entry at global index i < total */
__device__ __forceinline__ uint32_t sq_at(const SQueue &q, const SQView &v, uint32_t i) {
    uint32_t lo = 0, hi = kShards; /* largest s with pre[s] <= i */
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (v.pre[mid] <= i)
            lo = mid;
        else
            hi = mid;
    }
    return q.data[lo * q.cap + (i - v.pre[lo])];
}

/* Wave-wide search for a shard (starting at `from`) whose counter is below
 * its limit; lane l inspects shard (from + l) % kShards.  Returns kShards if
 * none.  The counters are read racily: the atomic that follows decides. */
__device__ __forceinline__ uint32_t find_shard(const uint32_t *ctr, const uint32_t *limit, uint32_t limit_const,
                                               uint32_t from) {
    const uint32_t lane = __lane_id();
    const uint32_t s = (from + lane) % kShards;
    bool has = false;
    if (lane < kShards) {
        const uint32_t lim = limit ? limit[s * kPad] : limit_const;
        has = ctr[s * kPad] < lim;
    }
    const unsigned long long m = __ballot(has);
    if (m == 0ull) return kShards;
    return (from + (uint32_t)(__ffsll((long long)m) - 1)) % kShards;
}

/*
 * Persistent-consumer fetch: idle lanes of the wave take entries from the
 * current shard (one atomic per refill); when the shard is drained the wave
 * looks for another one.  Returns true for lanes that received `value`.
 * `shard` and `done` are wave-uniform state owned by the caller.
 */
constexpr uint32_t kRefill = 16; /* refill once this many lanes of the wave are idle */
__device__ __forceinline__ bool sq_refill(const SQueue &q, bool idle, uint32_t &shard, bool &done, uint32_t &value) {
    unsigned long long im = __ballot(idle);
    if (done || (uint32_t)__popcll(im) < kRefill) return false;
    bool got = false;
    const uint32_t lane = __lane_id();
    while (im != 0ull && !done) {
        /* shard counts were final when this kernel started (their producers ran before it) */
        const uint32_t n = *sq_count(q, shard);
        const uint32_t req = (uint32_t)__popcll(im);
        const int leader = __ffsll((long long)im) - 1;
        uint32_t base = 0;
        if ((int)lane == leader) base = atomicAdd(sq_fetch(q, shard), req);
        base = __shfl(base, leader);
        const uint32_t take = base < n ? min(n - base, req) : 0u;
        const bool mine = ((im >> lane) & 1ull) != 0ull;
        const uint32_t rank = (uint32_t)__popcll(im & ((1ull << lane) - 1ull));
        const bool serve = mine && rank < take;
        if (serve) {
            value = q.data[shard * q.cap + base + rank];
            got = true;
        }
        im &= ~__ballot(serve); /* served lanes leave the idle mask */
        if (base + req >= n) {  /* drained: find another shard */
            const uint32_t nx = find_shard(q.fetch, q.count, 0u, shard);
            if (nx == kShards)
                done = true;
            else
                shard = nx;
        }
    }
    return got;
}

/* Lanes with `need` get the next items of the wave's current shard, then of other shards.  Returns true for
 * served lanes. */
__device__ __forceinline__ bool item_fetch(uint32_t *ctr, uint32_t total, uint32_t per, uint32_t chunk, bool need,
                                           uint32_t &shard, uint32_t &item) {
    unsigned long long im = __ballot(need);
    bool got = false;
    const uint32_t lane = __lane_id();
    while (im != 0ull) {
        const uint32_t skip = per - item_shard_size(total, per, chunk, shard);
        const uint32_t req = (uint32_t)__popcll(im);
        const int leader = __ffsll((long long)im) - 1;
        uint32_t base = 0;
        if ((int)lane == leader) base = atomicAdd(ctr + shard * kPad, req);
        base = __shfl(base, leader);
        const uint32_t take = base < per ? min(per - base, req) : 0u;
        const bool mine = ((im >> lane) & 1ull) != 0ull;
        const uint32_t rank = (uint32_t)__popcll(im & ((1ull << lane) - 1ull));
        const bool serve = mine && rank < take;
        if (serve) {
            item = item_at(per, chunk, shard, base + rank - skip);
            got = true;
        }
        im &= ~__ballot(serve);
        if (im != 0ull) {
            const uint32_t nx = find_shard(ctr, nullptr, per, shard);
            if (nx == kShards) break;
            shard = nx;
        }
    }
    return got;
}

}  // namespace vvpt
