/*
 * item_layout.h - how the work items of a launch window are dealt to the item shards of the wavefront loop.
 * Plain integer arithmetic, compiled for the host (tests, the host side of a render) and for the gfx950 kernels.
 */
#pragma once
#include <stdint.h>

#if defined(__HIPCC__)
#define VVPT_SHD __host__ __device__ __forceinline__
#else
#define VVPT_SHD inline
#endif

namespace vvpt {

constexpr uint32_t kShards = 64;

/*
 * Work items are split into kShards shards with one counter each, in one of two layouts:
 *   contiguous (chunk 0): shard s holds items [s*per, s*per + size_s) - neighbouring pixels stay together;
 *   chunked: chunk k (items [k*chunk, (k+1)*chunk)) belongs to shard k % kShards, so all shards walk the item
 *            order at the same pace and items early in the order finish first (a batched render puts its
 *            shortest jobs first).
 * Shard s's counter starts at per - size_s (the host sets it), so every shard is drained when its counter
 * reaches `per` = the largest shard size.
 */
VVPT_SHD uint32_t item_shard_size(uint32_t total, uint32_t per, uint32_t chunk, uint32_t s) {
    if (chunk == 0u) {
        const uint64_t first = (uint64_t)s * per;
        return first < total ? (uint32_t)(total - first < per ? total - first : per) : 0u;
    }
    const uint32_t full = total / chunk, rem = total % chunk;
    uint32_t n = (full / kShards + (s < full % kShards ? 1u : 0u)) * chunk;
    if (rem != 0u && full % kShards == s) n += rem;
    return n;
}
/* Item at position p (0 <= p < size_s) of shard s. */
VVPT_SHD uint32_t item_at(uint32_t per, uint32_t chunk, uint32_t s, uint32_t p) {
    if (chunk == 0u) return s * per + p;
    return ((p / chunk) * kShards + s) * chunk + p % chunk;
}

/*
 * Queue shards.  Every producer of a queue is a kernel whose wave with first input index i0 (a multiple of 64,
 * i0 < nslots) appends to shard (i0 / 64) % kShards, at most 64 entries per record kind it emits; one shard
 * therefore serves at most ceil(nslots / (64 kShards)) waves and receives at most 64 entries per wave and record
 * kind.  queue_shard_capacity is that bound (plus one wave of slack) for one record per slot; a queue that can
 * receive k records of one slot in one iteration needs k times as much.
 */
VVPT_SHD uint32_t queue_shard_capacity(uint64_t nslots) {
    return (uint32_t)(((nslots + 64u * kShards - 1u) / (64u * kShards)) * 64u + 64u);
}
constexpr uint32_t kExtendRecords = 1;    /* the slot's ray (each of the two extension queues) */
constexpr uint32_t kSecondaryRecords = 3; /* light-sample segment, emitter lookup of the previous and the last bounce */
constexpr uint32_t kShadowRecords = 2;    /* light-sample segment, 1 - alpha product in front of a found emitter */
constexpr uint32_t kQueryRecords = 1;     /* radiance-cache query */
/* Queue storage in units of kShards * queue_shard_capacity(nslots) entries. */
constexpr uint32_t kQueueBlocks = 2 * kExtendRecords + kSecondaryRecords + kShadowRecords + kQueryRecords;


}  // namespace vvpt
