/*
 * lists.hpp - work lists of several parts, read by whole waves.
 */
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace lyap {

__device__ __forceinline__ uint32_t uniform(uint32_t x)
{
    return __builtin_amdgcn_readfirstlane(x);
}

/* The chunks of up to 64 lists, held across a wave: lane j holds list j's
 * entry count and the chunks of lists 0..j (an inclusive scan), so a chunk
 * finds its list with one ballot. The counts come in one vector load rather
 * than a walk of dependent scalar loads at every wave's start. */
struct ChunkMap {
    uint32_t cnt;      /* lane j: entries of list j (0 past the lists) */
    uint32_t end;      /* lane j: chunks of lists 0..j */
    uint32_t total;    /* chunks of all lists */
};

__device__ __forceinline__ ChunkMap chunk_map(uint32_t cnt, uint32_t per, uint32_t lane)
{
    ChunkMap m;
    m.cnt = cnt;
    uint32_t x = (cnt + per - 1u) / per;
#pragma unroll
    for (uint32_t off = 1; off < 64u; off <<= 1) {
        const uint32_t y = (uint32_t)__shfl_up((int)x, off);
        if (lane >= off) x += y;
    }
    m.end = x;
    m.total = uniform((uint32_t)__shfl((int)x, 63));
    return m;
}

/* List p holding chunk c (< m.total), the chunks before p and p's entries.
 * Every lane of the wave takes part. */
__device__ __forceinline__ void chunk_find(const ChunkMap &m, uint32_t c, uint32_t per, uint32_t &p,
                                           uint32_t &acc, uint32_t &cnt)
{
    p = uniform((uint32_t)__popcll(__ballot(m.end <= c)));
    cnt = uniform((uint32_t)__shfl((int)m.cnt, (int)p));
    acc = uniform((uint32_t)__shfl((int)m.end, (int)p)) - (cnt + per - 1u) / per;
}

} /* namespace lyap */
