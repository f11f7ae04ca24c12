// Blocks of k_pairs_start: tiles of kPairTileSrc source items (one a thread) by
// kPairTileCut cut items, all in the grid's x.  The launchers bound the product
// of the counts, not each of them, and y holds 65,535 blocks: 12 source faces
// against more than 2,097,120 cut faces would not fit it.
//
// Usable on the host, where a test holds the launches to the device's limits.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mcgpu {

constexpr uint32_t kPairTileSrc = 256, kPairTileCut = 32;

__host__ __device__ inline uint32_t pair_src_tiles(uint32_t ns) { return (uint32_t)(((uint64_t)ns + kPairTileSrc - 1) / kPairTileSrc); }

inline uint64_t pair_blocks(uint32_t ns, uint32_t nc)
{
    return pair_src_tiles(ns) * (((uint64_t)nc + kPairTileCut - 1) / kPairTileCut);
}

// first source and cut item of a block
__host__ __device__ inline void pair_tile(uint32_t block, uint32_t ns, uint32_t* s, uint32_t* c)
{
    const uint32_t row = block / pair_src_tiles(ns);
    *s = (block - row * pair_src_tiles(ns)) * kPairTileSrc;
    *c = row * kPairTileCut;
}

} // namespace mcgpu
