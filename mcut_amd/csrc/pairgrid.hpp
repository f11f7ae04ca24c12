// Launch sizes that follow from more than one count.
//
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

// Rows of blocks for the raw boxes of a batch (k_batch_bbox), a column a mesh
// and a row a tile of its vertices: as many as the largest mesh's tiles, but no
// more blocks than kBatchBoxBlocks once every mesh has one, so that one large
// mesh among thousands does not launch its tiles for all of them (10 M vertices
// in 4,096 pairs: 20 M blocks).  Past that a block takes several tiles.
constexpr uint32_t kBatchBoxBlocks = 1u << 16;
inline uint32_t batch_box_rows(uint32_t npairs, uint32_t tiles)
{
    const uint64_t most = kBatchBoxBlocks / (2ull * npairs);
    return most < 1 ? 1u : most < tiles ? (uint32_t)most : tiles;
}

} // namespace mcgpu
