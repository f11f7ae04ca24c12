// Ranks of registry entries among runs of sorted keys: their places when a
// registry is put in order by counting (k_reg_tile_sort, k_reg_merge).
//
// Keys may repeat (a caller's list of pairs names a pair twice, or a soup with
// three faces on an edge is refused only after its kernels ran), and a place
// that two entries take leaves another unwritten, to be read as an index.  So
// equal keys keep their order, as in a stable sort: those of the run or tile
// that comes first go before the other's.
//
// Usable on the host, where a test holds the places to a stable sort.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mcgpu {

using RegKey = unsigned long long;

// place of the own-th of 16 keys among them
__host__ __device__ __forceinline__ uint32_t reg_rank16(const RegKey* group, uint32_t own, RegKey k)
{
    uint32_t below = 0;
#pragma unroll
    for (uint32_t q = 0; q < 16; ++q) below += group[q] < k || (q < own && group[q] == k);
    return below;
}

// keys of a sorted run of w (a power of two) that go before k, which belongs to
// a run after it (first) or before it.  No key is all ones (its face is below
// the face count): k + 1 does not wrap.
__host__ __device__ __forceinline__ uint32_t reg_rank_run(const RegKey* run, uint32_t w, bool first, RegKey k)
{
    const RegKey past = k + (first ? 1 : 0);
    uint32_t lo = 0;
    for (uint32_t h = w >> 1; h > 0; h >>= 1) lo += run[lo + h - 1] < past ? h : 0u;
    return lo + (run[lo] < past);
}

// the same for N sorted tiles of up to 4096 keys at once: 13 halvings cover
// 4096, every load unconditional (a load behind a branch is waited for at
// once), so that the N are in flight together.  len 0: no tile; lo: 0 before,
// the places after.
template <int N>
__host__ __device__ __forceinline__ void reg_rank_tiles(const RegKey* const (&tile)[N], const bool (&first)[N], uint32_t (&len)[N],
                                                        uint32_t (&lo)[N], RegKey k)
{
    RegKey past[N];
#pragma unroll
    for (int q = 0; q < N; ++q) past[q] = k + (first[q] ? 1 : 0);
    for (int step = 0; step < 13; ++step) {
        RegKey v[N];
#pragma unroll
        for (int q = 0; q < N; ++q) v[q] = tile[q][len[q] ? lo[q] + (len[q] >> 1) : 0];
#pragma unroll
        for (int q = 0; q < N; ++q) {
            const uint32_t half = len[q] >> 1;
            const bool right = len[q] && v[q] < past[q];
            lo[q] += right ? half + 1 : 0;
            len[q] = right ? len[q] - half - 1 : half;
        }
    }
}

} // namespace mcgpu
