// Host check of mcut_amd/csrc/pairgrid.hpp: the launches of k_pairs_start stay
// within the device's grid (2^31 - 1 blocks and 2^32 - 1 threads in x; all the
// blocks are in x, as y holds 65,535) for every pair of counts whose product its launchers allow, and
// its blocks cover every pair of items once; and those of k_batch_bbox do not
// grow with the product of the pairs and the largest mesh.
#include <cstdio>
#include <vector>

#include "pairgrid.hpp"

using namespace mcgpu;

int main()
{
    int bad = 0;
    auto fits = [&](uint32_t ns, uint32_t nc) {
        const uint64_t n = pair_blocks(ns, nc);
        if (n < 1 || n > 0x7fffffffull || n * kPairTileSrc > 0xffffffffull) {
            if (bad < 8) printf("%u x %u: %llu blocks\n", ns, nc, (unsigned long long)n);
            ++bad;
        }
    };
    for (int most : {22, 26}) // node pairs of the start levels; face pairs
        for (uint64_t ns = 1; ns <= 1ull << most; ns += 1 + ns / 7) {
            const uint32_t nc = (uint32_t)((1ull << most) / ns);
            fits((uint32_t)ns, nc);
            fits(nc, (uint32_t)ns);
        }
    for (uint32_t ns : {1u, 31u, 256u, 257u, 700u})
        for (uint32_t nc : {1u, 32u, 33u, 256u, 1000u}) {
            std::vector<int> seen((size_t)ns * nc, 0);
            for (uint32_t b = 0; b < pair_blocks(ns, nc); ++b) {
                uint32_t s0, c0;
                pair_tile(b, ns, &s0, &c0);
                bad += s0 >= ns || c0 >= nc;
                for (uint32_t s = s0; s < s0 + kPairTileSrc && s < ns; ++s)
                    for (uint32_t c = c0; c < c0 + kPairTileCut && c < nc; ++c) ++seen[(size_t)s * nc + c];
            }
            for (int n : seen) bad += n != 1;
        }
    // raw boxes of a batch: every mesh has a block, few are empty, y holds them
    for (uint32_t np : {1u, 2u, 96u, 320u, 4096u, 40000u, 1u << 20})
        for (uint32_t tiles : {1u, 2u, 25u, 245u, 2442u, 60000u, 300000u}) {
            const uint64_t rows = batch_box_rows(np, tiles), blocks = 2ull * np * rows;
            if (rows < 1 || rows > tiles || rows > 65535u || blocks > (2ull * np > (1u << 16) ? 2ull * np : 1u << 16)) {
                if (bad < 8) printf("%u pairs, %u tiles: %llu blocks\n", np, tiles, (unsigned long long)blocks);
                ++bad;
            }
        }
    printf("bad %d\n", bad);
    return bad != 0;
}
