// Host check of mcut_amd/csrc/regrank.hpp: the places that the registry's tile
// sort (groups of 16, runs merged two to one) and its merge across tiles give
// every entry, against a stable sort, with keys that repeat.  Prints, per
// input, the entries, those past the first of their key, and ok.
#include <algorithm>
#include <cstdio>
#include <numeric>
#include <random>
#include <vector>

#include "regrank.hpp"

using namespace mcgpu;

constexpr uint32_t kTile = 4096, kRunMax = 2048;

static std::vector<uint32_t> stable(const std::vector<RegKey>& k)
{
    std::vector<uint32_t> o(k.size()), place(k.size());
    std::iota(o.begin(), o.end(), 0u);
    std::stable_sort(o.begin(), o.end(), [&](uint32_t a, uint32_t b) { return k[a] < k[b]; });
    for (uint32_t i = 0; i < o.size(); ++i) place[o[i]] = i;
    return place;
}

// the runs of k_reg_tile_sort: the place of every entry of one tile
static std::vector<uint32_t> runs(const std::vector<RegKey>& key)
{
    const uint32_t cnt = (uint32_t)key.size(), P = cnt <= 16 ? 16u : 1u << (32 - __builtin_clz(cnt - 1));
    std::vector<RegKey> K(P), sk(P, ~0ull);
    std::vector<uint32_t> pos(P), at(P);
    for (uint32_t i = 0; i < P; ++i) sk[i] = K[i] = i < cnt ? key[i] : (1ull << 63) | i;
    for (uint32_t i = 0; i < P; ++i) pos[i] = (i & ~15u) + reg_rank16(&sk[i & ~15u], i & 15u, K[i]);
    for (uint32_t w = 16; w < cnt; w <<= 1) {
        for (uint32_t i = 0; i < P; ++i) sk[pos[i]] = K[i];
        for (uint32_t i = 0; i < P; ++i) {
            const uint32_t other = (pos[i] & ~(w - 1)) ^ w;
            at[i] = (pos[i] & ~(2 * w - 1)) + (pos[i] & (w - 1)) + reg_rank_run(&sk[other], w, (other & w) == 0, K[i]);
        }
        pos = at;
    }
    pos.resize(cnt);
    return pos;
}

// the ranks of k_reg_merge over sorted tiles
static std::vector<uint32_t> merged(const std::vector<RegKey>& key)
{
    constexpr int N = 8;
    const uint32_t n = (uint32_t)key.size(), ntiles = (n + kTile - 1) / kTile;
    std::vector<RegKey> s(n);
    std::vector<uint32_t> from(n), place(n);
    for (uint32_t t = 0; t < ntiles; ++t) { // each tile in (stable) order, whichever sort made it
        const uint32_t a = t * kTile, b = std::min(n, a + kTile);
        std::vector<RegKey> part(key.begin() + a, key.begin() + b);
        const std::vector<uint32_t> p = part.size() <= kRunMax ? runs(part) : stable(part);
        for (uint32_t i = a; i < b; ++i) s[a + p[i - a]] = key[i], from[a + p[i - a]] = i;
    }
    for (uint32_t i = 0; i < n; ++i) {
        const uint32_t t = i / kTile;
        uint32_t rank = i - t * kTile;
        for (uint32_t u0 = ntiles > 1 ? 0 : 1; u0 < ntiles; u0 += N) {
            const RegKey* tile[N];
            bool first[N];
            uint32_t lo[N], len[N];
            for (int q = 0; q < N; ++q) {
                const uint32_t u = u0 + q, base = u * kTile;
                const bool other = u < ntiles && u != t;
                tile[q] = s.data() + (other ? base : 0);
                first[q] = u < t;
                lo[q] = 0;
                len[q] = other ? std::min(n - base, kTile) : 0u;
            }
            reg_rank_tiles<N>(tile, first, len, lo, s[i]);
            for (int q = 0; q < N; ++q) rank += lo[q];
        }
        place[from[i]] = rank;
    }
    return place;
}

int main()
{
    std::mt19937_64 g(3);
    int bad = 0;
    for (uint32_t n : {1, 2, 3, 15, 16, 17, 31, 33, 50, 64, 65, 257, 1000, 1025, 2047, 2048, 4097, 9000, 40000})
        for (uint32_t distinct : {1u, 2u, std::max(1u, n / 16), std::max(1u, n / 2), n, 1u << 30}) {
            std::vector<RegKey> k(n);
            for (auto& x : k) x = distinct >> 30 ? g() >> 2 : g() % distinct;
            std::vector<RegKey> u = k;
            std::sort(u.begin(), u.end());
            const size_t repeats = n - (std::unique(u.begin(), u.end()) - u.begin());
            const std::vector<uint32_t> want = stable(k);
            const bool ok = merged(k) == want && (n > kRunMax || runs(k) == want);
            bad += !ok;
            printf("n=%u repeats=%zu %s\n", n, repeats, ok ? "ok" : "WRONG");
        }
    printf("bad %d\n", bad);
    return bad != 0;
}
