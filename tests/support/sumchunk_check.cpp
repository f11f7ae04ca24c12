// Host replica of the coordinate sums' kernels (k_head's tile sums, k_sum_items,
// k_sum_chain, k_sum_verify) over mcut_amd/csrc/sumseg.hpp: tiles of 64 chunks of
// 64 values, predictions added in the kernels' order, a tile's adds padded to
// 16, the chain with its rows of 16 adds, every chunk checked on its own start,
// and the values one by one from the first chunk that failed.
// Usage: sumchunk_check FILE, doubles; prints the chain's adds, the most of one
// chunk, the values replayed, and whether the sum is the left-to-right one.
#include <cmath>
#include <cstdio>
#include <vector>

#include "sumseg.hpp"

using namespace mcgpu;

constexpr size_t kThreads = 64, kTile = kThreads * kSumChunk;

static double tree(std::vector<double> t) // 64 lanes, __shfl_xor
{
    for (int o = 32; o > 0; o >>= 1) {
        std::vector<double> u(64);
        for (int i = 0; i < 64; ++i) u[i] = t[i] + t[i ^ o];
        t = u;
    }
    return t[0];
}

int main(int argc, char** argv)
{
    std::vector<double> x;
    FILE* f = argc > 1 ? fopen(argv[1], "rb") : nullptr;
    if (!f) return 2;
    for (double v; fread(&v, sizeof v, 1, f) == 1;) x.push_back(v);
    fclose(f);
    const size_t n = x.size(), tiles = (n + kTile - 1) / kTile;
    double want = 0.0;
    for (double v : x) want = want + v;

    std::vector<double> bsum(tiles);
    for (size_t b = 0; b < tiles; ++b) {
        double red[4];
        for (int w = 0; w < 4; ++w) {
            std::vector<double> t(64, 0.0);
            for (int l = 0; l < 64; ++l)
                for (size_t q = 0; q < kTile / 256; ++q) {
                    const size_t i = b * kTile + q * 256 + w * 64 + l;
                    t[l] += i < n ? x[i] : 0.0;
                }
            red[w] = tree(t);
        }
        bsum[b] = (red[0] + red[1]) + (red[2] + red[3]);
    }
    std::vector<std::vector<SumItem>> items(tiles * kThreads);
    std::vector<std::vector<double>> tadds(tiles);
    std::vector<size_t> off(tiles * kThreads), first(tiles);
    size_t most = 0, total = 0;
    for (size_t b = 0; b < tiles; ++b) {
        std::vector<double> t(64, 0.0);
        for (size_t q = 0; q < b; ++q) t[q % 64] += bsum[q];
        const double a0 = tree(t);
        std::vector<double> y(64, 0.0);
        for (size_t c = 0; c < kThreads; ++c)
            for (size_t k = 0; k < (size_t)kSumChunk; ++k) {
                const size_t i = b * kTile + c * kSumChunk + k;
                y[c] += i < n ? x[i] : 0.0;
            }
        for (int o = 1; o < 64; o <<= 1) { // __shfl_up
            std::vector<double> z = y;
            for (int l = o; l < 64; ++l) z[l] = y[l] + y[l - o];
            y = z;
        }
        for (size_t c = 0; c < kThreads; ++c) {
            const size_t g = b * kThreads + c, i0 = b * kTile + c * kSumChunk;
            SumWalk W;
            sum_restart(W, c ? a0 + y[c - 1] : a0);
            off[g] = tadds[b].size();
            auto emit = [&](const SumItem& it) {
                double a[kSumMaxAdds];
                const int k = sum_add_list(it, a);
                tadds[b].insert(tadds[b].end(), a, a + k);
                items[g].push_back(it);
            };
            for (size_t i = i0; i < i0 + kSumChunk && i < n; ++i) sum_step(W, x[i], emit);
            sum_close(W, emit);
            most = std::max(most, tadds[b].size() - off[g]);
        }
        while (tadds[b].size() % 16) tadds[b].push_back(0.0);
        first[b] = total;
        total += tadds[b].size();
    }
    std::vector<double> rows;
    double acc = 0.0;
    size_t k = 0;
    for (const auto& t : tadds)
        for (double a : t) {
            acc = acc + a;
            if (++k % 16 == 0) rows.push_back(acc);
        }
    size_t replayed = 0;
    for (size_t g = 0; g * kSumChunk < n && !replayed; ++g) {
        const size_t b = g / kThreads, o16 = off[g] & ~(size_t)15, row = (first[b] + o16) / 16;
        double s = row ? rows[row - 1] : 0.0;
        for (size_t q = o16; q < off[g]; ++q) s = s + tadds[b][q];
        const double start = s;
        bool ok = true;
        for (const SumItem& it : items[g]) {
            double end = s + it.p, d;
            bool odd;
            if (!sum_is_step(it)) ok &= sum_apply(it, s, &end, &d, &odd);
            s = end;
        }
        if (!ok) {
            replayed = n - g * kSumChunk;
            acc = start;
            for (size_t i = g * kSumChunk; i < n; ++i) acc = acc + x[i];
        }
    }
    const bool same = sum_bits(acc) == sum_bits(want) || (std::isnan(acc) && std::isnan(want));
    printf("n=%zu adds=%zu most=%zu replayed=%zu %s\n", n, total, most, replayed, same ? "ok" : "WRONG");
    return !same || most > (size_t)kSumChunkAdds;
}
