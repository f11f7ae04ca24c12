// Host check of mcut_amd/csrc/sumseg.hpp: sums composed from segments through
// two levels, with replays where a check fails, against the left-to-right sum.
// Prints, per input: name, values, items of each level, replayed values, ok.
#include <cmath>
#include <cstdio>
#include <functional>
#include <random>
#include <string>
#include <vector>

#include "sumseg.hpp"

using namespace mcgpu;

static double seq(const std::vector<double>& x, size_t a, size_t b, double s)
{
    for (size_t i = a; i < b; ++i) s = s + x[i];
    return s;
}

struct Result {
    size_t l1 = 0, l2 = 0, replayed = 0;
    double sum = 0;
    bool wrong = false;
};

static Result run(const std::vector<double>& x, size_t chunk, size_t groups, double off, double rel)
{
    Result R;
    std::vector<SumItem> l1, l2;
    std::vector<size_t> first;
    std::vector<std::pair<size_t, size_t>> starts; // a group's first item and first value
    // predicted starts from block sums in another order, pushed off by off + rel
    double pre = 0;
    for (size_t c = 0; c < x.size(); c += chunk) {
        const size_t e = std::min(x.size(), c + chunk);
        first.push_back(l1.size());
        SumWalk W;
        sum_restart(W, c ? pre * (1 + rel) + off : 0.0);
        auto emit = [&](const SumItem& it) { l1.push_back(it); };
        for (size_t i = c; i < e; ++i) sum_step(W, x[i], emit);
        sum_close(W, emit);
        double t = 0;
        for (size_t i = e; i-- > c;) t += x[i];
        pre += t;
    }
    first.push_back(l1.size());
    const size_t nc = first.size() - 1, per = (nc + groups - 1) / groups;
    for (size_t g = 0; g < nc; g += per) {
        const size_t a = first[g], b = first[std::min(nc, g + per)];
        starts.push_back({l2.size(), g * chunk});
        SumWalk W;
        sum_restart(W, sum_is_step(l1[a]) ? l1[a].q : l1[a].p);
        auto emit = [&](const SumItem& it) { l2.push_back(it); };
        for (size_t k = a; k < b; ++k) sum_compose(W, l1[k], emit);
        sum_close(W, emit);
    }
    R.l1 = l1.size();
    R.l2 = l2.size();
    // as the GPU does: every group on its real start, and from the first group
    // with an item that does not move with it the values one by one
    double s = 0.0;
    for (size_t g = 0; g < starts.size(); ++g) {
        const double at = s;
        bool ok = true;
        for (size_t k = starts[g].first; k < (g + 1 < starts.size() ? starts[g + 1].first : l2.size()) && ok; ++k) {
            double end = s + l2[k].p, d, a[kSumMaxAdds], w = s;
            bool odd;
            if (!sum_is_step(l2[k])) ok = sum_apply(l2[k], s, &end, &d, &odd);
            for (int q = 0, n = sum_add_list(l2[k], a); q < n; ++q) w = w + a[q];
            if (ok && sum_bits(w) != sum_bits(end) && !std::isnan(end)) {
                printf("the adds do not carry a start to its end\n");
                R.wrong = true;
            }
            s = end;
        }
        if (!ok) {
            R.replayed = x.size() - starts[g].second;
            s = seq(x, starts[g].second, x.size(), at);
            break;
        }
    }
    R.sum = s;
    return R;
}

int main()
{
    std::mt19937_64 g(11);
    std::normal_distribution<double> N;
    std::uniform_real_distribution<double> U(-1.0, 1.0);
    int bad = 0;
    auto check = [&](const std::string& name, const std::vector<double>& x, bool report) {
        const double want = seq(x, 0, x.size(), 0.0);
        for (size_t chunk : {7, 32, 64})
            for (size_t groups : {3, 64, 256})
                for (double rel : {0.0, 1e-13, 1e-6})
                    for (double off : {0.0, 1e-9, 0.37}) {
                        const Result R = run(x, chunk, groups, off, rel);
                        const bool ok = !R.wrong && (sum_bits(R.sum) == sum_bits(want) || (std::isnan(want) && std::isnan(R.sum)));
                        bad += !ok;
                        if (!ok || (report && chunk == 64 && groups == 64 && rel == 0 && off == 0))
                            printf("%s n=%zu l1=%zu l2=%zu replayed=%zu %s\n", name.c_str(), x.size(), R.l1, R.l2, R.replayed,
                                   ok ? "ok" : "WRONG");
                    }
    };
    auto make = [](size_t n, std::function<double(size_t)> f) {
        std::vector<double> x(n);
        for (size_t i = 0; i < n; ++i) x[i] = f(i);
        return x;
    };
    const double pi = std::acos(-1.0);
    for (size_t n : {1, 2, 63, 64, 65, 6000, 60000}) {
        const bool r = n == 60000;
        check("hover", make(n, [&](size_t) { return U(g); }), r);
        check("normal", make(n, [&](size_t) { return N(g); }), r);
        check("positive", make(n, [&](size_t) { return 1.0 + 0.5 * U(g); }), r);
        check("offset", make(n, [&](size_t) { return 0.4 + 0.02 * U(g); }), r);
        check("rings", make(n, [&](size_t i) { return std::sin(2 * pi * (double)(i % 64) / 64) * (1 + (double)(i / 64 % 16)); }), r);
        check("grid", make(n, [&](size_t i) { return (double)(i / 245); }), r);
        check("gridz", make(n, [&](size_t) { return std::rint(4096 * U(g)) / 4096; }), r);
        check("thirds", make(n, [&](size_t i) { return ((double)(i % 31) - 15.0) / 30.0; }), r);
        check("ties", make(n, [&](size_t) { return std::ldexp(1.0, 52) + (double)(g() % 4) + 0.5; }), r);
        check("halves", make(n, [&](size_t i) { return i == 0 ? std::ldexp(1.0, 53) : (double)(g() % 3) - 1.0 + 0.5; }), r);
        check("tiny", make(n, [&](size_t) { return N(g) * 1e-290; }), r);
        check("denormal", make(n, [&](size_t) { return N(g) * 1e-310; }), r);
        check("huge", make(n, [&](size_t) { return N(g) * 1e290; }), r);
        check("scales", make(n, [&](size_t) { return N(g) * std::pow(10.0, (double)(g() % 17) - 8); }), r);
        check("zeros", make(n, [&](size_t i) { return i % 5 ? 0.0 : U(g); }), r);
        check("cancel", make(n, [&](size_t i) { return (i & 1 ? -1 : 1) * (1.0 + (double)(i / 2) * 1e-3); }), r);
        check("walk", make(n, [&](size_t i) { return 3 * std::cos(i * 1e-3) + 1e-3 * U(g); }), r);
        check("powers", make(n, [&](size_t i) { return std::ldexp(i & 1 ? -1.0 : 1.0, (int)(i % 40) - 20); }), r);
        check("inf", make(n, [&](size_t i) { return i == n / 2 ? INFINITY : U(g); }), false);
        check("nan", make(n, [&](size_t i) { return i == n / 2 ? NAN : U(g); }), false);
    }
    printf("bad %d\n", bad);
    return bad != 0;
}
