// Left-to-right sums from segments that move with their start.
//
// The reference adds every coordinate of a mesh in order (preproc.cpp:2188-2202)
// and each step rounds, so the sum is a serial chain.  It parallelises because
// a stretch of steps moves rigidly with its start value: let a thread predict
// the partial sum a before its values and add them one after another (real
// adds, real roundings) to b.  A start a + d then ends at b + d, exactly, when
//   - d is a multiple of G, the unit in the last place of the largest binade
//     any partial sum of the stretch reaches (a itself is in that binade: the
//     stretch ends before a step that climbs above it), so every rounding grid
//     of the stretch divides d, and
//   - d lies in an interval [lo, hi] that keeps every partial sum where its
//     rounding grid is the predicted one:
//       an inexact step that ends at t in binade 2^E with unit u: t + d in
//       [2^E + u, 2^(E+1)] (mirrored below zero): the exact value is within
//       u/2 of it, and there the nearest double is the nearest multiple of u;
//       an exact step whose operands (moved by d) are multiples of g = min(G,
//       their lowest set bits): |t + d| <= 2^52 g, where every multiple of g is
//       a double, so the moved step is exact too, whatever its binade (sums
//       that cancel to noise or to zero, and sums of grid coordinates).
// A tie on the grid G resolves by the parity of d / G: an even d as predicted,
// an odd one to the other neighbour, after which the distance is even and every
// later tie resolves as predicted.  So the first tie alone counts: an odd d
// ends at b + d + tie G, tie being the side the prediction rounded away from.
// A climb, a sum on a power of two that neither rule covers, and sums outside
// [2^-900, 2^1000] stay single steps.  The kernels add the items of all chunks
// (7k for 164k values of a sphere) as one chain and check each on the start that
// it then has; from the first chunk with an item that does not move with its
// start the values are added one by one, so a bad prediction costs time and
// never a bit.  The items of a stretch are again a sequence of such steps, which
// the same walk could compose (sum_compose): on the device that cost what the
// shorter chain saved, so only a host test does it.
//
// Usable on the host, where a test holds it to the sequential sum.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mcgpu {

// a segment (p -> q, every start p + d to q + d for d in [lo, hi]; tie as above)
// or, with tie = kSumStep, a single step (+ p, predicted start q)
constexpr int kSumStep = 2;
struct SumItem {
    double p, q, lo, hi;
    int tie, pad;
};

__host__ __device__ inline uint64_t sum_bits(double x) { return __builtin_bit_cast(uint64_t, x); }
__host__ __device__ inline double sum_from_bits(uint64_t b) { return __builtin_bit_cast(double, b); }
__host__ __device__ inline int sum_exp(double x) { return (int)((sum_bits(x) >> 52) & 0x7ff); } // biased; 0 for 0
__host__ __device__ inline double sum_pow2(int e) { return sum_from_bits((uint64_t)e << 52); }   // biased
constexpr int kSumExpLo = 1023 - 900, kSumExpHi = 1023 + 1000;

// biased exponent of x's lowest set bit (x normal and not zero)
__host__ __device__ inline int sum_lowbit(double x)
{
    const uint64_t m = (sum_bits(x) & 0xfffffffffffffull) | 0x10000000000000ull;
    return sum_exp(x) - 52 + __builtin_ctzll(m);
}

__host__ __device__ inline bool sum_is_step(const SumItem& it) { return it.tie == kSumStep; }

struct SumWalk {
    double a, v;   // start and current value of the open segment
    double lo, hi; // interval of d so far
    int e;         // biased exponent of a: the segment's largest binade
    int tie;
    bool open;     // it holds a step
};

__host__ __device__ inline void sum_restart(SumWalk& W, double v)
{
    W.a = W.v = v;
    W.lo = -1.7976931348623157e308;
    W.hi = 1.7976931348623157e308;
    W.e = sum_exp(v);
    W.tie = 0;
    W.open = false;
}

template <class Emit>
__host__ __device__ inline void sum_close(SumWalk& W, Emit emit)
{
    if (W.open) emit(SumItem{W.a, W.v, W.lo, W.hi, W.tie, 0});
    W.open = false;
}

// The rule of exact steps for v + x = t with no rounding error: the interval
// that keeps |t + d| within 2^52 g.  False when it does not hold t itself.
__host__ __device__ inline bool sum_exact_rule(const SumWalk& W, double v, double x, double t, double* lo, double* hi)
{
    if (x == 0.0) { // nothing, whatever the start
        *lo = -1.7976931348623157e308;
        *hi = 1.7976931348623157e308;
        return true;
    }
    if (W.e < kSumExpLo) return false;
    int Eg = W.e - 52, l = sum_lowbit(x); // G and the operands' lowest set bits
    Eg = l < Eg ? l : Eg;
    if (v != 0.0) {
        l = sum_lowbit(v);
        Eg = l < Eg ? l : Eg;
    }
    if (!(sum_exp(t) < Eg + 52) || Eg + 52 < 1) return false;
    const double B = sum_pow2(Eg + 52); // |t| < B: the differences are multiples of g below 2^53 g, exact
    *lo = -B - t;
    *hi = B - t;
    return true;
}

// one step: value x.  The common case is straight-line code (the walk is a
// dependent chain on few waves); the exact rule is tried where the binade's
// would not do: on a power of two, at zero, or far below the segment's grid
// (sums that cancelled to noise, where its interval is as narrow as the noise).
template <class Emit>
__host__ __device__ inline void sum_step(SumWalk& W, double x, Emit emit)
{
    const double v = W.v, t = v + x;
    const double bb = t - v, err = (v - (t - bb)) + (x - bb); // the addition's exact error
    const int E = sum_exp(t);
    const bool range = E >= kSumExpLo && E < kSumExpHi;
    const int Ec = range ? E : 1023;
    const double u = sum_pow2(Ec - 52), at = t < 0.0 ? -t : t;
    const double in = (sum_pow2(Ec) + u) - at, out = sum_pow2(Ec + 1) - at;
    double l0 = t < 0.0 ? -out : in, h0 = t < 0.0 ? -in : out;
    const double ae = err < 0.0 ? -err : err;
    const bool edge = !range || in > 0.0; // no start but others than the predicted one
    bool keep = E <= W.e && !edge;
    if (keep && E == W.e && ae + ae == u && W.tie == 0) W.tie = err > 0.0 ? 1 : -1; // u is the grid here
    if (err == 0.0 && E <= W.e && (edge || x == 0.0 || E + 24 < W.e)) {
        double l = 0.0, h = 0.0;
        if (sum_exact_rule(W, v, x, t, &l, &h)) {
            l0 = l;
            h0 = h;
            keep = true;
        }
    }
    if (keep) {
        if (W.tie) { // the distance may have grown by the grid
            const double g = sum_pow2(W.e - 51);
            l0 = l0 + g;
            h0 = h0 - g;
        }
        W.v = t;
        W.lo = W.lo > l0 ? W.lo : l0;
        W.hi = W.hi < h0 ? W.hi : h0;
        W.open = true;
        return;
    }
    sum_close(W, emit);
    emit(SumItem{x, v, 0.0, 0.0, kSumStep, 0});
    sum_restart(W, t);
}

// Whether a start s is one the segment moves with; its end in *end, its
// distance from the predicted start in *d, and in *odd whether a tie segment's
// distance is odd.
__host__ __device__ inline bool sum_apply(const SumItem& it, double s, double* end, double* d, bool* odd)
{
    const double x = s - it.p;
    const double bv = s - x, av = x + bv;
    const double tail = (s - av) + (bv - it.p); // 0: the difference is exact
    const int e = sum_exp(it.p);
    bool ok = tail == 0.0 && it.lo <= x && x <= it.hi;
    double moved = x;
    *odd = false;
    if (x != 0.0) {
        ok = ok && e >= kSumExpLo;
        const double r = ok ? x * sum_pow2(2046 - (e - 52)) : 0.5; // x / G
        ok = ok && __builtin_rint(r) == r;
        if (it.tie != 0) {
            ok = ok && r < 1.0e15 && r > -1.0e15; // below 2^50: sum_add_list
            const double h = r * 0.5;
            *odd = ok && __builtin_rint(h) != h;
            if (*odd) moved = x + (it.tie > 0 ? sum_pow2(e - 52) : -sum_pow2(e - 52));
        }
    }
    *d = x;
    *end = it.q + moved;
    return ok;
}

// One item as adds that carry every start it moves with exactly to its end:
// start - p = d, d + q.  A tie segment's d is first taken to the multiple of 2G
// on its side: d + tie G / 2 is rounded to one by adding and taking away 1.5 2^53 G
// (e < kSumExpLo holds the predicted start alone: d = 0).
constexpr int kSumMaxAdds = 5;
// Adds of a chunk of 64 values, at most: a segment ends before a step or with
// the chunk, and every item covers a value, so there are up to 32 segments and
// 32 steps.
constexpr int kSumChunk = 64, kSumChunkAdds = kSumChunk / 2 * (kSumMaxAdds + 1);
__host__ __device__ inline int sum_add_list(const SumItem& it, double* a)
{
    if (sum_is_step(it)) {
        a[0] = it.p;
        return 1;
    }
    const int e = sum_exp(it.p);
    a[0] = -it.p;
    if (it.tie == 0 || e < kSumExpLo) {
        a[1] = it.q;
        return 2;
    }
    const double h = sum_pow2(e - 53), C = 1.5 * sum_pow2(e + 1);
    a[1] = it.tie > 0 ? h : -h;
    a[2] = C;
    a[3] = -C;
    a[4] = it.q;
    return 5;
}

// one item of the level below (no kernel composes items)
template <class Emit>
__host__ __device__ inline void sum_compose(SumWalk& W, const SumItem& it, Emit emit)
{
    if (sum_is_step(it)) {
        sum_step(W, it.p, emit);
        return;
    }
    double end, d;
    bool odd;
    const bool ok = sum_apply(it, W.v, &end, &d, &odd);
    const int e = sum_exp(it.p);
    if (ok && e <= W.e && sum_exp(end) <= W.e) {
        // lo and hi move by the segment's own distance from its prediction;
        // the differences are pushed inward past their rounding, and past the
        // grid that a tie may have added
        if (it.tie != 0 && e == W.e && W.tie == 0) W.tie = odd ? -it.tie : it.tie;
        const double g = W.tie ? sum_pow2(W.e - 51) : 0.0;
        double l = (it.lo - d) + g, h = (it.hi - d) - g;
        l = l + (l < 0.0 ? -l : l) * 9e-16;
        h = h - (h < 0.0 ? -h : h) * 9e-16;
        W.lo = W.lo > l ? W.lo : l;
        W.hi = W.hi < h ? W.hi : h;
        W.v = end;
        W.open = true;
        return;
    }
    sum_close(W, emit);
    emit(it);
    // the next item's start as best predicted; its real start decides
    sum_restart(W, ok ? end : it.q);
}

} // namespace mcgpu
