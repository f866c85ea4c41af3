// The running sum s <- fl(s + x_i), i in order, evaluated in parallel with the
// bits of the sequential loop.
//
// While s stays in one binade [2^e, 2^(e+1)) every partial sum is a multiple
// of u = 2^(e-52): s = S u with an integer S in [2^52, 2^53).  Adding x rounds
// S + x/u to the nearest integer, so it adds r = rint(x/u), whatever S is,
// unless x/u lies halfway between two integers: then the result is the even
// neighbour, which depends on the parity of S only.  A run of additions is
// therefore a map of the parity p of its start: it adds d + p D, where D = 0
// without a tie, and D = +1 or -1 after the first tie (from there on both
// starts have the same parity).  Maps compose associatively, so a workgroup
// scans them; all quantities are integers below 2^53, exact in doubles.  A
// run that could leave the binade (its path comes within two units of an
// end) is added one value at a time, and the scan goes on behind it in the
// new binade.
//
// The functions here compute one run's map and compose maps; they compile for
// the host too, where the tests compare them with the sequential loop.
#pragma once
#include <cmath>
#include <cstdint>
#include <cstring>

#ifdef __HIPCC__
#define LES_HD __host__ __device__ __forceinline__
#else
#define LES_HD inline
#endif

namespace les {

struct SumMap {
    double d;      // adds d from an even start, d + D from an odd one
    int D;
};
struct SumGrid {
    bool zero;          // s is zero, not finite or near the ends of the range
    bool odd;           // parity of S
    double scale, inv;  // sign(s) / u and its reciprocal
    double lo, hi;      // bounds of a path relative to S
    double S;
};

LES_HD bool sum_parity(double d) {   // of an integer below 2^53 in magnitude
    const double h = 0.5 * d;
    return h != floor(h);
}

LES_HD double sum_bits(uint64_t b) {
    double v;
    memcpy(&v, &b, 8);
    return v;
}

LES_HD SumGrid sum_grid(double s) {
    SumGrid g;
    uint64_t b;
    memcpy(&b, &s, 8);
    const int e = (int)((b >> 52) & 0x7ff);        // biased exponent
    g.zero = e < 123 || e > 1923;                  // |s| < 2^-900 or > 2^900, infinities, NaN
    if (g.zero) {
        g.odd = false;
        g.scale = g.inv = g.lo = g.hi = g.S = 0.0;
        return g;
    }
    const uint64_t sign = b & 0x8000000000000000ull;
    g.odd = (b & 1) != 0;
    g.scale = sum_bits(sign | ((uint64_t)(1023 + 52 + 1023 - e) << 52));
    g.inv = sum_bits(sign | ((uint64_t)(e - 52) << 52));
    g.S = s * g.scale;
    g.lo = 4503599627370496.0 + 2.0 - g.S;
    g.hi = 9007199254740992.0 - 2.0 - g.S;
    return g;
}

// The map of a run of N values on grid g, and bounds of its path relative to
// the start: no steps down (up) give mn = +inf (mx = -inf), no bound.  On a
// zero grid a run of zeros is the identity and anything else leaves the path's
// range.  The N values are rounded independently and summed in pairs; only a
// run with a tie walks its values.
template <int N>
LES_HD SumMap sum_run(const double* x, const SumGrid& g, double& mn, double& mx) {
    SumMap m{0.0, 0};
    mn = HUGE_VAL;
    mx = -HUGE_VAL;
    if (g.zero) {
        bool z = true;
#pragma unroll
        for (int j = 0; j < N; ++j) z = z && (x[j] == 0.0);
        if (!z) mx = HUGE_VAL;
        return m;
    }
    double r[N], dn[N], up[N];
    bool tie = false, down = false, rise = false;
#pragma unroll
    for (int j = 0; j < N; ++j) {
        const double z = x[j] * g.scale;           // x / u, exact
        r[j] = rint(z);
        tie = tie || (fabs(z - r[j]) == 0.5);
        down = down || (z < 0.0);
        rise = rise || (z > 0.0);
        dn[j] = fmin(r[j], 0.0);
        up[j] = fmax(r[j], 0.0);
    }
    if (tie) {
#pragma unroll 1
        for (int j = 0; j < N; ++j) {
            const double z = x[j] * g.scale, q = rint(z);
            if (fabs(z - q) == 0.5) {
                const double a = m.d + floor(z);
                const bool odd = sum_parity(a);
                m.d = odd ? a + 1.0 : a;
                if (m.D == 0) m.D = odd ? -1 : 1;
            } else {
                m.d += q;
            }
        }
    }
#pragma unroll
    for (int w = 1; w < N; w *= 2) {
#pragma unroll
        for (int j = 0; j + w < N; j += 2 * w) {
            r[j] += r[j + w];
            dn[j] += dn[j + w];
            up[j] += up[j + w];
        }
    }
    if (!tie) m.d = r[0];
    // rint and floor differ by one at a tie: N more on either side covers them
    const double pad = tie ? (double)N : 0.0;
    if (down) mn = dn[0] - pad;
    if (rise) mx = up[0] + pad;
    return m;
}

// first a, then b
LES_HD SumMap sum_then(const SumMap& a, const SumMap& b) {
    const bool odd = sum_parity(a.d);
    SumMap c;
    c.d = a.d + b.d + (double)(odd ? b.D : 0);
    c.D = (a.D != 0) ? a.D : (odd ? -b.D : b.D);
    return c;
}
LES_HD double sum_add(const SumMap& m, bool odd) { return m.d + (double)(odd ? m.D : 0); }

// whether a run whose start lies `at` beyond S stays inside the binade
LES_HD bool sum_inside(const SumGrid& g, double at, const SumMap& m, double mn, double mx) {
    return g.zero ? mx < 0.0 : (at + mn >= g.lo && at + mx <= g.hi && m.d == m.d);
}
LES_HD double sum_value(const SumGrid& g, double s, double at) { return g.zero ? s : (g.S + at) * g.inv; }

// When a chunk of values is scanned and when it is added one by one.  A scan
// takes as long as walking SUM_SCAN values (3.2 us against 4.5 ns a value).
// Sums of one sign leave a binade each time they double, and a scan reaches
// from one such point to the next; sums of mixed sign can stay about the end
// of a binade, where each scan advances a few values.  So the rest of a chunk
// is walked once its scans have fallen a scan's time behind a walk, two in the
// first chunk, where a sum of one sign stops several times; and with each such
// chunk in a row one, two, then four chunks are walked untried.  `cancels`
// says it of the first values at once: the sum is small beside the sum of the
// magnitudes.
constexpr int SUM_SCAN = 768, SUM_BACK = 4;
struct SumPace {
    int skip = 0, back = 1, credit = 0;
    LES_HD bool chunk(bool first) {   // scan this chunk?
        credit = first ? SUM_SCAN : 0;
        if (skip == 0) return true;
        --skip;
        return false;
    }
    LES_HD bool stopped(int added) {   // a scan ended at a stop, `added` values on: scan again?
        credit += added - SUM_SCAN;
        return credit >= -SUM_SCAN;
    }
    LES_HD void gave_up() {
        skip = back;
        back = (back < SUM_BACK) ? 2 * back : SUM_BACK;
    }
    LES_HD void finished() { back = (back > 1) ? back / 2 : 1; }
};
LES_HD bool sum_cancels(double s, double magnitudes) { return fabs(s) * 8.0 < magnitudes; }

}  // namespace les
