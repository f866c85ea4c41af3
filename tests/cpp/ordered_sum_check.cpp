// The scanned running sum (ordered_sum.hpp) against the sequential loop, bit
// for bit: runs of 16 values as the kernel's lanes take them, composed in
// order, over value distributions that meet every branch.
#include <cstdio>
#include <random>
#include <vector>
#include "../../overlappingbls_amd/csrc/ordered_sum.hpp"

using namespace les;

static long steps;   // runs added one value at a time

static double scanned(const std::vector<double>& x, int lanes) {
    const size_t n = x.size();
    double s = 0.0;
    for (size_t base = 0; base < n; base += (size_t)lanes * 16) {
        int start = 0;
        while (start < lanes) {
            const SumGrid g = sum_grid(s);
            SumMap pre{0.0, 0};
            int t = start;
            double run[16], mn, mx;
            for (; t < lanes; ++t) {
                for (int j = 0; j < 16; ++j) run[j] = base + (size_t)t * 16 + j < n ? x[base + (size_t)t * 16 + j] : 0.0;
                const SumMap m = sum_run<16>(run, g, mn, mx);
                if (!sum_inside(g, sum_add(pre, g.odd), m, mn, mx)) break;
                // as a scan composes: pairs first, then the prefix
                pre = sum_then(pre, m);
            }
            s = sum_value(g, s, sum_add(pre, g.odd));
            if (t < lanes) {
                for (int j = 0; j < 16; ++j) s += run[j];
                ++steps;
                ++t;
            }
            start = t;
        }
    }
    return s;
}

// composition is associative: (a b) c = a (b c) on random maps
static bool associative(std::mt19937_64& r) {
    for (int i = 0; i < 100000; ++i) {
        SumMap m[3];
        for (SumMap& a : m) a = {(double)((long)(r() % 2001) - 1000), (int)(r() % 3) - 1};
        // a map with D = 0 adds the same from either parity; a map with D != 0
        // ends on one parity
        const SumMap x = sum_then(sum_then(m[0], m[1]), m[2]), y = sum_then(m[0], sum_then(m[1], m[2]));
        if (x.d != y.d || x.D != y.D) return false;
    }
    return true;
}

int main() {
    std::mt19937_64 r(7);
    std::uniform_real_distribution<double> U(0.0, 1.0);
    std::normal_distribution<double> G(0.0, 1.0);
    int bad = associative(r) ? 0 : 1;
    if (bad) printf("composition is not associative\n");
    for (int kind = 0; kind < 13; ++kind)
        for (int rep = 0; rep < 40; ++rep) {
            const size_t n = 1 + r() % 70000;
            std::vector<double> x(n);
            const double c = (U(r) - 0.5) * 4.0;
            for (size_t i = 0; i < n; ++i) switch (kind) {
                case 0: x[i] = 20.0 + G(r); break;                       // speeds
                case 1: x[i] = 1.0 + 1e-6 * G(r); break;                 // temperatures
                case 2: x[i] = c; break;                                 // a uniform plane
                case 3: x[i] = 0.0; break;
                case 4: x[i] = -5.0 - U(r); break;                       // negative
                case 5: x[i] = G(r); break;                              // cancelling
                case 6: x[i] = std::ldexp((double)(r() % 7) - 1.0, -2); break;   // many ties, repeated values
                case 7: x[i] = std::ldexp(1.0, (int)(r() % 60) - 30); break;     // wide range
                case 8: x[i] = (i == n / 2) ? 1e300 : 1e-300 * U(r); break;
                case 9: x[i] = (i == n / 2) ? HUGE_VAL : U(r); break;
                case 10: x[i] = (i == n / 2) ? NAN : U(r); break;
                case 11: x[i] = (i % 3) ? 1.0 + std::ldexp((double)(r() & 1), -40) : std::ldexp(3.0, -38); break;
                default: x[i] = (i & 1) ? -c : c; break;                 // back to zero
            }
            volatile double s = 0.0;
            for (size_t i = 0; i < n; ++i) s = s + x[i];
            const double a = s, b = scanned(x, 1 << (r() % 9));
            if (memcmp(&a, &b, 8) && !(a != a && b != b)) {
                if (++bad < 10) printf("kind %d n %zu: %.17g against %.17g\n", kind, n, b, a);
            }
        }
    printf("%s\n", bad ? "different" : "equal");
    return bad != 0;
}
