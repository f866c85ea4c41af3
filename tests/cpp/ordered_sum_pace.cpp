// How a plane sum is scanned and walked (SumPace, ordered_sum.hpp), as the
// kernel does it: the bits of the sequential loop, and a cost, counted in
// walked values, that stays near a walk's for sums that cancel and near the
// scans' for sums of one sign.
#include <algorithm>
#include <cstdio>
#include <random>
#include <vector>
#include "../../overlappingbls_amd/csrc/ordered_sum.hpp"

using namespace les;

constexpr int RUN = 16, NT = 256, CHUNK = RUN * NT, HEAD = 512;

struct Cost {
    long scans = 0, walked = 0, tries = 0, worst = 0;   // tries: chunks given up; worst: a chunk's cost beyond a walk
};

static double chain(const std::vector<double>& x, Cost& c) {
    const long n = (long)x.size();
    auto at = [&](long i) { return i < n ? x[i] : 0.0; };
    SumPace pace;
    double s = 0.0;
    for (long base = 0; base < n; base += CHUNK) {
        const int lim = (int)std::min<long>((n - base + RUN - 1) / RUN, NT);
        int start = 0;
        const long before = c.walked + SUM_SCAN * c.scans;
        bool scan = pace.chunk(base == 0);
        if (base == 0) {
            start = HEAD / RUN;
            double a = 0.0;
            for (long i = 0; i < HEAD; ++i) s += x[i], a += fabs(x[i]);
            c.walked += HEAD;
            scan = !sum_cancels(s, a);
        }
        const bool tried = scan;
        while (scan && start < lim) {
            const SumGrid g = sum_grid(s);
            SumMap pre{0.0, 0};
            double run[RUN], mn, mx;
            int t = start;
            for (; t < lim; ++t) {
                for (int j = 0; j < RUN; ++j) run[j] = at(base + t * RUN + j);
                const SumMap m = sum_run<RUN>(run, g, mn, mx);
                if (!sum_inside(g, sum_add(pre, g.odd), m, mn, mx)) break;
                pre = sum_then(pre, m);
            }
            s = sum_value(g, s, sum_add(pre, g.odd));
            ++c.scans;
            if (t == lim) {
                start = lim;
                break;
            }
            for (int j = 0; j < RUN; ++j) s += run[j];
            scan = pace.stopped((t + 1 - start) * RUN);
            start = t + 1;
        }
        if (start < lim) {
            if (tried || base == 0) pace.gave_up(), ++c.tries;
            for (int t = start; t < lim; ++t)
                for (int j = 0; j < RUN; ++j) s += at(base + t * RUN + j);
            c.walked += std::min<long>((long)(lim - start) * RUN, n - base);
        } else if (tried) {
            pace.finished();
        }
        // the first chunk may fall a scan further behind
        const long cost = c.walked + SUM_SCAN * c.scans - before - std::min<long>(CHUNK, n - base);
        c.worst = std::max(c.worst, base ? cost : cost - SUM_SCAN);
    }
    return s;
}

int main() {
    std::mt19937_64 r(11);
    std::uniform_real_distribution<double> U(0.0, 1.0);
    std::normal_distribution<double> G(0.0, 1.0);
    int bad = 0;
    for (int kind = 0; kind < 9; ++kind)
        for (long n : {2304L, 4096L, 9216L, 16384L, 65536L, 82944L, 262144L}) {
            std::vector<double> x(n);
            const double c = 0.5 + U(r);
            for (long i = 0; i < n; ++i) switch (kind) {
                case 0: x[i] = 20.0 + G(r); break;                     // speeds
                case 1: x[i] = 1.0 + 1e-3 * G(r); break;               // temperatures
                case 2: x[i] = -c; break;                              // a uniform plane
                case 3: x[i] = 0.0; break;
                case 4: x[i] = G(r); break;                            // v, w without a mean
                case 5: x[i] = 0.3 + G(r); break;                      // and with one
                case 6: x[i] = sin(0.05 * i) + 0.2 * G(r); break;      // in long waves
                case 7: x[i] = (i & 1) ? -c : c; break;                // back to zero each time
                default: x[i] = (i == n / 2) ? NAN : G(r); break;
            }
            volatile double s = 0.0;
            for (long i = 0; i < n; ++i) s = s + x[i];
            Cost k;
            const double a = s, b = chain(x, k);
            if (memcmp(&a, &b, 8) && !(a != a && b != b)) ++bad, printf("kind %d n %ld: %.17g against %.17g\n", kind, n, b, a);
            // a chunk is at most a scan's time behind a walk before its last scan
            if (k.worst > 2 * SUM_SCAN) ++bad, printf("kind %d n %ld: %ld values behind\n", kind, n, k.worst);
            // where no scan pays, only every fifth chunk is tried from the third on
            const long chunks = (n + CHUNK - 1) / CHUNK;
            if (kind == 7 && k.tries > 3 + chunks / 5) ++bad, printf("kind %d n %ld: %ld tries\n", kind, n, k.tries);
            // one sign: only the head is walked; a stop for each doubling
            if (kind < 4 && (k.walked != HEAD || k.scans > chunks + 10))
                ++bad, printf("kind %d n %ld: walked %ld, %ld scans\n", kind, n, k.walked, k.scans);
        }
    printf("%s\n", bad ? "different" : "as expected");
    return bad != 0;
}
