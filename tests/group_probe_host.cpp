// Runs the lane-group search of csrc/group_probe.hpp on the host: for each group
// size and table length, targets below, between, at and past the entries, on tables
// with mass, without and with NaN.  Prints the first wrong answer, or "ok <searches>".
#include <cstdio>
#include <limits>
#include <vector>

#include "group_probe.hpp"

static int64_t search(const std::vector<double>& cum, double t, int lanes, bool& inside) {
    exafac::ProbeRange r{0, (int64_t)cum.size()};
    while (r.hi - r.lo > 1) {
        const int64_t step = exafac::probe_step(r, lanes);
        int first = -1;
        for (int l = lanes - 1; l >= 0; l--) {
            const int64_t at = exafac::probe_at(r, step, l);
            if (at < 0 || at >= (int64_t)cum.size()) inside = false;
            else if (cum[(size_t)at] > t) first = l;
        }
        if (!inside) return -1;
        r = exafac::probe_narrow(r, step, first);
    }
    return r.lo;
}

int main() {
    const double nan = std::numeric_limits<double>::quiet_NaN();
    long done = 0;
    for (int lanes : {8, 16, 32, 64}) {
        for (int64_t n = 1; n <= 5000; n += n < 300 ? 1 : 157) {
            for (int kind = 0; kind < 3; kind++) {   // ascending, no mass, NaN
                std::vector<double> cum((size_t)n);
                for (int64_t i = 0; i < n; i++) cum[(size_t)i] = kind == 0 ? (double)(i + 1) : kind == 1 ? 0.0 : nan;
                for (int64_t q = 0; q <= 2 * n + 2; q += n < 40 ? 1 : 1 + n / 20) {
                    const double t = 0.5 * (double)q;
                    // first entry past t, or the last one
                    const int64_t want = kind == 0 && q / 2 < n ? q / 2 : n - 1;
                    bool inside = true;
                    const int64_t got = search(cum, t, lanes, inside);
                    if (!inside || got != want) {
                        std::printf("lanes %d n %lld kind %d t %g: got %lld, want %lld\n", lanes, (long long)n, kind,
                                    t, (long long)got, (long long)want);
                        return 0;
                    }
                    done++;
                }
            }
        }
    }
    std::printf("ok %ld\n", done);
}
