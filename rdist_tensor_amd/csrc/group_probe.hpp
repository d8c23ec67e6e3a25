// Search of an ascending table by a group of lanes that probe as many positions a
// step (index arithmetic only; constexpr, so that it runs on the host as well).
#pragma once
#include <cstdint>

namespace exafac {

// The entries still searched.  After the first step the last one exceeds the target.
struct ProbeRange {
    int64_t lo, hi;
};

constexpr int64_t probe_step(ProbeRange r, int lanes) { return (r.hi - r.lo + lanes - 1) / lanes; }

// Position probed by `lane`: the last entry of its piece.
constexpr int64_t probe_at(ProbeRange r, int64_t step, int lane) {
    const int64_t at = r.lo + (int64_t)(lane + 1) * step - 1;
    return at < r.hi ? at : r.hi - 1;
}

// What is left when `first` is the lowest lane whose entry exceeds the target.  No
// such lane (first < 0: no mass, a NaN, or a target that rounding put past the
// total): the last entry.  Taking the last lane's piece instead would pass the end
// of the table wherever the pieces of fewer lanes cover it (65 entries, 64 lanes:
// pieces of 2, the last of them from entry 126).
constexpr ProbeRange probe_narrow(ProbeRange r, int64_t step, int first) {
    if (first < 0) return ProbeRange{r.hi - 1, r.hi};
    const int64_t lo = r.lo + (int64_t)first * step, hi = lo + step;
    return ProbeRange{lo, hi < r.hi ? hi : r.hi};
}

}  // namespace exafac
