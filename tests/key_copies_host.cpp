// Replays failing allocations into fill_key_copies (csrc/key_copies.hpp): prints,
// for each call, whether it succeeded and what the two buffers hold afterwards.
// Arguments: for each call, which of its two allocations fails (0: none, 1, 2).
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "key_copies.hpp"

static int g_fail = 0, g_alloc = 0;

struct Buf {
    std::vector<char> mem;
    bool held = false;
    bool try_ensure(std::size_t n) {
        if (held && mem.size() >= n) return true;
        if (++g_alloc == g_fail) return false;
        mem.assign(n, 'u');   // not initialised
        held = true;
        return true;
    }
    void release() {
        mem.clear();
        held = false;
    }
};

int main(int argc, char** argv) {
    Buf row, val;
    bool row_filled = false, val_filled = false;
    for (int a = 1; a < argc; a++) {
        // which allocation of this call fails; "v<k>": drop the values first, as
        // where only the rows were made for another type of them
        const char* arg = argv[a];
        if (*arg == 'v') {
            val.release();
            val_filled = false;
            arg++;
        }
        g_fail = std::atoi(arg);
        g_alloc = 0;
        const bool ok = exafac::fill_key_copies(row, row_filled, val, val_filled, 10, 8, [&](bool rows) {
            if (rows) row.mem.assign(row.mem.size(), 'r');
            val.mem.assign(val.mem.size(), 'v');
        });
        std::printf("%d %c%d %c%d\n", ok ? 1 : 0, row.held ? row.mem[0] : '-', row_filled ? 1 : 0,
                    val.held ? val.mem[0] : '-', val_filled ? 1 : 0);
    }
}
