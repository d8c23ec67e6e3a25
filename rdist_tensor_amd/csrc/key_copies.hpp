// Filling of a lookup's key-order copies (host logic, no HIP: the copies are
// buffers with try_ensure and release).
#pragma once
#include <cstddef>

namespace exafac {

// Makes `row` (4 bytes an entry) and `val` (val_bytes an entry) hold n entries in
// key order; fill(rows) enqueues the copy of the values, and of the rows where
// `rows`.  A buffer counts as filled only once its fill has been enqueued: an
// allocation alone says nothing, since the other one may have failed after it.
// Both are allocated before either is filled.  false: no room (nothing is filled,
// and no buffer is held that was not filled before).
template <class Buf, class Fill>
bool fill_key_copies(Buf& row, bool& row_filled, Buf& val, bool& val_filled, std::size_t n, std::size_t val_bytes,
                     Fill fill) {
    if (row_filled && val_filled) return true;
    if (!row.try_ensure(n * 4)) return false;
    if (!val.try_ensure(n * val_bytes)) {
        if (!row_filled) row.release();
        return false;
    }
    fill(!row_filled);
    row_filled = val_filled = true;
    return true;
}

}  // namespace exafac
