// sph_pinned.hpp -- which host columns a kernel may write (host code, no device headers).
#pragma once
#include <cstdint>

namespace sph {

// A pinned allocation that kernels reach at its host address; none: 0 bytes.
struct PinnedRange {
    const char* start = nullptr;
    int64_t bytes = 0;
    bool holds(const char* p, int64_t n) const { return p >= start && n <= bytes && p - start <= bytes - n; }
};

// Whether every column [dst, dst + bytes) of the table lies whole in one pinned allocation; range_of(p) is the
// one that holds the byte at p. Looking at a column's two ends is not enough: they may lie in two allocations
// with ordinary memory, which a kernel cannot reach, in between. A response is usually one allocation, so the
// last one found is looked at first.
template <class Col, class RangeOf>
bool columns_pinned(const Col* col, int n, RangeOf range_of)
{
    PinnedRange last;
    for (int i = 0; i < n; ++i) {
        const char* p = static_cast<const char*>(col[i].dst);
        if (last.holds(p, col[i].bytes)) continue;
        last = range_of(p);
        if (!last.holds(p, col[i].bytes)) return false;
    }
    return true;
}

}  // namespace sph
