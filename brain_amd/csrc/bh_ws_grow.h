// How a workspace grows (no HIP in here: the CPU tests compile it alone).
#pragma once
#include <algorithm>
#include <cstddef>

namespace bh {

struct WsBuf {
    int* ws = nullptr;
    size_t ints = 0;
};

// At least `ints` i32 in `b`. A replaced buffer is not freed: a graph captured
// earlier may still launch kernels that use it, and other streams' work need
// not be waited for. So a buffer at least doubles, up to `cap` ints: however
// slowly the sizes rise, all that is left behind is less than twice the buffer
// in use (but for growths for which there was only memory for the exact size).
// alloc(bytes) returns null when there is none; then `b` stays as it is.
template <class Alloc>
bool ws_grow(WsBuf& b, size_t ints, size_t cap, Alloc alloc) {
    if (b.ints >= ints) return true;
    for (const size_t want : {std::max(ints, std::min(2 * b.ints, cap)), ints}) {
        if (int* p = static_cast<int*>(alloc(want * sizeof(int)))) {
            b = WsBuf{p, want};
            return true;
        }
    }
    return false;
}

}  // namespace bh
