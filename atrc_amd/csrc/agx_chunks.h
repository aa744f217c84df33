// Parts of a call on n items that goes through buffers of at most `chunk` items.
#pragma once
#include <algorithm>
#include <cstddef>
#include <cstdint>

namespace agx {

// fn(first, count) for the parts of [0, n) in order, each of `chunk` items but the
// last; ends at the first non-zero result of fn and returns it, else 0.
template <class Fn> int for_each_chunk(uint32_t n, uint32_t chunk, Fn fn) {
    for (uint64_t first = 0; first < n; first += chunk)  // 64 bits: the last step may pass 2^32
        if (const int r = fn(size_t(first), uint32_t(std::min<uint64_t>(n - first, chunk)))) return r;
    return 0;
}

}  // namespace agx
