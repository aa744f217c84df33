// Device memory of the wavefront's path buffers, for sizing a pass.
#pragma once
#include <cstddef>

namespace agx {

// Bytes that one path in flight holds (PathBuffers): its state 120, two rays and
// their hits 88, queue entries 16; for each light a pending contribution, a
// shadow ray, its result and its queue entry; in scenes with media the medium
// sample, and for each light its segment.  An upper bound by less than a percent.
constexpr size_t path_bytes(int lights, bool media) {
    const size_t l = lights > 1 ? size_t(lights) : 1;
    return 226 + 49 * l + (media ? 48 + 16 * l : 0);
}

}  // namespace agx
