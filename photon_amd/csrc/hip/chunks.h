// A render in chunks of whole samples, as large as memory allows.
#pragma once

#include <algorithm>

#include "internal.h"

namespace phk {

// Work items (pixels x samples) a chunk may have at once and paths in flight; both are halved whenever a chunk does not
// find the device memory for them, down to kLeastSlots paths.
struct ChunkLimits {
    int64_t items, slots;
};
constexpr int64_t kLeastSlots = 1 << 16;

// Calls run(k0, k1, slots) for consecutive ranges of the `spp` samples, each of at most limits.items items (or one sample).
// run allocates before it adds anything to the image: a chunk that throws OutOfMemory is taken again, smaller, after
// release().
template <class Run, class Release>
void in_chunks(int64_t pixels, int spp, ChunkLimits limits, Run run, Release release) {
    for (int k0 = 0; k0 < spp;) {
        const int64_t left = spp - k0, most = std::max<int64_t>(1, limits.items / pixels);
        const int k1 = k0 + int(left / ((left + most - 1) / most));
        try {
            run(k0, k1, limits.slots);
            k0 = k1;
        } catch (const OutOfMemory&) {
            (void)hipGetLastError();
            if (limits.slots <= kLeastSlots) throw;
            limits.items /= 2;
            limits.slots /= 2;
            release();
        }
    }
}

}  // namespace phk
