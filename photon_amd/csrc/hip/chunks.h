// How a render runs for a launch configuration: the launch rule's sizes, renders in chunks of whole samples, as large as
// memory allows, and which configurations run alike.
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

// The rule of the default configuration (no path slots or sub-streams asked for), with its reasons at
// WavefrontEngine::render.
constexpr int64_t kChunkItems = int64_t(1) << 26, kChunkSlots = int64_t(1) << 23, kDirectItems = int64_t(1) << 20;
constexpr int kChunkGraph = 2;

inline bool default_launch(const ph_wavefront_config& c) { return c.sample_split == 1 && c.path_slots == 0; }

// A render of at most kDirectItems samples at the default launch runs a sample per lane.
inline bool runs_direct(const ph_wavefront_config& c, int64_t pixels, int spp) {
    return default_launch(c) && c.finish_percent > 0 && pixels * spp <= kDirectItems;
}

// Sub-streams per pixel: the largest divisor of spp not above the configured split.
inline int sub_streams(const ph_wavefront_config& c, int spp) {
    int split = 1;
    for (int k = 1; k <= std::min(c.sample_split, spp); k++)
        if (spp % k == 0) split = k;
    return split;
}

// The configuration with every field that this render does not look at set to one value: two configurations that give the
// same here run the same launches.
inline ph_wavefront_config effective_launch(ph_wavefront_config c, int64_t pixels, int spp, bool wide) {
    if (runs_direct(c, pixels, spp)) {
        c = ph_wavefront_config{};
        c.sample_split = c.finish_percent = 1;
        return c;
    }
    if (default_launch(c)) {
        c.graph_iterations = std::min(c.graph_iterations, kChunkGraph);
    } else {
        c.sample_split = sub_streams(c, spp);
        c.path_slots = int(std::min(c.path_slots > 0 ? int64_t(c.path_slots) : std::min<int64_t>(pixels, 1 << 22), pixels * c.sample_split));
    }
    if (wide && c.lds_nodes == 0) c.stack_depth = 0;  // the wide walk's stack has a depth of its own
    return c;
}

}  // namespace phk
