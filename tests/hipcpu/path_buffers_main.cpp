// The wavefront engine's path-state memory (photon_amd/csrc/hip/path_buffers.h) against allocations that fail.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <utility>

#include "chunks.h"
#include "path_buffers.h"

namespace phk {
int set_error(const std::string&) { return -1; }
}  // namespace phk

using namespace phk;

#define EXPECT(x)                                                   \
    do {                                                            \
        if (!(x)) {                                                 \
            std::fprintf(stderr, "line %d: %s\n", __LINE__, #x);    \
            std::exit(1);                                           \
        }                                                           \
    } while (0)

static bool holds(const PathBuffers& b, size_t n) {
    for (const DevBuf<int>* p : {&b.job, &b.pixel, &b.sample, &b.sample_end, &b.part, &b.q_ext, &b.q_shadow, &b.q_term, &b.q_miss})
        if (!p->ptr || p->count < n) return false;
    for (const DevBuf<int>& q : b.q_cls)
        if (!q.ptr || q.count < n) return false;
    for (const DevBuf<float4>* p : {&b.ro, &b.rd, &b.beta, &b.L, &b.hit, &b.so, &b.sd, &b.sc})
        if (!p->ptr || p->count < n) return false;
    const size_t chunks = size_t(kMaxCategories) * size_t(compact_chunks(int(n)));
    return b.rng.ptr && b.rng.count >= n && b.stage.ptr && b.stage.count >= n && b.partial.ptr && b.partial.count >= chunks && b.first_pos.ptr &&
           b.first_pos.count >= chunks;
}

// Every allocation of a growth fails in turn; the size that there was room for before is then asked for again.
static void failed_growth() {
    for (int fail = 0;; fail++) {
        PathBuffers b;
        b.make_room(5000);
        EXPECT(holds(b, 5000));
        hipcpu::mallocs_left = fail;
        bool threw = false;
        try {
            b.make_room(20000);
        } catch (const HipError&) {
            threw = true;
        }
        hipcpu::mallocs_left = -1;
        b.make_room(5000);
        EXPECT(holds(b, 5000));
        if (!threw) {
            EXPECT(fail > 20);
            return;
        }
    }
}

// Sizes in turn allocate in the first round only; a size beyond the kept ones is given back.
static void sizes_in_turn() {
    PathBuffers b;
    int first = 0;
    for (int round = 0; round < 3; round++) {
        for (int n : {4000, 16000, 48000}) {
            b.make_room(n);
            EXPECT(holds(b, size_t(n)));
        }
        if (round == 0) first = hipcpu::mallocs_made;
    }
    EXPECT(hipcpu::mallocs_made == first);
    EXPECT(b.capacity == 48000);
    b.capacity = PathBuffers::kKeptSlots + 1;  // as if so many had been asked for
    b.make_room(4000);
    EXPECT(b.capacity == 4000 && holds(b, 4000) && b.ro.count == 4000);
    b.make_sums(1000);
    first = hipcpu::mallocs_made;
    for (size_t n : {400, 1000, 1}) b.make_sums(n);
    EXPECT(hipcpu::mallocs_made == first && b.part_sums.count == 1000);
    b.make_sums(PathBuffers::kKeptSums + 1);
    b.make_sums(500);
    EXPECT(b.part_sums.count == 500);
    b.release();
    EXPECT(b.capacity == 0 && !b.part_sums.ptr && !b.ro.ptr && !b.q_cls[0].ptr);
}

// A render in chunks where at most `room` slots and items fit: every sample runs once, in order, in chunks that fit.
static void short_memory() {
    for (int64_t pixels : {1, 7, 1000, 300000, 3000000})
        for (int spp : {1, 2, 3, 64, 1000})
            for (int64_t room : {int64_t(1) << 40, int64_t(1) << 22, int64_t(200000), kLeastSlots - 1}) {
                int next = 0, failed = 0;
                bool threw = false, released = true;
                try {
                    in_chunks(
                        pixels, spp, ChunkLimits{int64_t(1) << 26, int64_t(1) << 23},
                        [&](int k0, int k1, int64_t slots) {
                            EXPECT(k0 == next && k1 > k0 && k1 <= spp && released);
                            EXPECT(k1 - k0 == 1 || (k1 - k0) * pixels <= int64_t(1) << 26);
                            if (std::min(slots, (k1 - k0) * pixels) > room) {
                                failed++;
                                released = false;
                                throw OutOfMemory("no room");
                            }
                            next = k1;
                        },
                        [&] { released = true; });
                } catch (const OutOfMemory&) {
                    threw = true;
                }
                EXPECT(threw ? room < kLeastSlots : next == spp);
                EXPECT(failed <= 8);
            }
}

static bool alike(const ph_wavefront_config& a, const ph_wavefront_config& b, int64_t pixels, int spp, bool wide) {
    const ph_wavefront_config x = effective_launch(a, pixels, spp, wide), y = effective_launch(b, pixels, spp, wide);
    return std::memcmp(&x, &y, sizeof(x)) == 0;
}

// Which configurations the tuner may not tell apart.
static void same_launches() {
    const ph_wavefront_config base{128, 24, 0, 16, 1, 1, 16, 16, 0, 1, 1, 1, 10};
    using Field = int32_t ph_wavefront_config::*;
    const std::pair<Field, int> changes[] = {{&ph_wavefront_config::block, 64},          {&ph_wavefront_config::stack_depth, 8},
                                             {&ph_wavefront_config::blocks_per_cu, 4},   {&ph_wavefront_config::refill_lanes, 32},
                                             {&ph_wavefront_config::ray_bins, 0},        {&ph_wavefront_config::xcd_parts, 8},
                                             {&ph_wavefront_config::lds_nodes, 128},     {&ph_wavefront_config::use_graph, 0},
                                             {&ph_wavefront_config::graph_iterations, 8}, {&ph_wavefront_config::finish_percent, 30}};
    for (const auto& [field, value] : changes) {
        ph_wavefront_config c = base;
        c.*field = value;
        EXPECT(alike(base, c, 1 << 18, 4, true) && alike(base, c, 1 << 18, 4, false));  // a sample per lane: nothing is looked at
        const bool depth = field == &ph_wavefront_config::stack_depth, graph = field == &ph_wavefront_config::graph_iterations;
        EXPECT(alike(base, c, 1 << 18, 5, true) == (depth || graph));
        EXPECT(alike(base, c, 1 << 18, 5, false) == graph);
        ph_wavefront_config slots = base, slots_c = c;
        slots.path_slots = slots_c.path_slots = 100000;
        EXPECT(alike(slots, slots_c, 1 << 18, 4, true) == depth);
        EXPECT(!alike(slots, slots_c, 1 << 18, 4, false));
        slots.lds_nodes = 64;  // the binary nodes' top in LDS: over the binary nodes
        slots_c.lds_nodes = std::max(64, slots_c.lds_nodes);
        EXPECT(!alike(slots, slots_c, 1 << 18, 4, true));
    }
    ph_wavefront_config c = base, d = base;
    c.finish_percent = 0;  // in bounces
    EXPECT(!alike(base, c, 1 << 18, 4, true));
    c = base;
    c.path_slots = 1 << 18, d.path_slots = 1 << 20;  // no more slots than items
    EXPECT(alike(c, d, 1 << 18, 4, true) && !alike(c, base, 1 << 18, 4, true));
    c.sample_split = 4, d.sample_split = 5;  // rounded down to a divisor
    EXPECT(!alike(c, d, 1 << 18, 4, true));  // now there are items for the slots
    d.path_slots = c.path_slots;
    EXPECT(alike(c, d, 1 << 18, 4, true) && !alike(c, d, 1 << 18, 20, true));
}

int main() {
    same_launches();
    short_memory();
    failed_growth();
    sizes_in_turn();
    std::puts("ok");
    return 0;
}
