// The wavefront engine's path-state memory (photon_amd/csrc/hip/path_buffers.h) against allocations that fail.
#include <cstdio>
#include <cstdlib>

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

int main() {
    short_memory();
    failed_growth();
    sizes_in_turn();
    std::puts("ok");
    return 0;
}
