// Device memory of the wavefront engine's paths in flight: one entry per path slot in each array.
#pragma once

#include "internal.h"

namespace phk {

constexpr int kClasses = 4;  // shading queues (material classes)
// Ordered compaction: a block of 256 threads covers 4096 slots, 16 consecutive slots per thread.
constexpr int kCompactThreads = 256, kCompactPerThread = 16, kCompactChunk = kCompactThreads * kCompactPerThread;
constexpr int kMaxCategories = 9;  // stages that one compaction tells apart

inline int compact_chunks(int n) { return (n + kCompactChunk - 1) / kCompactChunk; }

struct PathBuffers {
    DevBuf<int> job, pixel, sample, sample_end, part, q_ext, q_shadow, q_term, q_miss, q_cls[kClasses], partial, first_pos;
    DevBuf<uint8_t> stage;
    DevBuf<uint64_t> rng;
    DevBuf<float4> ro, rd, beta, L, hit, so, sd, sc;
    DevBuf<float4> part_sums;  // partial sums of a single render in sub-streams
    int capacity = 0;  // slots that every array has room for

    // Renders of changing sizes keep the largest one's arrays, up to this many slots (1.6 GB): 1920x1080 Cornell with 1 and
    // 4 samples in turn takes 3.9 ms a pair, 16.4 with arrays of the exact size. What a configuration asked
    // for beyond that is given back by the next smaller call.
    static constexpr int kKeptSlots = 1 << 23;
    static constexpr size_t kKeptSums = size_t(1) << 26;  // the same for partial sums (1 GB)

    // Whether make_room(n) would allocate (what points into the arrays is to be dropped before).
    bool moves(int n) const { return n > capacity || (n < capacity && capacity > kKeptSlots); }

    // Room for at least n slots. If an allocation fails there is room for none, and the next call allocates what is missing.
    void make_room(int n) {
        if (!moves(n)) return;
        capacity = 0;
        for (DevBuf<int>* b : {&job, &pixel, &sample, &sample_end, &part, &q_ext, &q_shadow, &q_term, &q_miss}) b->allocate(size_t(n));
        for (auto& q : q_cls) q.allocate(size_t(n));
        stage.allocate(size_t(n + 15) / 16 * 16);
        partial.allocate(size_t(kMaxCategories) * size_t(compact_chunks(n)));
        first_pos.allocate(size_t(kMaxCategories) * size_t(compact_chunks(n)));
        rng.allocate(size_t(n));
        for (DevBuf<float4>* b : {&ro, &rd, &beta, &L, &hit, &so, &sd, &sc}) b->allocate(size_t(n));
        capacity = n;
    }

    // Room for at least n partial sums.
    void make_sums(size_t n) {
        if (n > part_sums.count || part_sums.count > kKeptSums) part_sums.allocate(n);
    }

    void release() {
        capacity = 0;
        part_sums.release();
        for (DevBuf<int>* b : {&job, &pixel, &sample, &sample_end, &part, &q_ext, &q_shadow, &q_term, &q_miss, &partial, &first_pos}) b->release();
        for (auto& q : q_cls) q.release();
        stage.release();
        rng.release();
        for (DevBuf<float4>* b : {&ro, &rd, &beta, &L, &hit, &so, &sd, &sc}) b->release();
    }
};

}  // namespace phk
