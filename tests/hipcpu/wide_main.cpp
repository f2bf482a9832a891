// The walk over the wide nodes and the walk over the binary ones (photon_amd/csrc/hip/dwide.h, dtrace.h) with the wide
// nodes' build (wide_build.hip), compiled for the CPU through hip/hip_runtime.h into a library that tests call: the
// device's own arithmetic on rays in any number, without a GPU.
#define __builtin_amdgcn_readfirstlane(x) (x)
#define __builtin_amdgcn_ldexpf(x, e) __builtin_ldexpf(x, e)
#include "wide_build.cpp"

using namespace phd;

namespace phk {
int set_error(const std::string&) { return -1; }
}  // namespace phk

namespace {

// A walk's stack in ordinary memory, with the distances rounded where the device's are.
struct HostStack {
    static constexpr int kDepth = kWideLdsDepth;
    int links[kMaxStack];
    float distances[kMaxStack];
    void store_lds(int sp, int link, float t) {
        links[sp] = link;
        distances[sp] = __uint_as_float(__float_as_uint(t) & 0xffff0000u);
    }
    void store(int sp, int link, float t) {
        if (sp < kDepth) {
            store_lds(sp, link, t);
        } else {
            links[sp] = link;
            distances[sp] = t;
        }
    }
    void load(int sp, int& link, float& t) const {
        link = links[sp];
        t = distances[sp];
    }
    void store(int sp, int link) { links[sp] = link; }
    int load(int sp) const { return links[sp]; }
};

template <bool AnyHit>
void one_ray(const TraceScene& ts, const float* r, HitRec* out, int* again) {
    const f3 o = mk3(r[0], r[1], r[2]), d = mk3(r[3], r[4], r[5]);
    HostStack stack;
    BinaryWalk<AnyHit, false> b;
    b.start(o, d, r[6]);
    while (b.step(ts, stack)) {
    }
    WideWalk<AnyHit, false> w{};
    w.start(o, d, r[6]);
    while (w.step(ts, stack)) {
    }
    *again = !w.settled(ts);
    out[0] = b.hit;
    out[1] = *again ? b.hit : w.hit;
}

}  // namespace

// Each ray (7 floats) over both kinds of nodes: hits[2 i] the binary walk's, hits[2 i + 1] the wide walk's; again[i]:
// the wide walk left the ray to the binary one. Returns 0 if the scene has no wide nodes.
extern "C" __attribute__((visibility("default"))) int walk_both(const float* nodes, int num_nodes, const float* tris, int num_tris, const float* rays, int n, int anyhit, HitRec* hits, int* again) {
    phk::DevBuf<float4> dev_nodes, dev_tris;
    phk::WideNodes wide;
    dev_nodes.upload(nodes, size_t(num_nodes) * 4, nullptr);
    dev_tris.upload(tris, size_t(num_tris) * 3, nullptr);
    phk::build_wide_nodes(nullptr, dev_nodes.ptr, num_nodes, num_tris, wide);
    if (!wide.settled()) return 0;
    phk::mark_leaves(nullptr, dev_nodes.ptr, num_nodes, num_tris, dev_tris.ptr);
    DScene s{};
    s.nodes = dev_nodes.ptr;
    s.wide = wide.nodes.ptr;
    s.tris = dev_tris.ptr;
    s.num_nodes = num_nodes;
    s.num_tris = num_tris;
    const TraceScene ts = trace_scene(s);
    std::atomic<int> next{0};
    auto work = [&] {
        constexpr int kRun = 4096;
        for (int first; (first = next.fetch_add(kRun)) < n;)
            for (int i = first; i < std::min(n, first + kRun); i++) (anyhit ? one_ray<true> : one_ray<false>)(ts, rays + 7 * size_t(i), hits + 2 * size_t(i), again + i);
    };
    std::vector<std::thread> pool;
    for (int k = 1; k < 8; k++) pool.emplace_back(work);
    work();
    for (std::thread& t : pool) t.join();
    return num_nodes;
}
