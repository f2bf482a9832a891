// Traversal over four-wide nodes with quantised child boxes, for the rays whose answer does not depend
// on the order of the tests: the closest hit, and whether anything is hit at all.
//
// What bounds the walk over the binary nodes (dtrace.h) is work per ray: about 21 node steps and 3
// triangle tests, each a dependent round trip, each costing the wave the instructions of both kinds of
// step, and each node step four 16-byte loads per lane with 64 different addresses per wave. A wide node
// holds the boxes of up to four descendants of a binary node in the same 64 bytes, so a ray takes half
// the steps and half the loads.
//
// Measured, binary nodes against these: 4,194,304 camera rays into 262,144 triangles 0.99 / 0.44 ms; 1080p, 64
// samples, 1M triangles 96.8 / 79.5 ms (closest hits 3.4 / 2.6 ms a bounce); its one-sample 1600x900 frame
// 3.6 / 2.6 ms. The traversal kernels keep 8 waves per SIMD (64 VGPRs) and issue VALU instructions 87 % of the time.
//
// Wide node (64 bytes, four 16-byte loads):
//   [0]  origin.xyz, three signed exponent bytes: plane q of an axis lies at origin + q 2^exponent
//   [1]  lower x, upper x, lower y, upper y planes of the four children, a byte each
//   [2]  lower z, upper z, and two unused words
//   [3]  four links: interior (a wide node's index, its binary node's, >= 0) or leaf (bit 31, 5 bits triangles - 1, 26 bits
//        first triangle). An unused child has an inverted box and a sibling's link.
//
// The answer is the binary walk's, with the one exception below:
//   * Child planes are rounded outwards by at least 2^-10 of a quantisation step, and the ray's distances
//     to them are widened by 2^-21 of the distance to the origin plane: more than the rounding errors of
//     both walks' slab tests. So every box that the binary walk enters is entered here too (its boxes
//     nest, and its slab arithmetic is monotone in the planes).
//   * The walk may therefore test triangles that the binary walk does not reach. settled() tests the
//     winner's leaf box with the binary walk's own arithmetic; the ancestors' boxes then pass as well.
//   * Two hits within 2^-19 of each other could be told apart by the order of the binary walk's tests:
//     such a pair marks the ray.
//   * A ray that is marked, whose winner fails the box test, whose stack overflows or whose numbers are
//     too large for the bounds above is traced again over the binary nodes (a few in 100,000).
//   * Boxes from 2^-10 behind the closest hit on are not entered. A triangle in one of them can be the
//     binary walk's answer only if its computed distance lies that much before its own box, and if the
//     binary walk, in its order, came to it before the closest hit. Moller-Trumbore's relative error of
//     the distance is a few 2^-24 over |det| / (|e1| |e2| |d|), so such a triangle is seen edge-on to
//     within 2^-13: its distance, not the walk, is what is off. Aimed along random triangles' planes (1e-4
//     of a radian and less) up to 1 ray in 5,000 answers with the hit behind; at angles from 1e-4 on, from
//     1 to 100,000 extents away, none in 36 million. With 2^-19 instead of 2^-10 up to 1 in 20,000 of the
//     far ones did. 4M camera rays into 262,144 triangles 0.419 / 0.423 ms, 1080p render 70.5 ms with
//     either; 2^-8 costs 3 and 0.5 % more. Any-hit answers have no such exception: the ray's own limit culls
//     boxes.
#pragma once

#include "dtrace.h"

namespace phd {

constexpr int kWideLdsDepth = 12;                      // of them in LDS, in the traversal kernels
constexpr int kWideStack = 48;                          // stack entries (link and entry distance) per lane
constexpr int kWideCountShift = 26;                     // leaf links: triangles - 1 above, first triangle below
constexpr int kWideMaxLeaf = 32, kWideMaxTris = 1 << kWideCountShift;
constexpr float kWideReach = 1e15f;                     // largest coordinate the error bounds cover
constexpr float kTieAbove = 1.0f + 0x1p-19f, kTieBelow = 1.0f - 0x1p-19f;
constexpr float kCullAbove = 1.0f + 0x1p-10f;

// Overflow entries of a WideStack<Depth>; the binary walk's stack uses them too.
template <int Depth>
struct WideSpill {
    static_assert(Depth < kWideStack && kMaxStack - Depth <= 2 * (kWideStack - Depth));
    int v[2 * (kWideStack - Depth)];
};

// A lane's stack of links and entry distances: `Depth` of them in LDS, interleaved over the block's lanes, the
// rest in private memory. In LDS a distance is its upper 16 bits (rounded towards zero, so that it still bounds
// the box from below): 6 bytes an entry keep 12 entries and 32 waves on a CU.
using LdsShort = __attribute__((address_space(3))) uint16_t;

template <int Depth, int Block>
struct WideStack {
    static constexpr int kDepth = Depth;
    uint32_t first;      // LDS address of this lane's first link; its distances follow at half that offset
    uint32_t distances;  // what to add to half of a link's address (the same in every lane)
    PrivateInt* spill;
    PH_DEV WideStack(int* lds, int lane, int* spill_area) : spill((PrivateInt*)spill_area) {
        const uint32_t base = uint32_t(uintptr_t((LdsInt*)lds));
        first = base + 4 * uint32_t(lane);
        distances = base - base / 2 + 4 * Depth * Block;
    }
    PH_DEV LdsInt* link_at(uint32_t a) const { return (LdsInt*)uintptr_t(a); }
    PH_DEV LdsShort* distance_at(uint32_t a) const { return (LdsShort*)uintptr_t(a / 2 + distances); }
    PH_DEV uint32_t address(int sp) const { return first + uint32_t(sp) * (4 * Block); }
    // The entry is known to be one of the first `Depth`.
    PH_DEV void store_lds(int sp, int link, float t) {
        const uint32_t a = address(sp);
        *link_at(a) = link;
        *distance_at(a) = uint16_t(__float_as_uint(t) >> 16);
    }
    PH_DEV void store(int sp, int link, float t) {
        if (sp < Depth) {
            store_lds(sp, link, t);
        } else {
            spill[2 * (sp - Depth)] = link;
            spill[2 * (sp - Depth) + 1] = __float_as_int(t);
        }
    }
    PH_DEV void load(int sp, int& link, float& t) const {
        if (sp < Depth) {
            const uint32_t a = address(sp);
            link = *link_at(a);
            t = __uint_as_float(uint32_t(*distance_at(a)) << 16);
        } else {
            link = spill[2 * (sp - Depth)];
            t = __int_as_float(spill[2 * (sp - Depth) + 1]);
        }
    }
    // The binary walk's stack in the same memory (the links).
    PH_DEV LaneStack<Depth> binary() const { return LaneStack<Depth>((int*)link_at(first), Block, (int*)spill); }
};

// The traversal stack of a kernel whose blocks have `Block` lanes, for either walk: the LDS words of a block,
// the overflow area and the lane's handle. `Depth` entries per lane are in LDS.
template <int Block, int Depth, bool Wide>
struct StackShape {
    static constexpr int kWords = Depth * Block;
    using Spill = SpillArea<Depth>;
    using Stack = LaneStack<Depth>;
    static PH_DEV Stack make(int* lds, int lane, Spill& spill) { return Stack(lds + lane, Block, spill.v); }
};

template <int Block, int Depth>
struct StackShape<Block, Depth, true> {
    static constexpr int kWords = Depth * Block + Depth * Block / 2;
    using Spill = WideSpill<Depth>;
    using Stack = WideStack<Depth, Block>;
    static PH_DEV Stack make(int* lds, int lane, Spill& spill) { return Stack(lds, lane, spill.v); }
};

// mt_hit without the upper limit on t, which the caller applies.
PH_DEV bool mt_hit_any(f3 v0, f3 e1, f3 e2, f3 o, f3 d, float& t, float& u, float& v) { return mt_hit(v0, e1, e2, o, d, __builtin_inff(), t, u, v); }

PH_DEV float plane_byte(uint32_t w, int k) { return float((w >> (8 * k)) & 255u); }

// One ray's walk. `Unbounded`: the ray has no upper limit (tmax = kInf).
template <bool AnyHit, bool Unbounded>
struct WideWalk {
    static constexpr bool kSecond = true;  // a few rays are traced again
    f3 o, d, inv;
    float limit;  // boxes and triangles from here on are of no interest
    float tmax;   // the ray's own upper limit (unless Unbounded)
    int cur, sp;  // link being worked on; stack entries
    bool doubt;   // the answer may depend on the order of the tests, or was not found here
    HitRec hit;
    int leaf;  // of the hit triangle: its place in the binary nodes (2 node + side)

    PH_DEV void start(f3 o_, f3 d_, float tmax_) {
        o = o_;
        d = d_;
        inv = guarded_reciprocal(d_);
        limit = tmax = tmax_;
        cur = sp = 0;
        hit = HitRec{kInf, -1, 0.0f, 0.0f};
        leaf = 0;
        const float reach = fmaxf(fmaxf(fmaxf(fabsf(o.x), fabsf(o.y)), fabsf(o.z)), fmaxf(fmaxf(fabsf(d.x), fabsf(d.y)), fabsf(d.z)));
        const float sum = (o.x + o.y + o.z) + (d.x + d.y + d.z);  // NaN if any of them is
        doubt = !(reach <= kWideReach) || !(sum == sum);
        if (doubt) limit = -1.0f;  // no box is entered; the ray is traced again
    }
    PH_DEV int material_of(const TraceScene& ts) const { return __float_as_int(ldg(ts.tris + 3 * hit.tri).w); }
    PH_DEV float upper() const { return Unbounded ? kInf : (AnyHit ? limit : tmax); }

    // The boxes of the wide node (q0..q3): the nearest child entered is taken up, the others go on the stack.
    // False if none is entered.
    template <class Stack>
    PH_DEV bool visit_node(float4 q0, float4 q1, float4 q2, float4 q3, Stack& stack) {
        const uint32_t ex = __float_as_uint(q0.w);
        const float bx = __builtin_amdgcn_ldexpf(inv.x, int(int8_t(ex))), by = __builtin_amdgcn_ldexpf(inv.y, int(int8_t(ex >> 8))),
                    bz = __builtin_amdgcn_ldexpf(inv.z, int(int8_t(ex >> 16)));
        const float ax = (q0.x - o.x) * inv.x, ay = (q0.y - o.y) * inv.y, az = (q0.z - o.z) * inv.z;
        constexpr float kWiden = 0x1p-21f;
        const float nx = __builtin_fmaf(-kWiden, fabsf(ax), ax), fx = __builtin_fmaf(kWiden, fabsf(ax), ax);
        const float ny = __builtin_fmaf(-kWiden, fabsf(ay), ay), fy = __builtin_fmaf(kWiden, fabsf(ay), ay);
        const float nz = __builtin_fmaf(-kWiden, fabsf(az), az), fz = __builtin_fmaf(kWiden, fabsf(az), az);
        // The planes a ray meets first and last along each axis, by the sign of its direction.
        uint32_t wnx = __float_as_uint(q1.x), wfx = __float_as_uint(q1.y), wny = __float_as_uint(q1.z), wfy = __float_as_uint(q1.w);
        uint32_t wnz = __float_as_uint(q2.x), wfz = __float_as_uint(q2.y);
        if (inv.x < 0.0f) {
            const uint32_t t = wnx;
            wnx = wfx;
            wfx = t;
        }
        if (inv.y < 0.0f) {
            const uint32_t t = wny;
            wny = wfy;
            wfy = t;
        }
        if (inv.z < 0.0f) {
            const uint32_t t = wnz;
            wnz = wfz;
            wfz = t;
        }
        constexpr float kMissed = __builtin_inff();
        float key[4];
        int link[4] = {__float_as_int(q3.x), __float_as_int(q3.y), __float_as_int(q3.z), __float_as_int(q3.w)};
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const float tn = fmaxf(fmaxf(__builtin_fmaf(plane_byte(wnx, k), bx, nx), __builtin_fmaf(plane_byte(wny, k), by, ny)),
                                   fmaxf(__builtin_fmaf(plane_byte(wnz, k), bz, nz), 0.0f));
            const float tf = fminf(fminf(__builtin_fmaf(plane_byte(wfx, k), bx, fx), __builtin_fmaf(plane_byte(wfy, k), by, fy)),
                                   fminf(__builtin_fmaf(plane_byte(wfz, k), bz, fz), limit));
            key[k] = tn <= tf ? tn : kMissed;
        }
        auto order = [&](int a, int b) {
            const bool s = key[b] < key[a];
            const float ka = s ? key[b] : key[a], kb = s ? key[a] : key[b];
            const int la = s ? link[b] : link[a], lb = s ? link[a] : link[b];
            key[a] = ka;
            key[b] = kb;
            link[a] = la;
            link[b] = lb;
        };
        order(0, 1);
        order(2, 3);
        order(0, 2);
        if (!AnyHit) {
            order(1, 3);
            order(1, 2);
        }
        if (key[0] < kMissed) {
            cur = link[0];
            if (sp + 3 <= Stack::kDepth) {
                // Room in LDS for all three: an entry that is none is overwritten by the next.
#pragma unroll
                for (int k = 3; k >= 1; k--) {
                    stack.store_lds(sp, link[k], key[k]);
                    sp += key[k] < kMissed ? 1 : 0;
                }
            } else if (sp + 3 > kWideStack) {
                doubt = true;  // the ray is traced again
                if (!AnyHit) limit = -1.0f;
            } else {
#pragma unroll
                for (int k = 3; k >= 1; k--)
                    if (key[k] < kMissed) stack.store(sp++, link[k], key[k]);
            }
            return true;
        }
        return false;
    }

    // The triangle (q0..q2) of the leaf at `cur`. False if it was the leaf's last.
    PH_DEV bool visit_triangle(const TraceScene& ts, float4 q0, float4 q1, float4 q2) {
        const int tri = cur & (kWideMaxTris - 1);
        float t, u, v;
        if (mt_hit_any(xyz(q0), xyz(q1), xyz(q2), o, d, t, u, v) && t < limit) {
            bool cut = false;
            if (__float_as_int(q1.w) & PH_TRI_ALPHA_TESTED) cut = alpha_cut(*ts.full, tri, __float_as_int(q0.w), u, v);
            if (!cut) {
                if (AnyHit) {
                    hit.t = t;
                    hit.tri = tri;
                    leaf = __float_as_int(q2.w);
                    // the walk ends
                    sp = 0;
                    return false;
                }
                const bool first = hit.tri < 0;
                // A triangle near the closest hit so far marks the ray; one clearly in front of it, or the
                // first, starts afresh; one clearly behind it is of no interest.
                const bool clear = first || t < hit.t * kTieBelow;
                doubt = !clear && (doubt || (t <= hit.t * kTieAbove && tri != hit.tri));
                const bool nearer = first || t < hit.t;
                hit.t = nearer ? t : hit.t;
                hit.tri = nearer ? tri : hit.tri;
                hit.u = nearer ? u : hit.u;
                hit.v = nearer ? v : hit.v;
                leaf = nearer ? __float_as_int(q2.w) : leaf;
                limit = Unbounded ? hit.t * kCullAbove : fminf(hit.t * kCullAbove, tmax);
            }
        }
        if (((cur >> kWideCountShift) & (kWideMaxLeaf - 1)) == 0) return false;
        cur += 1 - (1 << kWideCountShift);
        return true;
    }

    // Takes up the nearest stack entry that can still matter. False if there is none.
    template <class Stack>
    PH_DEV bool pop(Stack& stack) {
        while (sp > 0) {
            float t;
            stack.load(--sp, cur, t);
            if (t <= limit) return true;
        }
        return false;
    }

    // One node or one triangle, as walk_step: every lane issues its loads before any lane uses them. False once the
    // walk is over. Letting lanes at a leaf wait until 8, 16 or 24 of them do measured 4 to 9 % slower in the render,
    // a node and then its leaf's triangle in one step 1 to 2 %.
    template <class Stack>
    PH_DEV bool step(const TraceScene& ts, Stack& stack) {
        const bool node = cur >= 0;
        const float4* p = node ? ts.wide + 4 * cur : ts.tris + 3 * (cur & (kWideMaxTris - 1));
        float4 q0 = ldg(p), q1 = ldg(p + 1), q2 = ldg(p + 2), q3 = ldg(node ? p + 3 : p);
        // The links are used last: without this the compiler moves their load behind the box tests, a second
        // round trip in every step.
        asm volatile("" : "+v"(q3.x), "+v"(q3.y), "+v"(q3.z), "+v"(q3.w));
        bool more;
        if (node)
            more = visit_node(q0, q1, q2, q3, stack);
        else
            more = visit_triangle(ts, q0, q1, q2);
        return more || pop(stack);
    }

    // After the walk: whether the answer is the binary walk's. If not, the ray is traced again over the binary nodes.
    PH_DEV bool settled(const TraceScene& ts) const {
        if (hit.tri < 0) return !doubt;
        const float4* box = ts.nodes + 2 * leaf;
        const float tl = slab(ldg(box), ldg(box + 1), o, inv, upper());
        const bool entered = tl != kInf && tl < upper();
        return AnyHit ? entered : entered && !doubt && tl <= hit.t * (1.0f + 0x1p-20f);
    }
};

// The whole query of one ray.
template <bool AnyHit, bool Unbounded, class Stack>
PH_DEV bool traverse_wide(const TraceScene& ts, f3 o, f3 d, float tmax, HitRec& hit, Stack& stack) {
    WideWalk<AnyHit, Unbounded> w;
    w.start(o, d, tmax);
    while (w.step(ts, stack)) {
    }
    hit = w.hit;
    if (!w.settled(ts)) {
        LaneStack<Stack::kDepth> s = stack.binary();
        BinaryWalk<AnyHit, false> b;
        b.start(o, d, tmax);
        while (b.step(ts, s)) {
        }
        hit = b.hit;
    }
    return hit.tri >= 0;
}

}  // namespace phd
