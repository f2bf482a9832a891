// The four-wide nodes of a scene (dwide.h), from its binary nodes.
//
// Wide node i is made from binary node i alone: starting with its two children, the interior child of the
// largest surface area is replaced by its own two children until there are four. So every node is one
// thread's work, and its place in the array is its binary node's, which its parent's link then needs no list
// for. The nodes that no walk reaches, since a wide node holds their children, stay as gaps: listing only the
// others, breadth first, took a block 0.6 ms of the upload of 1M triangles and made no walk faster (1080p render
// 70.8 ms listed, 71.0 in place; 4M rays 0.445 and 0.448; mixed serving 26.2 and 26.3).
#include "dwide.h"
#include "internal.h"

using namespace phd;

namespace phk {

namespace {

struct Child {
    f3 lo, hi;
    int link, count;  // as in the binary node
};

PH_DEV bool interior(const Child& c) { return c.count <= 0 && c.link >= 0; }

PH_DEV float half_area(const Child& c) {
    const f3 e = c.hi - c.lo;
    return e.x * e.y + e.y * e.z + e.z * e.x;
}

// The children of binary node `i`, in slots [n, n + 2) of `c` (those that exist); returns the new count.
PH_DEV int add_children(const float4* nodes, int i, Child* c, int n) {
    const float4 a = nodes[4 * i], b = nodes[4 * i + 1], e = nodes[4 * i + 2], f = nodes[4 * i + 3];
    const Child l{xyz(a), xyz(b), __float_as_int(a.w), __float_as_int(b.w)}, r{xyz(e), xyz(f), __float_as_int(e.w), __float_as_int(f.w)};
    if (l.count > 0 || l.link >= 0) c[n++] = l;
    if (r.count > 0 || r.link >= 0) c[n++] = r;
    return n;
}

// The up to four descendants of binary node `i` that its wide node holds.
PH_DEV int collapse(const float4* nodes, int num_nodes, int i, Child* c) {
    int n = add_children(nodes, i, c, 0);
    while (n < 4) {
        int best = -1;
        float area = -1.0f;
        for (int k = 0; k < n; k++)
            if (interior(c[k]) && c[k].link < num_nodes && !(half_area(c[k]) <= area)) {
                best = k;
                area = half_area(c[k]);
            }
        if (best < 0) break;
        const int node = c[best].link;
        c[best] = c[--n];
        n = add_children(nodes, node, c, n);
    }
    return n;
}

PH_DEV bool inside(const Child& c, const Child& box) {
    return c.lo.x >= box.lo.x && c.lo.y >= box.lo.y && c.lo.z >= box.lo.z && c.hi.x <= box.hi.x && c.hi.y <= box.hi.y && c.hi.z <= box.hi.z;
}

// Planes of one axis: the exponent of the step, the origin below the lowest plane, and each child's planes.
PH_DEV void quantise_axis(const float* lo, const float* hi, int n, float& origin, int& exponent, uint32_t& wlo, uint32_t& whi) {
    float a = lo[0], b = hi[0];
    for (int k = 1; k < n; k++) {
        a = fminf(a, lo[k]);
        b = fmaxf(b, hi[k]);
    }
    // A step of at least 1/250 of the extent, so that 255 of them hold it with one to spare at each end, and
    // of several ulps of the planes, so that the origin lies below them.
    const double need = fmax(fmax((double(b) - double(a)) / 250.0, 0x1p-21 * fmax(fabs(double(a)), fabs(double(b)))), 0x1p-60);
    exponent = ilogb(need) + 1;
    const double step = ldexp(1.0, exponent), per_step = ldexp(1.0, -exponent);
    origin = float(double(a) - step);
    wlo = whi = 0;
    for (int k = 0; k < 4; k++) {
        int ql = 255, qh = 0;  // an unused child: inverted
        if (k < n) {
            ql = max(0, int(floor((double(lo[k]) - double(origin)) * per_step - 0x1p-10)));
            qh = min(255, int(ceil((double(hi[k]) - double(origin)) * per_step + 0x1p-10)));
        }
        wlo |= uint32_t(ql) << (8 * k);
        whi |= uint32_t(qh) << (8 * k);
    }
}

// Makes wide node i, and checks that what it is made from lies within the format's limits (*beyond becomes nonzero where
// not). The binary nodes' boxes must nest: a wide node leaves out the boxes between its node and the descendants it
// holds, which the binary walk tests.
__global__ __launch_bounds__(256) void wide_node_kernel(const float4* nodes, int num_nodes, int num_tris, float4* wide, int* beyond) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= num_nodes) return;
    Child c[4];
    bool ok = true;
    const int sides = add_children(nodes, i, c, 0);
    for (int k = 0; k < sides; k++) {
        if (!interior(c[k]) || c[k].link >= num_nodes) continue;
        Child below[2];
        const int m = add_children(nodes, c[k].link, below, 0);
        for (int j = 0; j < m; j++) ok = ok && inside(below[j], c[k]);
    }
    const int n = collapse(nodes, num_nodes, i, c);
    int link[4];
    for (int k = 0; k < n; k++) {
        const f3 a = c[k].lo, b = c[k].hi;
        const float reach = fmaxf(fmaxf(fmaxf(fabsf(a.x), fabsf(a.y)), fabsf(a.z)), fmaxf(fmaxf(fabsf(b.x), fabsf(b.y)), fabsf(b.z)));
        const float sum = (a.x + a.y + a.z) + (b.x + b.y + b.z);
        ok = ok && reach <= kWideReach && sum == sum && a.x <= b.x && a.y <= b.y && a.z <= b.z;
        if (interior(c[k])) {
            ok = ok && c[k].link < num_nodes;
            link[k] = c[k].link;
        } else {
            ok = ok && c[k].count <= kWideMaxLeaf && c[k].link >= 0 && c[k].link <= num_tris - c[k].count;
            link[k] = int(0x80000000u | (uint32_t(c[k].count - 1) << kWideCountShift) | uint32_t(c[k].link));
        }
    }
    for (int k = n; k < 4; k++) link[k] = n > 0 ? link[0] : int(0x80000000u);
    if (!ok) {
        *beyond = 1;
        return;
    }
    float lo[3][4], hi[3][4];
    for (int k = 0; k < n; k++) {
        lo[0][k] = c[k].lo.x, lo[1][k] = c[k].lo.y, lo[2][k] = c[k].lo.z;
        hi[0][k] = c[k].hi.x, hi[1][k] = c[k].hi.y, hi[2][k] = c[k].hi.z;
    }
    if (n == 0)
        for (int a = 0; a < 3; a++) lo[a][0] = hi[a][0] = 0.0f;
    float origin[3];
    int e[3];
    uint32_t wl[3], wh[3];
    for (int a = 0; a < 3; a++) {
        quantise_axis(lo[a], hi[a], max(n, 1), origin[a], e[a], wl[a], wh[a]);
        if (n == 0) wl[a] = 0xffffffffu, wh[a] = 0;
    }
    const uint32_t ex = uint32_t(e[0] & 255) | uint32_t(e[1] & 255) << 8 | uint32_t(e[2] & 255) << 16;
    wide[4 * i] = make_float4(origin[0], origin[1], origin[2], __uint_as_float(ex));
    wide[4 * i + 1] = make_float4(__uint_as_float(wl[0]), __uint_as_float(wh[0]), __uint_as_float(wl[1]), __uint_as_float(wh[1]));
    wide[4 * i + 2] = make_float4(__uint_as_float(wl[2]), __uint_as_float(wh[2]), 0.0f, 0.0f);
    wide[4 * i + 3] = make_float4(__int_as_float(link[0]), __int_as_float(link[1]), __int_as_float(link[2]), __int_as_float(link[3]));
}

// Writes each triangle's leaf (2 * binary node + side) into the triangle's fourth unused word.
__global__ __launch_bounds__(256) void leaf_of_kernel(const float4* nodes, int num_nodes, int num_tris, float4* tris) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= num_nodes) return;
    for (int side = 0; side < 2; side++) {
        const int link = __float_as_int(nodes[4 * i + 2 * side].w), count = __float_as_int(nodes[4 * i + 2 * side + 1].w);
        if (count <= 0 || link < 0) continue;
        for (int k = 0; k < count && link + k < num_tris; k++) tris[3 * (link + k) + 2].w = __int_as_float(2 * i + side);
    }
}

}  // namespace

void build_wide_nodes(hipStream_t st, const float4* nodes, int num_nodes, int num_tris, WideNodes& wide) {
    wide.queued = false;
    if (num_nodes <= 0 || num_tris <= 0 || num_tris > kWideMaxTris) return;
    wide.nodes.allocate(size_t(num_nodes) * 4);
    if (!wide.beyond) PH_CHECK(hipHostMalloc(reinterpret_cast<void**>(&wide.beyond), sizeof(int), hipHostMallocDefault));
    *wide.beyond = 0;  // the stream of the last build has been waited for
    hipLaunchKernelGGL(wide_node_kernel, dim3((num_nodes + 255) / 256), dim3(256), 0, st, nodes, num_nodes, num_tris, wide.nodes.ptr, wide.beyond);
    PH_CHECK(hipGetLastError());
    wide.queued = true;
}

void mark_leaves(hipStream_t st, const float4* nodes, int num_nodes, int num_tris, float4* tris) {
    hipLaunchKernelGGL(leaf_of_kernel, dim3((num_nodes + 255) / 256), dim3(256), 0, st, nodes, num_nodes, num_tris, tris);
    PH_CHECK(hipGetLastError());
}

}  // namespace phk
