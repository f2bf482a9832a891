// The four-wide nodes of a scene (dwide.h), from its binary nodes.
//
// Wide node i is made from binary node i alone: starting with its two children, the interior child of the
// largest surface area is replaced by its own two children until there are four. So every node is one
// thread's work. Only the nodes that a walk from the root can reach are kept: a block lists them in
// breadth-first order (a wide node's interior children are neighbours), and the wide nodes are written
// in that order.
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

// Every binary node's interior children in its wide node (-1: none), and whether all of them and its leaves lie
// within the format's limits (status[1] becomes nonzero where not). The binary nodes' boxes must nest: a wide node
// leaves out the boxes between its node and the descendants it holds, which the binary walk tests.
__global__ __launch_bounds__(256) void wide_children_kernel(const float4* nodes, int num_nodes, int num_tris, int4* children, int* status) {
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
    int inner[4] = {-1, -1, -1, -1}, m = 0;
    for (int k = 0; k < n; k++) {
        const f3 a = c[k].lo, b = c[k].hi;
        const float reach = fmaxf(fmaxf(fmaxf(fabsf(a.x), fabsf(a.y)), fabsf(a.z)), fmaxf(fmaxf(fabsf(b.x), fabsf(b.y)), fabsf(b.z)));
        const float sum = (a.x + a.y + a.z) + (b.x + b.y + b.z);
        ok = ok && reach <= kWideReach && sum == sum && a.x <= b.x && a.y <= b.y && a.z <= b.z;
        if (interior(c[k])) {
            ok = ok && c[k].link < num_nodes;
            inner[m++] = c[k].link;
        } else {
            ok = ok && c[k].count <= kWideMaxLeaf && c[k].link >= 0 && c[k].link <= num_tris - c[k].count;
        }
    }
    if (!ok) atomicOr(status + 1, 1);
    children[i] = make_int4(inner[0], inner[1], inner[2], inner[3]);
}

constexpr int kListThreads = 1024;

// Lists the binary nodes whose wide nodes a walk reaches, breadth first from the root: list[k] is the
// binary node of wide node k, and first_child[k] the wide node of its first interior child (the others
// follow). One block: the frontier is taken 1024 nodes at a time, and a scan places each node's children.
// status[0] is the number of wide nodes.
__global__ __launch_bounds__(kListThreads) void wide_list_kernel(const int4* children, int num_nodes, int* list, int* first_child, int* status) {
    __shared__ int wave_total[kListThreads / 64];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    if (status[1]) return;
    if (t == 0) list[0] = 0;
    __syncthreads();
    int done = 0, total = 1;  // nodes whose children are listed; nodes listed
    while (done < total) {
        const int here = min(kListThreads, total - done);
        const int4 c = t < here ? children[list[done + t]] : make_int4(-1, -1, -1, -1);
        const int inner = (c.x >= 0) + (c.y >= 0) + (c.z >= 0) + (c.w >= 0);
        // Exclusive scan of the interior children over the block.
        int v = inner;
        for (int off = 1; off < 64; off <<= 1) {
            const int u = __shfl_up(v, off);
            if (lane >= off) v += u;
        }
        if (lane == 63) wave_total[wave] = v;
        __syncthreads();
        int before = 0, sum = 0;
        for (int w = 0; w < kListThreads / 64; w++) {
            if (w < wave) before += wave_total[w];
            sum += wave_total[w];
        }
        // A tree has no more interior children than nodes; anything else (a cycle) is left to the binary walk.
        if (total + sum > num_nodes) {
            if (t == 0) status[1] = 1;
            return;
        }
        const int at = total + before + v - inner;
        if (t < here) {
            first_child[done + t] = at;
            if (inner > 0) list[at] = c.x;
            if (inner > 1) list[at + 1] = c.y;
            if (inner > 2) list[at + 2] = c.z;
            if (inner > 3) list[at + 3] = c.w;
        }
        done += here;
        total += sum;
        __threadfence_block();
        __syncthreads();
    }
    if (t == 0) status[0] = total;
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
    const double step = ldexp(1.0, exponent);
    origin = float(double(a) - step);
    wlo = whi = 0;
    for (int k = 0; k < 4; k++) {
        int ql = 255, qh = 0;  // an unused child: inverted
        if (k < n) {
            ql = max(0, int(floor((double(lo[k]) - double(origin)) / step - 0x1p-10)));
            qh = min(255, int(ceil((double(hi[k]) - double(origin)) / step + 0x1p-10)));
        }
        wlo |= uint32_t(ql) << (8 * k);
        whi |= uint32_t(qh) << (8 * k);
    }
}

__global__ __launch_bounds__(256) void wide_node_kernel(const float4* nodes, int num_nodes, const int* list, const int* first_child, int count,
                                                        float4* wide) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= count) return;
    Child c[4];
    const int n = collapse(nodes, num_nodes, list[i], c);
    int link[4], at = first_child[i];
    for (int k = 0; k < 4; k++) {
        if (k >= n)
            link[k] = n > 0 ? link[0] : int(0x80000000u);
        else if (interior(c[k]))
            link[k] = at++;
        else
            link[k] = int(0x80000000u | (uint32_t(c[k].count - 1) << kWideCountShift) | uint32_t(c[k].link));
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

bool build_wide_nodes(hipStream_t st, const float4* nodes, int num_nodes, int num_tris, DevBuf<float4>& wide) {
    wide.release();
    if (num_nodes <= 0 || num_tris <= 0 || num_tris > kWideMaxTris) return false;
    DevBuf<int> list, first_child, status;
    DevBuf<int4> children;
    children.allocate(size_t(num_nodes));
    list.allocate(size_t(num_nodes));
    first_child.allocate(size_t(num_nodes));
    status.allocate(2);
    status.zero(st);
    hipLaunchKernelGGL(wide_children_kernel, dim3((num_nodes + 255) / 256), dim3(256), 0, st, nodes, num_nodes, num_tris, children.ptr, status.ptr);
    hipLaunchKernelGGL(wide_list_kernel, dim3(1), dim3(kListThreads), 0, st, children.ptr, num_nodes, list.ptr, first_child.ptr, status.ptr);
    PH_CHECK(hipGetLastError());
    int host[2] = {0, 0};  // wide nodes, limits exceeded
    PH_CHECK(hipMemcpyAsync(host, status.ptr, sizeof(host), hipMemcpyDeviceToHost, st));
    PH_CHECK(hipStreamSynchronize(st));
    if (host[1] || host[0] <= 0) return false;
    wide.allocate(size_t(host[0]) * 4);
    hipLaunchKernelGGL(wide_node_kernel, dim3((host[0] + 255) / 256), dim3(256), 0, st, nodes, num_nodes, list.ptr, first_child.ptr, host[0], wide.ptr);
    PH_CHECK(hipGetLastError());
    PH_CHECK(hipStreamSynchronize(st));  // the lists above are freed
    return true;
}

void mark_leaves(hipStream_t st, const float4* nodes, int num_nodes, int num_tris, float4* tris) {
    hipLaunchKernelGGL(leaf_of_kernel, dim3((num_nodes + 255) / 256), dim3(256), 0, st, nodes, num_nodes, num_tris, tris);
    PH_CHECK(hipGetLastError());
}

}  // namespace phk
