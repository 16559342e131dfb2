// ff_pack.hip -- a scene's traversal and shading arrays, packed on the GPU
// from a binary BVH (host SAH, linear or PLOC: one node format for all) and
// the caller's triangle arrays.
#include <hip/hip_runtime.h>

#include <rocprim/device/device_scan.hpp>
#include <rocprim/iterator/transform_iterator.hpp>

#include <stdint.h>

#include <algorithm>
#include <vector>

#include "ff_internal.h"

namespace ffk {
namespace {

constexpr uint32_t PK_BLOCK = 256;

// ---------------------------------------------- compressed wide records --
// One level of the wide tree: a thread per wide node gathers up to four
// children by opening, again and again, the child of the largest surface area
// (an interior node into its two children; a leaf of several triangles into
// halves, each with the leaf's own box), writes the node's record, its
// triangles' records and queues its wide children for the next level.
struct WItem {
    int32_t node;  // binary node
    int32_t a, b;  // leaf: its triangles' slots [a, b)
    uint32_t out;  // record index
};

__device__ __forceinline__ float half_area(const ffh::BvhNode& n) {
    float dx = n.bmax[0] - n.bmin[0], dy = n.bmax[1] - n.bmin[1], dz = n.bmax[2] - n.bmin[2];
    float a = (dx * dy + dy * dz) + dz * dx;
    return a >= 0.f ? a : 0.f;  // (inf * 0 of a box beyond the floats' range)
}
// bfloat16 bits of a value not above (dir < 0) or not below (dir > 0) x by at
// least the padding of the conservative plane test
__device__ __forceinline__ uint32_t bf16_out(double x, double tiny, int dir) {
    double p = x + (double)dir * (fabs(x) * 0x1p-16 + tiny);
    float f = (float)p;
    if (dir < 0 ? (double)f > p : (double)f < p) f = nextafterf(f, dir < 0 ? -INFINITY : INFINITY);
    uint32_t u = __float_as_uint(f), hi = u >> 16;
    bool away = (f < 0.f) == (dir < 0);  // rounding outwards grows the magnitude
    if ((u & 0xffffu) && away) hi += 1u;
    return hi;
}

// level 0: the root
__global__ void k_wide_root(const ffh::BvhNode* __restrict__ nodes, WItem* q) {
    const ffh::BvhNode r = nodes[0];
    WItem it{0, 0, -1, 0u};
    if (r.n_prims != 0) {
        it.a = r.offset;
        it.b = r.offset + r.n_prims;
    }
    q[0] = it;
}
__global__ __launch_bounds__(PK_BLOCK) void k_wide_level(const ffh::BvhNode* __restrict__ nodes,
                                                        const float* __restrict__ tris, const WItem* __restrict__ in,
                                                        const uint32_t* __restrict__ n_in, WItem* __restrict__ next,
                                                        uint32_t* n_next, uint32_t* groups, float4* __restrict__ rec) {
    const uint32_t n = *n_in;
    for (uint32_t i = blockIdx.x * PK_BLOCK + threadIdx.x; i < n; i += gridDim.x * PK_BLOCK) {
        WItem it = in[i];
        WItem c[4];
        float area[4];
        int m = 0;
        auto put = [&](int32_t node, int32_t a, int32_t b) {
            const ffh::BvhNode& nd = nodes[node];
            if (nd.n_prims != 0 && b < 0) {
                a = nd.offset;
                b = nd.offset + nd.n_prims;
            }
            c[m].node = node;
            c[m].a = a;
            c[m].b = b;
            area[m] = nd.n_prims != 0 && b - a == 1 ? -1.f : half_area(nd);
            m++;
        };
        auto open = [&](const WItem& w) {
            const ffh::BvhNode& nd = nodes[w.node];
            if (nd.n_prims == 0) {
                put(w.node + 1, 0, -1);
                put(nd.offset, 0, -1);
            } else if (w.b - w.a > 1) {
                int32_t mid = w.a + (w.b - w.a + 1) / 2;
                put(w.node, w.a, mid);
                put(w.node, mid, w.b);
            } else {
                put(w.node, w.a, w.b);
            }
        };
        open(it);
        while (m > 1 && m < 4) {
            int k = -1;
            float best = -1.f;
            for (int j = 0; j < m; j++)
                if (area[j] > best) {
                    best = area[j];
                    k = j;
                }
            if (k < 0) break;  // single triangles only
            WItem w = c[k];
            m--;
            c[k] = c[m];
            area[k] = area[m];
            open(w);
        }
        // wide children first
        int ni = 0;
        for (int j = 0; j < m; j++)
            if (area[j] >= 0.f) {
                WItem w = c[j];
                c[j] = c[ni];
                c[ni] = w;
                float t = area[j];
                area[j] = area[ni];
                area[ni] = t;
                ni++;
            }
        uint32_t g = 4u * atomicAdd(groups, 1u);
        const ffh::BvhNode& me = nodes[it.node];
        float org[3];
        double ext = 0.0;
        for (int a = 0; a < 3; a++) {
            org[a] = 0.5f * me.bmin[a] + 0.5f * me.bmax[a];
            ext = fmax(ext, (double)me.bmax[a] - (double)me.bmin[a]);
        }
        double tiny = ext * 0x1p-40 + 0x1p-100;
        uint32_t w[12];
        for (int a = 0; a < 3; a++)
            for (int h = 0; h < 2; h++) {
                uint32_t lo = 0u, hi = 0u;
                for (int q = 0; q < 2; q++) {
                    int k = 2 * h + q;
                    uint32_t l = 0x7f80u, u = 0xff80u;  // empty: (+inf, -inf)
                    if (k < m) {
                        const ffh::BvhNode& nd = nodes[c[k].node];
                        l = bf16_out((double)nd.bmin[a] - (double)org[a], tiny, -1);
                        u = bf16_out((double)nd.bmax[a] - (double)org[a], tiny, 1);
                    }
                    lo |= l << (16 * q);
                    hi |= u << (16 * q);
                }
                w[2 * a + h] = lo;
                w[6 + 2 * a + h] = hi;
            }
        float4* R = rec + (size_t)it.out * 4;
        R[0] = make_float4(org[0], org[1], org[2], __uint_as_float(g | ((uint32_t)ni << 29)));
        for (int q = 0; q < 3; q++)
            R[1 + q] = make_float4(__uint_as_float(w[4 * q]), __uint_as_float(w[4 * q + 1]),
                                   __uint_as_float(w[4 * q + 2]), __uint_as_float(w[4 * q + 3]));
        uint32_t dst = ni ? atomicAdd(n_next, (uint32_t)ni) : 0u;
        for (int k = 0; k < 4; k++) {
            if (k < ni) {
                WItem x = c[k];
                x.out = g + (uint32_t)k;
                next[dst + (uint32_t)k] = x;
                continue;
            }
            float4* L = rec + (size_t)(g + (uint32_t)k) * 4;
            if (k >= m) {  // no triangle: one without area, which nothing hits
                for (int q = 0; q < 4; q++) L[q] = make_float4(0.f, 0.f, 0.f, 0.f);
                continue;
            }
            const float* t = tris + (size_t)c[k].a * 9;
            const ffh::BvhNode& nd = nodes[c[k].node];
            L[0] = make_float4(t[0], t[1], t[2], t[3]);
            L[1] = make_float4(t[4], t[5], t[6], t[7]);
            L[2] = make_float4(t[8], __int_as_float(c[k].a), nd.bmin[0], nd.bmin[1]);
            L[3] = make_float4(nd.bmin[2], nd.bmax[0], nd.bmax[1], nd.bmax[2]);
        }
    }
}

// ---------------------------------------------------- binary tree records --
struct IsInterior {
    __host__ __device__ uint32_t operator()(const ffh::BvhNode& n) const { return n.n_prims == 0 ? 1u : 0u; }
};

// The reference's pre-order binary BVH re-packed, a record per interior node
// (numbered in pre-order, `rank`):
//  - 64-byte two-child records: both child boxes, the child refs and the split
//    axis.  Leaf refs are ~(first slot << 4 | count), count 15 meaning "read
//    leaf_count[first slot]".
//  - 128-byte 4-wide records: the boxes of the node's grandchildren, slots 0-1
//    under its first child, 2-3 under its second (a child that is a leaf keeps
//    its own box in the first slot of its pair and leaves the second empty),
//    plus the three split axes (node, first child, second child) that order
//    them: lo.x, lo.y, lo.z, hi.x, hi.y, hi.z of slots 0..3, refs, axes.  An
//    empty slot has the box (+inf, -inf), which every slab test misses, and
//    the ref of a leaf with no triangles.  The walk reaches every second level
//    of the tree; the records of the others are not read.
__global__ __launch_bounds__(PK_BLOCK) void k_pack_nodes(const ffh::BvhNode* __restrict__ nodes,
                                                        const uint32_t* __restrict__ rank, int32_t n_nodes,
                                                        float4* __restrict__ two, float4* __restrict__ four,
                                                        int32_t* __restrict__ leaf_count, float* __restrict__ root) {
    for (uint32_t t = blockIdx.x * PK_BLOCK + threadIdx.x; t < (uint32_t)n_nodes; t += gridDim.x * PK_BLOCK) {
        const int32_t i = (int32_t)t;
        const ffh::BvhNode me = nodes[i];
        auto ref_of = [&](int32_t j, const ffh::BvhNode& nd) -> int32_t {
            if (nd.n_prims == 0) return (int32_t)rank[j];
            int32_t c = nd.n_prims < 15 ? nd.n_prims : 15;
            return ~((nd.offset << 4) | c);
        };
        if (i == 0) {
            for (int a = 0; a < 3; a++) {
                root[a] = me.bmin[a];
                root[3 + a] = me.bmax[a];
            }
            root[6] = __int_as_float(ref_of(0, me));
            root[7] = 0.f;
        }
        if (me.n_prims != 0) {
            if (me.n_prims >= 15) leaf_count[me.offset] = me.n_prims;
            continue;
        }
        const int32_t kid[2] = {i + 1, me.offset};
        const ffh::BvhNode A = nodes[kid[0]], B = nodes[kid[1]];
        float4* w = two + (size_t)rank[i] * 4;
        w[0] = make_float4(A.bmin[0], A.bmin[1], A.bmin[2], A.bmax[0]);
        w[1] = make_float4(A.bmax[1], A.bmax[2], B.bmin[0], B.bmin[1]);
        w[2] = make_float4(B.bmin[2], B.bmax[0], B.bmax[1], B.bmax[2]);
        w[3] = make_float4(__int_as_float(ref_of(kid[0], A)), __int_as_float(ref_of(kid[1], B)),
                           __int_as_float((int)me.axis), 0.f);
        float lo[3][4], hi[3][4];
        int32_t ref[4], ax[4] = {(int32_t)me.axis, 0, 0, 0};
        for (int side = 0; side < 2; side++) {
            const ffh::BvhNode& C = side ? B : A;
            const bool in = C.n_prims == 0;
            if (in) ax[1 + side] = (int32_t)C.axis;
            for (int k = 0; k < 2; k++) {
                const int s = 2 * side + k;
                if (!in && k == 1) {
                    for (int a = 0; a < 3; a++) {
                        lo[a][s] = INFINITY;
                        hi[a][s] = -INFINITY;
                    }
                    ref[s] = -1;  // a leaf of zero triangles
                    continue;
                }
                const int32_t j = in ? (k == 0 ? kid[side] + 1 : C.offset) : kid[side];
                const ffh::BvhNode nd = nodes[j];
                for (int a = 0; a < 3; a++) {
                    lo[a][s] = nd.bmin[a];
                    hi[a][s] = nd.bmax[a];
                }
                ref[s] = ref_of(j, nd);
            }
        }
        float4* f = four + (size_t)rank[i] * 8;
        for (int a = 0; a < 3; a++) {
            f[a] = make_float4(lo[a][0], lo[a][1], lo[a][2], lo[a][3]);
            f[3 + a] = make_float4(hi[a][0], hi[a][1], hi[a][2], hi[a][3]);
        }
        f[6] = make_float4(__int_as_float(ref[0]), __int_as_float(ref[1]), __int_as_float(ref[2]),
                           __int_as_float(ref[3]));
        f[7] = make_float4(__int_as_float(ax[0]), __int_as_float(ax[1]), __int_as_float(ax[2]), 0.f);
    }
}

// reorder_primitives (CRT/kernel.cu:184-191,701-712): the triangles in slot
// order, as positions-only records v0 | e1 | e2 and as 64-byte shading records.
__global__ __launch_bounds__(PK_BLOCK) void k_pack_slots(const int32_t* __restrict__ ordered,
                                                        const float* __restrict__ pos, const float* __restrict__ nrm,
                                                        const float* __restrict__ uv, const float* __restrict__ tan_in,
                                                        const int32_t* __restrict__ mid,
                                                        const float* __restrict__ mats, int32_t n,
                                                        float* __restrict__ tris, float* __restrict__ attr,
                                                        uint32_t* __restrict__ mat, float* __restrict__ tan) {
    for (uint32_t i = blockIdx.x * PK_BLOCK + threadIdx.x; i < (uint32_t)n; i += gridDim.x * PK_BLOCK) {
        const size_t src = (size_t)ordered[i];
        const float* p = pos + src * 9;
        float* t = tris + (size_t)i * 9;
        for (int k = 0; k < 3; k++) {
            t[k] = p[k];
            t[3 + k] = p[3 + k] - p[k];
            t[6 + k] = p[6 + k] - p[k];
        }
        float* a = attr + (size_t)i * 16;
        for (int k = 0; k < 9; k++) a[k] = nrm[src * 9 + k];
        for (int k = 0; k < 6; k++) a[9 + k] = uv ? uv[src * 6 + k] : 0.f;
        const uint32_t m = (uint32_t)mid[src];
        const uint32_t word = m | ((uint32_t)(int)mats[(size_t)m * FF_MAT_FLOATS_DEV] << MAT_TYPE_SHIFT);
        a[15] = __uint_as_float(word);
        mat[i] = word;
        if (tan)
            for (int k = 0; k < 18; k++) tan[(size_t)i * 18 + k] = tan_in[src * 18 + k];
    }
}

uint32_t pack_grid(size_t n) { return (uint32_t)std::min<size_t>((n + PK_BLOCK - 1) / PK_BLOCK, 8192); }

}  // namespace

hipError_t upload_bvh(const std::vector<ffh::BvhNode>& nodes, const std::vector<int32_t>& ordered, int32_t max_depth,
                      const float* positions, DevBvh& out) {
    const size_t n = ordered.size();
    auto carve = [&](Carver c) {
        out.nodes = c.take<ffh::BvhNode>(nodes.size());
        out.ordered = c.take<int32_t>(n);
        out.pos = c.take<float>(9 * n);
        return c.off;
    };
    hipError_t e = hipMalloc(&out.mem, carve(Carver{}));
    if (e != hipSuccess) return e;
    carve(Carver{(char*)out.mem});
    out.n_nodes = (int32_t)nodes.size();
    out.max_depth = max_depth;
    out.max_leaf = 1;
    for (const ffh::BvhNode& b : nodes) out.max_leaf = std::max(out.max_leaf, (int32_t)b.n_prims);
    e = hipMemcpy(out.nodes, nodes.data(), nodes.size() * sizeof(ffh::BvhNode), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(out.ordered, ordered.data(), 4 * n, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(out.pos, positions, 36 * n, hipMemcpyHostToDevice);
    return e;
}

// (n triangles make a tree of at most 2n - 1 nodes)
static auto interior_flags(const ffh::BvhNode* nodes) {
    return rocprim::make_transform_iterator(nodes, IsInterior());
}
hipError_t upload_arrays(const SceneArrays& a, PackScratch& tmp) {
    const size_t n = (size_t)a.n;
    size_t scan_bytes = 0;
    hipError_t e = rocprim::exclusive_scan(nullptr, scan_bytes, interior_flags(nullptr), tmp.rank, 0u, 2 * n,
                                           rocprim::plus<uint32_t>(), nullptr);
    if (e != hipSuccess) return e;
    auto carve = [&](Carver c) {
        tmp.rank = c.take<uint32_t>(2 * n);
        tmp.nrm = c.take<float>(9 * n);
        tmp.uv = c.take<float>(a.uv ? 6 * n : 0);
        tmp.tan = c.take<float>(a.tan ? 18 * n : 0);
        tmp.mid = c.take<int32_t>(n);
        tmp.q0 = c.take<WItem>(n);
        tmp.q1 = c.take<WItem>(n);
        tmp.scan_tmp = c.take<char>(scan_bytes);
        return c.off;
    };
    e = hipMalloc(&tmp.mem, carve(Carver{}));
    if (e != hipSuccess) return e;
    carve(Carver{(char*)tmp.mem});
    e = hipMemcpy(tmp.nrm, a.nrm, 36 * n, hipMemcpyHostToDevice);
    if (e == hipSuccess && a.uv) e = hipMemcpy(tmp.uv, a.uv, 24 * n, hipMemcpyHostToDevice);
    if (e == hipSuccess && a.tan) e = hipMemcpy(tmp.tan, a.tan, 72 * n, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(tmp.mid, a.mid, 4 * n, hipMemcpyHostToDevice);
    return e;
}

hipError_t pack_scene(const DevBvh& bvh, const SceneArrays& a, PackScratch& tmp, ScenePack& out) {
    const size_t n = (size_t)a.n, n_int = ((size_t)bvh.n_nodes - 1) / 2;  // a full binary tree
    // a group with fewer than four children holds single triangles only, so
    // n triangles make at most 2n/3 + 1 groups
    const size_t groups = 1 + (2 * n + 2) / 3 + 1;
    int32_t split = 0;
    while ((1 << split) < bvh.max_leaf) split++;
    const int32_t max_levels = bvh.max_depth + split + 2;
    uint32_t* cnt = nullptr;  // [levels + 1] wide nodes of each level, then the groups handed out
    auto carve = [&](Carver c) {
        out.nodes = c.take<float4>(4 * n_int);
        out.nodes4 = c.take<float4>(8 * n_int);
        out.wide = c.take<float4>(16 * groups);
        out.attr = c.take<float4>(4 * n);
        out.leaf_count = c.take<int32_t>(n);
        out.root = c.take<float>(8);
        out.tris = c.take<float>(9 * n);
        out.mats = c.take<float>((size_t)FF_MAT_FLOATS_DEV * a.n_mats);
        out.mat = c.take<uint32_t>(n);
        float* tan = c.take<float>(a.tan ? 18 * n : 0);
        out.tan = a.tan ? tan : nullptr;
        cnt = c.take<uint32_t>((size_t)max_levels + 2);
        return c.off;
    };
    hipError_t e = hipSuccess;
    auto ok = [&](hipError_t x) { if (e == hipSuccess) e = x; return e == hipSuccess; };
    std::vector<uint32_t> h((size_t)max_levels + 2, 0u);
    h[0] = 1u;                       // level 0: the root
    h[(size_t)max_levels + 1] = 1u;  // groups: the root's own
    size_t scan_bytes = 0;
    auto interior = interior_flags(bvh.nodes);
    if (ok(rocprim::exclusive_scan(nullptr, scan_bytes, interior, tmp.rank, 0u, (size_t)bvh.n_nodes,
                                   rocprim::plus<uint32_t>(), nullptr)) &&
        ok(hipMalloc(&out.mem, carve(Carver{})))) {
        carve(Carver{(char*)out.mem});
        ok(hipMemcpy(out.mats, a.mats, sizeof(float) * FF_MAT_FLOATS_DEV * a.n_mats, hipMemcpyHostToDevice));
        ok(hipMemcpy(cnt, h.data(), h.size() * 4, hipMemcpyHostToDevice));
        ok(hipMemsetAsync(out.leaf_count, 0, 4 * n, nullptr));
        ok(rocprim::exclusive_scan(tmp.scan_tmp, scan_bytes, interior, tmp.rank, 0u, (size_t)bvh.n_nodes,
                                   rocprim::plus<uint32_t>(), nullptr));
    }
    if (e == hipSuccess) {
        hipLaunchKernelGGL(k_pack_slots, dim3(pack_grid(n)), dim3(PK_BLOCK), 0, nullptr, bvh.ordered, bvh.pos, tmp.nrm,
                           a.uv ? tmp.uv : nullptr, a.tan ? tmp.tan : nullptr, tmp.mid, out.mats, a.n, out.tris,
                           (float*)out.attr, out.mat, out.tan);
        hipLaunchKernelGGL(k_pack_nodes, dim3(pack_grid((size_t)bvh.n_nodes)), dim3(PK_BLOCK), 0, nullptr, bvh.nodes,
                           tmp.rank, bvh.n_nodes, out.nodes, out.nodes4, out.leaf_count, out.root);
        WItem *q0 = (WItem*)tmp.q0, *q1 = (WItem*)tmp.q1;
        hipLaunchKernelGGL(k_wide_root, dim3(1), dim3(1), 0, nullptr, bvh.nodes, q0);
        ok(hipGetLastError());
        // Four children to a node: a balanced tree ends after half the binary
        // tree's levels, so the rest is launched only if the tree goes on there
        // (of 82 k triangles 14 levels instead of 26 launched, 4.5 us each).
        size_t at_most = 1;
        int32_t l = 0;
        for (int32_t stop : {max_levels / 2 + 1, max_levels}) {
            for (stop = std::min(stop, max_levels); l < stop && e == hipSuccess; l++) {
                hipLaunchKernelGGL(k_wide_level, dim3(pack_grid(at_most)), dim3(PK_BLOCK), 0, nullptr, bvh.nodes,
                                   out.tris, q0, cnt + l, q1, cnt + l + 1, cnt + max_levels + 1, out.wide);
                ok(hipGetLastError());
                std::swap(q0, q1);
                at_most = std::min<size_t>(at_most * 4, n);
            }
            if (!ok(hipMemcpy(h.data(), cnt, h.size() * 4, hipMemcpyDeviceToHost)) || !h[(size_t)l]) break;
        }
        out.wide_levels = 0;
        while (e == hipSuccess && out.wide_levels < max_levels && h[(size_t)out.wide_levels]) out.wide_levels++;
    }
    if (tmp.mem) (void)hipFree(tmp.mem);
    tmp.mem = nullptr;
    if (e != hipSuccess && out.mem) {
        (void)hipFree(out.mem);
        out.mem = nullptr;
    }
    return e;
}

}  // namespace ffk
