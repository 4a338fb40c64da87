// Device build of a resident scene's wide BVH, the index of the FP32
// closest-hit walk: primitives sorted by Morton code, neighbouring clusters
// merged pairwise to a binary tree, that tree cut into 8-wide nodes and leaves
// of up to 4 primitives at the least expected cost, the nodes written level
// by level; then a sample of rays chooses between it and the kd-tree. Launches
// and read-backs bound it for small scenes, memory for large ones (364 bytes of
// scratch a primitive).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <string>
#include <vector>

#include "device/xt_bvhbuild.h"
#include "device/xt_kdbuild.h"
#include "xt_device.h"
#include "xt_scratch.h"

#define XT_TRY(expr)                                                                  \
    do {                                                                              \
        hipError_t e_ = (expr);                                                       \
        if (e_ != hipSuccess) {                                                       \
            d->err = std::string(#expr) + ": " + hipGetErrorString(e_);               \
            return XT_E_DEVICE;                                                       \
        }                                                                             \
    } while (0)

#define XT_LAUNCHED()                                                                 \
    do {                                                                              \
        hipError_t e_ = hipGetLastError();                                            \
        if (e_ != hipSuccess) {                                                       \
            d->err = std::string("kernel launch: ") + hipGetErrorString(e_);          \
            return XT_E_DEVICE;                                                       \
        }                                                                             \
    } while (0)

namespace {

constexpr uint32_t kProbeRays = 4096;
constexpr int kMaxRounds = 160;   // of pairwise merging; a scene that needs more keeps the kd-tree walk
constexpr uint32_t kMaxDepth = 24;  // the deepest stack of the trace kernel

// One block of scratch memory, cut into arrays.
struct Block {
    char *p = nullptr;
    size_t bytes = 0, at = 0;
    template <class T>
    T *take(size_t count) {
        T *q = (T *)(p + at);
        at += (count * sizeof(T) + 255) & ~(size_t)255;
        return q;
    }
};

int scan(xt_dev *d, const uint64_t *in, uint64_t *out, uint32_t n, uint64_t *tiles) {
    const uint32_t nt = (uint32_t)(((uint64_t)n + XT_KDB_TILE - 1) / XT_KDB_TILE);
    if (nt) hipLaunchKernelGGL(k_kdb_scan_tiles, dim3(nt), dim3(256), 0, d->stream, in, out, n, tiles);
    hipLaunchKernelGGL(k_kdb_scan_sums, dim3(1), dim3(256), 0, d->stream, tiles, nt, out + n);
    if (nt) hipLaunchKernelGGL(k_kdb_scan_add, dim3(nt), dim3(256), 0, d->stream, out, n, (const uint64_t *)tiles);
    XT_LAUNCHED();
    return XT_OK;
}

// Which index the FP32 walk of a scene takes, from what a sample of rays costs
// on each (k_bvb_probe). The kd-tree clips primitives and ends a ray at its
// first hit; the wide BVH is cheaper for each ray until many boxes overlap at
// one place: fields of crossing triangles, dense hair, meshes so far from the
// origin that the boxes' slack is large against their triangles. No figure of the
// primitives alone told these apart (the boxes' area over the primitives' is 3.4
// for meshes, 5 for every soup below, 8 to 230 for hair, and one large floor
// hides a scene of hair from it). The weights are fitted to frames of 512x512x4
// and 1024x1024x4 paths and 1 M random rays of 57 scenes; one of them (300 random
// triangles) goes to a walk that is more than 2% slower than the other, by 12%. Time on the
// BVH over time on the kd-tree (geometric mean), and the ratio of the two costs:
//   icosphere of 1.31 M triangles 0.41 (0.37), one of 0.33 M 3,000 radii from
//     the origin 0.99 (0.88), 10,000 radii 1.95 (3.1)
//   terrain 0.57 (0.37), 64 spheres 0.86 (0.55), 500 random boxes 1.02 (1.2)
//   1 M random triangles in a cube 700 times as wide 0.48 (0.37), 200 times 0.98
//     (0.88), 70 times 2.3 (3.1), 20 times 6.7 (15)
//   strands: 2,000 0.65 (0.50), 10,000 0.81 (0.82), 30,000 1.21 (1.50), 50,000
//     1.61 (2.31), these over a floor of two triangles 1.57 (2.22)
bool bvh_walk_is_cheaper(const BvbInfo &s, uint32_t rays) {
    const double bvh = (double)s.nodes + 0.8 * (double)s.bvh_tests + 2.0 * rays;
    const double kd = 4.0 * (double)s.leaves + 0.5 * (double)s.kd_tests;
    return bvh <= kd;
}

}  // namespace

// Builds the wide BVH of a resident scene whose primitives, kd-tree and bounds
// are in place, if the trace would rather walk it than the kd-tree: `view`
// then names its arrays, which join ds.allocs. Otherwise view.bvh stays null.
int xt_bvh_build_into(xt_dev *d, DevScene &ds, XtScratch &mem) {
    SceneView &v = ds.view;
    const uint32_t n = v.n_prims;
    v.bvh = nullptr;
    v.bvh_leaf = nullptr;
    v.bvh_refs = nullptr;
    if (n == 0) return XT_OK;
    if (!d->host_words) XT_TRY(hipHostMalloc((void **)&d->host_words, 8192, hipHostMallocDefault));
    const uint32_t sort_tiles = (n + XT_BVB_SORT_TILE - 1) / XT_BVB_SORT_TILE;
    const size_t scan_n = std::max<size_t>((size_t)n + 4096, 256ull * sort_tiles) + 1;
    const uint32_t scan_tiles = (uint32_t)((scan_n + XT_KDB_TILE) / XT_KDB_TILE) + 1;
    const uint32_t cap = n + 4096;  // wide nodes, the unused ones among siblings included
    const size_t caps[] = {sizeof(BvbInfo), 8ull * n, 8ull * n, 4ull * cap, 4ull * cap,
                           2ull * n * sizeof(BvbNode), 4ull * n, 8ull * scan_n, 8ull * scan_n, 8ull * scan_tiles,
                           32ull * cap, (size_t)cap * sizeof(XtWideNode), 2 * sizeof(BvbCtl)};
    Block B;
    for (size_t c : caps) B.bytes += (c + 255) & ~(size_t)255;
    int rc = mem.take((void **)&B.p, B.bytes);
    if (rc == XT_E_BUDGET) return XT_OK;
    if (rc) return rc;
    BvbInfo *info = B.take<BvbInfo>(1);
    uint64_t *key[2] = {B.take<uint64_t>(n), nullptr};
    key[1] = B.take<uint64_t>(n);
    uint32_t *val[2] = {B.take<uint32_t>(cap), nullptr};
    val[1] = B.take<uint32_t>(cap);
    BvbNode *nodes = B.take<BvbNode>(2ull * n);
    uint32_t *nn = B.take<uint32_t>(n);
    uint64_t *flags = B.take<uint64_t>(scan_n), *sums = B.take<uint64_t>(scan_n);
    uint64_t *tiles = B.take<uint64_t>(scan_tiles);
    uint32_t *children = B.take<uint32_t>(8ull * cap);
    XtWideNode *wide = B.take<XtWideNode>(cap);
    BvbCtl *ctl = B.take<BvbCtl>(2);

    hipLaunchKernelGGL(k_fill_u32, dim3(1), dim3(64), 0, d->stream, (uint32_t *)info, 0u, sizeof(BvbInfo) / 4);
    // Morton order
    float ext = 0.f;
    for (int a = 0; a < 3; ++a) ext = std::max(ext, v.kb_hi[a] - v.kb_lo[a]);
    const float scale = ext > 0.f ? 2097152.f / ext : 0.f;
    const unsigned nb = (n + 255) / 256;
    hipLaunchKernelGGL(k_bvb_keys, dim3(nb), dim3(256), 0, d->stream, v.prims, n,
                       make_float3(v.kb_lo[0], v.kb_lo[1], v.kb_lo[2]), scale, key[0], val[0], info);
    for (uint32_t pass = 0; pass < 8; ++pass) {
        const int a = (int)(pass & 1u);
        hipLaunchKernelGGL(k_bvb_count, dim3(sort_tiles), dim3(256), 0, d->stream, (const uint64_t *)key[a], n,
                           8u * pass, flags);
        rc = scan(d, flags, sums, 256u * sort_tiles, tiles);
        if (rc) return rc;
        hipLaunchKernelGGL(k_bvb_scatter, dim3(sort_tiles), dim3(256), 0, d->stream, (const uint64_t *)key[a],
                           (const uint32_t *)val[a], n, 8u * pass, (const uint64_t *)sums, key[a ^ 1], val[a ^ 1]);
    }
    // clusters; the sort's value arrays hold their ids from here on
    hipLaunchKernelGGL(k_bvb_leaves, dim3(nb), dim3(256), 0, d->stream, v.prims, (const uint32_t *)val[0], n, nodes,
                       val[1], ctl);
    XT_LAUNCHED();
    uint32_t m = n;  // an upper bound of the clusters left
    int c = 1, q = 0;
    for (int round = 0; m > XT_BVB_SMALL && round < kMaxRounds; ++round) {
        const unsigned g = grid_for(m, 256, 8192);
        hipLaunchKernelGGL(k_bvb_nearest, dim3(g), dim3(256), 0, d->stream, (const BvbNode *)nodes,
                           (const uint32_t *)val[c], (const BvbCtl *)(ctl + q), nn);
        hipLaunchKernelGGL(k_bvb_flags, dim3(g), dim3(256), 0, d->stream, (const BvbCtl *)(ctl + q),
                           (const uint32_t *)nn, m, flags);
        rc = scan(d, flags, sums, m, tiles);
        if (rc) return rc;
        hipLaunchKernelGGL(k_bvb_merge, dim3(g), dim3(256), 0, d->stream, nodes, 2u * n, (const uint32_t *)val[c],
                           (const uint32_t *)nn, (const uint64_t *)sums, (const uint64_t *)(sums + m),
                           (const BvbCtl *)(ctl + q), ctl + (q ^ 1), val[c ^ 1]);
        XT_LAUNCHED();
        c ^= 1;
        q ^= 1;
        if (round % 3 == 2) {
            XT_TRY(hipMemcpyAsync(d->host_words, ctl + q, sizeof(BvbCtl), hipMemcpyDeviceToHost, d->stream));
            XT_TRY(hipStreamSynchronize(d->stream));
            m = ((const BvbCtl *)d->host_words)->m;
        }
    }
    hipLaunchKernelGGL(k_bvb_small, dim3(1), dim3(XT_BVB_SMALL), 0, d->stream, nodes, 2u * n,
                       (const uint32_t *)val[c], (const BvbCtl *)(ctl + q), &info->root);
    XT_LAUNCHED();
    const BvbInfo *const host = (const BvbInfo *)d->host_words;
    XT_TRY(hipMemcpyAsync(d->host_words, info, sizeof(BvbInfo), hipMemcpyDeviceToHost, d->stream));
    XT_TRY(hipStreamSynchronize(d->stream));
    if (host->bad || host->root >= 2u * n) return XT_OK;  // boxes that are not finite, or not merged to one root

    // wide nodes, level by level
    uint32_t *items[2] = {val[0], val[1]}, *refs = nn;
    XT_TRY(hipMemcpyAsync(items[0], &info->root, 4, hipMemcpyDeviceToDevice, d->stream));
    uint32_t base = 0, prim_base = 0, count = 1, depth = 0;
    for (int a = 0; count > 0; a ^= 1) {
        if (++depth > kMaxDepth || (uint64_t)base + count > std::min(cap, XT_WIDE_MAX_NODES)) return XT_OK;
        const unsigned g = (count + 127) / 128;
        hipLaunchKernelGGL(k_bvb_cut, dim3(g), dim3(128), 0, d->stream, (const BvbNode *)nodes,
                           (const uint32_t *)items[a], count, children, flags);
        rc = scan(d, flags, sums, count, tiles);
        if (rc) return rc;
        hipLaunchKernelGGL(k_bvb_emit, dim3(g), dim3(128), 0, d->stream, (const BvbNode *)nodes,
                           (const uint32_t *)items[a], count, (const uint32_t *)children, (const uint64_t *)sums, base,
                           prim_base, n, cap, wide, items[a ^ 1], refs);
        XT_LAUNCHED();
        XT_TRY(hipMemcpyAsync(d->host_words, sums + count, 8, hipMemcpyDeviceToHost, d->stream));
        XT_TRY(hipStreamSynchronize(d->stream));
        const uint64_t t = ((const uint64_t *)d->host_words)[0];
        base += count;
        prim_base += (uint32_t)(t >> 32);
        count = (uint32_t)t;
        if (prim_base > n) {
            d->err = "wide BVH build: more primitives than the scene has";
            return XT_E_STATE;
        }
    }
    if (prim_base != n) {
        d->err = "wide BVH build: primitives missing";
        return XT_E_STATE;
    }
    SceneView w = v;
    w.bvh = (const uint4 *)wide;
    w.bvh_refs = refs;
    hipLaunchKernelGGL(k_bvb_probe, dim3(2 * kProbeRays / XT_BVB_PROBE), dim3(XT_BVB_PROBE), 0, d->stream, w, info);
    XT_LAUNCHED();
    XT_TRY(hipMemcpyAsync(d->host_words, info, sizeof(BvbInfo), hipMemcpyDeviceToHost, d->stream));
    // the scene's own arrays, allocated while the sample is walked
    const uint64_t node_bytes = (uint64_t)base * sizeof(XtWideNode), ref_bytes = (4ull * n + 255) & ~255ull;
    const uint64_t bytes = node_bytes + ref_bytes + 48ull * n;
    if (d->budget && d->used + bytes > d->budget) return XT_OK;
    struct Own {
        char *p = nullptr;
        ~Own() {
            if (p) (void)hipFree(p);
        }
    } own;
    if (hipMalloc((void **)&own.p, bytes) != hipSuccess) {  // as beyond the budget: the kd-tree is walked
        own.p = nullptr;
        (void)hipGetLastError();
        return XT_OK;
    }
    uint32_t *const own_refs = (uint32_t *)(own.p + node_bytes);
    float4 *const own_leaf = (float4 *)(own.p + node_bytes + ref_bytes);
    XT_TRY(hipMemcpyAsync(own.p, wide, node_bytes, hipMemcpyDeviceToDevice, d->stream));
    XT_TRY(hipMemcpyAsync(own_refs, refs, 4ull * n, hipMemcpyDeviceToDevice, d->stream));
    hipLaunchKernelGGL(k_bvb_records, dim3(grid_for(n, 256, 16384)), dim3(256), 0, d->stream, v.prims,
                       (const uint32_t *)refs, n, own_leaf);
    XT_LAUNCHED();
    XT_TRY(hipStreamSynchronize(d->stream));
    if (!bvh_walk_is_cheaper(*host, kProbeRays)) return XT_OK;
    ds.allocs.push_back(own.p);
    ds.bytes += bytes;
    d->used += bytes;
    ds.bvh_depth = depth;
    v.bvh = (const uint4 *)own.p;
    v.bvh_refs = own_refs;
    v.bvh_leaf = own_leaf;
    own.p = nullptr;
    return XT_OK;
}
