// Kernels of the wide BVH build (xt_bvhbuild.hip).
#pragma once
#include <hip/hip_runtime.h>

#include "xt_kernels.h"

#define XT_BVB_RADIUS 12      // neighbours looked at on each side
#define XT_BVB_SMALL 1024     // clusters that one block merges to the root
#define XT_BVB_SORT_TILE 2048 // keys per block of a sorting pass
#define XT_BVB_PROBE 8        // rays of a wave that walks the sample
#define XT_BVB_COST_PRIM 0.4f // a primitive test against an inner node visit

// A node of the binary tree. Nodes [0, n) are the primitives in Morton order.
struct BvbNode {
    float lo[3];
    uint32_t left;   // primitive: its soup index
    float hi[3];
    uint32_t right;
    float cost[7];   // cost[i - 1]: the cheapest forest of at most i roots for the subtree
    uint32_t pick;   // 3 bits per i = 1..7: roots given to the left child (0: as with i - 1 roots), bit 31: a leaf
    uint32_t count;  // primitives below
    uint32_t pad[3];
};
static_assert(sizeof(BvbNode) == 80, "BvbNode layout");

struct BvbCtl {
    uint32_t m, next;  // clusters, next binary node
};

// What a build reports to the host.
struct BvbInfo {
    uint32_t bad, root;  // whether a box is not finite; binary node of the root, or XT_NONE
    // of a sample of rays: wide nodes visited and primitives tested on the
    // BVH, leaves visited and primitives tested on the kd-tree
    unsigned long long nodes, bvh_tests, leaves, kd_tests;
};

__device__ __forceinline__ float bvb_area(const float lo[3], const float hi[3]) {
    const float x = hi[0] - lo[0], y = hi[1] - lo[1], z = hi[2] - lo[2];
    return x * y + y * z + z * x;
}

__device__ __forceinline__ uint64_t bvb_spread(uint32_t v) {  // 21 bits, two zeros between bits
    uint64_t x = v & 0x1fffffu;
    x = (x | x << 32) & 0x1f00000000ffffull;
    x = (x | x << 16) & 0x1f0000ff0000ffull;
    x = (x | x << 8) & 0x100f00f00f00f00full;
    x = (x | x << 4) & 0x10c30c30c30c30c3ull;
    x = (x | x << 2) & 0x1249249249249249ull;
    return x;
}

// FP32 box of a primitive: exact for triangles, rounded outward for spheres.
__device__ __forceinline__ void bvb_prim_box(const float4 *prims, uint32_t p, float lo[3], float hi[3]) {
    const float4 a = prims[3 * (size_t)p], b = prims[3 * (size_t)p + 1], c = prims[3 * (size_t)p + 2];
    const float av[3] = {a.x, a.y, a.z};
    if (XT_PRIM_TYPE(__float_as_uint(a.w)) == XT_PRIM_TRIANGLE) {
        const float bv[3] = {b.x, b.y, b.z}, cv[3] = {c.x, c.y, c.z};
        for (int k = 0; k < 3; ++k) {
            lo[k] = fminf(av[k], fminf(bv[k], cv[k]));
            hi[k] = fmaxf(av[k], fmaxf(bv[k], cv[k]));
        }
    } else {
        const float r = fabsf(b.x);
        for (int k = 0; k < 3; ++k) {
            const float pad = 4e-7f * (fabsf(av[k]) + r);
            lo[k] = av[k] - r - pad;
            hi[k] = av[k] + r + pad;
        }
    }
}

static __global__ __launch_bounds__(256) void k_bvb_keys(const float4 *prims, uint32_t n, float3 org, float scale,
                                                         uint64_t *key, uint32_t *val, BvbInfo *info) {
    const uint32_t p = blockIdx.x * 256 + threadIdx.x;
    if (p >= n) return;
    float lo[3], hi[3];
    bvb_prim_box(prims, p, lo, hi);
    const float ha = bvb_area(lo, hi);
    if (!(fabsf(ha) < 1e30f) || !(fabsf(lo[0]) < 1e30f) || !(fabsf(lo[1]) < 1e30f) || !(fabsf(lo[2]) < 1e30f))
        info->bad = 1;
    const float og[3] = {org.x, org.y, org.z};
    uint64_t k = 0;
    for (int a = 0; a < 3; ++a) {
        const float f = (0.5f * lo[a] + 0.5f * hi[a] - og[a]) * scale;
        const uint32_t q = (uint32_t)fminf(fmaxf(f, 0.f), 2097151.f);
        k |= bvb_spread(q) << a;
    }
    key[p] = k;
    val[p] = p;
}

// One pass of a least-significant-digit radix sort on 8 bits: digit counts of
// each tile (digit-major, so that their exclusive scan gives every tile's
// place for every digit), then the stable scatter.
static __global__ __launch_bounds__(256) void k_bvb_count(const uint64_t *key, uint32_t n, uint32_t shift,
                                                          uint64_t *counts) {
    __shared__ uint32_t h[256];
    h[threadIdx.x] = 0;
    __syncthreads();
    const uint32_t t0 = blockIdx.x * XT_BVB_SORT_TILE;
    for (uint32_t k = threadIdx.x; k < XT_BVB_SORT_TILE; k += 256)
        if (t0 + k < n) atomicAdd(&h[(uint32_t)(key[t0 + k] >> shift) & 255u], 1u);
    __syncthreads();
    counts[(size_t)threadIdx.x * gridDim.x + blockIdx.x] = h[threadIdx.x];
}

static __global__ __launch_bounds__(256) void k_bvb_scatter(const uint64_t *key, const uint32_t *val, uint32_t n,
                                                            uint32_t shift, const uint64_t *place, uint64_t *key_out,
                                                            uint32_t *val_out) {
    constexpr uint32_t PER = XT_BVB_SORT_TILE / 256;  // rounds of a wave over its quarter of the tile
    __shared__ uint32_t wh[4][256];
    const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
    for (uint32_t k = threadIdx.x; k < 4 * 256; k += 256) wh[k >> 8][k & 255u] = 0;
    __syncthreads();
    const uint32_t t0 = blockIdx.x * XT_BVB_SORT_TILE + w * (XT_BVB_SORT_TILE / 4);
    uint32_t rank[PER];
    for (uint32_t r = 0; r < PER; ++r) {
        const uint32_t i = t0 + r * 64 + lane;
        const bool in = i < n;
        const uint32_t dg = in ? (uint32_t)(key[i] >> shift) & 255u : 0u;
        unsigned long long same = __ballot(in);
        for (int b = 0; b < 8; ++b) {
            const unsigned long long m = __ballot((dg >> b) & 1u);
            same &= (dg >> b) & 1u ? m : ~m;
        }
        const uint32_t before = (uint32_t)__popcll(same & ((1ull << lane) - 1ull));
        uint32_t at = 0;
        if (in) at = wh[w][dg];
        rank[r] = at + before;
        __builtin_amdgcn_wave_barrier();
        if (in && before == 0) wh[w][dg] = at + (uint32_t)__popcll(same);
        __builtin_amdgcn_wave_barrier();
        __threadfence_block();
    }
    __syncthreads();
    {  // counts of the waves before
        uint32_t run = 0;
        for (int k = 0; k < 4; ++k) {
            const uint32_t c = wh[k][threadIdx.x];
            wh[k][threadIdx.x] = run;
            run += c;
        }
    }
    __syncthreads();
    for (uint32_t r = 0; r < PER; ++r) {
        const uint32_t i = t0 + r * 64 + lane;
        if (i >= n) continue;
        const uint64_t kk = key[i];
        const uint32_t dg = (uint32_t)(kk >> shift) & 255u;
        const uint32_t at = (uint32_t)place[(size_t)dg * gridDim.x + blockIdx.x] + wh[w][dg] + rank[r];
        if (at < n) {
            key_out[at] = kk;
            val_out[at] = val[i];
        }
    }
}

static __global__ __launch_bounds__(256) void k_bvb_leaves(const float4 *prims, const uint32_t *order, uint32_t n,
                                                           BvbNode *nodes, uint32_t *cl, BvbCtl *ctl) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i == 0) {
        ctl[0].m = n;
        ctl[0].next = n;
    }
    if (i >= n) return;
    BvbNode nd = {};
    const uint32_t p = order[i];
    bvb_prim_box(prims, p, nd.lo, nd.hi);
    nd.left = p;
    nd.right = XT_NONE;
    const float c = bvb_area(nd.lo, nd.hi) * XT_BVB_COST_PRIM;
    for (int k = 0; k < 7; ++k) nd.cost[k] = c;
    nd.pick = 0x80000000u;
    nd.count = 1;
    nodes[i] = nd;
    cl[i] = i;
}

// The cluster next to i that makes the smallest box with it, among the
// XT_BVB_RADIUS on each side (Meister, Bittner, "Parallel Locally-Ordered
// Clustering for Bounding Volume Hierarchy Construction", TVCG 2018). Equal
// areas go to the smaller i ^ j: an order of the pairs that both ends agree
// on, in which a run of equal boxes pairs up completely.
template <int BS>
__device__ __forceinline__ uint32_t bvb_nearest(const float (*box)[6], int at, int lo, int hi, uint32_t first) {
    float best = INFINITY;
    uint32_t bj = XT_NONE, bx = XT_NONE;
    for (int j = lo; j <= hi; ++j) {
        if (j == at) continue;
        float l[3], h[3];
        for (int a = 0; a < 3; ++a) {
            l[a] = fminf(box[at][a], box[j][a]);
            h[a] = fmaxf(box[at][3 + a], box[j][3 + a]);
        }
        const float ar = bvb_area(l, h);
        const uint32_t x = (first + (uint32_t)at) ^ (first + (uint32_t)j);
        if (ar < best || (ar == best && x < bx)) {
            best = ar;
            bj = first + (uint32_t)j;
            bx = x;
        }
    }
    return bj;
}

static __global__ __launch_bounds__(256) void k_bvb_nearest(const BvbNode *nodes, const uint32_t *cl,
                                                            const BvbCtl *ctl, uint32_t *nn) {
    constexpr int R = XT_BVB_RADIUS;
    __shared__ float box[256 + 2 * R][6];
    const uint32_t m = ctl->m;
    const uint32_t tiles = (m + 255) / 256;
    for (uint32_t t = blockIdx.x; t < tiles; t += gridDim.x) {
        const int b0 = (int)(t * 256) - R;
        for (int k = (int)threadIdx.x; k < 256 + 2 * R; k += 256) {
            const int i = b0 + k;
            if (i >= 0 && i < (int)m) {
                const BvbNode &nd = nodes[cl[i]];
                for (int a = 0; a < 3; ++a) {
                    box[k][a] = nd.lo[a];
                    box[k][3 + a] = nd.hi[a];
                }
            }
        }
        __syncthreads();
        const int i = (int)(t * 256 + threadIdx.x);
        if (i < (int)m) {
            const int at = (int)threadIdx.x + R;
            const int lo = max(at - R, -b0), hi = min(at + R, (int)m - 1 - b0);
            nn[i] = bvb_nearest<256>(box, at, lo, hi, (uint32_t)b0);
        }
        __syncthreads();
    }
}

// Cluster i of the next round: low word 1 if it stays (alone, or as the
// first of a merged pair), high word 1 if it heads a merged pair.
__device__ __forceinline__ uint64_t bvb_flag(const uint32_t *nn, uint32_t i) {
    const uint32_t j = nn[i];
    if (j != XT_NONE && nn[j] == i) return i < j ? (1ull << 32) | 1ull : 0ull;
    return 1ull;
}

static __global__ __launch_bounds__(256) void k_bvb_flags(const BvbCtl *ctl, const uint32_t *nn, uint32_t cap,
                                                          uint64_t *flags) {
    const uint32_t m = ctl->m;
    for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < cap; i += gridDim.x * 256)
        flags[i] = i < m ? bvb_flag(nn, i) : 0ull;
}

// The parent of two clusters, with the cheapest ways to cut it into at most
// 1..7 roots of wide nodes and leaves (the dynamic programme of the wide BVH
// paper: an inner root costs its area plus its best cut into 8).
__device__ __forceinline__ void bvb_join(BvbNode *nodes, uint32_t l, uint32_t r, uint32_t id) {
    const BvbNode L = nodes[l], R = nodes[r];
    BvbNode nd;
    for (int a = 0; a < 3; ++a) {
        nd.lo[a] = fminf(L.lo[a], R.lo[a]);
        nd.hi[a] = fmaxf(L.hi[a], R.hi[a]);
    }
    nd.left = l;
    nd.right = r;
    nd.count = L.count + R.count;
    const float area = bvb_area(nd.lo, nd.hi);
    float dist[9];
    uint32_t cut[9];
#pragma unroll
    for (int i = 2; i <= 8; ++i) {
        float b = INFINITY;
        uint32_t c = 1;
#pragma unroll
        for (int k = 1; k < i; ++k) {
            if (k > 7 || i - k > 7) continue;
            const float v = L.cost[k - 1] + R.cost[i - k - 1];
            if (v < b) {
                b = v;
                c = (uint32_t)k;
            }
        }
        dist[i] = b;
        cut[i] = c;
    }
    uint32_t pick = cut[8];
    float prev = area + dist[8];
    if (nd.count <= XT_WIDE_LEAF && area * XT_BVB_COST_PRIM * (float)nd.count <= prev) {
        prev = area * XT_BVB_COST_PRIM * (float)nd.count;
        pick |= 0x80000000u;
    }
    nd.cost[0] = prev;
#pragma unroll
    for (int i = 2; i <= 7; ++i) {
        if (dist[i] < prev) {
            prev = dist[i];
            pick |= cut[i] << (3 * (i - 1));
        }
        nd.cost[i - 1] = prev;
    }
    nd.pick = pick;
    nd.pad[0] = nd.pad[1] = nd.pad[2] = 0;
    nodes[id] = nd;
}

static __global__ __launch_bounds__(256) void k_bvb_merge(BvbNode *nodes, uint32_t cap, const uint32_t *cl,
                                                          const uint32_t *nn, const uint64_t *scan,
                                                          const uint64_t *total, const BvbCtl *ctl, BvbCtl *ctl_out,
                                                          uint32_t *cl_out) {
    const uint32_t m = ctl->m, next = ctl->next;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        ctl_out->m = (uint32_t)*total;
        ctl_out->next = next + (uint32_t)(*total >> 32);
    }
    for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < m; i += gridDim.x * 256) {
        const uint64_t f = bvb_flag(nn, i);
        if (!(uint32_t)f) continue;
        const uint32_t pos = (uint32_t)scan[i];
        uint32_t id = cl[i];
        if (f >> 32) {
            const uint32_t nid = next + (uint32_t)(scan[i] >> 32);
            if (nid < cap) {
                bvb_join(nodes, id, cl[nn[i]], nid);
                id = nid;
            }
        }
        if (pos < m) cl_out[pos] = id;
    }
}

// The last clusters, merged to the root by one block; root gets its node.
// Every round merges at least one pair, so the rounds end.
static __global__ __launch_bounds__(XT_BVB_SMALL) void k_bvb_small(BvbNode *nodes, uint32_t cap, const uint32_t *cl,
                                                                   const BvbCtl *ctl, uint32_t *root) {
    __shared__ float box[XT_BVB_SMALL][6];
    __shared__ uint32_t id[XT_BVB_SMALL], near[XT_BVB_SMALL];
    __shared__ uint32_t wsum[2][XT_BVB_SMALL / 64];
    const int t = (int)threadIdx.x;
    uint32_t m = ctl->m, next = ctl->next;
    if (m > XT_BVB_SMALL) {
        if (t == 0) *root = XT_NONE;
        return;
    }
    if (t < (int)m) {
        id[t] = cl[t];
        const BvbNode &nd = nodes[id[t]];
        for (int a = 0; a < 3; ++a) {
            box[t][a] = nd.lo[a];
            box[t][3 + a] = nd.hi[a];
        }
    }
    __syncthreads();
    for (int round = 0; m > 1 && round < XT_BVB_SMALL; ++round) {
        if (t < (int)m)
            near[t] = bvb_nearest<XT_BVB_SMALL>(box, t, max(t - XT_BVB_RADIUS, 0),
                                                min(t + XT_BVB_RADIUS, (int)m - 1), 0u);
        __syncthreads();
        uint64_t f = 0;
        uint32_t a = 0, b = 0;
        if (t < (int)m) {
            f = bvb_flag(near, (uint32_t)t);
            a = id[t];
            if (f >> 32) b = id[near[t]];
        }
        const bool stay = (uint32_t)f != 0u, pair = (f >> 32) != 0u;
        const unsigned long long ms = __ballot(stay), mp = __ballot(pair);
        if ((t & 63) == 0) {
            wsum[0][t >> 6] = (uint32_t)__popcll(ms);
            wsum[1][t >> 6] = (uint32_t)__popcll(mp);
        }
        __syncthreads();
        uint32_t ps = rank_in(ms), pp = rank_in(mp), ts = 0, tp = 0;
        for (int w = 0; w < XT_BVB_SMALL / 64; ++w) {
            if (w < (t >> 6)) {
                ps += wsum[0][w];
                pp += wsum[1][w];
            }
            ts += wsum[0][w];
            tp += wsum[1][w];
        }
        if (pair && next + pp < cap) {
            bvb_join(nodes, a, b, next + pp);
            a = next + pp;
        }
        __syncthreads();
        if (stay) {
            id[ps] = a;
            const BvbNode &nd = nodes[a];
            for (int k = 0; k < 3; ++k) {
                box[ps][k] = nd.lo[k];
                box[ps][3 + k] = nd.hi[k];
            }
        }
        m = ts;
        next += tp;
        __threadfence_block();
        __syncthreads();
    }
    if (t == 0) *root = m == 1 ? id[0] : XT_NONE;
}

// The cut of one inner root into at most 8 children, placed in slots:
// children[8 j + s] = binary node of slot s (XT_NONE: empty); counts[j] =
// nodes its children take (low word: 8, or 0 without inner children) and
// primitives of leaf children (high word). An item XT_NONE is a node that no
// child uses.
static __global__ __launch_bounds__(128) void k_bvb_cut(const BvbNode *nodes, const uint32_t *items, uint32_t n_items,
                                                        uint32_t *children, uint64_t *counts) {
    const uint32_t j = blockIdx.x * 128 + threadIdx.x;
    if (j >= n_items) return;
    const uint32_t id = items[j];
    if (id == XT_NONE) {
        counts[j] = 0;
        return;
    }
    const BvbNode nd = nodes[id];
    uint32_t ch[8], n = 0;
    if (nd.pick & 0x80000000u) {
        ch[n++] = id;  // a root that is a leaf itself
    } else {
        uint32_t sid[8], si[8], top = 0;
        const uint32_t k8 = nd.pick & 7u;
        sid[top] = nd.right;
        si[top++] = 8u - k8;
        sid[top] = nd.left;
        si[top++] = k8;
        while (top > 0) {
            const uint32_t c = sid[--top];
            uint32_t i = si[top];
            const BvbNode &q = nodes[c];
            uint32_t k = 0;
            if (q.right != XT_NONE)
                while (i > 1 && (k = (q.pick >> (3 * (i - 1))) & 7u) == 0u) --i;
            if (q.right == XT_NONE || i <= 1) {
                if (n < 8) ch[n++] = c;
                continue;
            }
            if (top + 2 <= 8) {
                sid[top] = q.right;
                si[top++] = i - k;
                sid[top] = q.left;
                si[top++] = k;
            }
        }
    }
    float cx[8], cy[8], cz[8];
    for (uint32_t c = 0; c < n; ++c) {
        const BvbNode &q = nodes[ch[c]];
        cx[c] = q.lo[0] + q.hi[0] - nd.lo[0] - nd.hi[0];
        cy[c] = q.lo[1] + q.hi[1] - nd.lo[1] - nd.hi[1];
        cz[c] = q.lo[2] + q.hi[2] - nd.lo[2] - nd.hi[2];
    }
    uint32_t placed = 0, taken = 0;
    uint32_t slot[8];
    for (uint32_t r = 0; r < n; ++r) {
        float best = INFINITY;
        uint32_t bc = 0, bs = 0;
        bool found = false;
        for (uint32_t c = 0; c < n; ++c) {
            if ((placed >> c) & 1u) continue;
            for (uint32_t s = 0; s < 8; ++s) {
                if ((taken >> s) & 1u) continue;
                const float v = (s & 1u ? -cx[c] : cx[c]) + (s & 2u ? -cy[c] : cy[c]) + (s & 4u ? -cz[c] : cz[c]);
                if (!found || v < best) {
                    best = v;
                    bc = c;
                    bs = s;
                    found = true;
                }
            }
        }
        placed |= 1u << bc;
        taken |= 1u << bs;
        slot[bc] = bs;
    }
    for (uint32_t s = 0; s < 8; ++s) children[8 * (size_t)j + s] = XT_NONE;
    uint32_t inner = 0, prims = 0;
    for (uint32_t c = 0; c < n; ++c) {
        const BvbNode &q = nodes[ch[c]];
        children[8 * (size_t)j + slot[c]] = ch[c];
        if (q.pick & 0x80000000u) prims += q.count;
        else ++inner;
    }
    counts[j] = (uint64_t)prims << 32 | (inner ? 8u : 0u);
}

// Writes the level's wide nodes [base, base + n_items), the next level's
// items and the leaves' primitives.
static __global__ __launch_bounds__(128) void k_bvb_emit(const BvbNode *nodes, const uint32_t *items, uint32_t n_items,
                                                         const uint32_t *children, const uint64_t *scan,
                                                         uint32_t base, uint32_t prim_base, uint32_t n_prims,
                                                         uint32_t cap, XtWideNode *out, uint32_t *next_items,
                                                         uint32_t *refs) {
    const uint32_t j = blockIdx.x * 128 + threadIdx.x;
    if (j >= n_items || base + j >= cap) return;
    XtWideNode w = {};
    if (items[j] == XT_NONE) {
        out[base + j] = w;
        return;
    }
    const BvbNode nd = nodes[items[j]];
    const uint32_t at = (uint32_t)scan[j], p0 = prim_base + (uint32_t)(scan[j] >> 32);
    float ext = 0.f;
    for (int a = 0; a < 3; ++a) {
        w.p[a] = nd.lo[a];
        ext = fmaxf(ext, nd.hi[a] - nd.lo[a]);
    }
    w.step = fmaxf(ext * (1.f / (XT_WIDE_GRID - 0.01f)), 1e-30f);
    const float inv = 1.f / w.step;
    uint32_t np = 0, inner = 0;
    for (uint32_t s = 0; s < 8; ++s) {
        const uint32_t c = children[8 * (size_t)j + s];
        if (c == XT_NONE) continue;
        const BvbNode &q = nodes[c];
        for (int a = 0; a < 3; ++a) {
            // one part in 2^20 covers the roundings of the division
            const float l = floorf((q.lo[a] - nd.lo[a]) * inv * (1.f - 1e-6f)), h = ceilf((q.hi[a] - nd.lo[a]) * inv * (1.f + 1e-6f));
            const _Float16 fl = (_Float16)fminf(fmaxf(l, 0.f), XT_WIDE_GRID), fh = (_Float16)fminf(fmaxf(h, 0.f), XT_WIDE_GRID);
            w.plane[a][s] = __builtin_bit_cast(uint16_t, fl);
            w.plane[3 + a][s] = __builtin_bit_cast(uint16_t, fh);
        }
        if (q.pick & 0x80000000u) {
            w.masks |= (1u | ((q.count - 1u) & 1u) << 8 | ((q.count - 1u) >> 1 & 1u) << 16) << s;
            // at most XT_WIDE_LEAF primitives below
            uint32_t stk[8], top = 0;
            stk[top++] = c;
            while (top > 0) {
                const BvbNode &x = nodes[stk[--top]];
                if (x.right == XT_NONE) {
                    if (p0 + np < n_prims) refs[p0 + np] = x.left;
                    ++np;
                } else if (top + 2 <= 8) {
                    stk[top++] = x.right;
                    stk[top++] = x.left;
                }
            }
        } else {
            w.masks |= 1u << (24 + s);
            inner = 1;
        }
    }
    if (inner)
        for (uint32_t s = 0; s < 8; ++s)
            if (at + s < cap)
                next_items[at + s] = (w.masks >> (24 + s)) & 1u ? children[8 * (size_t)j + s] : XT_NONE;
    w.child = inner ? base + n_items + at : 0u;
    w.prims = p0;
    out[base + j] = w;
}

// Leaf records in the tree's order: the primitive with its soup index as object word.
static __global__ __launch_bounds__(256) void k_bvb_records(const float4 *prims, const uint32_t *refs, uint32_t n,
                                                            float4 *leaf) {
    for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
        const uint32_t p = refs[i];
        const float4 a = prims[3 * (size_t)p];
        float4 b = prims[3 * (size_t)p + 1];
        b.w = __uint_as_float(p);
        leaf[3 * (size_t)i] = a;
        leaf[3 * (size_t)i + 1] = b;
        leaf[3 * (size_t)i + 2] = prims[3 * (size_t)p + 2];
    }
}

// ------------------------------------------------------------------- the choice

// Ray i of the sample: through or from a primitive drawn by i, in a random
// direction; even rays come from outside the scene, odd ones leave the
// primitive as a bounce ray does.
__device__ __forceinline__ RayF probe_ray(const SceneView &S, uint32_t i) {
    const uint32_t key = xt_stream(xt_mix32(i + 1u), 1u);
    const uint32_t p = xt_draw(key, 0) % S.n_prims;
    const float4 a = S.prims[3 * (size_t)p], b = S.prims[3 * (size_t)p + 1], c = S.prims[3 * (size_t)p + 2];
    const float z = 2.f * xt_unit32(xt_draw(key, 1)) - 1.f, phi = 6.2831853f * xt_unit32(xt_draw(key, 2));
    const float s = sqrtf(fmaxf(0.f, 1.f - z * z));
    RayF r;
    r.d = mk(s * cosf(phi), s * sinf(phi), z);
    f3 at;
    if (XT_PRIM_TYPE(__float_as_uint(a.w)) == XT_PRIM_TRIANGLE)
        at = mk((a.x + b.x + c.x) / 3.f, (a.y + b.y + c.y) / 3.f, (a.z + b.z + c.z) / 3.f);
    else at = add(mk(a.x, a.y, a.z), scl(r.d, fabsf(b.x)));
    r.origin = XT_NONE;
    r.self_t = 0.f;
    if (i & 1u) {
        r.o = at;
        r.origin = p;
    } else {
        const f3 ext = mk(S.kb_hi[0] - S.kb_lo[0], S.kb_hi[1] - S.kb_lo[1], S.kb_hi[2] - S.kb_lo[2]);
        r.o = sub(at, scl(r.d, sqrtf(dot3(ext, ext))));
    }
    return r;
}

struct ProbeTester {
    Tester32 t;
    uint32_t leaves, tests;
    __device__ __forceinline__ float limit() const { return t.limit(); }
    __device__ __forceinline__ void test_leaf_range(uint32_t k, uint32_t n) {
        ++leaves;
        tests += n;
        for (uint32_t j = 0; j < n; ++j) t.test(t.S.kd_refs[k + j]);
    }
};

__device__ __forceinline__ void probe_add(unsigned long long *to, uint32_t v) {
    for (int o = XT_BVB_PROBE / 2; o > 0; o >>= 1) v += (uint32_t)__shfl_xor((int)v, o);
    if (threadIdx.x == 0) atomicAdd(to, (unsigned long long)v);
}

// Walks the sample on both indexes, one lane a ray, and adds up the steps: the
// first half of the blocks on the kd-tree, the second half the same rays on the
// BVH. Bound by the longest chain of dependent loads, on the BVH and the kd-tree
// side by side, and by lanes that wait for each other: 4096 rays in waves of 8
// take two thirds of the time of 8192 in waves of 64 (four scenes' mean 448 to 297
// us, 0.1 ms of an upload of 20,493 triangles that takes 5.4).
static __global__ __launch_bounds__(XT_BVB_PROBE) void k_bvb_probe(const SceneView S, BvbInfo *out) {
    __shared__ uint2 kstk[(XT_KD_STACK + 1) * XT_BVB_PROBE];
    __shared__ uint32_t bstk[24 * XT_BVB_PROBE];
    const uint32_t half = gridDim.x / 2;
    const RayF r = probe_ray(S, (blockIdx.x % half) * XT_BVB_PROBE + threadIdx.x);
    Tester32 tst{S, r, tsmall_of(r.o), {}, make_shear(r.d)};
    seed_best(r, tst.best);
    for (uint32_t k = 0; k < S.n_planes; ++k)
        plane32(r.o, r.d, tst.tsmall, S.planes[k], XT_PLANE_BASE + k, tst.best);
    if (blockIdx.x < half) {
        ProbeTester kd{tst, 0, 0};
        (void)walk_kd<XT_KD_STACK>(S, kd, r.o, r.d, kstk + threadIdx.x, XT_BVB_PROBE, 1e-6f);
        probe_add(&out->leaves, kd.leaves);
        probe_add(&out->kd_tests, kd.tests);
        return;
    }

    // the walk of k_trace_bvh, one lane a ray
    const f3 inv = mk(rcp_dir(r.d.x), rcp_dir(r.d.y), rcp_dir(r.d.z));
    const f3 eta = box_slack(r.o, inv, slack_base(S));
    const uint32_t oct = octant_of(inv);
    uint32_t grp = 1u << oct, sp = threadIdx.x, nodes = 0, tests = 0;
    while (grp) {
        const uint32_t bit = (uint32_t)__builtin_ctz(grp);
        grp &= grp - 1u;
        const uint4 *nd = S.bvh + 8 * (size_t)((grp >> 8) + (bit ^ oct));
        const half8 *pl = (const half8 *)(nd + 2);
        const uint4 n1 = nd[1];
        ++nodes;
        const uint32_t nx = oct & 1u ? 3u : 0u, ny = oct & 2u ? 4u : 1u, nz = oct & 4u ? 5u : 2u;
        const uint32_t hits = wide_hits(*(const float4 *)nd, pl[nx], pl[ny], pl[nz], pl[3u - nx], pl[5u - ny],
                                        pl[7u - nz], r.o, inv, eta, tst.limit() * (1.f + 4e-6f));
        for (uint32_t lh = hits & n1.z & 0xffu; lh; lh &= lh - 1u) {
            const uint32_t slot = (uint32_t)__builtin_ctz(lh);
            const uint32_t below = n1.z & ((1u << slot) - 1u) * 0x010101u, cb = n1.z >> slot;
            const uint32_t k0 = n1.y + (uint32_t)__popc(below) + (uint32_t)__popc(below >> 16);
            const uint32_t n = 1u + ((cb >> 8) & 1u) + ((cb >> 15) & 2u);
            tests += n;
            for (uint32_t k = k0; k < k0 + n; ++k) tst.test(S.bvh_refs[k]);
        }
        const uint32_t ih = octant_order(hits & (n1.z >> 24), oct);
        if (ih) {
            if (grp & 0xffu) {
                bstk[sp] = grp;
                sp += XT_BVB_PROBE;
            }
            grp = ih | n1.x << 8;
        } else if (!(grp & 0xffu)) {
            grp = 0;
            if (sp >= XT_BVB_PROBE) {
                sp -= XT_BVB_PROBE;
                grp = bstk[sp];
            }
        }
    }
    probe_add(&out->nodes, nodes);
    probe_add(&out->bvh_tests, tests);
}
