// The FP32 closest-hit kernel over the wide BVH: persistent waves whose lanes
// walk on their own and get new rays as the kd-tree walk's do (xt_trace_kd.h).
// A camera ray of the 1.31 M-triangle icosphere visits 6 nodes and 1.5
// triangles here, against 25 nodes, 6 leaves and 3.2 triangles of the kd-tree
// (random rays 2.8 and 0.6, against 11 and 1.2), and the arrays it reads are
// 63 MB of triangles and 18 MB of nodes, against 289 MB and 54 MB.
//
// Once the queue is empty, idle lanes help: one takes the siblings that a
// walking lane has not visited yet, or the top of its stack, walks them with the
// ray's state and hands its closest hit back; the lanes of a ray share the
// closest distance. What bounds a queue of fewer rays than the card has lanes is
// the chain of dependent loads of the rays with the longest walks, and this
// shares them out: 100,003 terrain camera rays 115 to 86 us, a 333x211 depth
// frame 236 to 191, 256x256x4 paths 715 to 560, and the end of larger launches
// (4 M random rays 710 to 545, 1080p 16 spp paths 16.2 to 15.0 ms).
//
// Bound by VALU issue and by the return of its gathers: on the 1080p icosphere
// frame the vector units are busy 71% of the time, at 38 of 64 lanes, and the
// texture data units 81%, three quarters of that waiting for L1 and L2; on 4 M
// random rays 63% at 31 lanes, and 84%. What it
// measured, trace time of that frame's 72.1 M queries with the launches one
// after another: kd-tree walk 15.5 ms, this 9.4 ms; 4 M random rays 1256 to
// 718 us. With 80-byte nodes of 8-bit planes (48 conversions more per node)
// the walk issued 15% more instructions.
#pragma once
#include "xt_walk.h"

#define XT_W_KEEP 6    // sixteenths of the working lanes at which a phase of a turn ends (3: 3% slower, 8: 1%)
#define XT_W_FREE 32   // walked rays of a wave at which they are finished for their lanes to help (8: 4% slower at 72 K rays)
#define XT_W_FAR 1e3f     // scene extents up to which a ray's origin widens the boxes
#define XT_W_WAVES 4   // waves per SIMD: as many as the LDS of 10 KB a wave leaves room for

// Gathers records of PARTS 16-byte parts into LDS: record `rec` (an index) of
// every lane of `mask`, in the order of the lanes. Lane number rank finds its
// record at buf[PARTS * rank]. Neighbouring lanes load neighbouring parts, so
// that each 64 bytes of a record are one access of the vector L1. With 8 parts
// (a stride of 128 bytes) part p lies at place p ^ (rank & 7), so that lanes
// reading one part of their records spread over the LDS banks.
// Loaded lane by lane instead, the parts of one lane's record come in separate
// instructions whose 64 lanes touch 64 lines each: 1.6 times the accesses of
// the vector L1, at the same frame time as long as the work cursor set the pace.
template <uint32_t PARTS, class OFF>
__device__ __forceinline__ void gather_records(const void *base, uint32_t rec, unsigned long long mask, uint32_t lane,
                                               uint32_t rank, bool on, uint4 *buf) {
    const uint32_t n = (uint32_t)__popcll(mask);
    // the records' indices in rank order, where the records go afterwards
    uint32_t *const list = (uint32_t *)buf;
    if (on) list[rank] = rec;
    __builtin_amdgcn_wave_barrier();
    uint32_t id[PARTS] = {};
#pragma unroll
    for (uint32_t k = 0; k < PARTS; ++k)
        if (k == 0 || n * PARTS > 64u * k) id[k] = list[PARTS == 8 ? 8u * k + (lane >> 3) : (64u * k + lane) / PARTS];
    // every index is in a register before the first record part lands on the list
#pragma unroll
    for (uint32_t k = 0; k < PARTS; ++k) asm volatile("" ::"v"(id[k]) : "memory");
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    const uint32_t part8 = ((lane & 7u) ^ (lane >> 3)) * 16u;
#pragma unroll
    for (uint32_t k = 0; k < PARTS; ++k) {
        if (k == 0 || n * PARTS > 64u * k) {
            const uint32_t c = 64u * k + lane, r = c / PARTS, part = (c - r * PARTS) * 16u;
            if (PARTS == 8 ? (lane >> 3) + 8u * k < n : r < n) {
                const char *src = (const char *)base + ((OFF)id[k] * (OFF)(16u * PARTS) + (OFF)(PARTS == 8 ? part8 : part));
                __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)src,
                                                 (__attribute__((address_space(3))) void *)(buf + 64u * k), 16, 0, 0);
            }
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// A helper's result into its ray's: the closest hit as one more candidate, and
// what the helper deferred. The ray's decisions stay what they would be for one
// lane: candidates within the tie band go to the FP64 re-check.
__device__ __forceinline__ void merge_best(Best &b, uint32_t &rec, float t, uint32_t prim, uint32_t prec, float mark_t,
                                           uint32_t c0, uint32_t c1) {
    if (prim != XT_NONE) {
        const uint32_t was = b.prim;
        offer(b, t, prim);
        rec = b.prim != was ? prec : rec;
    }
    if (c0 != XT_NONE) defer(b, mark_t, c0);
    if (c1 == XT_CAND_OVERFLOW) b.c1 = c1;
    else if (c1 != XT_NONE) defer(b, mark_t, c1);
}

__device__ __forceinline__ float from_lane(float v, uint32_t src) {
    return __int_as_float(__builtin_amdgcn_ds_bpermute((int)(src << 2), __float_as_int(v)));
}
__device__ __forceinline__ uint32_t from_lane(uint32_t v, uint32_t src) {
    return (uint32_t)__builtin_amdgcn_ds_bpermute((int)(src << 2), (int)v);
}
__device__ __forceinline__ float lane_value(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

typedef _Float16 half8 __attribute__((ext_vector_type(8)));

// The slots of a node whose boxes the ray enters before lim: n0 the grid's
// origin and step, near and far planes by the ray's signs.
__device__ __forceinline__ uint32_t wide_hits(const float4 n0, half8 qnx, half8 qny, half8 qnz, half8 qfx, half8 qfy,
                                              half8 qfz, f3 o, f3 inv, f3 eta, float lim) {
    const float dx = n0.w * inv.x, dy = n0.w * inv.y, dz = n0.w * inv.z;
    const float px = n0.x - o.x, py = n0.y - o.y, pz = n0.z - o.z;
    const float anx = px * inv.x - eta.x, afx = px * inv.x + eta.x;
    const float any_ = py * inv.y - eta.y, afy = py * inv.y + eta.y;
    const float anz = pz * inv.z - eta.z, afz = pz * inv.z + eta.z;
    uint32_t hits = 0;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        const float t0 = fmaxf(fmaxf(fmaxf((float)qnx[c] * dx + anx, (float)qny[c] * dy + any_),
                                     (float)qnz[c] * dz + anz), 0.f);
        const float t1 = fminf(fminf(fminf((float)qfx[c] * dx + afx, (float)qfy[c] * dy + afy),
                                     (float)qfz[c] * dz + afz), lim);
        hits |= t0 <= t1 ? 1u << c : 0u;
    }
    return hits;
}

// Slot order to octant order: bit s to bit s ^ oct.
__device__ __forceinline__ uint32_t octant_order(uint32_t ih, uint32_t oct) {
    ih = (oct & 1u) ? ((ih << 1) & 0xaau) | ((ih >> 1) & 0x55u) : ih;
    ih = (oct & 2u) ? ((ih << 2) & 0xccu) | ((ih >> 2) & 0x33u) : ih;
    return (oct & 4u) ? ((ih << 4) & 0xf0u) | (ih >> 4) : ih;
}

// Sign bits of a direction, and by how much the walk widens boxes for it: in
// proportion to the coordinates, as FP32's misplacement is, but for origins
// within XT_W_FAR extents of the scene at most. From 1e6 extents away the slack
// would be the whole scene, and each ray would meet every box; FP32 tells no
// triangles apart from there.
__device__ __forceinline__ uint32_t octant_of(f3 inv) {
    return (inv.x < 0.f ? 1u : 0u) | (inv.y < 0.f ? 2u : 0u) | (inv.z < 0.f ? 4u : 0u);
}
struct SlackBase {
    float scene, far;  // slack of the scene's coordinates; the largest coordinate of an origin that slack is given for
};
__device__ __forceinline__ SlackBase slack_base(const SceneView &S) {
    float m = 0.f, ext = 0.f;
    for (int k = 0; k < 3; ++k) {
        m = fmaxf(m, fmaxf(fabsf(S.kb_lo[k]), fabsf(S.kb_hi[k])));
        ext = fmaxf(ext, S.kb_hi[k] - S.kb_lo[k]);
    }
    return {XT_W_SLACK * m, m + XT_W_FAR * ext};
}
__device__ __forceinline__ f3 box_slack(f3 o, f3 inv, SlackBase b) {
    const float e = XT_W_SLACK * fminf(fmaxf(fabsf(o.x), fmaxf(fabsf(o.y), fabsf(o.z))), b.far) + b.scene;
    return mk(e * fabsf(inv.x), e * fabsf(inv.y), e * fabsf(inv.z));
}

// Whether a ray can meet a primitive: one of no direction, or with a NaN or an
// infinity, passes the tests of boxes and none of a primitive.
__device__ __forceinline__ bool can_hit(f3 o, f3 d, float dk) {
    return dk != 0.f && fabsf(o.x) + fabsf(o.y) + fabsf(o.z) + fabsf(d.x) + fabsf(d.y) + fabsf(d.z) < INFINITY;
}

// STACK: the deepest a walk's stack gets, which the tree's depth bounds. A
// stack entry is the rest of a group of siblings: the hits not yet visited in
// octant order (bits 0-7) and the node of slot 0 (bits 8-31).
template <int STACK, int BS>
static __global__ __launch_bounds__(BS) __attribute__((amdgpu_waves_per_eu(XT_W_WAVES))) void k_trace_bvh(
    const SceneView S, const Queue in, const uint32_t *in_count, float4 *hit, uint32_t *retest_list,
    uint4 *recheck_list, const TraceCtl T) {
    Counters *const cnt = T.cnt;
    __shared__ uint32_t wstk[STACK * BS];
    __shared__ uint4 wbuf[BS / 64][64 * 8];
    uint32_t *const stk = wstk + threadIdx.x;
    const uint32_t n = *in_count;
    trace_open(T, n);
    const uint32_t lane = lane_id();
    const uint32_t waves = gridDim.x * (BS / 64);
    const uint32_t wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t wave = blockIdx.x * (BS / 64) + wid;
    uint4 *const buf = wbuf[wid];
    const float4 *const recs = S.kd_indexed ? S.prims : S.bvh_leaf;
    RaySource R;
    source_init(R, n, waves, T);
    bool more = true;
    const SlackBase slack = slack_base(S);

    bool alive = false, done = false;
    uint32_t ri = 0, origin = XT_NONE, oct = 0, kz = 0;
    f3 o = mk(0, 0, 0), inv = mk(0, 0, 0), eta = mk(0, 0, 0);
    float sx = 0.f, sy = 0.f, sz = 0.f;
    Best best = {};
    uint32_t grp = 0;                         // current group: hits (bits 0-7, octant order), node of slot 0 (8-31)
    uint32_t tbase = 0, lhit = 0, lmask = 0;  // leaf children hit and not yet tested, the node's leaves
    uint32_t tk = 0, tn = 0, best_rec = 0;    // primitives of the leaf in hand; the closest one's record
    uint32_t sp = 0;
    uint32_t own = lane;        // the lane whose ray this one walks
    float shared_t = INFINITY;  // closest hit of the ray's other lanes, when last seen

    for (;;) {
        int nw = __popcll(__builtin_amdgcn_ballot_w64(alive));
        const bool low = nw == 0 || (more && 64 - nw >= XT_REFILL_IDLE);
        bool fin = done && low;
        if (!more) {
            // what helpers without work have found goes to their rays
            unsigned long long hm = __builtin_amdgcn_ballot_w64(done && own != lane);
            if (hm) {
                do {
                    const int h = __builtin_ctzll(hm);
                    hm &= hm - 1ull;
                    const uint32_t to = __builtin_amdgcn_readlane(own, h);
                    const float t = lane_value(best.t, h), mt = lane_value(best.mark_t, h);
                    const uint32_t prim = __builtin_amdgcn_readlane(best.prim, h);
                    const uint32_t rec = __builtin_amdgcn_readlane(best_rec, h);
                    const uint32_t c0 = __builtin_amdgcn_readlane(best.c0, h);
                    const uint32_t c1 = __builtin_amdgcn_readlane(best.c1, h);
                    if (lane == to) merge_best(best, best_rec, t, prim, rec, mt, c0, c1);
                } while (hm);
                if (own != lane) {
                    done = false;
                    own = alive ? own : lane;
                }
            }
            fin = done && nw == 0;
            // rays that no helper walks any more are finished, for their lanes to help
            if (nw != 0 && __popcll(__builtin_amdgcn_ballot_w64(done)) >= XT_W_FREE) {
                unsigned long long busy = __builtin_amdgcn_ballot_w64(alive && own != lane), kept = 0;
                while (busy) {
                    kept |= 1ull << __builtin_amdgcn_readlane(own, __builtin_ctzll(busy));
                    busy &= busy - 1ull;
                }
                fin = done && !((kept >> lane) & 1ull);
            }
        }
        if (__builtin_amdgcn_ballot_w64(fin)) {
            bool mark = false, full = false;
            if (fin)
                finish_ray(S, in, hit, cnt, ri, o, origin, true, best, recs, best_rec, mark, full);
            if (__builtin_amdgcn_ballot_w64(mark)) {
                const bool rf = mark && full, rc = mark && !full;
                const uint32_t slot = wave_append(rf, &cnt->n[CNT_RETEST + T.par]);
                if (rf) retest_list[slot] = ri;
                const uint32_t cslot = wave_append(rc, &cnt->n[CNT_RECHECK + T.par]);
                if (rc) recheck_list[cslot] = make_uint4(ri, best.c0, best.c1, XT_NONE);
            }
            done = done && !fin;
        }
        if (low) {
            while (more) {
                const bool idle = !alive && !done;
                const unsigned long long m = __builtin_amdgcn_ballot_w64(idle);
                if (m == 0) break;
                if (R.cur == R.end && !source_next(R, cnt, wave)) {
                    more = false;
                    break;
                }
                const uint32_t rank = rank_in(m);
                const uint32_t left = R.end - R.cur, free_lanes = (uint32_t)__popcll(m);
                if (idle && rank < left) {
                    const uint32_t i = source_ray(R, R.cur + rank);
                    const float4 a = in.r0[i];
                    if (__float_as_uint(a.w) == XT_DEAD) {
                        hit[i] = make_float4(INFINITY, __uint_as_float(XT_NONE), 0.f, 0.f);
                    } else {
                        const float4 b = in.r1[i];
                        RayF r;
                        r.o = mk(a.x, a.y, a.z);
                        r.d = mk(b.x, b.y, b.z);
                        r.origin = __float_as_uint(a.w);
                        r.self_t = b.w;
                        ri = i;
                        o = r.o;
                        origin = r.origin;
                        seed_best(r, best);
                        const float tsmall = tsmall_of(o);
                        for (uint32_t k = 0; k < S.n_planes; ++k)
                            if (XT_PLANE_BASE + k != origin)
                                plane32(r.o, r.d, tsmall, S.planes[k], XT_PLANE_BASE + k, best);
                        const float dk = ray_shear(r.d, kz, sx, sy, sz);
                        inv = mk(rcp_dir(r.d.x), rcp_dir(r.d.y), rcp_dir(r.d.z));
                        eta = box_slack(o, inv, slack);
                        oct = octant_of(inv);
                        // the root as the only hit of a group above it
                        grp = 1u << oct;
                        lhit = tn = 0;
                        sp = 0;
                        shared_t = INFINITY;
                        alive = can_hit(o, r.d, dk);
                        done = !alive;
                    }
                }
                R.cur += left < free_lanes ? left : free_lanes;
            }
            nw = __popcll(__builtin_amdgcn_ballot_w64(alive));
        }
        if (!more && nw != 0) {
            // no ray is left: idle lanes take over parts of the walking lanes' trees
            const bool idle = !alive && !done;
            const uint32_t bits = (uint32_t)__popc(grp & 0xffu);
            const bool can = alive && (bits >= 2u || sp != 0u || ((lhit | tn) != 0u && grp != 0u));
            const unsigned long long im = __builtin_amdgcn_ballot_w64(idle), dm = __builtin_amdgcn_ballot_w64(can);
            if (im && dm) {
                const uint32_t ni = (uint32_t)__popcll(im), nd = (uint32_t)__popcll(dm), pairs = ni < nd ? ni : nd;
                const uint32_t ri_ = rank_in(im), rd = rank_in(dm);
                const bool give = can && rd < pairs, take = idle && ri_ < pairs;
                uint32_t gift = 0;
                if (give) {
                    if (bits >= 2u) {  // the siblings after the next one
                        const uint32_t low = grp & (0u - grp);
                        gift = grp ^ low;
                        grp = (grp & ~0xffu) | low;
                    } else if (sp) {
                        sp -= BS;
                        gift = stk[sp];
                    } else {
                        gift = grp;
                        grp = 0;
                    }
                }
                // lane r of `giver` holds the lane of rank r among the givers (at most 32)
                const uint32_t giver = (uint32_t)__builtin_amdgcn_ds_permute((int)((give ? rd : 63u) << 2), (int)lane);
                const uint32_t from = from_lane(giver, take ? ri_ : 63u);
                const uint32_t src = take ? from : lane;
                gift = from_lane(gift, src);
                const uint32_t pk = from_lane(oct | kz << 3 | own << 5, src);
                ri = from_lane(ri, src);
                origin = from_lane(origin, src);
                o = mk(from_lane(o.x, src), from_lane(o.y, src), from_lane(o.z, src));
                inv = mk(from_lane(inv.x, src), from_lane(inv.y, src), from_lane(inv.z, src));
                eta = mk(from_lane(eta.x, src), from_lane(eta.y, src), from_lane(eta.z, src));
                sx = from_lane(sx, src);
                sy = from_lane(sy, src);
                sz = from_lane(sz, src);
                best.t = from_lane(best.t, src);
                best.prim = from_lane(best.prim, src);
                best_rec = from_lane(best_rec, src);
                if (take) {
                    oct = pk & 7u;
                    kz = (pk >> 3) & 3u;
                    own = pk >> 5;
                    best.mark_t = INFINITY;
                    best.c0 = best.c1 = XT_NONE;
                    grp = gift;
                    lhit = tn = sp = 0;
                    alive = true;
                }
            }
            if (__builtin_amdgcn_ballot_w64(alive && own != lane)) {
                // the closest hit of all lanes of a ray ends each one's walk
                int *const tm = (int *)buf;
                tm[lane] = __float_as_int(INFINITY);
                __builtin_amdgcn_wave_barrier();
                if (alive || done) atomicMin(tm + own, __float_as_int(best.t));
                __builtin_amdgcn_wave_barrier();
                shared_t = __int_as_float(tm[own]);
                asm volatile("" ::"v"(shared_t) : "memory");
            }
            nw = __popcll(__builtin_amdgcn_ballot_w64(alive));
        }
        if (nw == 0) {
            if (!more && !__builtin_amdgcn_ballot_w64(done)) break;
            continue;
        }
        const int keep = (nw * XT_W_KEEP) >> 4;

        // inner nodes
        bool node = alive && (lhit | tn) == 0u;
        // LDS offsets of the near planes; the far ones lie 48 bytes above or below
        const uint32_t offx = oct & 1u ? 80u : 32u, offy = oct & 2u ? 96u : 48u, offz = oct & 4u ? 112u : 64u;
        do {
            const unsigned long long m = __builtin_amdgcn_ballot_w64(node);
            const uint32_t rank = rank_in(m);
            uint32_t idx = 0;
            if (node) {
                const uint32_t bit = (uint32_t)__builtin_ctz(grp);
                grp &= grp - 1u;  // hits are the lowest bits
                idx = (grp >> 8) + (bit ^ oct);
            }
            gather_records<8, uint32_t>(S.bvh, idx, m, lane, rank, node, buf);
            if (node) {
                const char *nd = (const char *)(buf + 8u * rank);
                const uint32_t sw = (rank & 7u) * 16u;
                const float4 n0 = *(const float4 *)(nd + sw);
                const uint4 n1 = *(const uint4 *)(nd + (16u ^ sw));
                const half8 qnx = *(const half8 *)(nd + (offx ^ sw)), qfx = *(const half8 *)(nd + ((112u - offx) ^ sw));
                const half8 qny = *(const half8 *)(nd + (offy ^ sw)), qfy = *(const half8 *)(nd + ((144u - offy) ^ sw));
                const half8 qnz = *(const half8 *)(nd + (offz ^ sw)), qfz = *(const half8 *)(nd + ((176u - offz) ^ sw));
                const uint32_t hits = wide_hits(n0, qnx, qny, qnz, qfx, qfy, qfz, o, inv, eta,
                                                fminf(best.t, shared_t) * (1.f + 4e-6f));
                lmask = n1.z;
                lhit = hits & lmask & 0xffu;
                tbase = n1.y;
                const uint32_t ih = octant_order(hits & (lmask >> 24), oct);
                if (ih) {
                    if (grp & 0xffu) {
                        stk[sp] = grp;
                        sp += BS;
                    }
                    grp = ih | n1.x << 8;
                } else if (!(grp & 0xffu)) {
                    grp = 0;
                    if (sp) {
                        sp -= BS;
                        grp = stk[sp];
                    }
                }
                node = lhit == 0u && grp != 0u;
                done = lhit == 0u && grp == 0u;
                alive = !done;
            }
        } while (__popcll(__builtin_amdgcn_ballot_w64(node)) > keep);

        // primitives
        bool leaf = alive && (lhit | tn) != 0u;
        for (;;) {
            const unsigned long long m = __builtin_amdgcn_ballot_w64(leaf);
            if (__popcll(m) <= keep) break;
            const uint32_t rank = rank_in(m);
            uint32_t prim = 0;
            if (leaf) {
                if (tn == 0u) {
                    const uint32_t slot = (uint32_t)__builtin_ctz(lhit);
                    lhit &= lhit - 1u;
                    // primitives of the leaf slots below: one each, and what the count bits add
                    const uint32_t below = lmask & __umul24((1u << slot) - 1u, 0x010101u);
                    tk = tbase + (uint32_t)__popc(below) + (uint32_t)__popc(below >> 16);
                    const uint32_t cb = lmask >> slot;
                    tn = 1u + ((cb >> 8) & 1u) + ((cb >> 15) & 2u);
                }
                prim = tk;
                if (S.kd_indexed) prim = S.bvh_refs[tk];
                ++tk;
                --tn;
            }
            gather_records<3, uint64_t>(recs, prim, m, lane, rank, leaf, buf);
            const uint32_t this_rec = prim;
            if (leaf) {
                const float4 *rec = (const float4 *)(buf + 3u * rank);
                const float4 a = rec[0], b = rec[1], c = rec[2];
                if (!S.kd_indexed) prim = __float_as_uint(b.w);
                if (prim != origin) {
                    const uint32_t was = best.prim;
                    if (XT_PRIM_TYPE(__float_as_uint(a.w)) == XT_PRIM_TRIANGLE) {
                        tri32_flat<true>(o, sx, sy, sz, kz, a, b, c, prim, best, inv, eta);
                    } else {
                        const float4 b4 = in.r1[ri];
                        sph32(o, mk(b4.x, b4.y, b4.z), tsmall_of(o), a, b, prim, best);
                    }
                    best_rec = best.prim != was ? this_rec : best_rec;
                }
                leaf = (lhit | tn) != 0u;
                done = !leaf && grp == 0u;
                alive = !done;
            }
        }
    }
}
