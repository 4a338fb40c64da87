// The FP32 closest-hit kernel over the kd-tree: persistent waves whose lanes
// walk on their own. Each turn of the main loop descends until few lanes are
// left above a leaf, tests leaf primitives until few have any, and pops; lanes
// whose ray is finished wait, and once XT_REFILL_IDLE of a wave's lanes do,
// their hits are written and they get new rays. With whole groups of 64 rays
// a wave ran as long as its longest ray: 10 of 64 lanes were active in the mean
// instruction (1080p icosphere frame, rocprofv3), 26 with the refill. The
// turn's phases end at 3 sixteenths of the working lanes (strands frame at 2: the
// same, at 4: 4% slower). What bounds a queue of about as many
// rays as the card has lanes is each ray's chain of dependent loads, 27 records
// of it on the strands: those of a leaf are loaded one ahead (50,000 strands,
// 512x512x4 paths 6.70 to 6.05 ms, 1024x1024x8 20.0 to 18.4, 2 M random rays
// 2.30 to 2.18; with whole groups of 64 rays and the same loads 6.2, 24.7, 3.0).
#pragma once
#include "xt_walk.h"

#define XT_KD_KEEP 3      // sixteenths of the working lanes at which a phase ends
#define XT_KD_WAVES 5     // waves per SIMD (strands frame at 4: 3% slower, at 6: 10%, for spills)
#define XT_KD_EPS 2e-6f   // relative widening of the walk's intervals

// kd-tree walk with a ring of the STACK newest far children per lane in LDS
// (one entry more: each step writes the far child behind the newest entry and
// keeps it only when both children are visited) and a restart from the root
// when older ones were overwritten. tmin and tmax are kept widened.
template <int STACK, int BS>
static __global__ __launch_bounds__(BS) __attribute__((amdgpu_waves_per_eu(XT_KD_WAVES))) void k_trace_kd(
    const SceneView S, const Queue in, const uint32_t *in_count, float4 *hit, uint32_t *retest_list,
    uint4 *recheck_list, const TraceCtl T) {
    Counters *const cnt = T.cnt;
    constexpr uint32_t SLOTS = STACK + 1;
    __shared__ uint2 kstk[SLOTS * BS];
    uint2 *const stk = kstk + threadIdx.x;
    const uint32_t n = *in_count;
    trace_open(T, n);
    const uint32_t waves = gridDim.x * (BS / 64);
    const uint32_t wave = __builtin_amdgcn_readfirstlane(blockIdx.x * (BS / 64) + (threadIdx.x >> 6));
    RaySource R;
    source_init(R, n, waves, T);
    bool more = true;

    const XtKdNode root = S.kd[0];
    const float4 *const recs = S.kd_indexed ? S.prims : S.kd_leaf;
    bool alive = false, done = false, ok = true;
    uint32_t ri = 0, origin = XT_NONE;
    f3 o = mk(0, 0, 0), inv = mk(0, 0, 0);
    float sx = 0.f, sy = 0.f, sz = 0.f;
    uint32_t kz = 0;
    Best best = {};
    uint32_t word = 3u, payload = 0u;
    float tmin = 0.f, tmax = 0.f;
    uint32_t off = 0;
    int count = 0, lost = 0;
    uint32_t steps = 0;

    for (;;) {
        int nw = __popcll(__builtin_amdgcn_ballot_w64(alive));
        if (nw == 0 || (more && 64 - nw >= XT_REFILL_IDLE)) {
            if (__builtin_amdgcn_ballot_w64(done)) {
                bool mark = false, full = false;
                if (done) finish_ray(S, in, hit, cnt, ri, o, origin, ok, best, S.prims, best.prim, mark, full);
                const bool rf = mark && full, rc = mark && !full;
                if (__builtin_amdgcn_ballot_w64(mark)) {
                    const uint32_t slot = wave_append(rf, &cnt->n[CNT_RETEST + T.par]);
                    if (rf) retest_list[slot] = ri;
                    const uint32_t cslot = wave_append(rc, &cnt->n[CNT_RECHECK + T.par]);
                    if (rc) recheck_list[cslot] = make_uint4(ri, best.c0, best.c1, XT_NONE);
                }
                done = false;
            }
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
                        const float dk = ray_shear(r.d, kz, sx, sy, sz);
                        inv = mk(rcp_dir(r.d.x), rcp_dir(r.d.y), rcp_dir(r.d.z));
                        seed_best(r, best);
                        const float tsmall = tsmall_of(o);
                        for (uint32_t k = 0; k < S.n_planes; ++k)
                            if (XT_PLANE_BASE + k != origin)
                                plane32(r.o, r.d, tsmall, S.planes[k], XT_PLANE_BASE + k, best);
                        ok = true;
                        steps = 0;
                        tmin = 0.f;
                        tmax = best.t;
                        alive = dk != 0.f && slab(o, inv, S.kb_lo, S.kb_hi, tmin, tmax, 1e-6f);
                        done = !alive;
                        tmax *= 1.f + XT_KD_EPS;
                        word = root.word;
                        payload = root.count;
                        off = 0;
                        count = lost = 0;
                    }
                }
                R.cur += left < free_lanes ? left : free_lanes;
            }
            nw = __popcll(__builtin_amdgcn_ballot_w64(alive));
            if (nw == 0) {
                if (!more && !__builtin_amdgcn_ballot_w64(done)) break;
                continue;
            }
        }

        // descent
        const int keep = (nw * XT_KD_KEEP) >> 4;
        bool node = alive && (word & 3u) != 3u;
        do {
            if (node) {
                const uint32_t c = word >> 2, axis = word & 3u;
                const uint4 pair = *(const uint4 *)(S.kd + c);
                const float split = __uint_as_float(payload);
                const float oo = axis == 0 ? o.x : (axis == 1 ? o.y : o.z);
                const float ii = axis == 0 ? inv.x : (axis == 1 ? inv.y : inv.z);
                const float tp = (split - oo) * ii;
                const bool neg = ii < 0.f;
                const bool only_near = tp > tmax, only_far = tp < tmin;
                const bool both = !(only_near || only_far);
                const uint32_t next = off == STACK * BS ? 0u : off + BS;
                stk[next] = make_uint2(c | (neg ? 0u : 1u), __float_as_uint(tmax));
                off = both ? next : off;
                count += both ? 1 : 0;
                lost = max(lost, count - STACK);
                tmax = both ? fminf(tmax, tp * (1.f + XT_KD_EPS)) : tmax;
                const bool upper = neg != only_far;
                word = upper ? pair.z : pair.x;
                payload = upper ? pair.w : pair.y;
                node = (word & 3u) != 3u;
            }
        } while (__popcll(__builtin_amdgcn_ballot_w64(node)) > keep);

        // the node a pop resumes with, loaded while the leaf is tested
        XtKdNode pre = root;
        if (alive && !node && count != lost) pre = S.kd[stk[off].x];

        // leaf primitives, each record loaded while the one before it is
        // tested (the empty asm ends the wait for a record before its test)
        bool leaf = alive && !node && payload != 0u;
        float4 na = {}, nb = {}, nc = {};
        uint32_t nrec = 0;
        if (leaf) {
            nrec = S.kd_indexed ? S.kd_refs[word >> 2] : word >> 2;
            const float4 *rec = recs + 3 * (size_t)nrec;
            na = rec[0];
            nb = rec[1];
            nc = rec[2];
        }
        while (__popcll(__builtin_amdgcn_ballot_w64(leaf)) > keep) {
            if (leaf) {
                const float4 a = na, b = nb, c = nc;
                const uint32_t prim = S.kd_indexed ? nrec : __float_as_uint(b.w);
                word += 4u;
                --payload;
                leaf = payload != 0u;
                if (leaf) {
                    nrec = S.kd_indexed ? S.kd_refs[word >> 2] : word >> 2;
                    const float4 *rec = recs + 3 * (size_t)nrec;
                    na = rec[0];
                    nb = rec[1];
                    nc = rec[2];
                }
                asm volatile("" ::"v"(c.x), "v"(c.y), "v"(c.z), "v"(c.w));
                if (prim != origin) {
                    if (XT_PRIM_TYPE(__float_as_uint(a.w)) == XT_PRIM_TRIANGLE) {
                        tri32_flat<false>(o, sx, sy, sz, kz, a, b, c, prim, best, inv, inv);
                    } else {
                        const float4 b4 = in.r1[ri];
                        sph32(o, mk(b4.x, b4.y, b4.z), tsmall_of(o), a, b, prim, best);
                    }
                }
            }
        }

        // pop
        if (alive && !node && payload == 0u) {
            ++steps;
            const float lim = best.t;
            if (lim <= tmax * (1.f - XT_KD_EPS)) {
                done = true;
            } else if (steps >= XT_MAX_STEPS) {
                done = true;
                ok = false;
            } else if (count == lost) {
                float r0 = 0.f, r1 = lim;
                if (lost == 0 || !slab(o, inv, S.kb_lo, S.kb_hi, r0, r1, 1e-6f) || tmax >= r1 * (1.f + XT_KD_EPS)) {
                    done = true;
                } else {
                    // entries were lost: restart from the root beyond the processed range
                    tmin = tmax * (1.f - 2.f * XT_KD_EPS);
                    tmax = r1 * (1.f + XT_KD_EPS);
                    word = root.word;
                    payload = root.count;
                    count = lost = 0;
                }
            } else {
                const float far_t = __uint_as_float(stk[off].y);
                off = off == 0u ? (uint32_t)(STACK * BS) : off - BS;
                --count;
                word = pre.word;
                payload = pre.count;
                tmin = tmax * (1.f - 2.f * XT_KD_EPS);
                tmax = fminf(far_t, lim * (1.f + XT_KD_EPS));
                // the popped range starts beyond the closest hit, and so do all
                // deeper (farther) entries
                done = tmin > tmax;
            }
            alive = !done;
        }
    }
}
