// Parts of the FP32 closest-hit kernels that the kd-tree walk and the wide BVH
// walk share: where a wave takes its rays from, a walked ray's hit record, and
// the triangle test in one straight line.
#pragma once

#define XT_STRETCH_LOG 12   // log2 of the rays of a stretch
#define XT_RUN_MAX 512u     // rays of the longest run a wave takes at once
#define XT_REFILL_IDLE 24   // a wave takes new rays once this many lanes are idle

// Where a wave's rays come from. Wave w first takes 64 consecutive rays, or, when
// the grid's waves could take more than there are, its equal share of them: the
// rays of a wave wait for each other's phases, and its idle lanes help (256x256x4
// paths 715 us with 64 a wave, 660 with equal shares). The rays beyond 64 times
// the grid's waves are cut into stretches of 2^sh
// dealt to the XCDs in turn (nseg = 8: one stretch each), each XCD's stretches
// with a cursor in a line of its own. A wave takes runs from its own XCD's
// cursor, shorter ones as the end comes near, and then from the others'.
//
// Atomics on one address take about 11 ns each, one after the other: one
// cursor that every wave asks for every 64 rays is 12.4 ms of the 72 million
// queries of the 1080p icosphere frame, and was the pace of the whole trace
// (ray order, lane use and memory traffic changed nothing). Eight cursors and
// runs of up to 512 rays leave 0.1 ms; a queue that one run per wave covers
// needs no atomic at all (100,003 rays: 219 to 120 us).
struct RaySource {
    uint32_t n, first, base, sh, len, par, xcd;  // rays, first dealt ray, log2 of a stretch (or, sh = 32, its length)
    uint32_t waves;                  // per XCD
    uint32_t cur, end;               // the run in hand: rays (first run), or positions on the XCD's stretches
    uint32_t seen;                   // the XCD's cursor when last seen
    uint32_t state;                  // 0: before the first run, 1: in it, 2: dealt runs
};

__device__ __forceinline__ void source_init(RaySource &R, uint32_t n, uint32_t waves, const TraceCtl &T) {
    const uint32_t nseg = T.nseg;
    R.n = n;
    R.par = T.par;
    R.first = waves * 64u < n ? 64u : (n + waves - 1u) / waves;
    R.base = waves * R.first < n ? waves * R.first : n;
    R.sh = nseg == 1u ? (uint32_t)XT_STRETCH_LOG : 32u;
    R.len = nseg == 1u ? 1u << XT_STRETCH_LOG : ((n - R.base) / 8u + 64u) & ~63u;
    R.xcd = __builtin_amdgcn_s_getreg(20 | 3 << 11) & 7u;  // XCC_ID
    R.waves = (waves + 7u) / 8u;
    R.cur = R.end = R.seen = R.state = 0;
}

// Rays on XCD x's stretches.
__device__ __forceinline__ uint32_t source_count(const RaySource &R, uint32_t x) {
    const uint32_t m = R.n - R.base, round = 8u * R.len;
    const uint32_t full = R.sh < 32u ? m >> (R.sh + 3u) : m / round;
    const uint32_t rest = m - full * round, before = x * R.len;
    const uint32_t more = rest > before ? (rest - before < R.len ? rest - before : R.len) : 0u;
    return full * R.len + more;
}

__device__ __forceinline__ uint32_t source_ray(const RaySource &R, uint32_t at) {
    if (R.state == 1u) return at;
    const uint32_t s = R.sh < 32u ? at >> R.sh : 0u;
    return R.base + (s * 8u + R.xcd) * R.len + (at - s * R.len);
}

// The next run for this wave into [cur, end); false when no ray is left.
__device__ __forceinline__ bool source_next(RaySource &R, Counters *cnt, uint32_t wave) {
    if (R.state == 0u) {
        R.state = 1u;
        R.cur = wave * R.first < R.n ? wave * R.first : R.n;
        R.end = R.n - R.cur < R.first ? R.n : R.cur + R.first;
        if (R.cur < R.end) return true;
    }
    R.state = 2u;
    if (R.base == R.n) return false;
    const uint32_t lane = lane_id();
    for (int tries = 0; tries < 16; ++tries) {
        const uint32_t total = source_count(R, R.xcd);
        if (R.seen < total) {
            uint32_t want = (total - R.seen) / (2u * R.waves) & ~63u;
            want = want < 64u ? 64u : (want > XT_RUN_MAX ? XT_RUN_MAX : want);
            uint32_t c = 0;
            if (lane == 0) c = atomicAdd(&cnt->cursor[R.par][R.xcd * XT_CURSOR_STRIDE], want);
            c = __builtin_amdgcn_readfirstlane(c);
            R.seen = c + want;
            if (c < total) {
                R.cur = c;
                R.end = total - c < want ? total : c + want;
                return true;
            }
        }
        // this XCD's stretches are dealt: go on with the next one that has rays left
        bool left = false;
        uint32_t at = 0;
        const uint32_t x = (R.xcd + 1u + lane) & 7u;
        if (lane < 8u) {
            at = __hip_atomic_load(&cnt->cursor[R.par][x * XT_CURSOR_STRIDE], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            left = at < source_count(R, x);
        }
        const unsigned long long m = __builtin_amdgcn_ballot_w64(left);
        if (m == 0) return false;
        const int k = __builtin_ctzll(m);
        R.seen = __builtin_amdgcn_readlane(at, k);
        R.xcd = (R.xcd + 1u + (uint32_t)k) & 7u;
    }
    return false;
}

__device__ __forceinline__ uint32_t rank_in(unsigned long long m) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// Writes a walked ray's hit: the closest triangle's t and barycentrics in
// FP64, or the FP32 record of a ray whose deferred candidates the FP64
// kernel decides: `mark` lists it, `full` for the whole re-test.
// recs[3 rec ..] is the closest primitive's record, if it is a primitive.
__device__ __forceinline__ void finish_ray(const SceneView &S, const Queue &in, float4 *hit, Counters *cnt,
                                           uint32_t ri, f3 o, uint32_t origin, bool ok, const Best &best,
                                           const float4 *recs, uint32_t rec, bool &mark, bool &full) {
    const float4 b4 = in.r1[ri];
    const f3 d = mk(b4.x, b4.y, b4.z);
    if (!ok) atomicAdd(&cnt->trace_fail, 1ull);
    // a deferred candidate matters only up to the closest hit (a miss
    // has t = INF, so compare only when something was deferred)
    mark = !ok || (best.mark_t != INFINITY && best.mark_t <= best.t * (1.f + XT_TIE));
    full = !ok || best.c1 == XT_CAND_OVERFLOW;
    float ht = best.t, hu = 0.f, hv = 0.f;
    if (!mark && best.prim < S.n_prims && !(b4.w > 0.f && best.prim == origin)) {
        const float4 *q = recs + 3 * (size_t)rec;
        const float4 a = q[0];
        // the closest triangle's t and barycentrics in FP64
        if (XT_PRIM_TYPE(__float_as_uint(a.w)) == XT_PRIM_TRIANGLE) tri_hit64(o, d, a, q[1], q[2], ht, hu, hv);
    }
    hit[ri] = make_float4(ht, __uint_as_float(best.prim), hu, hv);
}

// 1 / x within 1 ulp, +-1e30 near 0. It places boxes and planes alone: an ulp is
// a sixteenth of the boxes' slack (XT_W_SLACK) and of the kd walk's widening
// (XT_KD_EPS), and moves no hit.
__device__ __forceinline__ float rcp_dir(float x) {
    return fabsf(x) > 1e-30f ? __builtin_amdgcn_rcpf(x) : copysignf(1e30f, x);
}

// make_shear with the largest axis alone: axes kz + 1 and kz + 2 follow it
// (their swap for a negative d[kz] would only negate U, V, W and their sum).
// Returns d[kz], 0 for a ray of no direction, which meets no primitive.
__device__ __forceinline__ float ray_shear(f3 d, uint32_t &kz, float &sx, float &sy, float &sz) {
    const float ax = fabsf(d.x), ay = fabsf(d.y), az = fabsf(d.z);
    kz = ax > ay ? (ax > az ? 0u : 2u) : (ay > az ? 1u : 2u);
    const float dk = kz == 0u ? d.x : (kz == 1u ? d.y : d.z);
    sz = 1.f / dk;
    sx = (kz == 0u ? d.y : (kz == 1u ? d.z : d.x)) * sz;
    sy = (kz == 0u ? d.z : (kz == 1u ? d.x : d.y)) * sz;
    return dk;
}

// Where the ray enters the triangle's box, widened by half of eta; INFINITY
// when it passes it by.
__device__ __forceinline__ float tri_box_entry(f3 A, f3 B, f3 C, f3 inv, f3 eta) {
    float t0 = 0.f, t1 = INFINITY;
    const float v[3][3] = {{A.x, B.x, C.x}, {A.y, B.y, C.y}, {A.z, B.z, C.z}};
    const float iv[3] = {inv.x, inv.y, inv.z}, e[3] = {eta.x, eta.y, eta.z};
    for (int k = 0; k < 3; ++k) {
        const float p = fminf(v[k][0], fminf(v[k][1], v[k][2])) * iv[k];
        const float q = fmaxf(v[k][0], fmaxf(v[k][1], v[k][2])) * iv[k];
        t0 = fmaxf(t0, fminf(p, q) - 0.5f * e[k]);
        t1 = fminf(t1, fmaxf(p, q) + 0.5f * e[k]);
    }
    return t0 <= t1 ? t0 : INFINITY;
}

// tri32 and offer() in one straight line: the tests' rare outcomes (a
// deferral) share one branch. The same values, rounded alike, and the same
// decisions; but with BOX a grazed triangle is deferred from where the ray
// enters its box (rinv, eta: the ray's reciprocal direction and the slack of the
// walk's boxes) and not from the ray's origin: a walk that visits the tree in
// another order, and so tests other triangles behind the closest hit, decides
// alike which rays are re-checked.
template <bool BOX>
__device__ __forceinline__ void tri32_flat(const f3 o, float sx, float sy, float sz, uint32_t kz, const float4 a,
                                           const float4 b, const float4 c, uint32_t prim, Best &best, f3 rinv,
                                           f3 eta) {
    const uint32_t tf = __float_as_uint(a.w);
    const float tsmall = tsmall_of(o);
    const f3 A = sub(mk(a.x, a.y, a.z), o), B = sub(mk(b.x, b.y, b.z), o), C = sub(mk(c.x, c.y, c.z), o);
    const bool k0 = kz == 0u, k1 = kz == 1u;
    const float az = k0 ? A.x : (k1 ? A.y : A.z), bz = k0 ? B.x : (k1 ? B.y : B.z), cz = k0 ? C.x : (k1 ? C.y : C.z);
    const float ax = (k0 ? A.y : (k1 ? A.z : A.x)) - sx * az, ay = (k0 ? A.z : (k1 ? A.x : A.y)) - sy * az;
    const float bx = (k0 ? B.y : (k1 ? B.z : B.x)) - sx * bz, by = (k0 ? B.z : (k1 ? B.x : B.y)) - sy * bz;
    const float cx = (k0 ? C.y : (k1 ? C.z : C.x)) - sx * cz, cy = (k0 ? C.z : (k1 ? C.x : C.y)) - sy * cz;
    const float U = edge2(cx, by, cy, bx), V = edge2(ax, cy, ay, cx), W = edge2(bx, ay, by, ax);
    const float det = U + V + W;
    const float inv = 1.f / det;
    const float t = (U * az + V * bz + W * cz) * sz * inv;
    const float m = fminf(fminf(V * inv, W * inv), U * inv);
    const bool live = !(XT_PRIM_FLAGS(tf) & XT_PF_DEGENERATE);
    const bool graze = fabsf(det) * c.w < XT_GRAZE * fabsf(sz);
    const bool in_t = !(t < -tsmall || t > best.t * (1.f + XT_TIE)) && live && !graze;
    const bool in = in_t && !(m < 0.f);
    const bool near0 = t < tsmall;
    const bool cand = in && !near0 && prim != best.prim;
    const bool closer = t < best.t;
    const bool tie = fabsf(best.t - t) <= XT_TIE * fminf(t, best.t);
    const bool rare = (live && graze) || (in_t && m > -XT_BAND && m < XT_BAND) || (in && near0) || (cand && tie);
    const float old_t = best.t;
    const uint32_t old_prim = best.prim;
    if (cand && closer) {
        best.t = t;
        best.prim = prim;
    }
    if (rare) {
        if (graze) {
            const float at = BOX ? tri_box_entry(A, B, C, rinv, eta) : 0.f;
            if (at < INFINITY) defer(best, at, prim);
        } else {
            if (m > -XT_BAND && m < XT_BAND) defer(best, t, prim);
            if (in && near0) defer(best, fmaxf(t, 0.f), prim);
            if (cand && tie) defer(best, closer ? t : old_t, closer ? old_prim : prim);
        }
    }
}

