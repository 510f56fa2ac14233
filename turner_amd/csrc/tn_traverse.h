// tn_traverse.h -- device kd-tree traversal for gfx950 (wave64).
//
// The traversal restates KDTreeIntersection::intersect (lib/kdtree.cpp:515-607)
// for one ray per lane:
//   * zero direction components become 1e-5 for traversal only (:503-511);
//   * root slab test without a t >= 0 clamp (lib/intersection.h:105-128);
//   * near child = left iff d[axis] > 0, the three-way texit<t / t<tenter /
//     both decision of :540-564;
//   * leaves are tested with the unmodified ray, closest hit with strict <,
//     so the first of equal hits in visit order wins (:566-607).
// All of it is FP32 with the reference's operation order, IEEE division and
// no FMA contraction (the library is compiled with -ffp-contract=off), so
// hit ids and r/s/t are bit-identical to the reference's.
//
// GPU-specific machinery:
//   * nodes are 8 bytes (see DevNode in tn_host.h); a leaf holds an offset
//     and count into a 32-bit triangle-reference array.  The cooperative
//     traversal reads the same tree as 32-byte treelets of two levels;
//   * triangle records are 64 bytes (4 x float4: v0|uv, n|vv, u|uu, v|denom),
//     one L2 line per triangle for the per-lane gathers;
//   * the stack is a circular short stack of S entries in LDS, 8 bytes per
//     entry (node, texit): the entry's tenter is always the exit of the last
//     leaf processed, so it is not stored.  When entries are lost to
//     overflow, the traversal restarts from the root at the last leaf's exit
//     (kd-restart), which visits the remaining leaves in the same order;
//   * near-first early exit: traversal ends once the best hit lies before the
//     current leaf's exit by a 2^-16 relative margin (no later leaf can then
//     hold a strictly closer hit).  TN_ISECT_EXHAUSTIVE disables it;
//   * the traversal is a per-lane state machine (trav_init / trav_tick: a
//     few node steps or one triangle test per tick) so lanes in different
//     phases share a wave's instructions and a wave can hand finished lanes
//     new rays.
#pragma once

#include <hip/hip_runtime.h>

#include <cfloat>
#include <cstdint>

namespace tn {

constexpr uint32_t kInvalidId = 1u << 30;
// Hit record of a ray a traversal of a refined tree leaves to the reference
// tree (not a triangle id: ids are below 2^30).
constexpr uint32_t kFixId = 0xFFFFFFFFu;
constexpr float kDirEps = 0.00001f;  // lib/types.h:14
constexpr float kExitMargin = 1.0f + 1.0f / 65536.0f;
constexpr int kMaxRestarts = 4096;
// Leaves one ray may visit before its traversal is abandoned as incomplete
// (far above any real ray; bounds every traversal loop).
constexpr uint32_t kMaxLeafVisits = 1u << 22;

// Root of one tree in a packed forest (many scenes in one node / reference /
// triangle allocation): its first treelet and root box.
struct SceneRoot {
    float bmin[3];
    float bmax[3];
    uint32_t treelet;
};

struct SceneView {
    const uint2* nodes;  // of a single tree, for the per-lane kernels (else null)
    const uint4* treelets;  // the same tree two levels at a time (Treelet of tn_host.h, 2 uint4 each)
    const uint32_t* refs;
    const float4* tris;  // 4 per triangle
    // The same records once per triangle reference, in reference order, as
    // two arrays of halves: lra[2r..2r+1] = (v0, uv) (n, vv) and
    // lrb[2r..2r+1] = (u, uu) (v, denom) of triangle refs[r].  The pairs of a
    // leaf are then contiguous and need no reference lookup.
    const float4* lra;
    const float4* lrb;
    float bmin[3];
    float bmax[3];
    const SceneRoot* roots = nullptr;  // forest: per-scene roots (bmin/bmax unused)
};

struct TraversalCounters {
    uint32_t inner = 0, leaves = 0, refs = 0, tests = 0, restarts = 0;
    uint32_t full = 0;  // tests that read the whole 64-byte record
    bool incomplete = false;
};

struct Trav {
    float3 o, d, dinv;
    float tenter, texit, root_exit;
    uint32_t node;
    uint32_t leaf_off, leaf_left;  // triangle references still to test in the current leaf
    int head, count, restarts;
    uint32_t visits;  // leaves visited
    bool lost;
    uint32_t best_id;
    float best_r, best_s, best_t;
};

__device__ __forceinline__ float pick(float3 v, uint32_t ax) {
    return ax == 0 ? v.x : (ax == 1 ? v.y : v.z);
}

// True when num / den is certainly < 0: opposite signs and a quotient that
// cannot underflow to -0 (|num / den| >= 2^-100).  Lets a test reject
// without the division while giving exactly the division's verdict.
__device__ __forceinline__ bool certainly_negative(float num, float den) {
    return ((num < 0.f) != (den < 0.f)) && num != 0.f &&
           fabsf(num) >= fabsf(den) * 0x1p-100f;
}

// lib/intersection.h:40-49 + 63-89: plane, then barycentrics; no culling.
// A candidate is also rejected when r is not below `bound` (closest hit: the
// current best, which it must beat strictly) or, with ANY, above it.
// Returns 2 on a hit, 1 for a miss decided after reading the whole record,
// 0 for a miss decided from its first 32 bytes.  pa: the record's first half
// (v0, uv) (n, vv); pc: its second half (u, uu) (v, denom).
template <bool ANY>
__device__ __forceinline__ int leaf_test_ref(const float4* __restrict__ pa, const float4* __restrict__ pc,
                                             float3 o, float3 d, float bound, float& r, float& s, float& t) {
    const float4 a = pa[0];  // v0, uv
    const float4 b = pa[1];  // n, vv
    const float den = b.x * d.x + b.y * d.y + b.z * d.z;
    if (den == 0.f) return 0;  // r = lowest() < 0
    const float nom = b.x * (a.x - o.x) + b.y * (a.y - o.y) + b.z * (a.z - o.z);
    if (certainly_negative(nom, den)) return 0;
    if (!ANY) {
        // r = nom / den certainly >= bound (it cannot beat the current best):
        // compare against bound * den widened by 2^-20, far beyond the
        // rounding of the division and of the product.
        const float q = bound * den * (1.0f + 0x1p-20f);
        if (fabsf(q) >= 0x1p-100f && (den > 0.f ? nom >= q : nom <= q)) return 0;
    }
    const float rr = nom / den;
    if (rr < 0) return 0;
    if (ANY ? !(rr <= bound) : !(rr < bound)) return 0;
    const float4 c = pc[0];  // u, uu
    const float4 e = pc[1];  // v, denom
    const float px = o.x + rr * d.x, py = o.y + rr * d.y, pz = o.z + rr * d.z;
    const float wx = px - a.x, wy = py - a.y, wz = pz - a.z;
    const float wv = wx * e.x + wy * e.y + wz * e.z;
    const float wu = wx * c.x + wy * c.y + wz * c.z;
    const float snum = a.w * wv - b.w * wu;
    const float tnum = a.w * wu - c.w * wv;
    // The reference rejects on s < 0, t < 0 or 1 < s + t; the verdict does
    // not depend on the order of the checks, so decide what the numerators
    // decide before dividing: a negative quotient, or s + t above 1 by a
    // 2^-18 margin (s and t then have the sign of the denominator, so the
    // sum of the numerators carries only rounding error).
    if (certainly_negative(snum, e.w) || certainly_negative(tnum, e.w)) return 1;
    {
        const float sum = snum + tnum;
        const float q = e.w * (1.0f + 0x1p-18f);
        if (fabsf(q) >= 0x1p-100f && (e.w < 0.f ? sum < q : sum > q)) return 1;
    }
    const float ss = snum / e.w;
    if (ss < 0) return 1;
    const float tt = tnum / e.w;
    if (tt < 0 || 1 < ss + tt) return 1;
    r = rr;
    s = ss;
    t = tt;
    return 2;
}

// The same test for the cooperative traversal, where a wave runs every stage
// of it for whichever lanes are left, so a stage costs the same for one lane as
// for 64.  It makes no rejection before the plane's division (some lane always
// needs it) and hands out the numerators of s and t instead of the quotients:
// s = snum / denom and t = tnum / denom are needed for the final hit of a ray
// only.  The reference's verdict (s < 0, t < 0 or 1 < s + t reject) follows
// from the numerators when a quotient is certainly negative (it cannot
// underflow to -0) or the sum is above or below 1 by a 2^-18 margin, far beyond
// the rounding of the divisions and of the sum; the divisions decide the rest.
// (146 -> 100 VALU instructions per 64 pairs.)  With TIE (closest hit) returns
// 3 for a hit at exactly r == bound, which does not replace the best.
template <bool ANY, bool TIE>
__device__ __forceinline__ int pair_test_ref(const float4* __restrict__ pa, const float4* __restrict__ pc,
                                             float3 o, float3 d, float bound, bool whole, float& r, float& snum,
                                             float& tnum) {
    const float4 a = pa[0];  // v0, uv
    const float4 b = pa[1];  // n, vv
    typedef float v4 __attribute__((ext_vector_type(4)));
    const v4* second = reinterpret_cast<const v4*>(pc);
    v4 c = {}, e = {};
    if (whole) {
        c = second[0];
        e = second[1];
        asm volatile("" : "+v"(c), "+v"(e));  // read here, not where they are used
    }
    const float den = b.x * d.x + b.y * d.y + b.z * d.z;
    const float nom = b.x * (a.x - o.x) + b.y * (a.y - o.y) + b.z * (a.z - o.z);
    const float rr = nom / den;
    float uv = a.w, vv = b.w;
    asm volatile("" : "+v"(uv), "+v"(vv));  // read with the rest of their 16 bytes, not again below
    // a ray along the plane (den 0) has no hit: the quotient is infinite or NaN
    if (!(rr >= 0.f) || ((ANY || TIE) ? !(rr <= bound) : !(rr < bound)) || (ANY && den == 0.f)) return 0;
    if (!whole) {
        c = second[0];  // u, uu
        e = second[1];  // v, denom
    }
    const float px = o.x + rr * d.x, py = o.y + rr * d.y, pz = o.z + rr * d.z;
    const float wx = px - a.x, wy = py - a.y, wz = pz - a.z;
    const float wv = wx * e.x + wy * e.y + wz * e.z;
    const float wu = wx * c.x + wy * c.y + wz * c.z;
    snum = uv * wv - vv * wu;
    tnum = uv * wu - c.w * wv;
    const uint32_t sign = __float_as_uint(e.w) & 0x80000000u;
    const float s1 = __uint_as_float(__float_as_uint(snum) ^ sign), t1 = __uint_as_float(__float_as_uint(tnum) ^ sign);
    const float size = fabsf(e.w), sum = s1 + t1, tiny = size * -0x1p-100f;
    // NaN operands fail every comparison here and go on to the divisions
    const float one = size >= 0x1p-99f ? size : __builtin_nanf("");
    if (s1 < tiny || t1 < tiny || sum > one * (1.0f + 0x1p-18f)) return 1;
    if (!(s1 >= 0.f && t1 >= 0.f && sum < one * (1.0f - 0x1p-18f))) {
        const float ss = snum / e.w;
        if (ss < 0) return 1;
        const float tt = tnum / e.w;
        if (tt < 0 || 1 < ss + tt) return 1;
    }
    r = rr;
    return (TIE && !ANY && rr == bound) ? 3 : 2;
}

// Moeller & Trumbore 1997 in FP32 on the record's v0, e1 = u, e2 = v.
// Returns 2 on a hit, 1 on a miss (the test always reads v0, u and v).
template <bool ANY>
__device__ __forceinline__ int leaf_test_mt(const float4* __restrict__ pa, const float4* __restrict__ pc,
                                            float3 o, float3 d, float bound, float& r, float& s, float& t) {
    const float4 a = pa[0];
    const float4 c = pc[0];
    const float4 e = pc[1];
    const float px = d.y * e.z - d.z * e.y, py = d.z * e.x - d.x * e.z, pz = d.x * e.y - d.y * e.x;
    const float det = c.x * px + c.y * py + c.z * pz;
    if (det == 0.f) return 1;
    const float inv = 1.0f / det;
    const float tx = o.x - a.x, ty = o.y - a.y, tz = o.z - a.z;
    const float u = (tx * px + ty * py + tz * pz) * inv;
    if (u < 0.f || u > 1.f) return 1;
    const float qx = ty * c.z - tz * c.y, qy = tz * c.x - tx * c.z, qz = tx * c.y - ty * c.x;
    const float v = (d.x * qx + d.y * qy + d.z * qz) * inv;
    if (v < 0.f || u + v > 1.f) return 1;
    const float tt = (e.x * qx + e.y * qy + e.z * qz) * inv;
    if (tt < 0.f) return 1;
    if (ANY ? !(tt <= bound) : !(tt < bound)) return 1;
    r = tt;
    s = u;
    t = v;
    return 2;
}

// A direction with a zero component is traversed as if that component were
// 1e-5 (kdtree.cpp:503-511): the traversal path then bends away from the ray
// itself, and only the reference tree's own leaves reproduce the reference's
// result for it.
__device__ __forceinline__ bool needs_reference(float3 d) { return d.x == 0.f || d.y == 0.f || d.z == 0.f; }

// Fixes the direction and clips the ray to the root box (kdtree.cpp:519-535)
// of its scene (the tree of `scene` in a forest): the reciprocal direction and
// the parameters [tlo, thi] inside the box.  Returns false when the root box
// is missed.
__device__ __forceinline__ bool root_clip(const SceneView& sc, float3 o, float3 d, uint32_t scene, float3& dinv,
                                          float& tlo, float& thi) {
    float3 fd = d;
    if (fd.x == 0.f) fd.x = kDirEps;
    if (fd.y == 0.f) fd.y = kDirEps;
    if (fd.z == 0.f) fd.z = kDirEps;
    dinv = make_float3(1 / fd.x, 1 / fd.y, 1 / fd.z);
    const float3 di = dinv;
    float b0[3], b1[3];
    if (sc.roots) {
        const SceneRoot& R = sc.roots[scene];
        for (int k = 0; k < 3; ++k) {
            b0[k] = R.bmin[k];
            b1[k] = R.bmax[k];
        }
    } else {
        for (int k = 0; k < 3; ++k) {
            b0[k] = sc.bmin[k];
            b1[k] = sc.bmax[k];
        }
    }
    const float tx1 = (b0[0] - o.x) * di.x, tx2 = (b1[0] - o.x) * di.x;
    float lo = fminf(tx1, tx2), hi = fmaxf(tx1, tx2);
    const float ty1 = (b0[1] - o.y) * di.y, ty2 = (b1[1] - o.y) * di.y;
    lo = fmaxf(lo, fminf(ty1, ty2));
    hi = fminf(hi, fmaxf(ty1, ty2));
    const float tz1 = (b0[2] - o.z) * di.z, tz2 = (b1[2] - o.z) * di.z;
    lo = fmaxf(lo, fminf(tz1, tz2));
    hi = fminf(hi, fmaxf(tz1, tz2));
    tlo = lo;
    thi = hi;
    return !(hi < lo);
}

// Starts one ray of a per-lane traversal of a single tree.  Returns false when
// the root box is missed.
__device__ __forceinline__ bool trav_init(Trav& T, const SceneView& sc, float3 o, float3 d) {
    T.o = o;
    T.d = d;
    float lo, hi;
    const bool inside = root_clip(sc, o, d, 0, T.dinv, lo, hi);
    T.tenter = lo;
    T.texit = hi;
    T.root_exit = hi;
    T.node = 0;
    T.leaf_off = 0;
    T.leaf_left = 0;
    T.head = 0;
    T.count = 0;
    T.restarts = 0;
    T.visits = 0;
    T.lost = false;
    T.best_id = kInvalidId;
    T.best_r = FLT_MAX;
    T.best_s = 0.f;
    T.best_t = 0.f;
    return inside;
}

// One leaf per step: descend to the next leaf, test all of its triangles,
// then the early-exit check and the move to the next stack entry.  Returns
// true when the traversal is complete.
template <int S, bool EXH, bool MT, bool ANY, bool COUNT>
__device__ __forceinline__ bool trav_step(Trav& T, const SceneView& sc, float tmax_any, uint2* stk,
                                          int stride, TraversalCounters& cnt) {
    static_assert((S & (S - 1)) == 0, "stack size must be a power of two");
    uint32_t node = T.node;
    float tenter = T.tenter, texit = T.texit;
    uint2 nd = sc.nodes[node];
    while ((nd.y & 3u) != 3u) {
        if (COUNT) cnt.inner++;
        const uint32_t ax = nd.y & 3u;
        const float tt = (__uint_as_float(nd.x) - pick(T.o, ax)) * pick(T.dinv, ax);
        uint32_t nearn = node + 1, farn = nd.y >> 2;
        if (pick(T.d, ax) < 0.f) {  // fixed direction <= 0 (zeros become +1e-5)
            const uint32_t tmp = nearn;
            nearn = farn;
            farn = tmp;
        }
        if (texit < tt) {
            node = nearn;
        } else if (tt < tenter) {
            node = farn;
        } else {
            stk[T.head * stride] = make_uint2(farn, __float_as_uint(texit));
            T.head = (T.head + 1) & (S - 1);
            if (T.count < S) ++T.count;
            else T.lost = true;
            node = nearn;
            texit = tt;
        }
        nd = sc.nodes[node];
    }
    if (COUNT) cnt.leaves++;
    if (++T.visits > kMaxLeafVisits) {
        cnt.incomplete = true;
        return true;
    }
    const uint32_t off = nd.x, nref = nd.y >> 2;
    for (uint32_t k = 0; k < nref; ++k) {
        const uint32_t id = sc.refs[off + k];
        float rr, ss, tt;
        const float bound = ANY ? tmax_any : T.best_r;
        const float4* pa = sc.tris + 4 * (size_t)id;
        const int code = MT ? leaf_test_mt<ANY>(pa, pa + 2, T.o, T.d, bound, rr, ss, tt)
                            : leaf_test_ref<ANY>(pa, pa + 2, T.o, T.d, bound, rr, ss, tt);
        if (COUNT) {
            cnt.refs++;
            cnt.tests++;
            cnt.full += code >= 1 ? 1u : 0u;
        }
        if (code == 2) {
            T.best_r = rr;
            T.best_s = ss;
            T.best_t = tt;
            T.best_id = id;
            if (ANY) return true;
        }
    }
    if (!EXH) {
        if (!ANY && T.best_id != kInvalidId && T.best_r * kExitMargin < texit) return true;
        if (ANY && tmax_any * kExitMargin < texit) return true;
    }
    if (T.count == 0) {
        if (!T.lost || !(texit < T.root_exit)) return true;
        if (++T.restarts > kMaxRestarts) {
            cnt.incomplete = true;
            return true;
        }
        T.node = 0;
        T.tenter = texit;
        T.texit = T.root_exit;
        T.lost = false;
        return false;
    }
    T.head = (T.head - 1) & (S - 1);
    --T.count;
    const uint2 e = stk[T.head * stride];
    T.node = e.x;
    T.tenter = texit;
    T.texit = __uint_as_float(e.y);
    return false;
}

// Traversal schedules: one leaf per step (a wave runs its largest leaf) or
// ticks of a few node steps / one triangle test.
enum Schedule { kSchedLeaf = 0, kSchedTick = 1, kSchedCoop = 2 };

template <int SCHED, int S, bool EXH, bool MT, bool ANY, bool COUNT>
__device__ __forceinline__ bool trav_advance(Trav& T, const SceneView& sc, float tmax_any,
                                             uint2* stk, int stride, TraversalCounters& cnt);

constexpr int kDescendPerTick = 8;

// One tick of the traversal state machine: at most kDescendPerTick node
// steps towards the next leaf, then at most one triangle test, then -- when
// the leaf is exhausted -- the early-exit check and the move to the next
// stack entry.  Returns true when the traversal is complete.  Lanes of a
// wave advance through different phases in the same tick, so a wave never
// waits for the largest leaf among its lanes.
template <int S, bool EXH, bool MT, bool ANY, bool COUNT>
__device__ __forceinline__ bool trav_tick(Trav& T, const SceneView& sc, float tmax_any, uint2* stk,
                                          int stride, TraversalCounters& cnt) {
    static_assert((S & (S - 1)) == 0, "stack size must be a power of two");
    if (T.leaf_left == 0) {
        uint32_t node = T.node;
        float tenter = T.tenter, texit = T.texit;
        uint2 nd = sc.nodes[node];
        int steps = 0;
        while ((nd.y & 3u) != 3u && steps < kDescendPerTick) {
            if (COUNT) cnt.inner++;
            const uint32_t ax = nd.y & 3u;
            const float tt = (__uint_as_float(nd.x) - pick(T.o, ax)) * pick(T.dinv, ax);
            uint32_t nearn = node + 1, farn = nd.y >> 2;
            if (pick(T.d, ax) < 0.f) {  // fixed direction <= 0 (zeros become +1e-5)
                const uint32_t tmp = nearn;
                nearn = farn;
                farn = tmp;
            }
            if (texit < tt) {
                node = nearn;
            } else if (tt < tenter) {
                node = farn;
            } else {
                stk[T.head * stride] = make_uint2(farn, __float_as_uint(texit));
                T.head = (T.head + 1) & (S - 1);
                if (T.count < S) ++T.count;
                else T.lost = true;
                node = nearn;
                texit = tt;
            }
            nd = sc.nodes[node];
            ++steps;
        }
        T.node = node;
        T.tenter = tenter;
        T.texit = texit;
        if ((nd.y & 3u) != 3u) return false;  // still descending
        if (COUNT) cnt.leaves++;
        if (++T.visits > kMaxLeafVisits) {
            cnt.incomplete = true;
            return true;
        }
        T.leaf_off = nd.x;
        T.leaf_left = nd.y >> 2;
        if (T.leaf_left == 0) goto leaf_done;
    }
    {
        const uint32_t id = sc.refs[T.leaf_off];
        ++T.leaf_off;
        --T.leaf_left;
        float rr, ss, tt;
        const float bound = ANY ? tmax_any : T.best_r;
        const float4* pa = sc.tris + 4 * (size_t)id;
        const int code = MT ? leaf_test_mt<ANY>(pa, pa + 2, T.o, T.d, bound, rr, ss, tt)
                            : leaf_test_ref<ANY>(pa, pa + 2, T.o, T.d, bound, rr, ss, tt);
        if (COUNT) {
            cnt.refs++;
            cnt.tests++;
            cnt.full += code >= 1 ? 1u : 0u;
        }
        if (code == 2) {
            T.best_r = rr;
            T.best_s = ss;
            T.best_t = tt;
            T.best_id = id;
            if (ANY) return true;
        }
        if (T.leaf_left != 0) return false;
    }
leaf_done : {
    const float texit = T.texit;
    if (!EXH) {
        if (!ANY && T.best_id != kInvalidId && T.best_r * kExitMargin < texit) return true;
        if (ANY && tmax_any * kExitMargin < texit) return true;
    }
    if (T.count == 0) {
        if (!T.lost || !(texit < T.root_exit)) return true;
        if (++T.restarts > kMaxRestarts) {
            cnt.incomplete = true;
            return true;
        }
        T.node = 0;
        T.tenter = texit;
        T.texit = T.root_exit;
        T.lost = false;
        return false;
    }
    T.head = (T.head - 1) & (S - 1);
    --T.count;
    const uint2 e = stk[T.head * stride];
    T.node = e.x;
    T.tenter = texit;
    T.texit = __uint_as_float(e.y);
    return false;
}
}

template <int SCHED, int S, bool EXH, bool MT, bool ANY, bool COUNT>
__device__ __forceinline__ bool trav_advance(Trav& T, const SceneView& sc, float tmax_any,
                                             uint2* stk, int stride, TraversalCounters& cnt) {
    if (SCHED == kSchedTick) return trav_tick<S, EXH, MT, ANY, COUNT>(T, sc, tmax_any, stk, stride, cnt);
    return trav_step<S, EXH, MT, ANY, COUNT>(T, sc, tmax_any, stk, stride, cnt);
}

// Whole traversal of one ray (closest hit, or visibility up to tmax_any).
template <int S, bool EXH, bool MT, bool ANY, bool COUNT>
__device__ __forceinline__ uint32_t traverse(const SceneView& sc, float3 o, float3 d, float tmax_any,
                                             float& r_out, float& s_out, float& t_out, uint2* stk,
                                             int stride, TraversalCounters& cnt) {
    Trav T;
    if (!trav_init(T, sc, o, d)) return kInvalidId;
    while (!trav_step<S, EXH, MT, ANY, COUNT>(T, sc, tmax_any, stk, stride, cnt)) {
    }
    if (COUNT) cnt.restarts += T.restarts;
    r_out = T.best_r;
    s_out = T.best_s;
    t_out = T.best_t;
    return T.best_id;
}

// Wave64 helpers for lane refill.
__device__ __forceinline__ uint32_t lanes_below(uint64_t mask) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                     __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

// Inclusive scan (sum, or maximum with MAX) over the 64 lanes of a wave, all
// lanes active: row shifts by 1, 2, 4, 8 within each 16-lane row (lanes whose
// source falls outside the row add the identity 0), then lane 15 of each row
// into rows 1 and 3 and lane 31 into rows 2 and 3.  Six DPP instructions.
template <bool MAX>
__device__ __forceinline__ uint32_t wave_scan(uint32_t x) {
#define TN_SCAN_STEP(ctrl, rows, bound)                                                          \
    {                                                                                            \
        const uint32_t t = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, ctrl, rows, 0xf, bound); \
        x = MAX ? max(x, t) : x + t;                                                             \
    }
    TN_SCAN_STEP(0x111, 0xf, true)   // row_shr:1
    TN_SCAN_STEP(0x112, 0xf, true)   // row_shr:2
    TN_SCAN_STEP(0x114, 0xf, true)   // row_shr:4
    TN_SCAN_STEP(0x118, 0xf, true)   // row_shr:8
    TN_SCAN_STEP(0x142, 0xa, false)  // row_bcast:15
    TN_SCAN_STEP(0x143, 0xc, false)  // row_bcast:31
#undef TN_SCAN_STEP
    return x;
}

// LDS of one wave for the cooperative loop, one entry per lane: the key of
// the closest hit in the lane's leaf, the start markers of the pooled pairs of
// one round, the distance at which a second pair of the leaf was hit, and the
// barycentrics (or their numerators) of the best hit so far.
struct CoopLds {
    unsigned long long slot[64];
    uint32_t mark[64];
    uint32_t tie[64];
    float2 st[64];
};

// What a cooperative traversal hands to its caller for one ray: the closest
// hit (id kInvalidId, r FLT_MAX, s = t = 0 on a miss), or with ANY whether
// some triangle was hit (id).
struct CoopHit {
    float3 d;
    uint32_t id;
    float r, s, t;
    bool tie;         // another triangle was hit at exactly r (TIE)
    uint32_t visits;  // leaves visited (COUNT)
};

// One ray of the cooperative loop.  Its stack holds the entries base .. head-1
// of a circular array of S; base > 0 tells that entries were overwritten.
// node: treelet << 2 | (0: its root, 1: the left child, 2: the right child), or
// kDone.  Flags are bits of words, not bools: the compiler keeps a bool that
// lives across the loop as a lane mask and spends scalar instructions on
// merging it at every branch.
constexpr uint32_t kDone = 0xFFFFFFFFu;
struct CoopRay {
    float3 o, d, dinv;
    float tenter, texit, root_exit;
    uint32_t node, root;
    int head, base, restarts;
    uint32_t visits;  // leaves left behind, kTied: another triangle was hit at exactly best_r
    float best_r;
    uint32_t best_ref;  // reference slot of the best hit
};
constexpr uint32_t kTied = 0x80000000u;

// The decision of one node step of a lane's descent (kdtree.cpp:540-564): the
// near child is the left one iff the direction is positive along the axis;
// past: the near child only, before: the far child only, else both, and the
// far one goes on the stack.
struct NodeStep {
    float t;
    bool both, right;  // right: the child to go on with
};
__device__ __forceinline__ NodeStep node_step(const CoopRay& R, uint32_t split, uint32_t ax) {
    const float di = pick(R.dinv, ax);
    NodeStep n;
    n.t = (__uint_as_float(split) - pick(R.o, ax)) * di;
    const bool neg = __float_as_int(di) < 0;  // fixed direction <= 0 (zeros become +1e-5)
    const bool past = R.texit < n.t, before = n.t < R.tenter;
    n.both = !past && !before;
    n.right = neg != (before && !past);
    return n;
}

// Wave-cooperative traversal loop.  Every round, the lanes with a ray descend
// towards their next leaf; then the wave pools the (ray, triangle reference)
// pairs of the leaves its lanes have reached and tests them 64 at a time, so
// a round costs ceil(sum of leaf sizes / 64) tests instead of the largest
// leaf.  Pair p belongs to the lane whose range [excl, incl) of the prefix
// sum of leaf sizes holds it.  In the round of pairs base..base+63 every lane
// whose range meets the round writes its number at its first pair of the
// round; a prefix maximum of these markers over the lanes gives each pair its
// owner, whose ray is fetched with ds_bpermute.  A hit is
// folded into the owner's 64-bit LDS slot with atomicMin on (r, pair index):
// the minimum is the first of the leaf's closest hits in leaf order, i.e. the
// reference's strict-< scan (kdtree.cpp:587-605).  The lane whose key stands
// after its round's atomics leaves the barycentrics in the owner's entry, so
// the owner reads nothing but its slot.
//
// What bounds the loop: where the scene is cached, VALU issue; in launches that
// leave the chip idle, the chain of dependent reads of the longest rays.  On the
// 2^24-ray batch (1.31 M triangles, refined tree) no unit is full: SIMDs issue in
// 82 % of the cycles, for 49 % of the lanes, and 25.4 GB in 4.9 ms are 5.2 TB/s,
// where the reference tree's launch of the same kernel draws 6.45 (66 GB, SIMDs 66 %
// busy: that one is bound by the lines it reads).  Four rules keep all three short:
//   * a round's descent stops when at most a third of the wave's rays are
//     still on their way (they go on in the next round): the last lanes of a
//     round take most of its dependent node reads.  2^24 rays: 8.03 ms with
//     no limit, 6.76 (1/8), 6.65 (1/4), 6.68 (1/3), 6.72 (1/2); small and
//     ragged launches are fastest at 1/3;
//   * finished rays are written out and replaced once kRefill lanes wait: a
//     ray's start (three divisions) and end run for that many lanes at once
//     (2^24 rays: 7.39 ms at 1, 6.91 at 8, 6.80 at 16, 6.79 at 24; renders
//     lose 2 % at 24);
//   * the descent reads two levels at a time (treelets, 32 bytes: a node and
//     its children), so a leaf is about 2.4 dependent reads away instead of
//     4.8: 6.67 -> 5.52 ms, a million visibility queries against 82 k
//     triangles 366 -> 298 us, a 512^2 one-sample pass 2.91 -> 2.63 ms;
//   * no branches where some lane always takes either side, loop exits and
//     work ranges in scalar registers, no division for a pair that only needs
//     a verdict (pair_test_ref): a two-level step takes 60 VALU instructions
//     (was 90), a round of 64 pairs 95 (was 146); 298 -> 257 us, 2.63 -> 2.26
//     ms, 4099 rays 195 -> 153 us, the 2^24 batch 5.50 -> 5.36 ms.
//   whole: read a record's second half with the first instead of when the first
//                      half asks for it: a latency less per leaf, and twice the
//                      bytes per test.  For launches of at most a ray per lane,
//                      which wait for their slowest ray (512^2 one-sample pass
//                      2.035 -> 1.975 ms, guided 512^2 x 8 3.98 -> 3.94); always, the
//                      2^24 batch went 4.95 -> 6.17 ms, 1080p m 4 85.1 -> 93.3.  Not
//                      with TIE or on a refined tree, whose kernels spill with it
//                      (1080p 87.1 ms, 4099 rays 92 -> 93.5 us);
//   chunk(begin, end): called by all lanes of the wave; returns false when no
//                      work is left (may update begin/end);
//   load(k, o, d, tmax, scene), store(k, hit): per-ray I/O (scene: the ray's
//                      tree in a forest, 0 otherwise).
// TIE (closest hit, reference leaf test): hit.tie tells whether a second
// triangle was hit at exactly the final best distance (in the same leaf, or
// in a later leaf at the earlier best); the winner among such ties depends on
// the tree's visit order.
constexpr uint32_t kRefill = 16, kDescendTail = 3;

template <int S, bool EXH, bool MT, bool ANY, bool COUNT, bool TIE = false, class Chunk, class Load, class Store>
__device__ __forceinline__ void coop_loop(const SceneView& sc, uint2* stk, int stride, CoopLds* wl, bool whole, Chunk chunk,
                                          Load load, Store store, TraversalCounters& cnt) {
    static_assert(!TIE || (!ANY && !MT), "tie detection is for the reference leaf test's closest hit");
    static_assert(S > 0 && (S & (S - 1)) == 0, "the circular stack index wraps with & (S - 1)");
    const uint32_t lane = threadIdx.x & 63u;
    constexpr uint32_t kNone = 0xFFFFFFFFu;
    constexpr uint32_t kWalk = 0xFFFFFFFFu;  // leaf size of a lane that is still on its way
    auto uniform = [](uint32_t x) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)x); };
    uint32_t next = 0, end = 0, more = 1;  // the same in all lanes
    uint32_t ray = kNone;
    CoopRay R;
    R.node = kDone;
    float tmx = 0.f;
    for (;;) {
        uint64_t act = __ballot(R.node != kDone);
        uint32_t nact = uniform((uint32_t)__popcll(act));
        if (nact == 0 || (nact <= 64 - kRefill && (more | (uint32_t)(next < end)))) {
            if (ray != kNone && R.node == kDone) {
                CoopHit h;
                h.d = R.d;
                h.visits = R.visits & ~kTied;
                h.tie = TIE && (R.visits & kTied);
                h.id = kInvalidId;
                h.r = FLT_MAX;
                h.s = h.t = 0.f;
                if (R.best_ref != kNone) {
                    h.id = ANY ? 0u : sc.refs[R.best_ref];
                    if (!ANY) {
                        const float2 st = wl->st[lane];
                        const float denom = MT ? 1.f : sc.lrb[2 * (size_t)R.best_ref + 1].w;
                        h.r = R.best_r;
                        h.s = MT ? st.x : st.x / denom;
                        h.t = MT ? st.y : st.y / denom;
                    }
                }
                store(ray, h);
                ray = kNone;
            }
            if (next >= end && more) {
                more = uniform(chunk(next, end) ? 1u : 0u);
                next = uniform(next);
                end = uniform(end);
            }
            if (next < end) {
                const uint32_t k = next + lanes_below(~act);
                if (R.node == kDone && k < end) {
                    float3 o, d;
                    uint32_t scene = 0;
                    load(k, o, d, tmx, scene);
                    R.o = o;
                    R.d = d;
                    float lo, hi;
                    const bool inside = root_clip(sc, o, d, scene, R.dinv, lo, hi);
                    // node steps take the direction's sign from the reciprocal
                    // (d = -inf, NaN: as d < 0 decides)
                    R.dinv.x = copysignf(R.dinv.x, d.x < 0.f ? -1.f : 1.f);
                    R.dinv.y = copysignf(R.dinv.y, d.y < 0.f ? -1.f : 1.f);
                    R.dinv.z = copysignf(R.dinv.z, d.z < 0.f ? -1.f : 1.f);
                    R.tenter = lo;
                    R.texit = hi;
                    R.root_exit = hi;
                    R.root = sc.roots ? sc.roots[scene].treelet << 2 : 0u;
                    R.node = inside ? R.root : kDone;  // a miss is written out by the next refill
                    R.head = R.base = R.restarts = 0;
                    R.visits = 0;
                    R.best_r = FLT_MAX;
                    R.best_ref = kNone;
                    ray = k;
                }
                next = min(next + (64u - nact), end);
            } else if (nact == 0 && !more) {
                break;
            }
            act = __ballot(R.node != kDone);
            nact = uniform((uint32_t)__popcll(act));
            if (nact == 0) continue;
        }
        // phase 1: descend towards the next leaf, two levels per read
        uint32_t loff = 0, lcnt = R.node != kDone ? kWalk : 0u;
        const uint32_t tail = nact / kDescendTail;
        do {
            if (lcnt == kWalk) {
                // No branches but around the stack writes: every path through
                // them would be taken by some lane, and merging their results
                // costs moves.
                const uint32_t ref = R.node;
                const uint4* t = sc.treelets + 2 * (size_t)(ref >> 2);
                const uint4 a = t[0];                                    // root_x, left_x, right_x, root_y
                const uint2 b = *reinterpret_cast<const uint2*>(t + 1);  // left_y, right_y
                // the root, for lanes that enter there (a leaf root's children repeat it)
                const uint32_t ax0 = a.w & 3u;
                const bool root = (ref & 3u) == 0 && ax0 != 3u;
                const NodeStep n0 = node_step(R, a.x, ax0);
                const bool push0 = root && n0.both;
                if (push0)
                    stk[(R.head & (S - 1)) * stride] =
                        make_uint2(ref | (n0.right ? 1u : 2u), __float_as_uint(R.texit));
                R.head += push0 ? 1 : 0;
                R.texit = push0 ? n0.t : R.texit;
                // its child, or the child the lane enters at
                const bool right = root ? n0.right : (ref & 2u) != 0;
                const uint32_t x = right ? a.z : a.y, y = right ? b.y : b.x;
                const uint32_t ax1 = y & 3u;
                const bool inner = ax1 != 3u;
                const NodeStep n1 = node_step(R, x, ax1);
                const bool push1 = inner && n1.both;
                R.node = (y & ~3u) | (n1.right ? 4u : 0u);  // the children's treelets are a pair
                if (push1) stk[(R.head & (S - 1)) * stride] = make_uint2(R.node ^ 4u, __float_as_uint(R.texit));
                R.head += push1 ? 1 : 0;
                R.texit = push1 ? n1.t : R.texit;
                R.base = max(R.base, R.head - S);
                loff = x;
                lcnt = inner ? kWalk : y >> 2;
                if (COUNT) cnt.inner += (root ? 1u : 0u) + (inner ? 1u : 0u);
            }
        } while (uniform((uint32_t)__popcll(__ballot(lcnt == kWalk))) > tail);
        // R.node of a lane at its leaf is not kDone: its low bits come from a pair index
        const bool leaf = R.node != kDone && lcnt != kWalk;
        if (!leaf) lcnt = 0;
        if (COUNT && leaf) cnt.leaves++;
        // phase 2: pooled leaf tests
        const uint32_t incl = wave_scan<false>(lcnt);
        const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
        if (total) {
            const uint32_t excl = lcnt ? incl - lcnt : ~0u;  // no pairs: meets no round
            const uint32_t rbase = loff - excl;              // refs index of pair p of this lane: rbase + p
            const float bound_own = ANY ? tmx : R.best_r;
            wl->slot[lane] = ~0ull;
            if (TIE) wl->tie[lane] = ~0u;
            uint32_t base = 0;
            do {
                // the first pair of a round always has a marker, so 0 is free for "none"
                wl->mark[lane] = 0u;
                __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
                if (excl < base + 64u && incl > base) wl->mark[excl > base ? excl - base : 0u] = lane;
                __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
                const uint32_t item = base + lane;
                const int own = (int)wave_scan<true>(wl->mark[lane]);
                auto of_owner = [&](float x) {
                    return __int_as_float(__builtin_amdgcn_ds_bpermute(own << 2, __float_as_int(x)));
                };
                const uint32_t rb = (uint32_t)__builtin_amdgcn_ds_bpermute(own << 2, (int)rbase);
                const float3 ro = make_float3(of_owner(R.o.x), of_owner(R.o.y), of_owner(R.o.z));
                const float3 rd = make_float3(of_owner(R.d.x), of_owner(R.d.y), of_owner(R.d.z));
                const float bnd = of_owner(bound_own);
                if (item < total) {
                    const size_t r = rb + item;  // reference slot of the pair
                    float rr, ss, tt;  // barycentrics, or their numerators (pair_test_ref)
                    const int code = MT ? leaf_test_mt<ANY>(sc.lra + 2 * r, sc.lrb + 2 * r, ro, rd, bnd, rr, ss, tt)
                                        : pair_test_ref<ANY, TIE>(sc.lra + 2 * r, sc.lrb + 2 * r, ro, rd, bnd, whole, rr, ss, tt);
                    if (COUNT) {
                        cnt.refs++;
                        cnt.tests++;
                        cnt.full += whole || code >= 1 ? 1u : 0u;
                    }
                    if (code >= 2) {
                        if (ANY) {
                            wl->slot[own] = 0ull;
                        } else {
                            // r >= 0 here; -0 maps to +0 so the key orders like the reference's <
                            const uint32_t rbits = __float_as_uint(rr + 0.0f);
                            const unsigned long long key = ((unsigned long long)rbits << 32) | item;
                            atomicMin(&wl->slot[own], key);
                            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
                            const unsigned long long now = wl->slot[own];
                            if (now == key) {
                                if (!TIE || code == 2) wl->st[own] = make_float2(ss, tt);
                            } else if (TIE && (uint32_t)(now >> 32) == rbits) {
                                wl->tie[own] = rbits;  // another pair at the smallest distance
                            }
                        }
                    }
                }
                base += 64u;
            } while (base < total);
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            const unsigned long long key = wl->slot[lane];
            if (lcnt && key != ~0ull) {
                const uint32_t r = rbase + (uint32_t)key, rbits = (uint32_t)(key >> 32);
                if (ANY) {
                    R.best_ref = 0u;
                    R.node = kDone;
                } else {
                    const bool tied = TIE && wl->tie[lane] == rbits;
                    if (TIE && R.best_ref != kNone && rbits == __float_as_uint(R.best_r + 0.0f)) {
                        // The leaf's hits lie only at exactly the current best
                        // distance: the best stays; tied iff one of them is
                        // another triangle -- two or more of them (a triangle
                        // occurs once per leaf), or one that is not the best's
                        // (a triangle spanning several leaves is met again in
                        // later ones).
                        if (tied || sc.refs[r] != sc.refs[R.best_ref]) R.visits |= kTied;
                    } else {
                        R.best_r = __uint_as_float(rbits);
                        R.best_ref = r;
                        if (TIE) R.visits = (R.visits & ~kTied) | (tied ? kTied : 0u);
                        if (rbits == 0u) {  // a distance of zero keeps its sign
                            float ss, tt;
                            const float4 *pa = sc.lra + 2 * (size_t)r, *pc = sc.lrb + 2 * (size_t)r;
                            if (MT) leaf_test_mt<ANY>(pa, pc, R.o, R.d, bound_own, R.best_r, ss, tt);
                            else pair_test_ref<ANY, TIE>(pa, pc, R.o, R.d, bound_own, false, R.best_r, ss, tt);
                        }
                    }
                }
            }
        }
        // after the leaf (empty ones included): early exit, next stack entry or restart
        if (leaf && (!ANY || R.node != kDone)) {
            const float texit = R.texit;
            bool done = false;
            if (!EXH) done = (ANY ? tmx : R.best_r) * kExitMargin < texit;  // no hit: FLT_MAX, never below
            if (!done) {
                if (R.head == R.base) {
                    done = R.base == 0 || !(texit < R.root_exit);
                    if (!done && ++R.restarts > kMaxRestarts) {
                        cnt.incomplete = true;
                        done = true;
                    }
                    R.node = R.root;
                    R.texit = R.root_exit;
                    R.head = R.base = 0;
                } else {
                    --R.head;
                    const uint2 e = stk[(R.head & (S - 1)) * stride];
                    R.node = e.x;
                    R.texit = __uint_as_float(e.y);
                }
                R.tenter = texit;
                if (!done && (++R.visits & ~kTied) > kMaxLeafVisits) {
                    cnt.incomplete = true;
                    done = true;
                }
            }
            if (done) {
                if (COUNT) {
                    cnt.restarts += R.restarts;
                    // its last leaf, unless that is the one it was abandoned at
                    R.visits += (R.visits & ~kTied) <= kMaxLeafVisits ? 1u : 0u;
                }
                R.node = kDone;
            }
        }
    }
}

}  // namespace tn
