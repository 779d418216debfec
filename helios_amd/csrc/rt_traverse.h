// rt_traverse.h -- BVH traversal and launch helpers shared by the wavefront-persistent ray kernels.
//
//   trace_closest   stack traversal of the 64-byte BVH2 (both child boxes per node), LDS stack,
//                   closest hit with the reference acceptance rule (t > tmin, skip the origin
//                   primitive; R/shaders/common/bvh_traversal.glsl:68-170) and a canonical tie rule
//                   (equal t -> lower primitive index) instead of traversal order.
//   trace_any       occlusion query: any accepted hit with t <= tmax ends the traversal.  The direct
//                   pass only needs "occluded or not"; with the nearest periodic face as tmax this
//                   reproduces the reference decision (closest hit vs periodic face) exactly.
//   packet_any4     the same for the 64 rays of a wave over the BVH4 (packet_any: over the BVH2).
//   WaveQueue       work queue of a persistent launch.
//   LaneRay, lane_* resumable closest-hit traversal of one lane over the BVH2 (counting kernels, scenes
//                   without a block tree).
//   BlkRay, blk_*   the same over the block tree (rt_types.h).
// The kernels that use them are in rt_trace.hip (diffuse rays and gathers), rt_direct.hip (direct rays),
// rt_cast.hip (castRays, cameras) and rt_glass.hip (translucent covers).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include <cfloat>
#include <string>

#include "rt_internal.h"

namespace rt {

__device__ __forceinline__ float min3f(float a, float b, float c) { return fminf(fminf(a, b), c); }
__device__ __forceinline__ float max3f(float a, float b, float c) { return fmaxf(fmaxf(a, b), c); }

// traversal work counters (node fetches, primitive tests) of one lane.  The counter type also carries the
// traversal's flags MK: bit 0 = honour texture masks (off compiles the mask tests away for scenes without
// masks, keeping the leaf code and its register use as small as before masks existed), bit 1 = watertight
// intersection predicates instead of the reference's (rt_set_predicates).
template <int MK>
struct TCntT {
    uint32_t nodes, prims;
    static constexpr bool mask = (MK & RT_FL_MASK) != 0;
    static constexpr bool wt = (MK & RT_FL_WT) != 0;
    static constexpr int flags = MK;
};
// the same interface with every update compiled away (timed kernels)
struct NopCounter {
    __device__ __forceinline__ NopCounter operator++(int) { return *this; }
    __device__ __forceinline__ NopCounter &operator+=(uint32_t) { return *this; }
};
template <int MK>
struct NoCntT {
    NopCounter nodes, prims;
    static constexpr bool mask = (MK & RT_FL_MASK) != 0;
    static constexpr bool wt = (MK & RT_FL_WT) != 0;
    static constexpr int flags = MK;
};
template <bool COUNT, int MK>
using Cnt = typename std::conditional<COUNT, TCntT<MK>, NoCntT<MK>>::type;

struct RayPre {
    float ix, iy, iz, ox, oy, oz;
};

__device__ __forceinline__ RayPre ray_pre(v3f o, v3f d) {
    RayPre r;
    r.ix = fabsf(d.x) > 1e-30f ? 1.0f / d.x : 1e30f;
    r.iy = fabsf(d.y) > 1e-30f ? 1.0f / d.y : 1e30f;
    r.iz = fabsf(d.z) > 1e-30f ? 1.0f / d.z : 1e30f;
    r.ox = o.x * r.ix;
    r.oy = o.y * r.iy;
    r.oz = o.z * r.iz;
    return r;
}

// BVH nodes and primitive records do not change while a trace kernel runs: loading them through the
// constant address space lets the compiler use scalar loads when the index is wave-uniform (the
// packet traversal) and ordinary vector loads otherwise.
__device__ __forceinline__ float4 ldc(const float4 *p) {
#if defined(__HIP_DEVICE_COMPILE__)
    typedef __attribute__((address_space(4))) const float cfloat_t;
    const cfloat_t *q = (const cfloat_t *)(const float *)p;
    return make_float4(q[0], q[1], q[2], q[3]);
#else
    return *p;
#endif
}

// wave-uniform copy of a pointer (lets the compiler keep it, and addresses built from uniform
// indices, in scalar registers)
template <typename T>
__device__ __forceinline__ T *uptr(T *p) {
    uint64_t v = (uint64_t)p;
    uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
    uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return (T *)(((uint64_t)hi << 32) | lo);
}

// Load of a value at a wave-uniform address through the constant address space (scalar load).
template <typename T>
__device__ __forceinline__ T ldu(const T *p) {
#if defined(__HIP_DEVICE_COMPILE__)
    typedef __attribute__((address_space(4))) const T cT;
    return *(const cT *)p;
#else
    return *p;
#endif
}

// Intersect the primitive whose record is at r (recs: the scene's record array, which mask descriptors count
// from); returns its index and the hit.
template <bool CD, int MK = RT_FL_MASK>
__device__ __forceinline__ bool leaf_hit_at(const float4 *r, const float4 *recs, v3f o, v3f d, uint32_t skip,
                                            uint32_t &id, float &t) {
    float4 r0 = ldc(r);
    uint32_t tag = __float_as_uint(r0.w);
    id = tag & RT_ID_BITS;
    bool patch = (tag & RT_PATCH_BIT) != 0;
    const bool masked = (MK & RT_FL_MASK) && !CD && (tag & RT_MASK_BIT) != 0;
    float4 r1 = ldc(r + 1), r2 = ldc(r + 2);
    // a voxel is a box that castRays hits (CollisionDetection_RayTracing.cpp:1625-1711) and the radiation
    // traversal never does (bvh_traversal.glsl:118-140 tests patches, tiles and triangles only)
    if (CD && (tag & RT_VOXEL_BIT)) return voxel_hit_cd(r0, r1, o, d, t) && id != skip;
    float4 r3 = (patch || masked) ? ldc(r + 3) : make_float4(0.f, 0.f, 0.f, 0.f);
    float ua, ub;
    bool hit = isect_rec_uv<CD, (MK & RT_FL_WT) != 0>(r0, r1, r2, r3, patch, o, d, t, ua, ub) && id != skip &&
               (CD || !(tag & RT_VOXEL_BIT));
    // texture mask (bvh_traversal.glsl:143-148): a transparent texel lets the ray pass
    if (masked && hit) hit = mask_hit_opaque(recs, __float_as_uint(r3.w), patch, ua, ub, r1.w, r2.w);
    return hit;
}

// leaf_hit_at() for the primitive in leaf slot k
template <bool CD, int MK = RT_FL_MASK>
__device__ __forceinline__ bool leaf_hit_p(const float4 *recs, uint32_t k, v3f o, v3f d, uint32_t skip, uint32_t &id,
                                           float &t) {
    return leaf_hit_at<CD, MK>(recs + (size_t)k * 4, recs, o, d, skip, id, t);
}

template <bool CD, int MK = RT_FL_MASK>
__device__ __forceinline__ bool leaf_hit(const DevScene &sc, uint32_t k, v3f o, v3f d, uint32_t skip, uint32_t &id,
                                         float &t) {
    return leaf_hit_p<CD, MK>(sc.rec, k, o, d, skip, id, t);
}

template <bool CD, int MK = RT_FL_MASK>
__device__ __forceinline__ void test_leaf(const float4 *recs, uint32_t k, v3f o, v3f d, float tmin, uint32_t skip,
                                          float &best_t, uint32_t &best, uint32_t &best_slot) {
    uint32_t id;
    float t;
    // castRays takes a patch or triangle beyond 1e-6 and a voxel at 1e-6 or beyond
    // (CD/src/CollisionDetection_RayTracing.cpp:1562, 1595, 1681)
    if (leaf_hit_p<CD, MK>(recs, k, o, d, skip, id, t) &&
        (t > tmin || (CD && t == tmin && (__float_as_uint(ldc(recs + (size_t)k * 4).w) & RT_VOXEL_BIT)))) {
        if (t < best_t || (t == best_t && best != RT_MISS && id < best)) {
            best_t = t;
            best = id;
            best_slot = k;
        }
    }
}

// slab tests of both children of node ni against [.., tlim]
struct NodeTest {
    float tn0, tn1;
    uint32_t c0, c1;
    bool h0, h1;
};

__device__ __forceinline__ NodeTest node_test_p(const float4 *nodes, uint32_t ni, const RayPre &rp, float tlim) {
    const float4 *nd = nodes + (size_t)ni * 4;
    float4 n0 = ldc(nd), n1 = ldc(nd + 1), n2 = ldc(nd + 2), n3 = ldc(nd + 3);
    float ax = fmaf(n0.x, rp.ix, -rp.ox), bx = fmaf(n0.y, rp.ix, -rp.ox);
    float ay = fmaf(n0.z, rp.iy, -rp.oy), by = fmaf(n0.w, rp.iy, -rp.oy);
    float az = fmaf(n1.x, rp.iz, -rp.oz), bz = fmaf(n1.y, rp.iz, -rp.oz);
    float tn0 = max3f(fminf(ax, bx), fminf(ay, by), fminf(az, bz));
    float tf0 = min3f(fmaxf(ax, bx), fmaxf(ay, by), fmaxf(az, bz));
    float cx = fmaf(n1.z, rp.ix, -rp.ox), dx = fmaf(n1.w, rp.ix, -rp.ox);
    float cy = fmaf(n2.x, rp.iy, -rp.oy), dy = fmaf(n2.y, rp.iy, -rp.oy);
    float cz = fmaf(n2.z, rp.iz, -rp.oz), dz = fmaf(n2.w, rp.iz, -rp.oz);
    float tn1 = max3f(fminf(cx, dx), fminf(cy, dy), fminf(cz, dz));
    float tf1 = min3f(fmaxf(cx, dx), fmaxf(cy, dy), fmaxf(cz, dz));
    NodeTest r;
    r.tn0 = tn0;
    r.tn1 = tn1;
    // tn <= tf && tf >= 0 && tn <= tlim, as one comparison (tlim >= 0; NaN only ever widens the test)
    r.h0 = fmaxf(tn0, 0.f) <= fminf(tf0, tlim);
    r.h1 = fmaxf(tn1, 0.f) <= fminf(tf1, tlim);
    r.c0 = __float_as_uint(n3.x);
    r.c1 = __float_as_uint(n3.y);
    return r;
}

// Closest accepted hit (t > tmin, t < tstart, ties -> lower primitive index).
template <bool CD, int STK, typename C>
__device__ uint32_t trace_closest(const DevScene &sc, v3f o, v3f d, float tmin, uint32_t skip, float tstart,
                                  float &t_out, uint32_t &slot_out, uint32_t *stk, uint32_t stride, int *err,
                                  C &cnt) {
    float best_t = tstart;
    uint32_t best = RT_MISS, best_slot = RT_MISS;
    // scene fields in registers: the stack stores below go through a generic pointer, and the compiler
    // would otherwise reload them from the descriptor on every step
    const float4 *nodes = sc.node, *recs = sc.rec;
    const uint32_t nleaf = sc.nleaf;
    if (nleaf <= 1) {
        if (nleaf == 1) { cnt.prims++; test_leaf<CD, C::flags>(recs, 0, o, d, tmin, skip, best_t, best, best_slot); }
        t_out = best_t;
        slot_out = best_slot;
        return best;
    }
    RayPre rp = ray_pre(o, d);
    uint32_t ni = 0;
    int sp = 0;
    // every internal node is entered at most once per trace; the cap only guards malformed trees
    uint32_t budget = nleaf + 8;
    while (true) {
        if (budget-- == 0 || ni >= nleaf - 1) {
            atomicOr(err, 2);
            break;
        }
        cnt.nodes++;
        NodeTest nt = node_test_p(nodes, ni, rp, best_t);
        bool l0 = (nt.c0 & RT_LEAF_BIT) != 0, l1 = (nt.c1 & RT_LEAF_BIT) != 0;
        if (nt.h0 && l0) { cnt.prims++; test_leaf<CD, C::flags>(recs, nt.c0 & ~RT_LEAF_BIT, o, d, tmin, skip, best_t, best, best_slot); }
        if (nt.h1 && l1) { cnt.prims++; test_leaf<CD, C::flags>(recs, nt.c1 & ~RT_LEAF_BIT, o, d, tmin, skip, best_t, best, best_slot); }
        bool g0 = nt.h0 && !l0, g1 = nt.h1 && !l1;
        if (g0 && g1) {
            bool first0 = nt.tn0 <= nt.tn1;
            if (sp >= STK) {
                atomicOr(err, 1);
                break;
            }
            stk[(uint32_t)sp * stride] = first0 ? nt.c1 : nt.c0;
            sp++;
            ni = first0 ? nt.c0 : nt.c1;
        } else if (g0) {
            ni = nt.c0;
        } else if (g1) {
            ni = nt.c1;
        } else {
            if (sp == 0) break;
            sp--;
            ni = stk[(uint32_t)sp * stride];
        }
    }
    t_out = best_t;
    slot_out = best_slot;
    return best;
}

// Any accepted radiation-predicate hit with tmin < t <= tmax?
template <int STK, typename C>
__device__ bool trace_any(const DevScene &sc, v3f o, v3f d, float tmin, uint32_t skip, float tmax, uint32_t *stk,
                          uint32_t stride, int *err, C &cnt) {
    uint32_t id;
    float t;
    const float4 *nodes = sc.node, *recs = sc.rec;
    const uint32_t nleaf = sc.nleaf;
    if (nleaf <= 1) {
        if (nleaf == 1) {
            cnt.prims++;
            return leaf_hit_p<false, C::flags>(recs, 0, o, d, skip, id, t) && t > tmin && t <= tmax;
        }
        return false;
    }
    RayPre rp = ray_pre(o, d);
    uint32_t ni = 0;
    int sp = 0;
    uint32_t budget = nleaf + 8;
    while (true) {
        if (budget-- == 0 || ni >= nleaf - 1) {
            atomicOr(err, 2);
            return false;
        }
        cnt.nodes++;
        NodeTest nt = node_test_p(nodes, ni, rp, tmax);
        bool l0 = (nt.c0 & RT_LEAF_BIT) != 0, l1 = (nt.c1 & RT_LEAF_BIT) != 0;
        if (nt.h0 && l0) {
            cnt.prims++;
            if (leaf_hit_p<false, C::flags>(recs, nt.c0 & ~RT_LEAF_BIT, o, d, skip, id, t) && t > tmin && t <= tmax) return true;
        }
        if (nt.h1 && l1) {
            cnt.prims++;
            if (leaf_hit_p<false, C::flags>(recs, nt.c1 & ~RT_LEAF_BIT, o, d, skip, id, t) && t > tmin && t <= tmax) return true;
        }
        bool g0 = nt.h0 && !l0, g1 = nt.h1 && !l1;
        if (g0 && g1) {
            bool first0 = nt.tn0 <= nt.tn1;
            if (sp >= STK) {
                atomicOr(err, 1);
                return false;
            }
            stk[(uint32_t)sp * stride] = first0 ? nt.c1 : nt.c0;
            sp++;
            ni = first0 ? nt.c0 : nt.c1;
        } else if (g0) {
            ni = nt.c0;
        } else if (g1) {
            ni = nt.c1;
        } else {
            if (sp == 0) return false;
            sp--;
            ni = stk[(uint32_t)sp * stride];
        }
    }
}

// Wave-coherent any-hit query: the 64 lanes (rays of one primitive towards one source, hence nearly
// parallel and close together) walk the BVH together.  The node index and the stack are wave-uniform
// (node fetched once per wave through scalar loads, stack in a per-wave LDS column); every lane tests
// the child boxes and primitives itself and stops searching at its first accepted hit.  A lane reaches
// every node whose box chain it intersects, so its answer equals the per-lane traversal's.
template <int STK, typename C>
__device__ bool packet_any(const DevScene &sc, v3f o, v3f d, float tmin, uint32_t skip, float tmax, bool active,
                           uint32_t *wstk, int *err, C &cnt) {
    bool act = active, found = false;
    uint32_t id;
    float t;
    if (sc.nleaf <= 1) {
        if (sc.nleaf == 1 && act) {
            cnt.prims++;
            found = leaf_hit<false, C::flags>(sc, 0, o, d, skip, id, t) && t > tmin && t <= tmax;
        }
        return found;
    }
    RayPre rp = ray_pre(o, d);
    const float4 *nodes = uptr(sc.node), *recs = uptr(sc.rec);
    const uint32_t nleaf = __builtin_amdgcn_readfirstlane(sc.nleaf);
    uint32_t ni = 0;
    uint32_t sp = 0;
    uint32_t budget = nleaf + 8;
    while (__ballot(act) != 0) {
        ni = __builtin_amdgcn_readfirstlane(ni);
        if (budget-- == 0 || ni >= nleaf - 1) {
            atomicOr(err, 2);
            break;
        }
        if (act) cnt.nodes++;  // per-ray visits (one fetch serves the whole wave)
        NodeTest nt = node_test_p(nodes, ni, rp, tmax);
        uint32_t c0 = __builtin_amdgcn_readfirstlane(nt.c0), c1 = __builtin_amdgcn_readfirstlane(nt.c1);
        nt.c0 = c0;
        nt.c1 = c1;
        bool l0 = (nt.c0 & RT_LEAF_BIT) != 0, l1 = (nt.c1 & RT_LEAF_BIT) != 0;
        bool h0 = act && nt.h0, h1 = act && nt.h1;
        if (l0 && h0) {
            cnt.prims++;
            if (leaf_hit_p<false, C::flags>(recs, nt.c0 & ~RT_LEAF_BIT, o, d, skip, id, t) && t > tmin && t <= tmax) {
                found = true;
                act = false;
            }
        }
        if (l1 && h1 && act) {
            cnt.prims++;
            if (leaf_hit_p<false, C::flags>(recs, nt.c1 & ~RT_LEAF_BIT, o, d, skip, id, t) && t > tmin && t <= tmax) {
                found = true;
                act = false;
            }
        }
        bool g0 = !l0 && __ballot(h0 && act) != 0;
        bool g1 = !l1 && __ballot(h1 && act) != 0;
        if (g0 && g1) {
            // nearer child first, as seen by the wave's first still-searching lane
            uint64_t m = __ballot(act && nt.tn0 <= nt.tn1);
            uint64_t a = __ballot(act);
            bool first0 = (m & (a & (~a + 1))) != 0;
            if (sp >= STK) {
                atomicOr(err, 1);
                break;
            }
            wstk[sp] = first0 ? nt.c1 : nt.c0;  // same value from every lane
            sp++;
            ni = first0 ? nt.c0 : nt.c1;
        } else if (g0) {
            ni = nt.c0;
        } else if (g1) {
            ni = nt.c1;
        } else {
            if (sp == 0) break;
            sp--;
            ni = wstk[sp];
        }
    }
    return found;
}

// Slab test of one child box of a BVH4 node.
__device__ __forceinline__ void slab4(float lx, float hx, float ly, float hy, float lz, float hz, const RayPre &rp,
                                      float &tn, float &tf) {
    float ax = fmaf(lx, rp.ix, -rp.ox), bx = fmaf(hx, rp.ix, -rp.ox);
    float ay = fmaf(ly, rp.iy, -rp.oy), by = fmaf(hy, rp.iy, -rp.oy);
    float az = fmaf(lz, rp.iz, -rp.oz), bz = fmaf(hz, rp.iz, -rp.oz);
    tn = max3f(fminf(ax, bx), fminf(ay, by), fminf(az, bz));
    tf = min3f(fmaxf(ax, bx), fmaxf(ay, by), fmaxf(az, bz));
}

// Ascending compare-exchange of two (key, link) pairs held in scalar registers.
__device__ __forceinline__ void cswap(float &ka, uint32_t &la, float &kb, uint32_t &lb) {
    bool sw = kb < ka;
    float k = sw ? kb : ka;
    uint32_t l = sw ? lb : la;
    kb = sw ? ka : kb;
    lb = sw ? la : lb;
    ka = k;
    la = l;
}

// packet_any() on the BVH4: one 128-byte node per step (two scalar loads), four child boxes tested by every
// lane.  Leaf children are tested by the lanes whose box test passed; internal children hit by any still
// searching lane are visited nearest-first as seen by the wave's first searching lane (a sorting network on
// at most four scalar keys), the others pushed on the per-wave LDS stack.  A lane still reaches every node
// whose box chain it intersects, so each lane's answer equals the single-ray traversal's.
#define RT_WSTK4 128
template <typename C>
__device__ bool packet_any4(const DevScene &sc, v3f o, v3f d, float tmin, uint32_t skip, float tmax, bool active,
                            uint32_t *wstk, int *err, C &cnt) {
    bool act = active, found = false;
    uint32_t id;
    float t;
    if (sc.nleaf <= 1) {
        if (sc.nleaf == 1 && act) {
            cnt.prims++;
            found = leaf_hit<false, C::flags>(sc, 0, o, d, skip, id, t) && t > tmin && t <= tmax;
        }
        return found;
    }
    RayPre rp = ray_pre(o, d);
    const float4 *nodes = uptr(sc.node4), *recs = uptr(sc.rec);
    const uint32_t nn4 = __builtin_amdgcn_readfirstlane(sc.nnode4);
    uint32_t ni = 0, sp = 0;
    uint32_t budget = nn4 + 8;
    while (__ballot(act) != 0) {
        ni = __builtin_amdgcn_readfirstlane(ni);
        if (budget-- == 0 || ni >= nn4) {
            atomicOr(err, 2);
            break;
        }
        if (act) cnt.nodes++;
        const float4 *nd = nodes + (size_t)ni * 8;
        const float4 lx = ldc(nd), hx = ldc(nd + 1), ly = ldc(nd + 2), hy = ldc(nd + 3);
        const float4 lz = ldc(nd + 4), hz = ldc(nd + 5), lk = ldc(nd + 6);
        uint32_t lnk[4];
        lnk[0] = __builtin_amdgcn_readfirstlane(__float_as_uint(lk.x));
        lnk[1] = __builtin_amdgcn_readfirstlane(__float_as_uint(lk.y));
        lnk[2] = __builtin_amdgcn_readfirstlane(__float_as_uint(lk.z));
        lnk[3] = __builtin_amdgcn_readfirstlane(__float_as_uint(lk.w));
        float tn[4], tf[4];
        slab4(lx.x, hx.x, ly.x, hy.x, lz.x, hz.x, rp, tn[0], tf[0]);
        slab4(lx.y, hx.y, ly.y, hy.y, lz.y, hz.y, rp, tn[1], tf[1]);
        slab4(lx.z, hx.z, ly.z, hy.z, lz.z, hz.z, rp, tn[2], tf[2]);
        slab4(lx.w, hx.w, ly.w, hy.w, lz.w, hz.w, rp, tn[3], tf[3]);
        bool h[4];
#pragma unroll
        for (int k = 0; k < 4; k++) h[k] = fmaxf(tn[k], 0.f) <= fminf(tf[k], tmax);  // unused slots never pass
        // leaf children: a wave-uniform branch per leaf, the test itself predicated per lane
#pragma unroll
        for (int k = 0; k < 4; k++) {
            if (lnk[k] & RT_LEAF_BIT) {
                const bool want = h[k] && act;
                if (__ballot(want) != 0) {
                    cnt.prims += want ? 1u : 0u;
                    const bool hit = leaf_hit_p<false, C::flags>(recs, lnk[k] & ~RT_LEAF_BIT, o, d, skip, id, t) && t > tmin &&
                                     t <= tmax;
                    const bool take = want && hit;
                    found = found || take;
                    act = act && !take;
                }
            }
        }
        const uint64_t am = __ballot(act);
        if (am == 0) break;
        const uint32_t leader = (uint32_t)__builtin_ctzll(am);
        // internal children some searching lane hits, keyed by the leader's entry distance
        float key[4];
        uint32_t lk4[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            bool inner = !(lnk[k] & RT_LEAF_BIT);
            bool any = inner && __ballot(h[k] && act) != 0;
            const int kk = __builtin_amdgcn_readlane(__float_as_int(h[k] ? tn[k] : 3.0e38f), (int)leader);
            key[k] = any ? __int_as_float(kk) : INFINITY;
            lk4[k] = any ? lnk[k] : 0xFFFFFFFFu;
        }
        cswap(key[0], lk4[0], key[1], lk4[1]);
        cswap(key[2], lk4[2], key[3], lk4[3]);
        cswap(key[0], lk4[0], key[2], lk4[2]);
        cswap(key[1], lk4[1], key[3], lk4[3]);
        cswap(key[1], lk4[1], key[2], lk4[2]);
        const uint32_t m = (lk4[0] != 0xFFFFFFFFu) + (lk4[1] != 0xFFFFFFFFu) + (lk4[2] != 0xFFFFFFFFu) +
                           (lk4[3] != 0xFFFFFFFFu);
        if (m == 0) {
            if (sp == 0) break;
            sp--;
            ni = wstk[sp];
        } else {
            if (sp + m - 1 > RT_WSTK4) {
                atomicOr(err, 1);
                break;
            }
            if (m >= 4) wstk[sp++] = lk4[3];
            if (m >= 3) wstk[sp++] = lk4[2];
            if (m >= 2) wstk[sp++] = lk4[1];
            ni = lk4[0];
        }
    }
    return found;
}

// R/shaders/common/periodic_boundary.glsl:28-59
__device__ __forceinline__ float isect_bbox_face(const BBoxFace &f, v3f o, v3f d) {
    v3f n = mk3(f.n[0], f.n[1], f.n[2]);
    v3f v0 = mk3(f.v0[0], f.v0[1], f.v0[2]);
    float denom = dot3(d, n);
    if (fabsf(denom) < 1e-8f) return -1.0f;
    float t = rdiv(dot3(sub3(v0, o), n), denom);
    if (t <= 1e-5f || t > 1e8f) return -1.0f;
    v3f p = add3(o, mul3(d, t));
    v3f dd = sub3(p, v0);
    float da = dot3(dd, mk3(f.a[0], f.a[1], f.a[2]));
    float db = dot3(dd, mk3(f.b[0], f.b[1], f.b[2]));
    if (da > 0.0f && da < f.aa && db > 0.0f && db < f.bb) return t;
    return -1.0f;
}

// nearest periodic face strictly below tlim (periodic_boundary.glsl:84-92); returns its t or -1
__device__ __forceinline__ float nearest_face(const DevScene &sc, v3f o, v3f d, float tlim) {
    float bt = tlim;
    int cf = -1;
    for (uint32_t f = 0; f < sc.nbbox; f++) {
        float t = isect_bbox_face(sc.bbox[f], o, d);
        if (t > 0.0f && t < bt) { bt = t; cf = (int)f; }
    }
    return cf < 0 ? -1.0f : bt;
}

// The same with the faces read through scalar loads (sc wave-uniform, its faces do not change)
__device__ __forceinline__ float nearest_face_u(const DevScene &sc, uint32_t nbbox, v3f o, v3f d, float tlim) {
    float bt = tlim;
    bool any = false;
    for (uint32_t f = 0; f < nbbox; f++) {
        BBoxFace F;
        const float *src = (const float *)&sc.bbox[f];
        float *dst = (float *)&F;
#pragma unroll
        for (int k = 0; k < (int)(sizeof(BBoxFace) / 4); k++) dst[k] = ldu(src + k);
        const float t = isect_bbox_face(F, o, d);
        if (t > 0.0f && t < bt) { bt = t; any = true; }
    }
    return any ? bt : -1.0f;
}

// wrapped origin for a face hit at distance bt (periodic_boundary.glsl:94-111)
__device__ __forceinline__ v3f wrap_at(const DevScene &sc, v3f o, v3f d, float bt) {
    v3f hp = add3(o, mul3(d, bt));
    const float eps = 1e-5f;
    float wx = sc.dom[1] - sc.dom[0], wy = sc.dom[3] - sc.dom[2];
    v3f w = hp;
    if (sc.px && fabsf(hp.x - sc.dom[0]) <= eps) w.x += wx - eps;
    else if (sc.px && fabsf(hp.x - sc.dom[1]) <= eps) w.x -= wx - eps;
    else if (sc.py && fabsf(hp.y - sc.dom[2]) <= eps) w.y += wy - eps;
    else if (sc.py && fabsf(hp.y - sc.dom[3]) <= eps) w.y -= wy - eps;
    return w;
}

// Occlusion towards a collimated source with periodic wraps (direct_raygen.comp:603-672 without
// translucent covers).  The reference wraps when the nearest periodic face is strictly closer than
// the closest hit, and is occluded otherwise if anything was hit; "some hit with t <= t_face" is the
// same decision, so an any-hit query suffices.  32 wraps without resolution count as unoccluded.
template <int STK, typename C>
__device__ __forceinline__ bool occluded(const DevScene &sc, v3f o, v3f d, float tmin, uint32_t skip, uint32_t *stk,
                                         uint32_t stride, int *err, C &cnt) {
    v3f cur = o;
    for (int step = 0; step < 32; ++step) {
        float tf = sc.nbbox ? nearest_face(sc, cur, d, 1e30f) : -1.0f;
        float tmax = tf > 0.f ? tf : 1e30f;
        if (trace_any<STK>(sc, cur, d, tmin, skip, tmax, stk, stride, err, cnt)) return true;
        if (tf <= 0.f) return false;
        cur = wrap_at(sc, cur, d, tf);
    }
    return false;
}

// occluded() for a whole wave with packet_any4() (packet_any() when the scene has no usable BVH4); each
// lane keeps its own wrap state.
template <int STK, typename C>
__device__ __forceinline__ bool packet_occluded(const DevScene &sc, v3f o, v3f d, float tmin, uint32_t skip,
                                                bool active, uint32_t *wstk, uint32_t *wstk4, int *err, C &cnt) {
    v3f cur = o;
    bool need = active, occl = false;
    for (int step = 0; step < 32; ++step) {
        if (__ballot(need) == 0) break;
        float tf = (need && sc.nbbox) ? nearest_face(sc, cur, d, 1e30f) : -1.0f;
        float tmax = tf > 0.f ? tf : 1e30f;
        bool f = sc.node4 ? packet_any4(sc, cur, d, tmin, skip, tmax, need, wstk4, err, cnt)
                          : packet_any<STK>(sc, cur, d, tmin, skip, tmax, need, wstk, err, cnt);
        if (need) {
            if (f) { occl = true; need = false; }
            else if (tf <= 0.f) need = false;
            else cur = wrap_at(sc, cur, d, tf);
        }
    }
    return occl;
}

// A wave's view of the work queue of a persistent launch: items [0, total) in chunks of `chunk`.  What bounds a
// queue is its atomics on one address, 11.3 ns each and one after the other: more than a whole item of the direct
// kernel takes the chip (225 rays of a primitive over an occlusion grid, 5 ns) or one of a gather.  So
// - a launch with at most one chunk a wave uses none: wave w takes chunk w (1,601 primitives: four gathers 0.202
//   to 0.057 ms, direct 0.060 to 0.027);
// - a launch of RT_QUEUE_SPLIT chunks a wave or more splits the items into RT_QUEUES segments, each with its own
//   counter in its own line.  A workgroup starts on the segment of its XCD (workgroups go to the XCDs in turn), so
//   an XCD's L2 holds one range of the leaf order instead of an eighth of every range, and goes on to the other
//   segments in turn once its own is empty (401,600 primitives x 64 directions: direct 297 to 136 ms; five gathers of
//   1 M primitives 58 to 24).  Larger chunks on one counter did the same for these but cost the diffuse kernel
//   and small scenes up to half their time.
// Looking at a counter before adding to it, past the first segment, made the direct kernel 4 % slower.
// All members are wave-uniform.
struct WaveQueue {
    uint32_t *ctr;
    uint32_t total, chunk, seg, mask, q, left;
    __device__ __forceinline__ WaveQueue(uint32_t *counter, uint32_t total_, uint32_t chunk_)
        : ctr(counter), total(total_), chunk(chunk_) {
        const uint64_t waves = (uint64_t)gridDim.x * (blockDim.x >> 6);
        const bool split = gridDim.x >= RT_QUEUES && (uint64_t)total >= RT_QUEUE_SPLIT * waves * chunk;
        mask = split ? RT_QUEUES - 1u : 0u;
        seg = split ? (total + RT_QUEUES - 1u) / RT_QUEUES : total;
        q = blockIdx.x & mask;
        left = mask + 1u;
        if (waves * chunk >= total) {
            ctr = nullptr;
            q = __builtin_amdgcn_readfirstlane(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6));
        }
    }
    // Adds the chunk to counter word w from lane 0 alone and returns its old value.  (Where all lanes add, the compiler
    // sums them first, in a loop of 64 scalar steps, and one lane adds the sum: 11.3 ns a fetch of a busy counter either
    // way, 12.0 for a 64-bit one, but with four waves on the chip a fetch takes a wave 2.4 us where lane 0's takes 0.4.)
    __device__ __forceinline__ uint32_t fetch(uint32_t *w) const {
        uint32_t x = 0;
        if ((threadIdx.x & 63) == 0) x = __hip_atomic_fetch_add(w, chunk, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return __builtin_amdgcn_readfirstlane(x);
    }
    // The next items [b, e) of this wave; false once all are taken.
    __device__ __forceinline__ bool take(uint32_t &b, uint32_t &e) {
        if (!ctr) {
            const uint64_t x = (uint64_t)q * chunk;
            if (left == 0u || x >= total) return false;
            left = 0u;
            b = (uint32_t)x;
            e = min(b + chunk, total);
            return true;
        }
        while (left != 0u) {
            const uint32_t x = fetch(ctr + q * RT_QUEUE_STRIDE);
            const uint32_t lo = q * seg;
            if (x < seg && lo + x < total) {
                b = lo + x;
                e = min(b + chunk, min(lo + seg, total));
                return true;
            }
            left--;
            q = (q + 1u) & mask;
        }
        return false;
    }
};

template <typename J>
__device__ __forceinline__ uint32_t find_job(const J *jobs, uint32_t njobs, uint32_t item) {
    uint32_t lo = 0, hi = njobs;  // last job with item_begin <= item
    while (hi - lo > 1) {
        uint32_t mid = (lo + hi) >> 1;
        if (jobs[mid].item_begin <= item) lo = mid; else hi = mid;
    }
    return lo;
}

__device__ __forceinline__ uint32_t wave_sum_u32(uint32_t v) {
    for (int off = 32; off >= 1; off >>= 1) v += (uint32_t)__shfl_xor((int)v, off, 64);
    return v;
}

// Sum of k rays of strength s, each added once: k s is exact in double (k < 2^24), then rounded to float.
__device__ __forceinline__ float lit_sum(uint32_t k, float s) { return (float)((double)k * (double)s); }

__device__ __forceinline__ void wave_reduce(ksum &k) {
    for (int off = 32; off >= 1; off >>= 1) {
        float os = __shfl_xor(k.s, off, 64);
        float oc = __shfl_xor(k.c, off, 64);
        k.merge(os, oc);
    }
}

__device__ __forceinline__ bool traced_type(uint32_t t) { return t == 0 || t == 1 || t == 3; }

template <int MK>
__device__ __forceinline__ void add_stats(unsigned long long *, const NoCntT<MK> &, uint32_t) {}
template <int MK>
__device__ __forceinline__ void add_stats(unsigned long long *stats, const TCntT<MK> &c, uint32_t rays) {
    if (stats) {
        atomicAdd(&stats[0], (unsigned long long)c.nodes);
        atomicAdd(&stats[1], (unsigned long long)c.prims);
        atomicAdd(&stats[2], (unsigned long long)rays);
    }
}

// lanes still traversing below which a wave hands out new rays; lanes waiting at a leaf that start a leaf phase;
// stack entries of the resumable traversals kept in LDS (the rest in private memory)
#ifndef RT_REFILL_BELOW
#define RT_REFILL_BELOW 48
#endif
#ifndef RT_LEAF_BATCH
#define RT_LEAF_BATCH 16
#endif
#ifndef RT_DIFFUSE_LDS_STACK
#define RT_DIFFUSE_LDS_STACK 16
#endif

// Resumable closest-hit traversal state of one lane (BVH2), for kernels that refill finished lanes.
struct LaneRay {
    v3f o, d;
    RayPre rp;
    float best_t;
    uint32_t best, ni, budget;
    int sp;
};

__device__ __forceinline__ void lane_start(LaneRay &L, uint32_t nleaf) {
    L.rp = ray_pre(L.o, L.d);
    L.best_t = 1e30f;
    L.best = RT_MISS;
    L.ni = 0;
    L.sp = 0;
    L.budget = nleaf + 8;
}

// Starts the closest-hit trace of L.o, L.d; returns false when it is already complete (a scene with at
// most one traced primitive needs no node steps), as trace_closest() with tstart = 1e30.
template <typename C>
__device__ __forceinline__ bool lane_begin(LaneRay &L, const float4 *recs, uint32_t nleaf, float tmin, uint32_t skip,
                                           C &cnt) {
    lane_start(L, nleaf);
    if (nleaf > 1) return true;
    uint32_t slot_unused;
    if (nleaf == 1) { cnt.prims++; test_leaf<false, C::flags>(recs, 0, L.o, L.d, tmin, skip, L.best_t, L.best, slot_unused); }
    return false;
}

// LDS pointer: accesses compile to ds_read/ds_write (a generic pointer chosen between LDS and private
// memory would compile to slower flat accesses that also wait on vector memory)
#if defined(__HIP_DEVICE_COMPILE__)
typedef __attribute__((address_space(3))) uint32_t lds_u32;
typedef __attribute__((address_space(3))) float lds_f32;
// device-memory values (a pointer read from a job descriptor is generic, and loads through it go the slower flat way)
typedef __attribute__((address_space(1))) uint32_t g_u32;
typedef __attribute__((address_space(1))) float g_f32;
#else
typedef uint32_t lds_u32;
typedef float lds_f32;
typedef uint32_t g_u32;
typedef float g_f32;
#endif

// Traversal entries are inner nodes or leaves (RT_LEAF_BIT).  The stack holds its first LSTK entries in
// LDS (stk, lane stride `stride`) and the rest, up to STK, in the lane's private array ovf (deep stacks
// are rare; LDS per wave bounds the occupancy).  lane_pop() returns true when the stack is empty.
template <int STK, int LSTK>
__device__ __forceinline__ bool lane_pop(LaneRay &L, const lds_u32 *stk, const uint32_t *ovf, uint32_t stride) {
    if (L.sp == 0) return true;
    L.sp--;
    if (LSTK >= STK || L.sp < LSTK) L.ni = stk[(uint32_t)L.sp * stride];
    else L.ni = ovf[L.sp - LSTK];
    return false;
}

// Visit the inner node L.ni: both child boxes against [0, best_t]; the nearer hit child (inner or leaf)
// becomes the next entry and the farther one is pushed.  Returns true when the traversal has ended.
template <int STK, int LSTK, typename C>
__device__ __forceinline__ bool lane_node(const float4 *nodes, uint32_t nleaf, LaneRay &L, lds_u32 *stk, uint32_t *ovf,
                                          uint32_t stride, int *err, C &cnt) {
    if (L.budget-- == 0 || L.ni >= nleaf - 1) {
        atomicOr(err, 2);
        return true;
    }
    cnt.nodes++;
    NodeTest nt = node_test_p(nodes, L.ni, L.rp, L.best_t);
    if (nt.h0 && nt.h1) {
        bool first0 = nt.tn0 <= nt.tn1;
        if (L.sp >= STK) {
            atomicOr(err, 1);
            return true;
        }
        const uint32_t far = first0 ? nt.c1 : nt.c0;
        if (LSTK >= STK || L.sp < LSTK) stk[(uint32_t)L.sp * stride] = far;
        else ovf[L.sp - LSTK] = far;
        L.sp++;
        L.ni = first0 ? nt.c0 : nt.c1;
    } else if (nt.h0) {
        L.ni = nt.c0;
    } else if (nt.h1) {
        L.ni = nt.c1;
    } else {
        return lane_pop<STK, LSTK>(L, stk, ovf, stride);
    }
    return false;
}

// Test the leaf entry L.ni (closest accepted hit, ties to the lower primitive index), then pop.
template <int STK, int LSTK, typename C>
__device__ __forceinline__ bool lane_leaf(const float4 *recs, LaneRay &L, float tmin, uint32_t skip,
                                          const lds_u32 *stk, const uint32_t *ovf, uint32_t stride, C &cnt) {
    cnt.prims++;
    uint32_t slot_unused;
    test_leaf<false, C::flags>(recs, L.ni & ~RT_LEAF_BIT, L.o, L.d, tmin, skip, L.best_t, L.best, slot_unused);
    return lane_pop<STK, LSTK>(L, stk, ovf, stride);
}

// ------------------------------------------------------------------------------------------------
// block tree (rt_types.h): resumable per-lane traversal
// ------------------------------------------------------------------------------------------------
// One lane's ray: origin, direction, reciprocal direction and origin x reciprocal, closest hit so far, the
// next link to visit (RT_BLK_DONE: none left) and the rows in use of the lane's stack.
struct BlkRay {
    v3f o, d;
    float ix, iy, iz, ox, oy, oz;
    uint32_t sx, sy, sz;  // byte selectors of the near bounds (blk_node_step)
    float best_t;
    uint32_t best, ni, sp;
};

// A lane's stack: row r < ROWS in the wave's LDS array (lane stride 4 B, row stride 4 x `stride`), rows from ROWS on
// in the lane's private array `ovf`, whose entry 0 is row ROWS - 2 (see the pushes).  Row 0 holds RT_BLK_DONE, so
// taking the top entry of an empty stack ends the trace without a test of its own.  The tree's depth bounds the
// rows (3 per level): a tree that needs more than RT_STACK has wide links, one that needs more than RT_STACK_WIDE is
// not built.
constexpr int blk_ovf(int rows, int flags) { return ((flags & RT_FL_WIDE) ? RT_STACK_WIDE : RT_STACK) + 5 - rows; }
// The block at a link (whose low bits may hold RT_BLK_REC)
template <int FL>
__device__ __forceinline__ const char *blk_at(const char *blk, uint32_t link) {
    if constexpr ((FL & RT_FL_WIDE) != 0) return blk + ((uint64_t)(link & ~3u) << 4);
    else return blk + (link & ~63u);
}
template <int ROWS>
__device__ __forceinline__ uint32_t blk_pop(BlkRay &L, const lds_u32 *stk, const uint32_t *ovf, uint32_t stride) {
    L.sp--;
    uint32_t v = stk[min(L.sp, (uint32_t)ROWS - 1u) * stride];
    if (L.sp >= (uint32_t)ROWS) v = ovf[L.sp - (ROWS - 2)];
    return v;
}

// Reciprocal of a component of a unit direction for the box tests of a ray that starts within the scene: any value
// within a few ulps does (a box is padded by 4e-6 of the scene's extent); a component near 0 gives a slab +-1e18 times
// as far as the origin is from its planes, beyond every hit.  Rays of other lengths or origins: see k_cast.
__device__ __forceinline__ float blk_rcp(float d) {
    return copysignf(fminf(__builtin_amdgcn_rcpf(fabsf(d)), 1e18f), d);
}

__device__ __forceinline__ void blk_start(BlkRay &L, lds_u32 *stk) {
    L.ox = L.o.x * L.ix;
    L.oy = L.o.y * L.iy;
    L.oz = L.o.z * L.iz;
    L.best_t = 1e30f;
    L.best = RT_MISS;
    L.ni = 0u;
    L.sp = 1u;
    stk[0] = RT_BLK_DONE;
}

// The direction's part of a ray: reciprocals and near-bound selectors
__device__ __forceinline__ void blk_direction(BlkRay &L, float ix, float iy, float iz) {
    L.ix = ix;
    L.iy = iy;
    L.iz = iz;
    L.sx = ix >= 0.f ? 0x0C020C00u : 0x0C060C04u;
    L.sy = iy >= 0.f ? 0x0C020C00u : 0x0C060C04u;
    L.sz = iz >= 0.f ? 0x0C020C00u : 0x0C060C04u;
}

// Lanes set in a wave-uniform mask, counted on the scalar unit (the compiler compares __popcll()'s 64-bit result in
// vector registers)
__device__ __forceinline__ int wave_popc(uint64_t m) {
#if defined(__HIP_DEVICE_COMPILE__)
    int r;
    asm("s_bcnt1_i32_b64 %0, %1" : "=s"(r) : "s"(m) : "scc");
    return r;
#else
    return __popcll(m);
#endif
}

#if defined(__HIP_DEVICE_COMPILE__)
__device__ __forceinline__ int max3i(int a, int b, int c) { int r; asm("v_max3_i32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c)); return r; }
__device__ __forceinline__ int min3i(int a, int b, int c) { int r; asm("v_min3_i32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c)); return r; }
__device__ __forceinline__ int med3i(int a, int b, int c) { int r; asm("v_med3_i32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c)); return r; }
#else
__device__ __forceinline__ int max3i(int a, int b, int c) { return max(max(a, b), c); }
__device__ __forceinline__ int min3i(int a, int b, int c) { return min(min(a, b), c); }
__device__ __forceinline__ int med3i(int a, int b, int c) { return max(min(a, b), min(max(a, b), c)); }
#endif
// a 16-bit half of w read as a half-precision number, times m plus a (one v_fma_mix_f32)
__device__ __forceinline__ float fma_lo(uint32_t w, float m, float a) {
    return fmaf((float)__builtin_bit_cast(_Float16, (uint16_t)w), m, a);
}
__device__ __forceinline__ float fma_hi(uint32_t w, float m, float a) {
    return fmaf((float)__builtin_bit_cast(_Float16, (uint16_t)(w >> 16)), m, a);
}

// Keeps the loads of a node together: the offset they share stays in its register until v has been computed from
// what the last of them returns.  A load into its own address register ends the clause (the compiler puts an s_nop
// before it); other waves' loads then run between this one and the first two and have often evicted the block from the
// vL1D: 20 M rays over 5 M primitives take 7.6 ms that way and 6.7 ms with the three loads in one clause.  Only k_cast
// needs it: the other kernels' registers fall so that the loads stay together, and their order of instructions without
// the hold measured 0.2 % better (k_diffuse).
__device__ __forceinline__ void keep_until(uint32_t offset, float &v) {
#if defined(__HIP_DEVICE_COMPILE__)
    asm("" : "+v"(v) : "v"(offset));
#endif
}

// Visit the node block L.ni: four child boxes against [0, best_t]; the hit children are pushed farthest first and
// the nearest (or, with none hit, the stack's top entry) becomes the next link.
//
// The step is written for the cycles of its vector instructions (see k_diffuse): fma, mul, add and bit operations
// take 2.4 to 3.0 cycles of a SIMD here against 4.1 to 4.5 for min/max, compares, selects, shifts, permutes and
// v_fma_mix and 4.7 for byte conversions (measured at 8 waves per SIMD).  So:
// - a child bound q decodes in t-space as q (s / dir) + (o - ray origin) / dir with the axis' step s.  v_perm takes the
//   bounds nearer the origin of two children from the lower or upper word (the ray's selector says which) as two
//   half-precision numbers q 2^-24 (a byte under a zero byte is that denormal), and v_fma_mix multiplies and adds with
//   the 2^24 in the stored step: 36 instructions, 160 cycles, for the 24 bounds against 54 and 210 with selects, byte
//   conversions and fma;
// - each hit child is one 32-bit key, the bits of its entry distance with the low byte replaced by its link code
//   (v_perm), so the order of four children takes eight min / med / max and no selects of links, and a link is
//   base + the key's low byte;
// - pushes need no branches: the three farthest keys are stored above the stack's top whether they are hits or
//   not (a key that is not lies above the new top).  Keys of missed children are 0x80000000: the smallest as int,
//   so last in the descending order, and above every hit as unsigned, so never the nearest.
template <int ROWS, int FL, bool HOLD = false>
__device__ __forceinline__ void blk_node_step(const char *blk, BlkRay &L, lds_u32 *stk, uint32_t *ovf, uint32_t stride) {
    const uint4 *nd = (const uint4 *)((FL & RT_FL_WIDE) ? blk + ((uint64_t)L.ni << 4) : blk + L.ni);
    const uint4 a = nd[0], b = nd[1], c = nd[2];
    // the entry a pop would take, read beside the node
    const uint32_t sp0 = L.sp;
    uint32_t popv = stk[min(sp0 - 1u, (uint32_t)ROWS - 1u) * stride];
    // the three steps: the word itself, and its two low bytes shifted to the exponent (rt_types.h)
    const float Ax = __uint_as_float(a.w) * L.ix, Ay = fabsf(__uint_as_float(a.w << 23)) * L.iy,
                Az = __uint_as_float(a.w << 15) * L.iz;
    float Bx = fmaf(__uint_as_float(a.x), L.ix, -L.ox);
    const float By = fmaf(__uint_as_float(a.y), L.iy, -L.oy), Bz = fmaf(__uint_as_float(a.z), L.iz, -L.oz);
    if constexpr (HOLD) keep_until(L.ni, Bx);
    float tn[4], tf[4];
#pragma unroll
    for (int k = 0; k < 2; k++) {
        // children k and k + 2: byte k and k + 2 of the bound words
        const uint32_t o = 0x00010001u * (uint32_t)k;
        const uint32_t nx = __builtin_amdgcn_perm(b.y, b.x, L.sx + o), fx = __builtin_amdgcn_perm(b.x, b.y, L.sx + o);
        const uint32_t ny = __builtin_amdgcn_perm(b.w, b.z, L.sy + o), fy = __builtin_amdgcn_perm(b.z, b.w, L.sy + o);
        const uint32_t nz = __builtin_amdgcn_perm(c.y, c.x, L.sz + o), fz = __builtin_amdgcn_perm(c.x, c.y, L.sz + o);
        tn[k] = fmaxf(max3f(fma_lo(nx, Ax, Bx), fma_lo(ny, Ay, By), fma_lo(nz, Az, Bz)), 0.f);
        tf[k] = fminf(min3f(fma_lo(fx, Ax, Bx), fma_lo(fy, Ay, By), fma_lo(fz, Az, Bz)), L.best_t);
        tn[k + 2] = fmaxf(max3f(fma_hi(nx, Ax, Bx), fma_hi(ny, Ay, By), fma_hi(nz, Az, Bz)), 0.f);
        tf[k + 2] = fminf(min3f(fma_hi(fx, Ax, Bx), fma_hi(fy, Ay, By), fma_hi(fz, Az, Bz)), L.best_t);
    }
    int key[4];
    uint32_t n = sp0 - 1u;  // becomes the rows in use after the step
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const bool h = tn[k] <= tf[k];
        // bytes 3..1 of tn over byte k of the codes
        const uint32_t kb = __builtin_amdgcn_perm(__float_as_uint(tn[k]), c.z, 0x07060500u + (uint32_t)k);
        key[k] = h ? (int)kb : (int)0x80000000u;
        n += h ? 1u : 0u;
    }
    const int hi = max3i(key[0], key[1], key[2]), mid = med3i(key[0], key[1], key[2]), lo = min3i(key[0], key[1], key[2]);
    const uint32_t e0 = (uint32_t)max(hi, key[3]), e1 = (uint32_t)med3i(hi, mid, key[3]), e2 = (uint32_t)med3i(mid, lo, key[3]);
    const uint32_t nearest = min(min(min((uint32_t)key[0], (uint32_t)key[1]), (uint32_t)key[2]), (uint32_t)key[3]);
    const uint32_t base = c.w;
    const uint32_t l0 = base + (e0 & 0xFFu), l1 = base + (e1 & 0xFFu), l2 = base + (e2 & 0xFFu);
    if (sp0 + 3u <= (uint32_t)ROWS) {
        lds_u32 *top = stk + sp0 * stride;
        top[0] = l0;
        top[stride] = l1;
        top[2 * stride] = l2;
    } else {
        // near the end of the LDS rows (some lane of a wave in a quarter of the steps): the private array takes the
        // entries, without branches, and LDS its rows among them
        uint32_t *o = ovf + (sp0 - (ROWS - 2));
        o[0] = l0;
        o[1] = l1;
        o[2] = l2;
        if (sp0 < (uint32_t)ROWS) stk[sp0 * stride] = l0;
        if (sp0 + 1u < (uint32_t)ROWS) stk[(sp0 + 1u) * stride] = l1;
        if (sp0 > (uint32_t)ROWS) popv = ovf[sp0 - 1u - (ROWS - 2)];
    }
    L.ni = (int)nearest >= 0 ? base + (nearest & 0xFFu) : popv;
    L.sp = n;
}

// Closest-hit test of the record at link (ties to the lower primitive index)
template <bool CD, int MK>
__device__ __forceinline__ void blk_leaf(const char *blk, const float4 *recs, uint32_t link, BlkRay &L, float tmin,
                                         uint32_t skip, uint32_t &slot) {
    uint32_t id;
    float t;
    const float4 *r = (const float4 *)blk_at<MK>(blk, link);
    // castRays takes a patch or triangle beyond 1e-6 and a voxel at 1e-6 or beyond
    // (CD/src/CollisionDetection_RayTracing.cpp:1562, 1595, 1681)
    if (leaf_hit_at<CD, MK>(r, recs, L.o, L.d, skip, id, t) &&
        (t > tmin || (CD && t == tmin && (__float_as_uint(ldc(r).w) & RT_VOXEL_BIT)))) {
        if (t < L.best_t || (t == L.best_t && L.best != RT_MISS && id < L.best)) {
            L.best_t = t;
            L.best = id;
            slot = link;
        }
    }
}

// The result does not depend on the visiting order: a primitive hit at t <= the final closest t lies in
// boxes whose entry distance is <= t <= every intermediate best_t, so no step culls it, and the tie rule
// is order-free.  The entries visited equal trace_closest()'s up to that order.

static __global__ void k_zero_u64(unsigned long long *p) { *p = 0ull; }

static __global__ void k_zero_queue(uint32_t *p) { p[threadIdx.x] = 0u; }

// ------------------------------------------------------------------------------------------------
// launchers
// ------------------------------------------------------------------------------------------------
static inline uint32_t grid_for(const LaunchCfg &cfg, int ncu, uint32_t total, uint32_t wpb) {
    uint64_t g = (uint64_t)cfg.blocks_per_cu * (uint64_t)ncu;
    uint64_t per_block = (uint64_t)wpb * std::max(cfg.chunk, 1u);
    uint64_t need = (total + per_block - 1) / per_block;
    if (g > need) g = need;
    if (g < 1) g = 1;
    return (uint32_t)g;
}

#define LCHECK()                                                                        \
    do {                                                                                \
        hipError_t e_ = hipGetLastError();                                              \
        if (e_ != hipSuccess) {                                                         \
            set_error(std::string("kernel launch failed: ") + hipGetErrorString(e_));    \
            return -1;                                                                  \
        }                                                                               \
    } while (0)

// LDS stack depth chosen from the BVH depth: 32 entries (32 KB per 256-lane block, 5 blocks per CU)
// when the tree allows it, else 64.
#define PICK_STK(depth, CALL32, CALL64) \
    do {                                 \
        if ((depth) + 1 <= 32) { CALL32; } else { CALL64; } \
    } while (0)

// Runs f(std::integral_constant<int, FL>) for the traversal flags fl (RT_FL_*): one kernel instance per flag set.
template <typename F>
static void with_flags(int fl, F &&f) {
    switch (fl & (RT_FL_MASK | RT_FL_WT)) {
        case 0: f(std::integral_constant<int, 0>{}); break;
        case RT_FL_MASK: f(std::integral_constant<int, RT_FL_MASK>{}); break;
        case RT_FL_WT: f(std::integral_constant<int, RT_FL_WT>{}); break;
        default: f(std::integral_constant<int, RT_FL_MASK | RT_FL_WT>{}); break;
    }
}
// the counting variants always compile the mask tests in (a scene without masks skips them at run time)
static inline int counting_flags(int fl) { return (fl & RT_FL_WT) | RT_FL_MASK; }

}  // namespace rt
