// rt_direct.hip -- direct-ray kernels: occlusion grids, BVH4 packets and non-collimated sources.
#include "rt_traverse.h"

namespace rt {

// two neighbouring words, two neighbouring list entries in one load
typedef uint32_t u32x2_a4 __attribute__((ext_vector_type(2), aligned(4)));
typedef uint32_t u32x4_a8 __attribute__((ext_vector_type(4), aligned(8)));

// Occlusion of one shadow ray through the source's grid: test the primitives binned in the cell of the
// origin's projection with the BVH traversal's predicate (t in (1e-4, 1e30], not the origin primitive) and
// stop at the first hit.  Non-periodic scenes only (the grid is not built otherwise).
// Candidate range [b, e) of the grid cell holding origin o's projection.
__device__ __forceinline__ void grid_cell(const SunGrid &G, v3f o, uint32_t &b, uint32_t &e) {
    const float qu = o.x * G.u[0] + o.y * G.u[1] + o.z * G.u[2];
    const float qv = o.x * G.v[0] + o.y * G.v[1] + o.z * G.v[2];
    float fx = floorf((qu - G.g0u) * G.inv_cs), fy = floorf((qv - G.g0v) * G.inv_cs);
    const int cx = fx < 0.f ? 0 : (fx > (float)(G.nx - 1) ? (int)(G.nx - 1) : (int)fx);
    const int cy = fy < 0.f ? 0 : (fy > (float)(G.ny - 1) ? (int)(G.ny - 1) : (int)fy);
    const uint32_t c = (uint32_t)cy * G.nx + (uint32_t)cx;
    const u32x2_a4 be = *(const u32x2_a4 *)(G.start + c);
    b = be.x - G.sbase;
    e = be.y - G.sbase;
}

// Candidates p and p + 1 (when p + 1 < e) of a cell list: is either accepted as an occluder?  Both
// candidates' loads are issued before either test (the list entry -> record chain is latency-bound); a slot
// that is out of the list or unfilled loads record 0 and is ignored.  An entry is one 8-byte load (slot and
// key), and a record's fourth float4 (the patch plane normal, the mask descriptor) is loaded only for the
// entries flagged as needing it, so a triangle candidate costs four vector loads instead of six.  A
// candidate whose depth key (an upper bound of the depth of its points along the source direction, padded
// by 1e-5 of the scene's largest coordinate) is below the ray origin's depth lies wholly behind the origin:
// no FP32 hit of it can have t > 1e-4 (the FP32 errors of t, of the key and of the depth are a few ulps of
// that coordinate), so it is skipped without loading its record.
// Returns 1 when a candidate occludes the ray, 2 when the list holds no further occluder (its next key is below
// the origin's depth), else 0.
template <typename C>
__device__ __forceinline__ int grid_pair(const uint2 *ents, float depth, const float4 *recs, uint32_t nleaf,
                                         uint32_t p, uint32_t e, v3f o, v3f d, uint32_t skip, C &cnt) {
    const bool two = p + 1 < e;
    const uint2 e0 = ents[p];
    const uint2 e1 = two ? ents[p + 1] : make_uint2(RT_MISS, __float_as_uint(-INFINITY));
    const float key0 = __uint_as_float(e0.y), key1 = __uint_as_float(e1.y);
    const uint32_t k0 = e0.x & RT_GRID_SLOT, k1 = e1.x & RT_GRID_SLOT;
    const bool v0 = e0.x != RT_MISS && k0 < nleaf && !(key0 < depth);
    const bool v1 = e1.x != RT_MISS && k1 < nleaf && !(key1 < depth);
    const float4 *q0 = recs + (size_t)(v0 ? k0 : 0u) * 4, *q1 = recs + (size_t)(v1 ? k1 : 0u) * 4;
    const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
    const float4 a0 = ldc(q0), a1 = ldc(q0 + 1), a2 = ldc(q0 + 2);
    const float4 a3 = (v0 && (e0.x & RT_GRID_REC3)) ? ldc(q0 + 3) : zero;
    const float4 b0 = ldc(q1), b1 = ldc(q1 + 1), b2 = ldc(q1 + 2);
    const float4 b3 = (v1 && (e1.x & RT_GRID_REC3)) ? ldc(q1 + 3) : zero;
    const uint32_t ta = __float_as_uint(a0.w), tb = __float_as_uint(b0.w);
    float t0, t1, ua0, ub0, ua1, ub1;
    bool h0 = v0 && isect_rec_uv<false, C::wt>(a0, a1, a2, a3, (ta & RT_PATCH_BIT) != 0, o, d, t0, ua0, ub0) &&
              (ta & RT_ID_BITS) != skip && t0 > 1e-4f && t0 <= 1e30f;
    bool h1 = v1 && isect_rec_uv<false, C::wt>(b0, b1, b2, b3, (tb & RT_PATCH_BIT) != 0, o, d, t1, ua1, ub1) &&
              (tb & RT_ID_BITS) != skip && t1 > 1e-4f && t1 <= 1e30f;
    if (C::mask && h0 && (ta & RT_MASK_BIT))
        h0 = mask_hit_opaque(recs, __float_as_uint(a3.w), (ta & RT_PATCH_BIT) != 0, ua0, ub0, a1.w, a2.w);
    if (C::mask && h1 && (tb & RT_MASK_BIT))
        h1 = mask_hit_opaque(recs, __float_as_uint(b3.w), (tb & RT_PATCH_BIT) != 0, ua1, ub1, b1.w, b2.w);
    cnt.prims += (v0 ? 1u : 0u) + ((v1 && !h0) ? 1u : 0u);  // the tests a one-at-a-time scan makes
    if (h0 || h1) return 1;
    return (!(key0 >= depth) || (two && !(key1 >= depth))) ? 2 : 0;
}

// ------------------------------------------------------------------------------------------------
// direct rays
// ------------------------------------------------------------------------------------------------
// COUNT: the counting variant (stats != nullptr) traces every ray on its own (per-lane LDS stack, or the
// occlusion grid's lists when the job has one) so the counters hold single-ray node visits and primitive
// tests -- the algorithmic work per ray -- rather than the packet's visits.  The other variant takes the
// launches without grids and walks the BVH4 in packets.  Both make the same occlusion decision for every ray.
#ifndef RT_DIRECT_REFILL
#define RT_DIRECT_REFILL 24
#endif
// Origin of direct ray r of primitive i (stratified sample, then the texture-mask rejection when the
// primitive has a mask: mdi = its descriptor, RT_MISS = none); false when the ray is dropped.
__device__ __forceinline__ bool direct_origin(const float4 *recs, uint32_t mdi, uint32_t i, uint32_t r, uint32_t d,
                                              uint32_t seed, bool patch, float &spx, float &spy) {
    uint32_t st;
    direct_sample_st(i, r % d, r / d, d, seed, patch, spx, spy, st);
    return mdi == RT_MISS || origin_mask(recs, mdi, patch, false, st, spx, spy);
}

// Waves per SIMD the compiler must fit the unmasked direct kernel into: 7 (72 VGPRs, 6 without the bound)
// takes the orchard's 64-sun direct pass from 407 to 393 ms; 8 spills in the candidate loop (419 ms)
#ifndef RT_DIRECT_WAVES_PER_EU
#define RT_DIRECT_WAVES_PER_EU 7
#endif
template <int WPB, int STK, bool COUNT, int MK>
__global__ __launch_bounds__(WPB * 64, (COUNT || MK) ? 1 : RT_DIRECT_WAVES_PER_EU) void k_direct(const DirectJob *__restrict__ jobs, uint32_t njobs, uint32_t total,
                                                     uint32_t *counter, uint32_t chunk, int *err,
                                                     unsigned long long *stats) {
    __shared__ uint32_t wstk_all[COUNT ? STK * WPB * 64 : STK * WPB];
    __shared__ uint32_t wstk4_all[COUNT ? 1 : RT_WSTK4 * WPB];
    uint32_t *wstk = COUNT ? wstk_all + threadIdx.x : wstk_all + (threadIdx.x >> 6) * STK;
    uint32_t *wstk4 = COUNT ? wstk4_all : wstk4_all + (threadIdx.x >> 6) * RT_WSTK4;
    const uint32_t lane = threadIdx.x & 63;
    Cnt<COUNT, MK> cnt{};
    uint32_t nray = 0;
    WaveQueue wq(counter, total, chunk);
    for (uint32_t first, end; wq.take(first, end);) {
        for (uint32_t item = first; item < end; ++item) {
            // job, scene and primitive data are wave-uniform: scalar loads keep them out of VGPRs
            uint32_t j = find_job(jobs, njobs, item);
            const DirectJob &J = jobs[j];
            const DevScene &sc = *ldu(&J.sc);
            uint32_t i = item - ldu(&J.item_begin);
            const uint32_t *jorder = ldu(&J.order);
            if (jorder) i = ldu(jorder + i);
            i = __builtin_amdgcn_readfirstlane(i);
            uint32_t ty = ldu(ldu(&sc.type) + i);
            float sum_out = 0.f;
            bool top = true;
            const SunGrid *grid = COUNT ? ldu(&J.grid) : nullptr;
            const float4 *recs = ldu(&sc.rec);
            const uint32_t *mdesc = ldu(&sc.mdesc);
            const uint32_t mdi = (MK && mdesc) ? ldu(mdesc + i) : RT_MISS;
            if (traced_type(ty)) {
                float4 n4 = ldu(ldu(&sc.nrm) + i);
                v3f n = mk3(n4.x, n4.y, n4.z);
                uint32_t tw = __float_as_uint(n4.w);
                v3f dir = nrm3(mk3(ldu(&J.sdir[0]), ldu(&J.sdir[1]), ldu(&J.sdir[2])));
                uint32_t d = ldu(&J.d), Nrays = d * d;
                float strength = rdiv(fabsf(dot3(n, dir)), (float)Nrays);
                top = dot3(dir, n) > 0.0f;
                if (!(tw == 3 || (!top && tw == 0))) {
                    bool patch = ty == 0 || ty == 3;
                    float tm[12];
                    const float *Tp = ldu(&sc.T) + (size_t)i * 16;
#pragma unroll
                    for (int q = 0; q < 12; q++) tm[q] = ldu(Tp + q);
                    // every ray of the primitive carries the same strength: the lit rays are counted and the
                    // sum is count x strength, rounded once (exact up to that rounding)
                    uint32_t lit = 0;
                    const uint32_t seed = ldu(&J.seed);
                    if (COUNT && grid) {
                        // Occlusion grid: each lane scans its ray's cell list two candidates per step.  A lane
                        // whose ray ends (occluder found, or list exhausted: lit) takes the primitive's next
                        // ray; idle lanes are refilled together once fewer than RT_DIRECT_REFILL lanes still
                        // scan (every ray is tested exactly as on its own; only the ray -> lane assignment
                        // and the summation grouping differ).
                        const SunGrid &G = *grid;
                        const uint2 *ents = G.ents;
                        const uint32_t nleaf = ldu(&sc.nleaf);
                        const float gw0 = G.w[0], gw1 = G.w[1], gw2 = G.w[2];
                        uint32_t r = lane, pc = 0, pe = 0;
                        v3f o = mk3(0.f, 0.f, 0.f);
                        float depth = 0.f;  // origin depth along the source direction
                        bool act = r < Nrays;
                        if (act) {
                            float spx, spy;
                            act = direct_origin(recs, mdi, i, r, d, seed, patch, spx, spy);
                            o = xform3(tm, spx, spy, 0.0f);
                            grid_cell(G, o, pc, pe);
                            depth = o.x * gw0 + o.y * gw1 + o.z * gw2;
                            cnt.nodes++;
                            nray++;
                        }
                        uint32_t qnext = min(64u, Nrays);
                        while (true) {
                            const uint32_t floor_lanes = qnext < Nrays ? RT_DIRECT_REFILL : 1u;
                            while (true) {
                                if (act) {
                                    const int res = pc >= pe ? 2
                                                             : grid_pair(ents, depth, recs, nleaf, pc, pe, o, dir, i, cnt);
                                    if (res == 2) lit++;
                                    if (res != 0) act = false;
                                    else pc += 2;
                                }
                                if ((uint32_t)__popcll(__ballot(act)) < floor_lanes) break;
                            }
                            const uint64_t idle = __ballot(!act);
                            if (qnext >= Nrays) {
                                if (idle == ~0ull) break;
                                continue;
                            }
                            const uint32_t rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(idle >> 32),
                                                                            __builtin_amdgcn_mbcnt_lo((uint32_t)idle, 0u));
                            const uint32_t take = min((uint32_t)__popcll(idle), Nrays - qnext);
                            if (!act && rank < take) {
                                r = qnext + rank;
                                float spx, spy;
                                act = direct_origin(recs, mdi, i, r, d, seed, patch, spx, spy);
                                o = xform3(tm, spx, spy, 0.0f);
                                grid_cell(G, o, pc, pe);
                                depth = o.x * gw0 + o.y * gw1 + o.z * gw2;
                                cnt.nodes++;
                                nray++;
                            }
                            qnext += take;
                        }
                    } else {
                        for (uint32_t base = 0; base < Nrays; base += 64) {
                            uint32_t r = base + lane;
                            bool need = r < Nrays;
                            v3f o = mk3(0.f, 0.f, 0.f);
                            if (need) {
                                float spx, spy;
                                need = direct_origin(recs, mdi, i, r, d, seed, patch, spx, spy);
                                o = xform3(tm, spx, spy, 0.0f);
                                nray++;
                            }
                            bool occl;
                            if (COUNT) occl = need && occluded<STK>(sc, o, dir, 1e-4f, i, wstk, WPB * 64, err, cnt);
                            else occl = packet_occluded<STK>(sc, o, dir, 1e-4f, i, need, wstk, wstk4, err, cnt);
                            if (need && !occl) lit++;
                        }
                    }
                    sum_out = lit_sum(wave_sum_u32(lit), strength);
                }
            }
            if (lane == 0) {
                float *out = ldu(&J.out);
                out[(size_t)i * 2 + 0] = top ? sum_out : 0.f;
                out[(size_t)i * 2 + 1] = top ? 0.f : sum_out;
            }
        }
    }
    add_stats(stats, cnt, nray);
}

// Collimated direct rays when every job of the launch has an occlusion grid.  The lanes of a wave are refilled
// across the primitives of a job, as the diffuse kernel refills them: a lane whose ray ends takes the next
// ray of the open primitive, or of the next primitive of the wave's work queue, so no lane idles until the
// longest ray of one primitive ends.  Each primitive with rays in flight holds a slot of the wave's ring in
// LDS that counts its lit rays; the primitive's sums are written once its last ray has ended.  A job change
// (another direction, grid and output) waits until the rays in flight have ended.  Every ray is tested
// exactly as in k_direct, and the sums are the same count x strength.
// The vector ALU bounds it (1,001,600 primitives x 225 rays x 64 directions, 14.4 G rays: 2.2e11 wave instructions in
// 302 ms, one per SIMD every 3.4 cycles; 401,600 primitives: 122 ms), so lanes must not idle and work that decides
// nothing must not run:
// - rays are generated up to 64 at a time with every lane active, into the wave's LDS queue, together with the first
//   two entries of their cell's list; a ray with nothing above it is counted lit there and never queued;
// - a lane tests one candidate a step (two a step tested the second in vain whenever the first hit), and the
//   origin's own entry, known by its leaf slot, is passed over without loading its record;
// - a cell's start and end are one 8-byte load and a pair of entries one 16-byte load (2.5e9 load instructions
//   where two candidates a step took 3.8e9).
// The smaller batch's direct pass took 136 ms with two candidates a step and rays generated by the lanes being refilled,
// 121 ms so.  Refills start below RT_DQ_REFILL scanning lanes (32 to 56 swept: 40 best by 2 %).
// The lists are sorted by descending key (SunGrid), which the scan's end relies on.
#define RT_DQ_SLOTS 8
#ifndef RT_DQ_REFILL
#define RT_DQ_REFILL 40
#endif
template <int WPB, int MK>
__global__ __launch_bounds__(WPB * 64, MK ? 1 : RT_DIRECT_WAVES_PER_EU) void k_direct_q(const DirectJob *__restrict__ jobs,
                                                                                        uint32_t njobs, uint32_t total,
                                                                                        uint32_t *counter, uint32_t chunk) {
    typedef Cnt<false, MK> C;
    __shared__ uint32_t ring_all[3 * RT_DQ_SLOTS * WPB];  // per wave: lit count, primitive, strength of each slot
    __shared__ float4 qo_all[64 * WPB];                   // queued rays: origin, depth along the source direction,
    __shared__ uint4 qe_all[64 * WPB];                    // the next two list entries
    __shared__ uint2 qp_all[64 * WPB];                    // and the list positions after them
    uint32_t *lit = ring_all + (threadIdx.x >> 6) * 3 * RT_DQ_SLOTS;
    uint32_t *sprim = lit + RT_DQ_SLOTS;
    float *sstr = (float *)(lit + 2 * RT_DQ_SLOTS);
    const uint32_t lane = threadIdx.x & 63, qbase = threadIdx.x & ~63u;
    // work queue (wave-uniform)
    WaveQueue wq(counter, total, chunk);
    uint32_t it = 0, it_end = 0;
    bool drained = false;
    // job (wave-uniform): loaded when the wave first takes one of its items
    uint32_t jcur = RT_MISS, jbegin = 0, jend = 0, d = 0, Nrays = 0, seed = 0, nleaf = 0;
    const DevScene *scp = nullptr;
    const SunGrid *grid = nullptr;
    const uint32_t *order = nullptr;
    const uint2 *ents = nullptr;
    const float4 *recs = nullptr;
    bool leaf_items = false;
    float *out = nullptr;
    v3f dir = mk3(0.f, 0.f, 0.f);
    // open primitive, the batch of its rays in the queue (wave-uniform) and the slots in use (bit mask; a slot's
    // bit 8 + k: its sums are lit from the top)
    uint32_t op_i = 0, op_own = RT_MISS, op_next = 0, op_cnt = 0, op_slot = 0, op_mdi = RT_MISS, slots = 0;
    uint32_t q_next = 0, q_cnt = 0;
    bool op_patch = false;
    // lane: its ray (origin, depth, current and following list entry, next list position and end), primitive, the
    // primitive's leaf slot and ring slot
    bool act = false;
    v3f o = mk3(0.f, 0.f, 0.f);
    float depth = 0.f;
    uint32_t ex = RT_MISS, ek = 0, nx = RT_MISS, nk = 0, pn = 0, pe = 0, my_i = 0, my_own = 0, my_slot = 0;
    while (true) {
        bool blocked = false;
        while (true) {
            const uint64_t idle = __builtin_amdgcn_ballot_w64(!act);
            if (idle == 0) break;
            if (q_next == q_cnt) {
                if (op_next == op_cnt) {
                    // the open primitive has no rays left: open the next item of the queue
                    if (it == it_end) {
                        if (drained) break;
                        if (!wq.take(it, it_end)) { drained = true; it = it_end = 0; break; }
                    }
                    if (jcur == RT_MISS || it < jbegin || it >= jend) {
                        if (idle != ~0ull || (slots & 0xFFu) != 0) { blocked = true; break; }
                        jcur = find_job(jobs, njobs, it);
                        const DirectJob &J = jobs[jcur];
                        jbegin = ldu(&J.item_begin);
                        jend = jcur + 1 < njobs ? ldu(&jobs[jcur + 1].item_begin) : total;
                        scp = ldu(&J.sc);
                        grid = ldu(&J.grid);
                        order = ldu(&J.order);
                        out = ldu(&J.out);
                        d = ldu(&J.d);
                        Nrays = d * d;
                        seed = ldu(&J.seed);
                        dir = nrm3(mk3(ldu(&J.sdir[0]), ldu(&J.sdir[1]), ldu(&J.sdir[2])));
                        nleaf = ldu(&scp->nleaf);
                        ents = ldu(&grid->ents);
                        recs = ldu(&scp->rec);
                        leaf_items = order != nullptr && order == ldu(&scp->order);
                    }
                    if ((slots & 0xFFu) == 0xFFu) { blocked = true; break; }
                    uint32_t i = it - jbegin;
                    op_own = leaf_items && i < nleaf ? i : RT_MISS;
                    if (order) i = ldu(order + i);
                    i = __builtin_amdgcn_readfirstlane(i);
                    it++;
                    const uint32_t ty = ldu(ldu(&scp->type) + i);
                    const float4 n4 = ldu(ldu(&scp->nrm) + i);
                    const v3f n = mk3(n4.x, n4.y, n4.z);
                    const uint32_t tw = __float_as_uint(n4.w);
                    const bool top = dot3(dir, n) > 0.0f;
                    if (!traced_type(ty) || tw == 3 || (!top && tw == 0)) {
                        if (lane == 0) { out[(size_t)i * 2] = 0.f; out[(size_t)i * 2 + 1] = 0.f; }
                        continue;
                    }
                    const uint32_t sl = (uint32_t)__builtin_ctz(~slots & 0xFFu);
                    slots |= (1u << sl) | (top ? (0x100u << sl) : 0u);
                    lit[sl] = 0u;
                    sprim[sl] = i;
                    sstr[sl] = rdiv(fabsf(dot3(n, dir)), (float)Nrays);
                    const uint32_t *mdesc = ldu(&scp->mdesc);
                    op_mdi = (MK && mdesc) ? ldu(mdesc + i) : RT_MISS;
                    op_i = i;
                    op_next = 0;
                    op_cnt = Nrays;
                    op_slot = sl;
                    op_patch = ty == 0 || ty == 3;
                    continue;
                }
                // generate the next batch of the open primitive's rays; those whose cell lists nothing above them
                // are lit, the others enter the queue with their first two entries
                const uint32_t left = op_cnt - op_next, batches = (left + 63u) >> 6;
                const uint32_t cnt = (left + batches - 1u) / batches, r = op_next + lane;
                op_next += cnt;
                bool islit = false, enter = false;
                v3f p = mk3(0.f, 0.f, 0.f);
                float pd = 0.f;
                uint4 e2 = make_uint4(RT_MISS, 0u, RT_MISS, 0u);
                uint32_t b = 0, e = 0;
                if (lane < cnt) {
                    float spx, spy;
                    if (direct_origin(recs, op_mdi, op_i, r, d, seed, op_patch, spx, spy)) {
                        float tm[12];
                        const float *Tp = ldu(&scp->T) + (size_t)op_i * 16;
#pragma unroll
                        for (int q = 0; q < 12; q++) tm[q] = ldu(Tp + q);
                        p = xform3(tm, spx, spy, 0.0f);
                        grid_cell(*grid, p, b, e);
                        pd = p.x * grid->w[0] + p.y * grid->w[1] + p.z * grid->w[2];
                        if (b < e) {
                            const u32x4_a8 v = *(const u32x4_a8 *)(ents + b);
                            e2 = make_uint4(v.x, v.y, v.z, v.w);
                            enter = __uint_as_float(e2.y) >= pd;
                            if (b + 1 >= e) e2.z = RT_MISS;
                        }
                        islit = !enter;
                    }
                }
                const uint64_t mlit = __builtin_amdgcn_ballot_w64(islit), menter = __builtin_amdgcn_ballot_w64(enter);
                if (lane == 0 && mlit) atomicAdd(&lit[op_slot], (uint32_t)wave_popc(mlit));
                if (enter) {
                    const uint32_t at = qbase + __builtin_amdgcn_mbcnt_hi((uint32_t)(menter >> 32),
                                                                          __builtin_amdgcn_mbcnt_lo((uint32_t)menter, 0u));
                    qo_all[at] = make_float4(p.x, p.y, p.z, pd);
                    qe_all[at] = e2;
                    qp_all[at] = make_uint2(b + 2, e);
                }
                q_next = 0;
                q_cnt = (uint32_t)wave_popc(menter);
                __builtin_amdgcn_wave_barrier();
                continue;
            }
            const uint32_t rank =
                __builtin_amdgcn_mbcnt_hi((uint32_t)(idle >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)idle, 0u));
            const uint32_t take = min((uint32_t)wave_popc(idle), q_cnt - q_next);
            if (!act && rank < take) {
                const uint32_t at = qbase + q_next + rank;
                const float4 q = qo_all[at];
                const uint4 e2 = qe_all[at];
                const uint2 pp = qp_all[at];
                o = mk3(q.x, q.y, q.z);
                depth = q.w;
                ex = e2.x; ek = e2.y; nx = e2.z; nk = e2.w;
                pn = pp.x;
                pe = pp.y;
                my_i = op_i;
                my_own = op_own;
                my_slot = op_slot;
                act = true;
            }
            q_next += take;
        }
        // write the sums of the primitives none of whose rays remain (the open one once all its rays are out)
        for (uint32_t pend = slots & 0xFFu; pend != 0u; pend &= pend - 1u) {
            const uint32_t sl = (uint32_t)__builtin_ctz(pend);
            if (sl == op_slot && (op_next < op_cnt || q_next < q_cnt)) continue;
            if (__builtin_amdgcn_ballot_w64(act && my_slot == sl) != 0) continue;
            const uint32_t i = sprim[sl];
            const float sum = lit_sum(lit[sl], sstr[sl]);
            const bool top = (slots >> (8 + sl)) & 1u;
            if (lane == 0) {
                out[(size_t)i * 2] = top ? sum : 0.f;
                out[(size_t)i * 2 + 1] = top ? 0.f : sum;
            }
            slots &= ~((1u << sl) | (0x100u << sl));
        }
        if (__builtin_amdgcn_ballot_w64(act) == 0) {
            if (drained && op_next == op_cnt && q_next == q_cnt && (slots & 0xFFu) == 0u) break;
            continue;
        }
        // trace until fewer than RT_DQ_REFILL lanes scan (all of them when no ray can be handed out)
        const uint32_t floor_lanes =
            (blocked || (drained && op_next == op_cnt && q_next == q_cnt)) ? 1u : RT_DQ_REFILL;
        do {
            if (act) {
                // the entries after this pair, while its last record is on the way
                u32x4_a8 f = {RT_MISS, 0u, RT_MISS, 0u};
                const bool fetch = nx == RT_MISS && pn < pe;
                if (fetch) f = *(const u32x4_a8 *)(ents + pn);
                const uint32_t k = ex & RT_GRID_SLOT;
                bool hit = false;
                if (k != my_own && k < nleaf) {
                    const float4 *q = recs + (size_t)k * 4;
                    const float4 a0 = ldc(q), a1 = ldc(q + 1), a2 = ldc(q + 2);
                    const float4 a3 = (ex & RT_GRID_REC3) ? ldc(q + 3) : make_float4(0.f, 0.f, 0.f, 0.f);
                    const uint32_t tag = __float_as_uint(a0.w);
                    float t, ua, ub;
                    hit = isect_rec_uv<false, C::wt>(a0, a1, a2, a3, (tag & RT_PATCH_BIT) != 0, o, dir, t, ua, ub) &&
                          (tag & RT_ID_BITS) != my_i && t > 1e-4f && t <= 1e30f;
                    if (C::mask && hit && (tag & RT_MASK_BIT))
                        hit = mask_hit_opaque(recs, __float_as_uint(a3.w), (tag & RT_PATCH_BIT) != 0, ua, ub, a1.w, a2.w);
                }
                if (fetch) {
                    ex = f.x; ek = f.y;
                    nx = pn + 1 < pe ? f.z : RT_MISS;
                    nk = f.w;
                    pn += 2;
                } else {
                    ex = nx; ek = nk;  // RT_MISS when the list has ended
                    nx = RT_MISS;
                }
                if (hit) act = false;
                else if (ex == RT_MISS || !(__uint_as_float(ek) >= depth)) {
                    atomicAdd(&lit[my_slot], 1u);
                    act = false;
                }
            }
        } while ((uint32_t)wave_popc(__builtin_amdgcn_ballot_w64(act)) >= floor_lanes);
    }
}

// Occlusion of a ray towards a non-collimated source, literally as the reference loop
// (direct_raygen.comp:603-628 without glass covers): closest hit, periodic wrap when a face is strictly
// nearer, and a hit at or beyond the distance from the original origin to the source centre does not block.
template <int STK, typename C>
__device__ __forceinline__ bool source_occluded(const DevScene &sc, v3f o, v3f d, uint32_t skip, float dist0,
                                                uint32_t *stk, uint32_t stride, int *err, C &cnt) {
    v3f cur = o;
    for (int step = 0; step < 32; ++step) {
        float t;
        uint32_t slot;
        uint32_t h = trace_closest<false, STK>(sc, cur, d, 1e-4f, skip, 1e30f, t, slot, stk, stride, err, cnt);
        if (sc.nbbox) {
            float bt = nearest_face(sc, cur, d, t);
            if (bt > 0.f) { cur = wrap_at(sc, cur, d, bt); continue; }
        }
        if (h == RT_MISS) return false;
        return t < dist0;
    }
    return false;
}

// The same over the block tree.  Without periodic faces the question is only whether some accepted hit lies before
// dist0: the trace starts with dist0 as its closest distance and ends at the first hit.
template <int ROWS, int MK>
__device__ __forceinline__ bool source_occluded_blk(const DevScene &sc, const char *blk, const float4 *recs, v3f o, v3f d,
                                                    uint32_t skip, float dist0, lds_u32 *stk, uint32_t *ovf,
                                                    uint32_t stride, uint32_t max_steps, int *err) {
    if (!(dist0 > 0.f)) return false;
    const bool any = sc.nbbox == 0;
    BlkRay L;
    L.o = o;
    L.d = d;
    blk_direction(L, blk_rcp(d.x), blk_rcp(d.y), blk_rcp(d.z));
    for (int step = 0; step < 32; ++step) {
        blk_start(L, stk);
        if (any) L.best_t = fminf(L.best_t, dist0);
        uint32_t left = max_steps;
        while (L.ni != RT_BLK_DONE) {
            while (!(L.ni & RT_BLK_REC) && left != 0u) {
                blk_node_step<ROWS, MK>(blk, L, stk, ovf, stride);
                left--;
            }
            if (left == 0u) {
                atomicOr(err, 2);
                return false;
            }
            if (L.ni == RT_BLK_DONE) break;
            uint32_t slot_unused;
            blk_leaf<false, MK>(blk, recs, L.ni, L, 1e-4f, skip, slot_unused);
            if (any && L.best != RT_MISS) return true;
            L.ni = blk_pop<ROWS>(L, stk, ovf, stride);
        }
        if (any) return false;
        const float bt = nearest_face(sc, L.o, d, L.best_t);
        if (!(bt > 0.f)) return L.best != RT_MISS && L.best_t < dist0;
        L.o = wrap_at(sc, L.o, d, bt);
    }
    return false;
}

// Direct rays towards sphere, sun-sphere, rectangle and disk sources (direct_raygen.comp:482-561): one
// wave per (job, primitive), d*d stratified origins as k_direct, per-ray direction, strength and lit face,
// per-lane closest-hit traversal.  Items [item_lo, item_lo + nitems) of jobs whose item_begin ascend.
// BLK: over the block tree (every launch that does not count, unless the scene lacks one or its links are wide).  The
// binary tree's stacks take 32 or 64 KB of LDS a workgroup, two waves a SIMD at 64, and its trace goes on to the closest
// hit; the block tree's take RT_SRC_ROWS rows, 17 KB (24 rows: the same time), and four waves a SIMD fit.  Three lamps
// over 20,100 primitives x 256 rays, the whole pass by pass solve: 9.29 to 8.57 ms.  The quadrature of a sphere's
// strength, 200 divisions a ray, is the larger part of what is left.
#ifndef RT_SRC_ROWS
#define RT_SRC_ROWS 17
#endif
template <int STK, bool COUNT, int MK, bool BLK>
__global__ __launch_bounds__(256) void k_direct_src(const DirectJob *__restrict__ jobs, uint32_t njobs, uint32_t item_lo,
                                                    uint32_t nitems, uint32_t *counter, int *err,
                                                    unsigned long long *stats) {
    __shared__ uint32_t stk_all[(BLK ? RT_SRC_ROWS : STK) * 256];
    uint32_t *stk = stk_all + threadIdx.x;
    uint32_t ovf[BLK ? blk_ovf(RT_SRC_ROWS, MK) : 1];
    const uint32_t lane = threadIdx.x & 63;
    Cnt<COUNT, MK> cnt{};
    uint32_t nray = 0;
    WaveQueue wq(counter, nitems, 1u);
    for (uint32_t first, end; wq.take(first, end);) {
        const uint32_t item = item_lo + first;
        const DirectJob &J = jobs[find_job(jobs, njobs, item)];
        const DevScene &sc = *J.sc;
        uint32_t i = item - J.item_begin;
        if (J.order) i = J.order[i];
        const uint32_t ty = sc.type[i];
        ksum top_acc, bot_acc;
        top_acc.init();
        bot_acc.init();
        if (traced_type(ty)) {
            const float4 n4 = sc.nrm[i];
            const v3f n = mk3(n4.x, n4.y, n4.z);
            const uint32_t tw = __float_as_uint(n4.w);
            const bool patch = ty == 0 || ty == 3;
            const uint32_t d = J.d, Nrays = d * d;
            float tm[12];
            const float *Tp = sc.T + (size_t)i * 16;
#pragma unroll
            for (int q = 0; q < 12; q++) tm[q] = Tp[q];
            const v3f sp3 = mk3(J.sdir[0], J.sdir[1], J.sdir[2]);
            for (uint32_t base = 0; base < Nrays; base += 64) {
                const uint32_t r = base + lane;
                if (r >= Nrays) continue;
                float spx, spy;
                uint32_t st;
                direct_sample_st(i, r % d, r / d, d, J.seed, patch, spx, spy, st);
                const uint32_t mdi = (MK && sc.mdesc) ? sc.mdesc[i] : RT_MISS;
                if (MK && mdi != RT_MISS && !origin_mask(sc.rec, mdi, patch, false, st, spx, spy)) continue;
                const v3f o = xform3(tm, spx, spy, 0.0f);
                for (uint32_t k = 0; k < J.skip_draws; k++) (void)rnd24(st);
                nray++;
                v3f dir;
                float strength;
                if (!source_ray(J.stype, J.sdir, J.width, J.rot, o, n, Nrays, st, dir, strength)) continue;
                const bool top = dot3(dir, n) > 0.0f;
                if (tw == 3 || (!top && tw == 0)) continue;
                const v3f dv = sub3(sp3, o);
                const float dist0 = rsqrt_cr(dot3(dv, dv));
                if constexpr (BLK) {
                    if (source_occluded_blk<RT_SRC_ROWS, MK>(sc, (const char *)sc.blk, sc.rec, o, dir, i, dist0,
                                                             (lds_u32 *)stk_all + threadIdx.x, ovf, 256u,
                                                             sc.nnode4 + 8u, err))
                        continue;
                } else if (source_occluded<STK>(sc, o, dir, i, dist0, stk, 256u, err, cnt)) continue;
                if (top) top_acc.add(strength);
                else bot_acc.add(strength);
            }
        }
        wave_reduce(top_acc);
        wave_reduce(bot_acc);
        if (lane == 0) {
            J.out[(size_t)i * 2 + 0] = top_acc.value();
            J.out[(size_t)i * 2 + 1] = bot_acc.value();
        }
    }
    add_stats(stats, cnt, nray);
}

template <int MK>
static int launch_direct_t(const DirectJob *jobs, uint32_t njobs, uint32_t total, uint32_t depth, uint32_t *counter,
                           int *err, unsigned long long *stats, const LaunchCfg &cfg, int ncu, hipStream_t st,
                           bool grids) {
    if (total == 0) return 0;
    const uint32_t ch = std::max(cfg.chunk, 1u);
    k_zero_queue<<<1, RT_QUEUE_WORDS, 0, st>>>(counter);
    uint32_t wpb = cfg.waves_per_block;
    uint32_t g = grid_for(cfg, ncu, total, wpb);
    if (grids && !stats) {
        switch (wpb) {
            case 1: k_direct_q<1, MK><<<g, 64, 0, st>>>(jobs, njobs, total, counter, ch); break;
            case 2: k_direct_q<2, MK><<<g, 128, 0, st>>>(jobs, njobs, total, counter, ch); break;
            default: k_direct_q<4, MK><<<g, 256, 0, st>>>(jobs, njobs, total, counter, ch); break;
        }
        LCHECK();
        return 0;
    }
    if (stats) {
        // counting variant: per-lane stacks, 4 waves per block
        PICK_STK(depth, (k_direct<4, 32, true, MK><<<g, 256, 0, st>>>(jobs, njobs, total, counter, ch, err, stats)),
                 (k_direct<4, 64, true, MK><<<g, 256, 0, st>>>(jobs, njobs, total, counter, ch, err, stats)));
        LCHECK();
        return 0;
    }
    switch (wpb) {
        case 1: PICK_STK(depth, (k_direct<1, 32, false, MK><<<g, 64, 0, st>>>(jobs, njobs, total, counter, ch, err, stats)),
                         (k_direct<1, 64, false, MK><<<g, 64, 0, st>>>(jobs, njobs, total, counter, ch, err, stats))); break;
        case 2: PICK_STK(depth, (k_direct<2, 32, false, MK><<<g, 128, 0, st>>>(jobs, njobs, total, counter, ch, err, stats)),
                         (k_direct<2, 64, false, MK><<<g, 128, 0, st>>>(jobs, njobs, total, counter, ch, err, stats))); break;
        default: PICK_STK(depth, (k_direct<4, 32, false, MK><<<g, 256, 0, st>>>(jobs, njobs, total, counter, ch, err, stats)),
                          (k_direct<4, 64, false, MK><<<g, 256, 0, st>>>(jobs, njobs, total, counter, ch, err, stats))); break;
    }
    LCHECK();
    return 0;
}

int launch_direct(const DirectJob *jobs, uint32_t njobs, uint32_t total, uint32_t depth, uint32_t *counter, int *err,
                  unsigned long long *stats, const LaunchCfg &cfg, int ncu, hipStream_t st, int flags) {
    int rc = 0;
    with_flags(stats ? counting_flags(flags) : flags, [&](auto fl) {
        rc = launch_direct_t<decltype(fl)::value>(jobs, njobs, total, depth, counter, err, stats, cfg, ncu, st,
                                                  (flags & RT_FL_GRIDS) != 0);
    });
    return rc;
}

template <int MK>
static int launch_direct_src_t(const DirectJob *jobs, uint32_t njobs, uint32_t item_lo, uint32_t nitems,
                               uint32_t depth, uint32_t *counter, int *err, unsigned long long *stats, int ncu,
                               hipStream_t st, bool blk) {
    if (nitems == 0) return 0;
    k_zero_queue<<<1, RT_QUEUE_WORDS, 0, st>>>(counter);
    blk = blk && !stats;
    uint64_t g64 = std::min<uint64_t>((uint64_t)(blk ? 8 : 4) * ncu, ((uint64_t)nitems + 3) / 4);
    uint32_t g = (uint32_t)std::max<uint64_t>(g64, 1);
    if (blk) k_direct_src<1, false, MK, true><<<g, 256, 0, st>>>(jobs, njobs, item_lo, nitems, counter, err, stats);
    else if (stats)
        PICK_STK(depth, (k_direct_src<32, true, MK, false><<<g, 256, 0, st>>>(jobs, njobs, item_lo, nitems, counter, err, stats)),
                 (k_direct_src<64, true, MK, false><<<g, 256, 0, st>>>(jobs, njobs, item_lo, nitems, counter, err, stats)));
    else
        PICK_STK(depth, (k_direct_src<32, false, MK, false><<<g, 256, 0, st>>>(jobs, njobs, item_lo, nitems, counter, err, stats)),
                 (k_direct_src<64, false, MK, false><<<g, 256, 0, st>>>(jobs, njobs, item_lo, nitems, counter, err, stats)));
    LCHECK();
    return 0;
}

int launch_direct_src(const DirectJob *jobs, uint32_t njobs, uint32_t item_lo, uint32_t nitems, uint32_t depth,
                      uint32_t *counter, int *err, unsigned long long *stats, int ncu, hipStream_t st, int flags) {
    int rc = 0;
    with_flags(stats ? counting_flags(flags) : flags, [&](auto fl) {
        rc = launch_direct_src_t<decltype(fl)::value>(jobs, njobs, item_lo, nitems, depth, counter, err, stats, ncu, st,
                                                      (flags & RT_FL_BLK) && !(flags & RT_FL_WIDE));
    });
    return rc;
}

int launch_direct_jobs(const DirectJob *hjobs, const DirectJob *jobs, uint32_t njobs, uint32_t total, uint32_t depth,
                       uint32_t *counter, int *err, unsigned long long *stats, const LaunchCfg &cfg, int ncu,
                       hipStream_t st, int flags) {
    uint32_t ncol = 0;
    while (ncol < njobs && hjobs[ncol].stype == 0) ncol++;
    for (uint32_t k = ncol; k < njobs; k++)
        if (hjobs[k].stype == 0) {
            set_error("internal: collimated direct jobs must precede the other source types");
            return -1;
        }
    // the collimated jobs' launch runs the queue kernel when each of them has an occlusion grid
    bool grids = ncol > 0;
    for (uint32_t k = 0; k < ncol; k++) grids = grids && hjobs[k].grid != nullptr;
    const int cflags = grids ? (flags | RT_FL_GRIDS) : (flags & ~RT_FL_GRIDS);
    if (ncol == njobs) return launch_direct(jobs, njobs, total, depth, counter, err, stats, cfg, ncu, st, cflags);
    if (ncol == 0) return launch_direct_src(jobs, njobs, 0, total, depth, counter, err, stats, ncu, st, flags);
    const uint32_t split = hjobs[ncol].item_begin;
    if (split > total) {
        set_error("internal: direct job items out of order");
        return -1;
    }
    if (launch_direct(jobs, ncol, split, depth, counter, err, stats, cfg, ncu, st, cflags)) return -1;
    return launch_direct_src(jobs + ncol, njobs - ncol, split, total - split, depth, counter, err, stats, ncu, st,
                             flags);
}

}  // namespace rt
