// rt_trace.hip -- diffuse / scattering trace and the gathers over its hit table.
#include "rt_traverse.h"

namespace rt {

// ------------------------------------------------------------------------------------------------
// diffuse / scattering rays -> hit words
// ------------------------------------------------------------------------------------------------
// A wave keeps 64 rays in flight; a lane whose traversal ends writes its hit word and takes another ray, and
// the wave opens the next primitive of the work queue when the current one has no rays left, so lanes do not
// idle for the longest ray of a fixed group of 64.  Every ray is traced exactly as on its own, over up to 32
// periodic wraps (diffuse_raygen.comp:498-560); only the assignment of rays to lanes and steps differs.
//
// k_diffuse walks the block tree.  Two units of a CU bound it together (SQ and TA counters, 83 ms a pass of the
// 1,001,600-primitive orchard, 439 M rays): the vector ALU (one instruction per SIMD every 3.3 cycles, where those of
// a node step take 2.4 to 4.7) and the vL1D's address unit (busy 80 % of the pass; a load instruction whose lanes lie on
// different lines takes it 45 cycles for 64 lanes whatever its width).  So a node is three 16-byte loads
// (rt_types.h), its step is short (blk_node_step()), and the rest keeps as many lanes as it can in each instruction
// (0.66 of them):
// - Rays are generated up to 64 at a time with every lane active, into the wave's LDS queue (local sample point
//   and world direction, 20 B a ray): the hashing, square roots and divisions of a ray (about 1,500 cycles a
//   wave) ran for the 19 lanes being refilled on average when each refill generated its own rays.  A
//   primitive's rays are split into equal batches (450 rays: 8 of 56 or 57).
// - A lane that reaches a record parks it and goes on with its next link, so it keeps taking node steps; it
//   waits only at a second record or with no links left.  Once RT_LEAF_BATCH_PARKED lanes wait, every parked
//   record is tested, one per lane, and the node phase goes on (6 to 16 lanes swept: 8 best, 16 3 % slower).
// - Refills start below RT_BLK_REFILL traversing lanes (40 to 58 swept: 48 best on all scenes).
// A pass of that orchard took 110 ms over 64-byte nodes with explicit links, 83 ms so (the masked kernel on 140,000
// texture-masked patches, 1,024 rays: 95 to 65 ms).  LDS per wave: RT_BLK_ROWS stack rows and the queue's five; 17 rows
// let 28 waves share the CU's 160 KB.  A step that finds 14 entries or more on a lane goes on in private memory; 17 rows
// against 15 with 8 waves: 427 and 431 ms for the orchard's five passes, 21 rows with 6 waves 459, 26 with 5 waves 506.
#ifndef RT_LEAF_BATCH_PARKED
#define RT_LEAF_BATCH_PARKED 8
#endif
#ifndef RT_BLK_REFILL
#define RT_BLK_REFILL 48
#endif
#ifndef RT_BLK_ROWS
#define RT_BLK_ROWS 17
#endif
// Waves per SIMD the compiler must fit the kernel into.  At 7 the plain kernel spills no registers and the masked one two
// or three.  Watertight predicates: 6, where their larger leaf test spills three (with masks 7 to 14, at 7 waves 19 to 25:
// 70,000 texture-masked patches x 400 rays 11.9 ms either way).
#ifndef RT_DIFFUSE_WAVES_PER_EU
#define RT_DIFFUSE_WAVES_PER_EU 7
#endif
#ifndef RT_DIFFUSE_WAVES_PER_EU_WT
#define RT_DIFFUSE_WAVES_PER_EU_WT 6
#endif
// rr / n and rr % n of a ray number rr < n * n: a multiply by ceil(2^32 / n) is exact while n^3 < 2^32
__device__ __forceinline__ void ray_cell(uint32_t rr, uint32_t n, uint32_t inv, uint32_t &lx, uint32_t &ly) {
    ly = n - 2u < 1598u ? __umulhi(rr, inv) : rr / n;
    lx = rr - ly * n;
}

template <int WPB, int MK>
__global__ __launch_bounds__(WPB * 64, (MK & RT_FL_WT) ? RT_DIFFUSE_WAVES_PER_EU_WT : RT_DIFFUSE_WAVES_PER_EU)
void k_diffuse(const DiffuseJob *__restrict__ job, uint32_t total, uint32_t *counter, uint32_t chunk, int *err) {
    constexpr int ROWS = RT_BLK_ROWS;
    __shared__ uint32_t stk_all[ROWS * WPB * 64];
    __shared__ float queue_all[5 * WPB * 64];
    // stack rows beyond the LDS part, in private memory
    uint32_t ovf[blk_ovf(ROWS, MK)];
    lds_u32 *stk = (lds_u32 *)stk_all + threadIdx.x;
    const uint32_t stride = WPB * 64;
    const uint32_t lane = threadIdx.x & 63;
    // the wave's queue: entry e of component c at queue[c * 64 + e]
    lds_f32 *queue = (lds_f32 *)queue_all + (threadIdx.x >> 6) * 320u;
    // job and scene (wave-uniform, scalar loads)
    const DevScene &sc = *ldu(&job->sc);
    const float4 *recs = ldu(&sc.rec), *nrm = ldu(&sc.nrm), *frame = ldu(&sc.frame);
    const char *blk = (const char *)ldu(&sc.blk);
    const float *T = ldu(&sc.T);
    const uint32_t *type = ldu(&sc.type);
    const uint32_t *mdesc = ldu(&sc.mdesc);
    const uint32_t nbbox = ldu(&sc.nbbox);
    const uint32_t n = ldu(&job->n), nn = n * n, seed = ldu(&job->seed);
    const uint32_t inv = n > 1u ? (uint32_t)((0x100000000ull + n - 1u) / n) : 0u;
    const uint32_t faces = ldu(&job->faces) ? ldu(&job->faces) : 3u;
    const uint32_t item_begin = ldu(&job->item_begin);
    const uint32_t *order = ldu(&job->order);
    uint32_t *hits = ldu(&job->hits);
    // a pass of the traversal loop takes at most one trace of each lane: more node steps than that mean a
    // malformed tree
    const uint32_t max_steps = (uint32_t)min(64ull * (ldu(&sc.nnode4) + 8ull), 0xFFFFFFFFull);
    // work queue, open primitive and its ray queue (wave-uniform); the primitive's frame and transform are
    // reloaded (scalar) whenever rays are generated or taken, so they hold no registers across the traversal
    WaveQueue wq(counter, total, chunk);
    uint32_t it = 0, it_end = 0;
    bool drained = false;
    uint32_t op_i = 0, op_next = 0, op_cnt = 0, op_base = 0, op_m = RT_MISS;
    uint32_t q_next = 0, q_cnt = 0, q_ray = 0;
    bool patch = false, flip = false;
    // lane state: busy = holds a ray (its trace has ended when L.ni is RT_BLK_DONE and no record is parked)
    bool busy = false;
    BlkRay L;
    L.o = L.d = mk3(0.f, 0.f, 0.f);
    blk_direction(L, 0.f, 0.f, 0.f);
    L.ox = L.oy = L.oz = 0.f;
    L.best_t = 0.f;
    L.best = RT_MISS;
    L.ni = RT_BLK_DONE;
    L.sp = 1u;
    uint32_t my_i = 0, my_r = 0, wraps = 0;
    uint32_t pend = 0u;   // link of the parked record of the lanes in mpend
    uint64_t mpend = 0u;  // lanes with a parked record (none outside the traversal loop)
    while (true) {
        // finish lanes whose traversal ended: periodic wrap (at most 32 traces), else write
        if (busy && L.ni == RT_BLK_DONE) {
            bool done = true;
            if (nbbox) {
                float bt = nearest_face_u(sc, nbbox, L.o, L.d, L.best_t);
                if (bt > 0.f && wraps < 31) {
                    L.o = wrap_at(sc, L.o, L.d, bt);
                    wraps++;
                    blk_start(L, stk);
                    done = false;
                }
            }
            if (done) {
                uint32_t word = RT_MISS;
                if (L.best != RT_MISS) {
                    float4 hn = nrm[L.best];
                    bool hit_top = dot3(mk3(hn.x, hn.y, hn.z), L.d) < 0.0f;
                    word = L.best | (hit_top ? 0u : RT_HIT_BOTTOM);
                }
                hits[(size_t)my_i * 2 * nn + my_r] = word;
                busy = false;
            }
        }
        // refill idle lanes
        while (true) {
            const uint64_t idle = __builtin_amdgcn_ballot_w64(!busy);
            if (idle == 0) break;
            if (q_next == q_cnt) {
                if (op_next == op_cnt) {
                    // open the next primitive of the work queue
                    if (it == it_end) {
                        if (drained) break;
                        if (!wq.take(it, it_end)) { drained = true; it = it_end = 0; break; }
                    }
                    uint32_t i = it - item_begin;
                    if (order) i = ldu(order + i);
                    i = __builtin_amdgcn_readfirstlane(i);
                    it++;
                    uint32_t *w = hits + (size_t)i * 2 * nn;
                    const uint32_t ty = ldu(type + i);
                    if (!traced_type(ty)) {
                        for (uint32_t r = lane; r < 2 * nn; r += 64) w[r] = RT_NOT_LAUNCHED;
                        continue;
                    }
                    const uint32_t tw = __float_as_uint(ldu(&nrm[i].w));
                    const bool s0 = (faces & 1u) != 0, s1 = ((faces >> 1) & 1u) != 0 && tw != 0;
                    if (!s0) for (uint32_t r = lane; r < nn; r += 64) w[r] = RT_NOT_LAUNCHED;
                    if (!s1) for (uint32_t r = nn + lane; r < 2 * nn; r += 64) w[r] = RT_NOT_LAUNCHED;
                    op_i = i;
                    op_m = (MK && mdesc) ? ldu(mdesc + i) : RT_MISS;
                    op_next = 0;
                    op_cnt = ((s0 ? 1u : 0u) + (s1 ? 1u : 0u)) * nn;
                    op_base = s0 ? 0u : nn;
                    patch = ty == 0 || ty == 3;
                    flip = tw == 1;
                    continue;
                }
                // generate the next batch of the open primitive's rays
                const uint32_t left = op_cnt - op_next, batches = (left + 63u) >> 6;
                q_cnt = (left + batches - 1u) / batches;
                q_next = 0;
                q_ray = op_base + op_next;
                op_next += q_cnt;
                if (lane < q_cnt) {
                    const uint32_t r = q_ray + lane;
                    const uint32_t slot = r >= nn ? 1u : 0u;  // slot 0 = top launch (face 1), slot 1 = bottom (face 0)
                    uint32_t lx, ly;
                    ray_cell(r - slot * nn, n, inv, lx, ly);
                    float spx, spy;
                    v3f dl;
                    if (diffuse_sample_m(op_i, lx, ly, n, seed, patch, recs, op_m, spx, spy, dl)) {
                        const float4 fr = ldu(frame + op_i);
                        v3f dir = frame_rotate(dl, fr.x, fr.y, fr.z, fr.w);
                        if (slot == 1 && flip) dir = mk3(-dir.x, -dir.y, -dir.z);
                        queue[lane] = spx;
                        queue[64 + lane] = spy;
                        queue[128 + lane] = dir.x;
                        queue[192 + lane] = dir.y;
                        queue[256 + lane] = dir.z;
                    } else {
                        // origin on transparent texels: the ray is dropped (adds nothing to the gather); the lane
                        // that takes this entry stays idle and takes another
                        hits[(size_t)op_i * 2 * nn + r] = RT_NOT_LAUNCHED;
                        queue[128 + lane] = 2.0f;
                    }
                }
                __builtin_amdgcn_wave_barrier();
                continue;
            }
            const uint32_t rank =
                __builtin_amdgcn_mbcnt_hi((uint32_t)(idle >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)idle, 0u));
            const uint32_t take = min((uint32_t)__popcll(idle), q_cnt - q_next);
            if (!busy && rank < take) {
                const uint32_t e = q_next + rank;
                const float dx = queue[128 + e];
                if (!MK || dx != 2.0f) {
                    float tm[12];
                    const float *Tp = T + (size_t)op_i * 16;
#pragma unroll
                    for (int q = 0; q < 12; q++) tm[q] = ldu(Tp + q);
                    L.o = xform3(tm, queue[e], queue[64 + e], 0.0f);
                    L.d = mk3(dx, queue[192 + e], queue[256 + e]);
                    blk_direction(L, blk_rcp(L.d.x), blk_rcp(L.d.y), blk_rcp(L.d.z));
                    blk_start(L, stk);
                    my_i = op_i;
                    my_r = q_ray + e;
                    wraps = 0;
                    busy = true;
                }
            }
            q_next += take;
        }
        if (__builtin_amdgcn_ballot_w64(busy) == 0) break;  // queue empty and nothing in flight
        // traverse until fewer than RT_BLK_REFILL lanes (once the queue is empty: no lane) still do
        const uint32_t floor_lanes = drained ? 1u : RT_BLK_REFILL;
        uint32_t steps = 0;
        while (true) {
            while (true) {
                const uint64_t mpark = __builtin_amdgcn_ballot_w64((L.ni & RT_BLK_REC) != 0u) &
                                       ~__builtin_amdgcn_ballot_w64(L.ni == RT_BLK_DONE) & ~mpend;
                mpend |= mpark;
                if (__builtin_amdgcn_inverse_ballot_w64(mpark)) {
                    pend = L.ni;
                    L.ni = blk_pop<ROWS>(L, stk, ovf, stride);
                }
                const bool inner = !(L.ni & RT_BLK_REC);
                const uint64_t minner = __builtin_amdgcn_ballot_w64(inner);
                if (minner == 0 || wave_popc(mpend & ~minner) >= RT_LEAF_BATCH_PARKED) break;
                if (++steps > max_steps) {
                    atomicOr(err, 2);
                    L.ni = RT_BLK_DONE;
                    break;
                }
                if (inner) blk_node_step<ROWS, MK>(blk, L, stk, ovf, stride);
            }
            if (__builtin_amdgcn_inverse_ballot_w64(mpend)) {
                uint32_t slot_unused;
                blk_leaf<false, MK>(blk, recs, pend, L, 1e-5f, my_i, slot_unused);
            }
            mpend = 0;
            if ((uint32_t)wave_popc(__builtin_amdgcn_ballot_w64(L.ni != RT_BLK_DONE)) < floor_lanes) break;
        }
    }
}

// The same over the binary tree: the counting variant (COUNT), whose node visits and primitive tests are the
// canonical work measure, and scenes without a block tree.  Traversal alternates a node phase (inner-node
// steps until RT_LEAF_BATCH lanes wait at a leaf) and a leaf phase.
template <int WPB, int STK, bool COUNT, int MK>
__global__ __launch_bounds__(WPB * 64) void k_diffuse_bin(const DiffuseJob *__restrict__ job, uint32_t total, uint32_t *counter,
                                                           uint32_t chunk, int *err, unsigned long long *stats) {
    constexpr int LSTK = STK < RT_DIFFUSE_LDS_STACK ? STK : RT_DIFFUSE_LDS_STACK;
    __shared__ uint32_t stk_all[LSTK * WPB * 64];
    // overflow entries: sized for the deepest stack (RT_STACK) so the array stays in private memory
    // instead of being promoted to registers, which would cost the occupancy the small LDS part buys
    uint32_t ovf[STK > LSTK ? RT_STACK - LSTK : 1];
    lds_u32 *stk = (lds_u32 *)stk_all + threadIdx.x;
    const uint32_t stride = WPB * 64;
    const uint32_t lane = threadIdx.x & 63;
    Cnt<COUNT, MK> cnt{};
    uint32_t nray = 0;
    // job and scene (wave-uniform, scalar loads)
    const DevScene &sc = *ldu(&job->sc);
    const float4 *nodes = ldu(&sc.node), *recs = ldu(&sc.rec), *nrm = ldu(&sc.nrm), *frame = ldu(&sc.frame);
    const float *T = ldu(&sc.T);
    const uint32_t *type = ldu(&sc.type);
    const uint32_t *mdesc = ldu(&sc.mdesc);
    const uint32_t nleaf = ldu(&sc.nleaf), nbbox = ldu(&sc.nbbox);
    const uint32_t n = ldu(&job->n), nn = n * n, seed = ldu(&job->seed);
    const uint32_t faces = ldu(&job->faces) ? ldu(&job->faces) : 3u;
    const uint32_t item_begin = ldu(&job->item_begin);
    const uint32_t *order = ldu(&job->order);
    uint32_t *hits = ldu(&job->hits);
    // work queue and open primitive (wave-uniform); the primitive's frame and transform are reloaded
    // (scalar) whenever rays are generated, so they hold no registers across the traversal
    WaveQueue wq(counter, total, chunk);
    uint32_t it = 0, it_end = 0;
    bool drained = false;
    uint32_t op_i = 0, op_next = 0, op_cnt = 0, op_base = 0, op_m = RT_MISS;
    bool patch = false, flip = false;
    // lane state: busy = holds a ray, trav = its traversal has not ended
    bool busy = false, trav = false;
    LaneRay L;
    L.o = L.d = mk3(0.f, 0.f, 0.f);
    lane_start(L, nleaf);
    uint32_t my_i = 0, my_r = 0, wraps = 0;
    while (true) {
        // finish lanes whose traversal ended: periodic wrap (at most 32 traces), else write
        if (busy && !trav) {
            bool done = true;
            if (nbbox) {
                float bt = nearest_face(sc, L.o, L.d, L.best_t);
                if (bt > 0.f && wraps < 31) {
                    L.o = wrap_at(sc, L.o, L.d, bt);
                    wraps++;
                    trav = lane_begin(L, recs, nleaf, 1e-5f, my_i, cnt);
                    done = false;
                }
            }
            if (done) {
                uint32_t word = RT_MISS;
                if (L.best != RT_MISS) {
                    float4 hn = nrm[L.best];
                    bool hit_top = dot3(mk3(hn.x, hn.y, hn.z), L.d) < 0.0f;
                    word = L.best | (hit_top ? 0u : RT_HIT_BOTTOM);
                }
                hits[(size_t)my_i * 2 * nn + my_r] = word;
                busy = false;
            }
        }
        // refill idle lanes
        while (true) {
            const uint64_t idle = __ballot(!busy);
            if (idle == 0) break;
            if (op_next == op_cnt) {
                // open the next primitive of the queue
                if (it == it_end) {
                    if (drained) break;
                    if (!wq.take(it, it_end)) { drained = true; it = it_end = 0; break; }
                }
                uint32_t i = it - item_begin;
                if (order) i = ldu(order + i);
                i = __builtin_amdgcn_readfirstlane(i);
                it++;
                uint32_t *w = hits + (size_t)i * 2 * nn;
                const uint32_t ty = ldu(type + i);
                if (!traced_type(ty)) {
                    for (uint32_t r = lane; r < 2 * nn; r += 64) w[r] = RT_NOT_LAUNCHED;
                    continue;
                }
                const uint32_t tw = __float_as_uint(ldu(&nrm[i].w));
                const bool s0 = (faces & 1u) != 0, s1 = ((faces >> 1) & 1u) != 0 && tw != 0;
                if (!s0) for (uint32_t r = lane; r < nn; r += 64) w[r] = RT_NOT_LAUNCHED;
                if (!s1) for (uint32_t r = nn + lane; r < 2 * nn; r += 64) w[r] = RT_NOT_LAUNCHED;
                op_i = i;
                op_m = (MK && mdesc) ? ldu(mdesc + i) : RT_MISS;
                op_next = 0;
                op_cnt = ((s0 ? 1u : 0u) + (s1 ? 1u : 0u)) * nn;
                op_base = s0 ? 0u : nn;
                patch = ty == 0 || ty == 3;
                flip = tw == 1;
                continue;
            }
            const uint32_t rank =
                __builtin_amdgcn_mbcnt_hi((uint32_t)(idle >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)idle, 0u));
            const uint32_t take = min((uint32_t)__popcll(idle), op_cnt - op_next);
            if (!busy && rank < take) {
                const uint32_t r = op_base + op_next + rank;
                const uint32_t slot = r >= nn ? 1u : 0u;  // slot 0 = top launch (face 1), slot 1 = bottom (face 0)
                const uint32_t rr = r - slot * nn;
                float spx, spy;
                v3f dl;
                if (diffuse_sample_m(op_i, rr % n, rr / n, n, seed, patch, recs, op_m, spx, spy, dl)) {
                    float tm[12];
                    const float *Tp = T + (size_t)op_i * 16;
#pragma unroll
                    for (int q = 0; q < 12; q++) tm[q] = ldu(Tp + q);
                    const float4 fr = ldu(frame + op_i);
                    L.o = xform3(tm, spx, spy, 0.0f);
                    v3f dir = frame_rotate(dl, fr.x, fr.y, fr.z, fr.w);
                    if (slot == 1 && flip) dir = mk3(-dir.x, -dir.y, -dir.z);
                    L.d = dir;
                    my_i = op_i;
                    my_r = r;
                    wraps = 0;
                    nray++;
                    busy = true;
                    trav = lane_begin(L, recs, nleaf, 1e-5f, my_i, cnt);
                } else {
                    // origin on transparent texels: the ray is dropped (adds nothing to the gather); the lane
                    // stays idle and takes another ray
                    hits[(size_t)op_i * 2 * nn + r] = RT_NOT_LAUNCHED;
                }
            }
            op_next += take;
        }
        if (__ballot(busy) == 0) break;  // queue empty and nothing in flight
        // traverse until fewer than RT_REFILL_BELOW lanes (once the queue is empty: no lane) still traverse
        // node phase: inner-node steps until no lane needs one or RT_LEAF_BATCH lanes wait at a leaf; leaf
        // phase: the waiting lanes test their leaves together (the intersection code runs with many lanes
        // active instead of once per node step for the few lanes that reached a leaf)
        const uint32_t floor_lanes = drained ? 1u : RT_REFILL_BELOW;
        while (true) {
            while (true) {
                const bool inner = trav && !(L.ni & RT_LEAF_BIT);
                const uint64_t mi = __ballot(inner);
                if (mi == 0 || (uint32_t)__popcll(__ballot(trav && !inner)) >= RT_LEAF_BATCH) break;
                if (inner && lane_node<STK, LSTK>(nodes, nleaf, L, stk, ovf, stride, err, cnt))
                    trav = false;
            }
            while (true) {
                const bool leaf = trav && (L.ni & RT_LEAF_BIT);
                if (__ballot(leaf) == 0) break;
                if (leaf && lane_leaf<STK, LSTK>(recs, L, 1e-5f, my_i, stk, ovf, stride, cnt)) trav = false;
            }
            if ((uint32_t)__popcll(__ballot(trav)) < floor_lanes) break;
        }
    }
    add_stats(stats, cnt, nray);
}

// ------------------------------------------------------------------------------------------------
// gather: lanes over rays (few channels)
// ------------------------------------------------------------------------------------------------
// Direction of diffuse ray r (face slot r / nn) of primitive i, regenerated from the pass seed exactly as
// the trace kernel generated it: the gather weighs a sky hit by the sky distribution in that direction.
__device__ __forceinline__ v3f diffuse_dir(const DevScene &sc, uint32_t i, uint32_t r, uint32_t n, uint32_t seed) {
    const uint32_t nn = n * n, slot = r >= nn ? 1u : 0u, rr = r - slot * nn;
    const uint32_t ty = sc.type[i];
    const uint32_t mdi = sc.mdesc ? sc.mdesc[i] : RT_MISS;
    float spx, spy;
    v3f dl;
    (void)diffuse_sample_m(i, rr % n, rr / n, n, seed, ty == 0 || ty == 3, sc.rec, mdi, spx, spy, dl);
    const float4 fr = sc.frame[i];
    v3f dir = frame_rotate(dl, fr.x, fr.y, fr.z, fr.w);
    if (slot == 1 && __float_as_uint(sc.nrm[i].w) == 1u) dir = mk3(-dir.x, -dir.y, -dir.z);
    return dir;
}

// Sums of N lane-private compensated accumulators over the wave (N a power of two up to 64): while more than one
// accumulator is left, a step hands half of them to the lane's partner and merges the other half, so N accumulators
// take N - 1 merges and then one per remaining step instead of 6 N.  On return lane l holds the sum of accumulator
// i whose bits are l's lowest log2(N) bits in reverse order.
template <int HALF, int OFF, int N>
__device__ __forceinline__ void reduce_halves(ksum (&v)[N], uint32_t lane) {
    if constexpr (HALF >= 1) {
        const bool up = (lane & (uint32_t)OFF) != 0u;
#pragma unroll
        for (int j = 0; j < HALF; j++) {
            const float gs = up ? v[j].s : v[j + HALF].s, gc = up ? v[j].c : v[j + HALF].c;
            v[j].s = up ? v[j + HALF].s : v[j].s;
            v[j].c = up ? v[j + HALF].c : v[j].c;
            v[j].merge(__shfl_xor(gs, OFF, 64), __shfl_xor(gc, OFF, 64));
        }
        reduce_halves<HALF / 2, OFF * 2>(v, lane);
    } else if constexpr (OFF < 64) {
        v[0].merge(__shfl_xor(v[0].s, OFF, 64), __shfl_xor(v[0].c, OFF, 64));
        reduce_halves<0, OFF * 2>(v, lane);
    }
}
template <int N>
__device__ __forceinline__ ksum wave_reduce_many(ksum (&v)[N], uint32_t lane) {
    reduce_halves<N / 2, 1>(v, lane);
    return v[0];
}

constexpr int pow2_up(int n) { int p = 1; while (p < n) p *= 2; return p; }

// One primitive per wave, lanes over its rays, NC channels (the jobs' C).  A lane's row -- the C-vector of a primitive
// anywhere in the scene -- is loaded whole, in as few instructions as its width needs: such a load costs the vL1D's
// address path about 0.67 cycles a lane whatever its width up to 16 B.  SKY: the sky is anisotropic.  ACCT: also
// record the pass's incident and sky flux densities and the sky-bound ray counts (GatherJob.acct, .miss) for the
// energy bookkeeping.  Both are separate instances, so the plain gather carries no extra registers.
// The channel count is exact up to 16: a kernel for the next power of two loaded and added channels that are not
// there.  Five passes of 1 M primitives x 450 rays, 3 channels: 24.1 to 11.9 ms; three passes of 200,000 x 100 rays:
// 4 channels 2.04 to 1.43 ms, 8 channels 3.75 to 1.44.  k_gather_chan (lanes over the channels) takes 5.2 ms for these
// passes at 9 to 17 channels and this kernel 1.60, 1.62 and 1.81 at 9, 12 and 16 (112 registers, none spilled).  The rule
// stops at 16 because the instances do; where the other kernel becomes the better one has not been measured.
template <int NC, bool SKY, bool ACCT>
__global__ __launch_bounds__(256) void k_gather_rays(const GatherJob *__restrict__ jobs, uint32_t njobs, uint32_t total,
                                                     uint32_t *counter, uint32_t chunk) {
    constexpr int N = pow2_up(2 * NC);  // accumulators: 2 c + face slot
    constexpr int NS = ACCT ? pow2_up(NC) : 1;
    const uint32_t lane = threadIdx.x & 63;
    WaveQueue wq(counter, total, chunk);
    for (uint32_t first, end; wq.take(first, end);) {
        for (uint32_t item = first; item < end; ++item) {
            const GatherJob &J = jobs[find_job(jobs, njobs, item)];
            uint32_t i = item - ldu(&J.item_begin);
            const uint32_t *order = ldu(&J.order);
            if (order) i = ldu(order + i);
            i = __builtin_amdgcn_readfirstlane(i);
            const DevScene *sc = ldu(&J.sc);
            if (!traced_type(ldu(ldu(&sc->type) + i))) continue;
            const uint32_t n = ldu(&J.n), nn = n * n;
            const g_u32 *w = (const g_u32 *)(ldu(&J.hits) + (size_t)i * 2 * nn);
            const g_f32 *otop = (const g_f32 *)ldu(&J.out_top), *obot = (const g_f32 *)ldu(&J.out_bot),
                        *dfl = (const g_f32 *)ldu(&J.dflux);
            ksum acc[N], asky[NS];
            uint32_t mt = 0, mb = 0;
#pragma unroll
            for (int k = 0; k < N; k++) acc[k].init();
#pragma unroll
            for (int k = 0; k < NS; k++) asky[k].init();
            // one face at a time: an accumulator index that depends on the ray would put the array in memory
#pragma unroll
            for (int f = 0; f < 2; f++)
                for (uint32_t r = (uint32_t)f * nn + lane; r < (uint32_t)(f + 1) * nn; r += 64) {
                    const uint32_t word = w[r];
                    if (word == RT_NOT_LAUNCHED) continue;
                    const bool miss = word == RT_MISS;
                    if (ACCT && miss) { if (f) mb++; else mt++; }
                    const g_f32 *src = miss ? dfl : ((word & RT_HIT_BOTTOM) ? obot : otop) + (size_t)(word & ~RT_HIT_BOTTOM) * NC;
                    float row[NC];
#pragma unroll
                    for (int c = 0; c < NC; c++) row[c] = src[c];
                    if (SKY && miss) {
                        // anisotropic sky: fd(direction) x diffuse flux (diffuse_raygen.comp:613-625)
                        const v3f dir = diffuse_dir(*sc, i, r, n, ldu(&J.seed));
                        const float *sky = ldu(&J.sky);
#pragma unroll
                        for (int c = 0; c < NC; c++) row[c] = sky_weight(dir, sky + 9 * c) * row[c];
                    }
#pragma unroll
                    for (int c = 0; c < NC; c++) {
                        acc[2 * c + f].add(row[c]);
                        if (ACCT && miss) asky[ACCT ? c : 0].add(row[c]);
                    }
                }
            const float strength = rdiv(1.0f, (float)nn);
            // lane l: accumulator k (bits of l reversed) = channel k / 2, face slot k % 2; the two faces of a channel
            // lie N / 2 lanes apart
            const ksum mine = wave_reduce_many<N>(acc, lane);
            const float I1 = mine.value() * strength, I0 = __shfl_xor(I1, N / 2, 64);
            float Is = 0.f;
            if (ACCT) {
                // (channel k / 2 lands in the lanes whose lowest bits are that channel's reversed: the same lanes)
                Is = wave_reduce_many<NS>(asky, lane).value() * strength;
                for (int off = 32; off > 0; off >>= 1) { mt += __shfl_xor(mt, off); mb += __shfl_xor(mb, off); }
                if (lane == 0) { J.miss[(size_t)i * 2] = mt; J.miss[(size_t)i * 2 + 1] = mb; }
            }
            const uint32_t k = __brev(lane) >> (32 - __builtin_ctz((unsigned)N));
            const uint32_t c = k >> 1;
            if (lane < (uint32_t)(N / 2) && c < (uint32_t)NC) {
                const bool act = J.active[c] != 0;
                if (act) {
                    const uint32_t B = ldu(&J.B), b = c % B;
                    float rho = J.rho[(size_t)i * B + b], tau = J.tau[(size_t)i * B + b];
                    size_t q = (size_t)i * NC + c;
                    J.in[q] += (I1 + I0) * (1.0f - rho - tau);
                    J.st[q] += I1 * rho + I0 * tau;
                    J.sb[q] += I1 * tau + I0 * rho;
                }
                if (ACCT) {
                    const size_t q = ((size_t)i * NC + c) * 2;
                    J.acct[q] = act ? I1 + I0 : 0.f;
                    J.acct[q + 1] = act ? Is : 0.f;
                }
            }
        }
    }
}

// ------------------------------------------------------------------------------------------------
// gather: lanes over channels (many channels, e.g. suns x bands of a diurnal batch)
// ------------------------------------------------------------------------------------------------
#ifndef RT_GATHER_UNROLL
#define RT_GATHER_UNROLL 4
#endif
// Waves per SIMD of the channel-parallel gather: 8 (64 VGPRs, a few spills) took the diurnal series'
// gathers from 180 to 166 ms against the 5 the compiler's register use allowed.
#ifndef RT_GATHER_WAVES_PER_EU
#define RT_GATHER_WAVES_PER_EU 8
#endif
template <int CB, bool ACCT>
__global__ __launch_bounds__(256, RT_GATHER_WAVES_PER_EU) void k_gather_chan(const GatherJob *__restrict__ jobs, uint32_t njobs, uint32_t total,
                                                     uint32_t *counter, uint32_t chunk) {
    const uint32_t lane = threadIdx.x & 63;
    WaveQueue wq(counter, total, chunk);
    for (uint32_t first, end; wq.take(first, end);) {
        for (uint32_t item = first; item < end; ++item) {
            uint32_t j = find_job(jobs, njobs, item);
            const GatherJob &J = jobs[j];
            uint32_t i = item - J.item_begin;
            if (J.order) i = J.order[i];
            uint32_t ty = J.sc->type[i];
            if (!traced_type(ty)) continue;
            uint32_t nn = J.n * J.n, C = J.C;
            const uint32_t *w = J.hits + (size_t)i * 2 * nn;
            ksum acc[2][CB];
            ksum asky[ACCT ? CB : 1];
            uint32_t mt = 0, mb = 0;
#pragma unroll
            for (int k = 0; k < CB; k++) {
                acc[0][k].init();
                acc[1][k].init();
            }
#pragma unroll
            for (int k = 0; k < (ACCT ? CB : 1); k++) asky[k].init();
            const float *dfl = J.dflux, *otop = J.out_top, *obot = J.out_bot;
            const float *sky = J.sky;
            for (uint32_t base = 0; base < 2 * nn; base += 64) {
                uint32_t mine = base + lane < 2 * nn ? w[base + lane] : RT_NOT_LAUNCHED;
                uint32_t cnt = min(64u, 2 * nn - base);
                if (ACCT) {
                    mt += (uint32_t)__popcll(__ballot(mine == RT_MISS && base + lane < nn));
                    mb += (uint32_t)__popcll(__ballot(mine == RT_MISS && base + lane >= nn));
                }
                // anisotropic sky: each lane regenerates the direction of its own ray if it missed; the
                // directions are broadcast with the words
                v3f mdir = mk3(0.f, 0.f, 1.f);
                if (sky && mine == RT_MISS) mdir = diffuse_dir(*J.sc, i, base + lane, J.n, J.seed);
                // RT_GATHER_UNROLL hit words per step: every row (the hit primitive's radiation_out C-vector,
                // or the sky fluxes for a miss) is loaded before any is summed, so that many rows are in
                // flight per wave; the sums take them in ray order.  A face slot that was not launched adds
                // nothing (its value is 0, which leaves a compensated sum unchanged).
                for (uint32_t q0 = 0; q0 < cnt; q0 += RT_GATHER_UNROLL) {
                    float v[RT_GATHER_UNROLL][CB];
#pragma unroll
                    for (int u = 0; u < RT_GATHER_UNROLL; u++) {
                        const uint32_t q = q0 + u;
                        const uint32_t word = q < cnt ? __builtin_amdgcn_readlane(mine, q) : RT_NOT_LAUNCHED;
                        const bool skip = word == RT_NOT_LAUNCHED;
                        const float *src = word == RT_MISS ? dfl
                                           : ((word & RT_HIT_BOTTOM) ? obot : otop) + (size_t)(word & ~RT_HIT_BOTTOM) * C;
#pragma unroll
                        for (int k = 0; k < CB; k++) {
                            uint32_t c = lane + 64 * k;
                            v[u][k] = (!skip && c < C) ? src[c] : 0.f;
                        }
                        if (sky && word == RT_MISS) {
                            const v3f dq = mk3(__shfl(mdir.x, q), __shfl(mdir.y, q), __shfl(mdir.z, q));
#pragma unroll
                            for (int k = 0; k < CB; k++) {
                                uint32_t c = lane + 64 * k;
                                if (c < C) v[u][k] = sky_weight(dq, sky + 9 * c) * v[u][k];
                            }
                        }
                    }
#pragma unroll
                    for (int u = 0; u < RT_GATHER_UNROLL; u++) {
                        const uint32_t slot = base + q0 + u >= nn ? 1u : 0u;
#pragma unroll
                        for (int k = 0; k < CB; k++) {
                            if (slot) acc[1][k].add(v[u][k]); else acc[0][k].add(v[u][k]);
                        }
                        if (ACCT) {
                            const uint32_t q = q0 + u;
                            const bool is_miss = q < cnt && __builtin_amdgcn_readlane(mine, q) == RT_MISS;
#pragma unroll
                            for (int k = 0; k < (ACCT ? CB : 1); k++)
                                if (is_miss) asky[k].add(v[u][k]);
                        }
                    }
                }
            }
            float strength = rdiv(1.0f, (float)nn);
            if (ACCT && lane == 0) { J.miss[(size_t)i * 2] = mt; J.miss[(size_t)i * 2 + 1] = mb; }
#pragma unroll
            for (int k = 0; k < CB; k++) {
                uint32_t c = lane + 64 * k;
                if (ACCT && c < C) {
                    const size_t q = ((size_t)i * C + c) * 2;
                    const bool act = J.active[c] != 0;
                    J.acct[q] = act ? (acc[0][k].value() * strength + acc[1][k].value() * strength) : 0.f;
                    J.acct[q + 1] = act ? asky[ACCT ? k : 0].value() * strength : 0.f;
                }
                if (c >= C || !J.active[c]) continue;
                float I1 = acc[0][k].value() * strength, I0 = acc[1][k].value() * strength;
                uint32_t b = c % J.B;
                float rho = J.rho[(size_t)i * J.B + b], tau = J.tau[(size_t)i * J.B + b];
                size_t qq = (size_t)i * C + c;
                J.in[qq] += (I1 + I0) * (1.0f - rho - tau);
                J.st[qq] += I1 * rho + I0 * tau;
                J.sb[qq] += I1 * tau + I0 * rho;
            }
        }
    }
}

int launch_diffuse(const DiffuseJob *job, uint32_t total, uint32_t depth, uint32_t *counter, int *err,
                   unsigned long long *stats, const LaunchCfg &cfg, int ncu, hipStream_t st, int flags) {
    if (total == 0) return 0;
    if (depth + 1 > RT_STACK) {
        set_error("BVH depth " + std::to_string(depth) + " exceeds the traversal stack (" + std::to_string(RT_STACK) + ")");
        return -1;
    }
    const uint32_t ch = std::max(cfg.chunk, 1u);
    k_zero_queue<<<1, RT_QUEUE_WORDS, 0, st>>>(counter);
    uint32_t wpb = cfg.waves_per_block;
    uint32_t g = grid_for(cfg, ncu, total, wpb);
    if (stats) {
        // counting variant: 4 waves per block
        with_flags(counting_flags(flags), [&](auto fl) {
            k_diffuse_bin<4, RT_STACK, true, decltype(fl)::value><<<g, 256, 0, st>>>(job, total, counter, ch, err, stats);
        });
        LCHECK();
        return 0;
    }
    with_flags(flags, [&](auto fl) {
        constexpr int FL = decltype(fl)::value;
        // the rarer kernels come with two waves a workgroup alone: as many waves a CU as the configuration asks for
        LaunchCfg two = cfg;
        two.blocks_per_cu = std::max(1u, cfg.blocks_per_cu * wpb / 2u);
        const uint32_t g2 = grid_for(two, ncu, total, 2);
        if (!(flags & RT_FL_BLK)) {
            k_diffuse_bin<2, RT_STACK, false, FL><<<g2, 128, 0, st>>>(job, total, counter, ch, err, stats);
            return;
        }
        if (flags & RT_FL_WIDE) {
            k_diffuse<2, FL | RT_FL_WIDE><<<g2, 128, 0, st>>>(job, total, counter, ch, err);
            return;
        }
        switch (wpb) {
            case 1: k_diffuse<1, FL><<<g, 64, 0, st>>>(job, total, counter, ch, err); break;
            case 2: k_diffuse<2, FL><<<g, 128, 0, st>>>(job, total, counter, ch, err); break;
            default: k_diffuse<4, FL><<<g, 256, 0, st>>>(job, total, counter, ch, err); break;
        }
    });
    LCHECK();
    return 0;
}

template <bool SKY, bool ACCT>
static int launch_gather_t(const GatherJob *jobs, uint32_t njobs, uint32_t total, uint32_t cmax, uint32_t *counter,
                           uint32_t g, uint32_t ch, hipStream_t st) {
    if (cmax <= 16)
        switch (cmax) {
            case 1: k_gather_rays<1, SKY, ACCT><<<g, 256, 0, st>>>(jobs, njobs, total, counter, ch); break;
            case 2: k_gather_rays<2, SKY, ACCT><<<g, 256, 0, st>>>(jobs, njobs, total, counter, ch); break;
            case 3: k_gather_rays<3, SKY, ACCT><<<g, 256, 0, st>>>(jobs, njobs, total, counter, ch); break;
            case 4: k_gather_rays<4, SKY, ACCT><<<g, 256, 0, st>>>(jobs, njobs, total, counter, ch); break;
            case 5: k_gather_rays<5, SKY, ACCT><<<g, 256, 0, st>>>(jobs, njobs, total, counter, ch); break;
            case 6: k_gather_rays<6, SKY, ACCT><<<g, 256, 0, st>>>(jobs, njobs, total, counter, ch); break;
            case 7: k_gather_rays<7, SKY, ACCT><<<g, 256, 0, st>>>(jobs, njobs, total, counter, ch); break;
            case 8: k_gather_rays<8, SKY, ACCT><<<g, 256, 0, st>>>(jobs, njobs, total, counter, ch); break;
            case 9: k_gather_rays<9, SKY, ACCT><<<g, 256, 0, st>>>(jobs, njobs, total, counter, ch); break;
            case 10: k_gather_rays<10, SKY, ACCT><<<g, 256, 0, st>>>(jobs, njobs, total, counter, ch); break;
            case 11: k_gather_rays<11, SKY, ACCT><<<g, 256, 0, st>>>(jobs, njobs, total, counter, ch); break;
            case 12: k_gather_rays<12, SKY, ACCT><<<g, 256, 0, st>>>(jobs, njobs, total, counter, ch); break;
            case 13: k_gather_rays<13, SKY, ACCT><<<g, 256, 0, st>>>(jobs, njobs, total, counter, ch); break;
            case 14: k_gather_rays<14, SKY, ACCT><<<g, 256, 0, st>>>(jobs, njobs, total, counter, ch); break;
            case 15: k_gather_rays<15, SKY, ACCT><<<g, 256, 0, st>>>(jobs, njobs, total, counter, ch); break;
            case 16: k_gather_rays<16, SKY, ACCT><<<g, 256, 0, st>>>(jobs, njobs, total, counter, ch); break;
            default: break;
        }
    else if (cmax <= 64) k_gather_chan<1, ACCT><<<g, 256, 0, st>>>(jobs, njobs, total, counter, ch);
    else if (cmax <= 128) k_gather_chan<2, ACCT><<<g, 256, 0, st>>>(jobs, njobs, total, counter, ch);
    else if (cmax <= 192) k_gather_chan<3, ACCT><<<g, 256, 0, st>>>(jobs, njobs, total, counter, ch);
    else if (cmax <= 256) k_gather_chan<4, ACCT><<<g, 256, 0, st>>>(jobs, njobs, total, counter, ch);
    else {
        set_error("more than 256 channels in one gather");
        return -1;
    }
    LCHECK();
    return 0;
}

int launch_gather(const GatherJob *jobs, uint32_t njobs, uint32_t total, uint32_t cmax, uint32_t *counter,
                  const LaunchCfg &cfg, int ncu, hipStream_t st, bool acct, bool sky) {
    if (total == 0) return 0;
    const uint32_t ch = std::max(cfg.chunk, 1u);
    k_zero_queue<<<1, RT_QUEUE_WORDS, 0, st>>>(counter);
    uint32_t g = grid_for(cfg, ncu, total, 4);
    if (acct)
        return sky ? launch_gather_t<true, true>(jobs, njobs, total, cmax, counter, g, ch, st)
                   : launch_gather_t<false, true>(jobs, njobs, total, cmax, counter, g, ch, st);
    return sky ? launch_gather_t<true, false>(jobs, njobs, total, cmax, counter, g, ch, st)
               : launch_gather_t<false, false>(jobs, njobs, total, cmax, counter, g, ch, st);
}

}  // namespace rt
