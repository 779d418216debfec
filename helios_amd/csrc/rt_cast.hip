// rt_cast.hip -- castRays, camera, pixel-label and debug kernels.
#include "rt_traverse.h"

namespace rt {

// ------------------------------------------------------------------------------------------------
// castRaysSoA
// ------------------------------------------------------------------------------------------------
// One closest-hit leaf test with the CollisionDetection predicates (tmin 1e-6, nothing skipped), keeping the
// hit's leaf slot for the normal, then pop.
template <int STK, int LSTK, typename C>
__device__ __forceinline__ bool lane_leaf_cd(const float4 *recs, LaneRay &L, uint32_t &slot, const lds_u32 *stk,
                                             const uint32_t *ovf, uint32_t stride, C &cnt) {
    cnt.prims++;
    test_leaf<true, C::flags>(recs, L.ni & ~RT_LEAF_BIT, L.o, L.d, 1e-6f, RT_MISS, L.best_t, L.best, slot);
    return lane_pop<STK, LSTK>(L, stk, ovf, stride);
}

// Next chunk of rays of a wave (wave-uniform 64-bit work counter), fetched by lane 0 (see WaveQueue::fetch): 1,000 rays
// into 20,000 primitives 177 to 169 us a call, long launches the same.  One counter serves: a chunk's 64 rays take a
// launch of 20 M rays over 5 M primitives 21 ns, the counter 12.
__device__ __forceinline__ unsigned long long wave_chunk64(unsigned long long *counter, uint32_t chunk) {
    unsigned long long f = 0;
    if ((threadIdx.x & 63) == 0)
        f = __hip_atomic_fetch_add(counter, (unsigned long long)chunk, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)f);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(f >> 32));
    return ((unsigned long long)hi << 32) | lo;
}

// Result of a cast ray: the hit's UUID, distance and normal; a miss leaves distance and normal untouched.
// rr: the hit's record (read on a hit only).
__device__ __forceinline__ void cast_result(unsigned long long my_r, uint32_t h, float best_t, const float4 *rr, v3f o, v3f d,
                                            const uint32_t *uuid, float *T, float *N, uint32_t *U) {
    if (h == RT_MISS) {
        U[my_r] = RT_MISS;
        return;
    }
    U[my_r] = uuid[h];
    T[my_r] = best_t;
    const float4 r0 = rr[0], r1 = rr[1], r2 = rr[2], r3 = rr[3];
    const uint32_t tag = __float_as_uint(r0.w);
    const bool patch = (tag & RT_PATCH_BIT) != 0;
    // CD/src/CollisionDetection_RayTracing.cpp:1572-1585: normal of cross(v1-v0, v2-v0), facing
    // the origin; a voxel's is the outward normal of the face hit (1685-1711), not turned
    v3f nn;
    bool ok;
    if (tag & RT_VOXEL_BIT) {
        nn = voxel_normal_cd(r0, r1, add3(o, mul3(d, best_t)));
        ok = false;
    } else if (patch) {
        nn = mk3(r3.x, r3.y, r3.z);
        v3f raw = cross3(mk3(r1.x, r1.y, r1.z), add3(mk3(r1.x, r1.y, r1.z), mk3(r2.x, r2.y, r2.z)));
        ok = rsqrt_cr(raw.x * raw.x + raw.y * raw.y + raw.z * raw.z) > 1e-8f;
    } else {
        nn = cross3(mk3(r1.x, r1.y, r1.z), mk3(r2.x, r2.y, r2.z));
        float mag = rsqrt_cr(nn.x * nn.x + nn.y * nn.y + nn.z * nn.z);
        ok = mag > 1e-8f;
        if (ok) nn = mul3(nn, rdiv(1.0f, mag));
    }
    if (ok) {
        v3f ip = add3(o, mul3(d, best_t));
        v3f to = sub3(o, ip);
        if (nn.x * to.x + nn.y * to.y + nn.z * to.z < 0) nn = mul3(nn, -1.0f);
    } else if (!(tag & RT_VOXEL_BIT)) {
        nn = nrm3(mk3(-d.x, -d.y, -d.z));
    }
    N[my_r * 3] = nn.x;
    N[my_r * 3 + 1] = nn.y;
    N[my_r * 3 + 2] = nn.z;
}

#ifndef RT_CAST_WAVES_PER_EU
#define RT_CAST_WAVES_PER_EU 1
#endif
// stack rows in LDS: 20 KB a workgroup, which eight of them fill the CU's 160 KB with
#ifndef RT_CAST_ROWS
#define RT_CAST_ROWS 20
#endif
// castRaysSoA (CD/src/CollisionDetection_RayTracing.cpp:551-680, 980-1080): closest hit of each ray with
// the CD predicates.  Persistent waves take chunks of rays from a counter and keep 64 rays in flight: a lane
// whose trace ends writes its result and takes the chunk's next ray; traversal runs in node and leaf phases.
// Each ray is traced exactly as on its own.  Over the block tree (blk_node_step).
template <int WPB, int MK>
__global__ __launch_bounds__(WPB * 64, RT_CAST_WAVES_PER_EU) void k_cast(const DevScene *__restrict__ scp, uint64_t n, const float *__restrict__ O,
                                              const float *__restrict__ D, float maxd, float *__restrict__ T,
                                              float *__restrict__ N, uint32_t *__restrict__ U,
                                              unsigned long long *counter, uint32_t chunk, int *err) {
    constexpr int ROWS = RT_CAST_ROWS;
    __shared__ uint32_t stk_all[ROWS * WPB * 64];
    uint32_t ovf[blk_ovf(ROWS, MK)];
    lds_u32 *stk = (lds_u32 *)stk_all + threadIdx.x;
    const uint32_t stride = WPB * 64;
    const DevScene &sc = *scp;
    const float4 *recs = ldu(&sc.rec);
    const char *blk = (const char *)ldu(&sc.blk);
    const uint32_t *uuid = ldu(&sc.uuid);
    const float tstart = maxd > 0.f ? maxd : FLT_MAX;
    // a pass of the traversal loop takes at most one trace of each lane: more node steps than that mean a
    // malformed tree
    const uint32_t max_steps = (uint32_t)min(64ull * (ldu(&sc.nnode4) + 8ull), 0xFFFFFFFFull);
    unsigned long long q_next = 0, q_end = 0, my_r = 0;
    bool drained = false, busy = false;
    BlkRay L;
    L.o = L.d = mk3(0.f, 0.f, 0.f);
    blk_direction(L, 0.f, 0.f, 0.f);
    L.ox = L.oy = L.oz = 0.f;
    L.best_t = 0.f;
    L.best = RT_MISS;
    L.ni = RT_BLK_DONE;
    L.sp = 1u;
    uint32_t slot = 0u;
    while (true) {
        // finished lanes write their result
        if (busy && L.ni == RT_BLK_DONE) {
            cast_result(my_r, L.best, L.best_t, (const float4 *)blk_at<MK>(blk, slot), L.o, L.d, uuid, T, N, U);
            busy = false;
        }
        // idle lanes take the next rays of the wave's chunk
        while (true) {
            const uint64_t idle = __builtin_amdgcn_ballot_w64(!busy);
            if (idle == 0) break;
            if (q_next == q_end) {
                if (drained) break;
                const unsigned long long f = wave_chunk64(counter, chunk);
                if (f >= n) { drained = true; break; }
                q_next = f;
                q_end = f + chunk < n ? f + chunk : n;
            }
            const uint32_t rank =
                __builtin_amdgcn_mbcnt_hi((uint32_t)(idle >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)idle, 0u));
            const uint32_t left = (uint32_t)(q_end - q_next);
            const uint32_t take = min((uint32_t)__popcll(idle), left);
            if (!busy && rank < take) {
                const unsigned long long r = q_next + rank;
                L.o = mk3(O[r * 3], O[r * 3 + 1], O[r * 3 + 2]);
                L.d = mk3(D[r * 3], D[r * 3 + 1], D[r * 3 + 2]);
                // A cast ray may start far outside the scene, where an ulp of the reciprocal counts: divide.  Its
                // direction may have any length (distances count in lengths of it), so what makes a component
                // near 0 is its size against the largest one: its slab then reaches 1e18 times as far as the
                // ray's own distances (1e30 at most, as ray_pre()).
                const float lim = fminf(1e18f * __builtin_amdgcn_rcpf(max3f(fabsf(L.d.x), fabsf(L.d.y), fabsf(L.d.z))), 1e30f);
                blk_direction(L, copysignf(fminf(1.0f / fabsf(L.d.x), lim), L.d.x),
                              copysignf(fminf(1.0f / fabsf(L.d.y), lim), L.d.y),
                              copysignf(fminf(1.0f / fabsf(L.d.z), lim), L.d.z));
                blk_start(L, stk);
                L.best_t = tstart;
                my_r = r;
                busy = true;
            }
            q_next += take;
        }
        if (__builtin_amdgcn_ballot_w64(busy) == 0) break;  // queue empty and nothing in flight
        const uint32_t floor_lanes = drained ? 1u : RT_REFILL_BELOW;
        uint32_t steps = 0;
        while (true) {
            while (true) {
                const bool inner = !(L.ni & RT_BLK_REC);
                const uint64_t minner = __builtin_amdgcn_ballot_w64(inner);
                if (minner == 0 || wave_popc(__builtin_amdgcn_ballot_w64(L.ni != RT_BLK_DONE) & ~minner) >= RT_LEAF_BATCH) break;
                if (++steps > max_steps) {
                    atomicOr(err, 2);
                    L.ni = RT_BLK_DONE;
                    break;
                }
                if (inner) blk_node_step<ROWS, MK, true>(blk, L, stk, ovf, stride);
            }
            while (true) {
                const bool leaf = (L.ni & RT_BLK_REC) && L.ni != RT_BLK_DONE;
                if (__builtin_amdgcn_ballot_w64(leaf) == 0) break;
                if (leaf) {
                    blk_leaf<true, MK>(blk, recs, L.ni, L, 1e-6f, RT_MISS, slot);
                    L.ni = blk_pop<ROWS>(L, stk, ovf, stride);
                }
            }
            if ((uint32_t)wave_popc(__builtin_amdgcn_ballot_w64(L.ni != RT_BLK_DONE)) < floor_lanes) break;
        }
    }
}

// The same over the binary tree: the counting variant (COUNT), whose node visits are the canonical work measure,
// and scenes without a block tree.
template <int STK, bool COUNT, int MK>
__global__ __launch_bounds__(256) void k_cast_bin(const DevScene *__restrict__ scp, uint64_t n, const float *__restrict__ O,
                                                  const float *__restrict__ D, float maxd, float *__restrict__ T,
                                                  float *__restrict__ N, uint32_t *__restrict__ U,
                                                  unsigned long long *counter, int *err, unsigned long long *stats) {
    constexpr int LSTK = STK < RT_DIFFUSE_LDS_STACK ? STK : RT_DIFFUSE_LDS_STACK;
    __shared__ uint32_t stk_all[LSTK * 256];
    uint32_t ovf[STK > LSTK ? RT_STACK - LSTK : 1];
    lds_u32 *stk = (lds_u32 *)stk_all + threadIdx.x;
    const uint32_t stride = 256;
    const DevScene &sc = *scp;
    const float4 *nodes = ldu(&sc.node), *recs = ldu(&sc.rec);
    const uint32_t *uuid = ldu(&sc.uuid);
    const uint32_t nleaf = ldu(&sc.nleaf);
    const float tstart = maxd > 0.f ? maxd : FLT_MAX;
    Cnt<COUNT, MK> cnt{};
    uint32_t nray = 0;
    unsigned long long q_next = 0, q_end = 0, my_r = 0;
    bool drained = false, busy = false, trav = false;
    LaneRay L;
    L.o = L.d = mk3(0.f, 0.f, 0.f);
    lane_start(L, nleaf);
    uint32_t slot = RT_MISS;
    while (true) {
        // finished lanes write their result
        if (busy && !trav) {
            cast_result(my_r, L.best, L.best_t, recs + (size_t)slot * 4, L.o, L.d, uuid, T, N, U);
            busy = false;
        }
        // idle lanes take the next rays of the wave's chunk
        while (true) {
            const uint64_t idle = __ballot(!busy);
            if (idle == 0) break;
            if (q_next == q_end) {
                if (drained) break;
                const unsigned long long f = wave_chunk64(counter, 64u);
                if (f >= n) { drained = true; break; }
                q_next = f;
                q_end = f + 64 < n ? f + 64 : n;
            }
            const uint32_t rank =
                __builtin_amdgcn_mbcnt_hi((uint32_t)(idle >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)idle, 0u));
            const uint32_t left = (uint32_t)(q_end - q_next);
            const uint32_t take = min((uint32_t)__popcll(idle), left);
            if (!busy && rank < take) {
                const unsigned long long r = q_next + rank;
                L.o = mk3(O[r * 3], O[r * 3 + 1], O[r * 3 + 2]);
                L.d = mk3(D[r * 3], D[r * 3 + 1], D[r * 3 + 2]);
                lane_start(L, nleaf);
                L.best_t = tstart;
                slot = RT_MISS;
                trav = nleaf > 1;
                if (nleaf == 1) { cnt.prims++; test_leaf<true, MK>(recs, 0, L.o, L.d, 1e-6f, RT_MISS, L.best_t, L.best, slot); }
                my_r = r;
                busy = true;
                nray++;
            }
            q_next += take;
        }
        if (__ballot(busy) == 0) break;  // queue empty and nothing in flight
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
                if (leaf && lane_leaf_cd<STK, LSTK>(recs, L, slot, stk, ovf, stride, cnt)) trav = false;
            }
            if ((uint32_t)__popcll(__ballot(trav)) < floor_lanes) break;
        }
    }
    add_stats(stats, cnt, nray);
}

// ------------------------------------------------------------------------------------------------
// cameras (camera_raygen.comp, pixel_label_raygen.comp)
// ------------------------------------------------------------------------------------------------
// Closest hit of a camera ray with up to 10 periodic wraps (camera_raygen.comp:266-285); a ray still
// crossing faces after the 10th trace counts as a miss.  depth accumulates the distance of the wraps.
// trace_closest() with radiation predicates and a hybrid stack: entries below LSTK in LDS (stride
// 256), deeper ones in the private array ovf.
template <int LSTK, int STK, typename C>
__device__ __forceinline__ uint32_t trace_closest_hyb(const DevScene &sc, v3f o, v3f d, float tmin, float &t_out,
                                                      lds_u32 *stk, uint32_t *ovf, int *err, C &cnt) {
    float best_t = 1e30f;
    uint32_t best = RT_MISS, best_slot = RT_MISS;
    const float4 *nodes = sc.node, *recs = sc.rec;
    const uint32_t nleaf = sc.nleaf;
    if (nleaf <= 1) {
        if (nleaf == 1) { cnt.prims++; test_leaf<false, C::flags>(recs, 0, o, d, tmin, RT_MISS, best_t, best, best_slot); }
        t_out = best_t;
        return best;
    }
    RayPre rp = ray_pre(o, d);
    uint32_t ni = 0;
    int sp = 0;
    uint32_t budget = nleaf + 8;
    while (true) {
        if (budget-- == 0 || ni >= nleaf - 1) {
            atomicOr(err, 2);
            break;
        }
        cnt.nodes++;
        NodeTest nt = node_test_p(nodes, ni, rp, best_t);
        bool l0 = (nt.c0 & RT_LEAF_BIT) != 0, l1 = (nt.c1 & RT_LEAF_BIT) != 0;
        if (nt.h0 && l0) { cnt.prims++; test_leaf<false, C::flags>(recs, nt.c0 & ~RT_LEAF_BIT, o, d, tmin, RT_MISS, best_t, best, best_slot); }
        if (nt.h1 && l1) { cnt.prims++; test_leaf<false, C::flags>(recs, nt.c1 & ~RT_LEAF_BIT, o, d, tmin, RT_MISS, best_t, best, best_slot); }
        bool g0 = nt.h0 && !l0, g1 = nt.h1 && !l1;
        if (g0 && g1) {
            bool first0 = nt.tn0 <= nt.tn1;
            if (sp >= STK) {
                atomicOr(err, 1);
                break;
            }
            const uint32_t far = first0 ? nt.c1 : nt.c0;
            if (sp < LSTK) stk[(uint32_t)sp * 256u] = far;
            else ovf[sp - LSTK] = far;
            sp++;
            ni = first0 ? nt.c0 : nt.c1;
        } else if (g0) {
            ni = nt.c0;
        } else if (g1) {
            ni = nt.c1;
        } else {
            if (sp == 0) break;
            sp--;
            ni = sp < LSTK ? stk[(uint32_t)sp * 256u] : ovf[sp - LSTK];
        }
    }
    t_out = best_t;
    return best;
}

#ifndef RT_CAMERA_LDS_STACK
#define RT_CAMERA_LDS_STACK 16
#endif

template <int STK, typename CT>
__device__ __forceinline__ uint32_t camera_trace(const DevScene &sc, v3f &o, v3f d, float &t, float &depth,
                                                 lds_u32 *stk, uint32_t *ovf, int *err, CT &cnt) {
    constexpr int LSTK = STK < RT_CAMERA_LDS_STACK ? STK : RT_CAMERA_LDS_STACK;
    uint32_t hit = RT_MISS;
    depth = 0.0f;
    for (int wrap = 0; wrap < 10; ++wrap) {
        hit = trace_closest_hyb<LSTK, STK>(sc, o, d, 1e-5f, t, stk, ovf, err, cnt);
        if (sc.nbbox == 0) break;
        const float bt = nearest_face(sc, o, d, t);
        if (!(bt > 0.f)) break;
        depth += bt;
        o = wrap_at(sc, o, d, bt);
        hit = RT_MISS;
    }
    return hit;
}

// Pixel of this thread: each wave takes an 8 x 8 block of the tile (blocks row by row), so the rays of
// a wave leave through neighbouring pixels and traverse much the same nodes.
__device__ __forceinline__ bool camera_pixel(const CameraLaunch &c, uint32_t &px, uint32_t &py) {
    const uint32_t q = blockIdx.x * 256u + threadIdx.x;
    const uint32_t blk = q >> 6, lane = q & 63u, bx = (c.res_x + 7u) >> 3;
    px = (blk % bx) * 8u + (lane & 7u);
    py = (blk / bx) * 8u + (lane >> 3);
    return px < c.res_x && py < c.res_y;
}

// Prague sky pattern (sky_distribution.glsl:60-90), or 1 (isotropic) when its normalisation is not positive.
__device__ __forceinline__ float cam_sky_weight(v3f d, const float *sun, const float *prm) {
    if (!(prm[3] > 0.0f)) return 1.0f;
    return sky_prague(d, sun[0], sun[1], sun[2], prm);
}

// Radiance of the sources a camera ray meets before tmax, for band b, summed in source order
// (camera_raygen.comp:349-377 on a hit, 431-455 on a miss, where collimated and sun-sphere sources add the
// solar disk's radiance when the ray lies within it).
__device__ __forceinline__ float cam_source_radiance(const CameraLaunch &c, v3f o, v3f d, uint32_t b, float tmax,
                                                     bool miss) {
    float rad = 0.0f;
    for (uint32_t s = 0; s < c.S; s++) {
        const float flux = c.flux[(size_t)s * c.B + b];
        if (flux <= 0.0f) continue;
        const uint32_t ty = c.src_type[s];
        const v3f sp = mk3(c.src_pos[3 * s], c.src_pos[3 * s + 1], c.src_pos[3 * s + 2]);
        const float *w = c.src_width + 2 * s;
        float cosang;
        if (ty == 0u || ty == 2u) {
            if (miss && d.x * c.sun[0] + d.y * c.sun[1] + d.z * c.sun[2] >= c.solar_cos && c.solar_rad[b] > 0.0f)
                rad += c.solar_rad[b];
        } else if (ty == 1u) {
            const float r = w[0] * 0.5f;
            if (cam_sphere_visible(o, d, sp, r, tmax)) rad += rdiv(rdiv(flux, 4.0f * RT_PI_F * r * r), RT_PI_F);
        } else if (ty == 3u) {
            if (cam_planar_visible(false, o, d, sp, w, c.src_rot + 9 * s, tmax, cosang))
                rad += rdiv(rdiv(flux, w[0] * w[1]) * cosang, RT_PI_F);
        } else if (ty == 4u) {
            const float r = w[0];
            if (cam_planar_visible(true, o, d, sp, w, c.src_rot + 9 * s, tmax, cosang))
                rad += rdiv(rdiv(flux, RT_PI_F * r * r) * cosang, RT_PI_F);
        }
    }
    return rad;
}

// Blinn-Phong specular term of a camera hit on primitive h for band b (camera_raygen.comp:362-409): for
// each source, the radiation it delivered to h in the direct launch (radiation_specular) times the
// camera's weight for that source and band and a Fresnel reflectance of 0.25; if positive, times the
// primitive's scale (mode 2, else 1), (n . h)^e (e + 2) / (2 pi samples), with h the half vector between
// the light direction (a collimated or sun-sphere source's direction, else towards the source's centre
// from the hit point) and the reversed view direction, and n the primitive's stored normal.  0 when the
// primitive's exponent is not positive.  FP32, the reference's operation order.
__device__ __forceinline__ float cam_specular(const CameraLaunch &c, v3f o, v3f d, float t, uint32_t h, uint32_t b,
                                              v3f n) {
    float acc = 0.0f;
    const float e = c.spec_exp[h];
    if (!(e > 0.0f)) return 0.0f;
    for (uint32_t s = 0; s < c.S; s++) {
        float spec = c.spec[((size_t)s * c.spec_P + h) * c.B + b];
        spec = spec * (c.fcam[(size_t)s * c.B + b] * 0.25f);
        if (!(spec > 0.0f)) continue;
        const uint32_t ty = c.src_type[s];
        v3f L = mk3(c.src_pos[3 * s], c.src_pos[3 * s + 1], c.src_pos[3 * s + 2]);
        if (!(ty == 0u || ty == 2u)) L = sub3(L, add3(o, mul3(d, t)));
        L = nrm3(L);
        const v3f hv = nrm3(sub3(L, d));
        const float scale = c.spec_mode == 2u ? c.spec_scale[h] : 1.0f;
        const float ch = fmaxf(0.0f, hv.x * n.x + hv.y * n.y + hv.z * n.z);
        acc += rdiv(spec * scale * powf(ch, e) * (e + 2.0f), (float)c.spp * 2.0f * RT_PI_F);
    }
    return acc;
}

// Camera pixels: one thread per pixel of the tile traces its antialiasing samples in order and adds
// their contributions to camera_radiation[b][pixel] (a fixed order, so a render is reproducible; the
// reference adds the samples with float atomics).  The lanes of a wave stay on the same sample: starting a lane's next
// sample while the others still traverse measured slower on the orchard image (1,094 against 1,460 Mrays/s), because
// lanes drift to different samples and the wave loses the coherence of neighbouring pixels' rays.
template <int STK, bool COUNT, int MK, bool SPEC>
__global__ __launch_bounds__(256) void k_camera(CameraLaunch c, int *err, unsigned long long *stats) {
    constexpr int LSTK = STK < RT_CAMERA_LDS_STACK ? STK : RT_CAMERA_LDS_STACK;
    __shared__ uint32_t stk_all[LSTK * 256];
    uint32_t ovf[STK > LSTK ? RT_STACK - LSTK : 1];
    lds_u32 *stk = (lds_u32 *)stk_all + threadIdx.x;
    uint32_t px, py;
    if (!camera_pixel(c, px, py)) return;
    const DevScene &sc = *c.sc;
    const uint32_t ii = c.off_x + px, jj = c.off_y + py;
    const size_t pix = (size_t)jj * c.full_x + ii, npix = (size_t)c.full_x * c.full_y;
    const float strength = rdiv(1.0f, (float)c.spp);
    const uint32_t dimx = c.res_x * c.res_y, indx = c.res_x * py + px;
    Cnt<COUNT, MK> cnt{};
    for (uint32_t smp = 0; smp < c.spp; smp++) {
        uint32_t st = tea16(indx + dimx * smp, c.seed);
        const float Rx = rnd24(st), Ry = rnd24(st);
        float lx = 0.f, ly = 0.f;
        if (c.lens > 0.0f) unit_disk(rnd24(st), rnd24(st), lx, ly);
        v3f o, d;
        camera_ray(c.pos[0], c.pos[1], c.pos[2], c.st, c.ct, c.sp, c.cp, c.focal, c.lens, c.aspect, c.viewplane, ii,
                   jj, c.full_x, c.full_y, Rx, Ry, lx, ly, o, d);
        float t, depth;
        const uint32_t h = camera_trace<STK>(sc, o, d, t, depth, stk, ovf, err, cnt);
        if (h != RT_MISS) {
            const float4 n4 = sc.nrm[h];
            const bool face = n4.x * d.x + n4.y * d.y + n4.z * d.z < 0.0f;  // true: top face hit
            const bool top = face || sc.type[h] == 4u;
            for (uint32_t b = 0; b < c.B; b++) {
                const float srad = cam_source_radiance(c, o, d, b, t, false);
                float surf = (top ? c.out_top : c.out_bot)[(size_t)h * c.B + b] * strength;
                if (srad > 0.0f) surf += srad * strength;
                if (SPEC) surf += cam_specular(c, o, d, t, h, b, mk3(n4.x, n4.y, n4.z));
                c.pixels[(size_t)b * npix + pix] += rdiv(surf, RT_PI_F);
            }
        } else {
            for (uint32_t b = 0; b < c.B; b++) {
                float rad = cam_source_radiance(c, o, d, b, 1e30f, true);
                if (rad <= 0.0f && c.sky_rad[b] > 0.0f) rad = c.sky_rad[b] * cam_sky_weight(d, c.sun, c.sky_params + 4 * b);
                if (c.emis[b] != 0u && c.cam_dflux[b] > 0.0f) rad += rdiv(c.cam_dflux[b], RT_PI_F);
                if (rad > 0.0f) c.pixels[(size_t)b * npix + pix] += rad * strength;
            }
        }
    }
    add_stats(stats, cnt, c.spp);
}

// Pixel labels (pixel_label_raygen.comp:80-155): the pixel-centre pinhole ray's hit UUID + 1 (0 = sky) and
// its depth along the view direction (-1 on a miss).
template <int STK, int MK>
__global__ __launch_bounds__(256) void k_pixel_label(CameraLaunch c, int *err) {
    constexpr int LSTK = STK < RT_CAMERA_LDS_STACK ? STK : RT_CAMERA_LDS_STACK;
    __shared__ uint32_t stk_all[LSTK * 256];
    uint32_t ovf[STK > LSTK ? RT_STACK - LSTK : 1];
    lds_u32 *stk = (lds_u32 *)stk_all + threadIdx.x;
    uint32_t px, py;
    if (!camera_pixel(c, px, py)) return;
    const DevScene &sc = *c.sc;
    const uint32_t ii = c.off_x + px, jj = c.off_y + py;
    const size_t pix = (size_t)jj * c.full_x + ii;
    v3f o, d;
    camera_ray(c.pos[0], c.pos[1], c.pos[2], c.st, c.ct, c.sp, c.cp, c.focal, 0.0f, c.aspect, c.viewplane, ii, jj,
               c.full_x, c.full_y, 0.5f, 0.5f, 0.0f, 0.0f, o, d);
    float t, depth;
    NoCntT<MK> cnt{};
    const uint32_t h = camera_trace<STK>(sc, o, d, t, depth, stk, ovf, err, cnt);
    if (h != RT_MISS) {
        c.labels[pix] = sc.uuid[h] + 1u;
        const v3f fwd = camera_rotate(mk3(1.0f, 0.0f, 0.0f), c.st, c.ct, c.sp, c.cp);
        c.depths[pix] = fabsf(dot3(fwd, d)) * (depth + t);
    } else {
        c.depths[pix] = -1.0f;
    }
}

// ------------------------------------------------------------------------------------------------
// parity hooks: generated diffuse rays, and radiation-predicate traces of arbitrary rays
// ------------------------------------------------------------------------------------------------
__global__ void k_debug_rays(const DevScene *__restrict__ scp, uint32_t n, uint32_t seed, float *__restrict__ out) {
    const DevScene &sc = *scp;
    uint32_t nn = n * n;
    uint64_t g = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= (uint64_t)sc.P * 2 * nn) return;
    uint32_t i = (uint32_t)(g / (2 * nn)), r = (uint32_t)(g % (2 * nn));
    uint32_t slot = r >= nn ? 1u : 0u, rr = r - slot * nn;
    uint32_t ty = sc.type[i];
    bool patch = ty == 0 || ty == 3;
    uint32_t tw = __float_as_uint(sc.nrm[i].w);
    float4 fr = sc.frame[i];
    float spx, spy;
    v3f dl;
    float *w = out + g * 6;
    const uint32_t mdi = sc.mdesc ? sc.mdesc[i] : RT_MISS;
    if (!diffuse_sample_m(i, rr % n, rr / n, n, seed, patch, sc.rec, mdi, spx, spy, dl)) {
        for (int k = 0; k < 6; k++) w[k] = __uint_as_float(0x7FC00000u);  // dropped ray: NaN
        return;
    }
    v3f o = xform3(sc.T + (size_t)i * 16, spx, spy, 0.0f);
    v3f dir = frame_rotate(dl, fr.x, fr.y, fr.z, fr.w);
    if (slot == 1 && tw == 1) dir = mk3(-dir.x, -dir.y, -dir.z);
    w[0] = o.x; w[1] = o.y; w[2] = o.z; w[3] = dir.x; w[4] = dir.y; w[5] = dir.z;
}

template <int MK>
__global__ __launch_bounds__(256) void k_debug_trace(const DevScene *__restrict__ scp, uint32_t n,
                                                     const float *__restrict__ rays, const uint32_t *__restrict__ skip,
                                                     float tmin, int brute, uint32_t *__restrict__ hit,
                                                     float *__restrict__ tout, int *err) {
    __shared__ uint32_t stk_all[RT_STACK * 256];
    TCntT<MK> cnt{0, 0};
    uint32_t *stk = stk_all + threadIdx.x;
    const DevScene &sc = *scp;
    uint32_t r = blockIdx.x * 256 + threadIdx.x;
    if (r >= n) return;
    v3f o = mk3(rays[r * 6], rays[r * 6 + 1], rays[r * 6 + 2]);
    v3f d = mk3(rays[r * 6 + 3], rays[r * 6 + 4], rays[r * 6 + 5]);
    float t = 1e30f;
    uint32_t h = RT_MISS, slot;
    if (brute) {
        for (uint32_t k = 0; k < sc.nleaf; k++) test_leaf<false, MK>(sc.rec, k, o, d, tmin, skip[r], t, h, slot);
    } else {
        h = trace_closest<false, RT_STACK>(sc, o, d, tmin, skip[r], 1e30f, t, slot, stk, 256, err, cnt);
    }
    hit[r] = h;
    tout[r] = t;
}

int launch_debug_rays(const DevScene *sc, uint32_t P, uint32_t n, uint32_t seed, float *out, hipStream_t st) {
    uint64_t tot = (uint64_t)P * 2 * n * n;
    if (tot == 0) return 0;
    k_debug_rays<<<(uint32_t)((tot + 255) / 256), 256, 0, st>>>(sc, n, seed, out);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) { set_error(std::string("kernel launch failed: ") + hipGetErrorString(e)); return -1; }
    return 0;
}

int launch_debug_trace(const DevScene *sc, uint32_t n, const float *rays, const uint32_t *skip, float tmin, int brute,
                       uint32_t *hit, float *t, int *err, hipStream_t st, int flags) {
    if (n == 0) return 0;
    with_flags(flags | RT_FL_MASK, [&](auto fl) {
        k_debug_trace<decltype(fl)::value><<<(n + 255) / 256, 256, 0, st>>>(sc, n, rays, skip, tmin, brute, hit, t, err);
    });
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) { set_error(std::string("kernel launch failed: ") + hipGetErrorString(e)); return -1; }
    return 0;
}

int launch_camera(const CameraLaunch &c, uint32_t depth, bool labels, int *err, unsigned long long *stats,
                  hipStream_t st, int flags) {
    if ((uint64_t)c.res_x * c.res_y == 0) return 0;
    // one wave per 8 x 8 pixel block, four waves per workgroup
    const uint64_t blocks = (uint64_t)((c.res_x + 7) / 8) * ((c.res_y + 7) / 8);
    const uint32_t g = (uint32_t)((blocks + 3) / 4);
    if (labels)
        with_flags(flags, [&](auto fl) {
            constexpr int FL = decltype(fl)::value;
            PICK_STK(depth, (k_pixel_label<32, FL><<<g, 256, 0, st>>>(c, err)),
                     (k_pixel_label<64, FL><<<g, 256, 0, st>>>(c, err)));
        });
    else if (stats)
        with_flags(counting_flags(flags), [&](auto fl) {
            constexpr int FL = decltype(fl)::value;
            if (c.spec)
                PICK_STK(depth, (k_camera<32, true, FL, true><<<g, 256, 0, st>>>(c, err, stats)),
                         (k_camera<64, true, FL, true><<<g, 256, 0, st>>>(c, err, stats)));
            else
                PICK_STK(depth, (k_camera<32, true, FL, false><<<g, 256, 0, st>>>(c, err, stats)),
                         (k_camera<64, true, FL, false><<<g, 256, 0, st>>>(c, err, stats)));
        });
    else
        // the specular term is a separate instantiation: inlined unconditionally it costs the plain
        // kernel 3 VGPRs and one wave per SIMD (78 -> 81 registers)
        with_flags(flags, [&](auto fl) {
            constexpr int FL = decltype(fl)::value;
            if (c.spec)
                PICK_STK(depth, (k_camera<32, false, FL, true><<<g, 256, 0, st>>>(c, err, nullptr)),
                         (k_camera<64, false, FL, true><<<g, 256, 0, st>>>(c, err, nullptr)));
            else
                PICK_STK(depth, (k_camera<32, false, FL, false><<<g, 256, 0, st>>>(c, err, nullptr)),
                         (k_camera<64, false, FL, false><<<g, 256, 0, st>>>(c, err, nullptr)));
        });
    LCHECK();
    return 0;
}

int launch_cast(const DevScene *sc, uint32_t depth, uint64_t n, const float *o, const float *d, float maxd, float *t,
                float *nrm, uint32_t *uuid, unsigned long long *counter, int *err, unsigned long long *stats,
                int ncu, hipStream_t st, int flags) {
    if (n == 0) return 0;
    if (depth + 1 > RT_STACK) {
        set_error("BVH depth " + std::to_string(depth) + " exceeds the traversal stack (" + std::to_string(RT_STACK) + ")");
        return -1;
    }
    k_zero_u64<<<1, 1, 0, st>>>(counter);
    const uint64_t chunks = (n + 63) / 64;
    const uint32_t g = (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>((uint64_t)8 * ncu, (chunks + 3) / 4));
    // castRays ignores texture masks (as CollisionDetection does); only the predicate flag applies
    with_flags(flags & RT_FL_WT, [&](auto fl) {
        constexpr int FL = decltype(fl)::value & RT_FL_WT;
        if (stats) k_cast_bin<RT_STACK, true, FL><<<g, 256, 0, st>>>(sc, n, o, d, maxd, t, nrm, uuid, counter, err, stats);
        else if ((flags & RT_FL_BLK) && (flags & RT_FL_WIDE))
            k_cast<4, FL | RT_FL_WIDE><<<g, 256, 0, st>>>(sc, n, o, d, maxd, t, nrm, uuid, counter, 64u, err);
        else if (flags & RT_FL_BLK) k_cast<4, FL><<<g, 256, 0, st>>>(sc, n, o, d, maxd, t, nrm, uuid, counter, 64u, err);
        else k_cast_bin<RT_STACK, false, FL><<<g, 256, 0, st>>>(sc, n, o, d, maxd, t, nrm, uuid, counter, err, nullptr);
    });
    LCHECK();
    return 0;
}

}  // namespace rt
