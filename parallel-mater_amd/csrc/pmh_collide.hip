// SPDX-License-Identifier: MIT
// Predictor, proxies, broadphase, narrowphase and the contact cache on
// gfx950, and the world step that chains them with the AVBD solve.
//
// Broadphase: the reference filters every proxy overlap (inclusive float
// AABB test) with the rules of pm_filter_rigid_spatial_candidates and
// orders pairs by (body, identity) (geometry.slang:829-947).  Here the
// proxies of bodies no larger than the largest dynamic proxy go into a
// uniform hash grid (cell = 1.0625 x that extent, keyed by the cell of the
// proxy's minimum corner, so any overlapping pair is found among the 27
// neighbouring cells); larger static proxies (floors, walls) form a short
// list every query scans.  Each dynamic body sorts its kept candidates, and
// an exclusive scan over the per-body counts emits the pairs in ascending
// code a*n+b.  The overlap test is the same comparison on the same floats,
// so the pair set and order equal the reference's bit for bit.
//
// Narrowphase: analytic spheres/capsules use closed forms, one thread per
// pair; convex meshes with <= 96 indices take the reference's SAT + face
// clipping path (rigid_convex_face_manifold and its swept variant,
// geometry.slang:1606-1853) on 16 lanes per pair.  Mesh pairs the face path
// declines take the triangle-pair path (leaf-pair candidates or BVH
// traversal): a screen of the leaf bounds, one thread per pair, then a
// wavefront or a block per pair that is left.
#include "pmh_internal.hpp"
#include "pmh_lanes.hpp"
#include "pmh_world.hpp"

#include <algorithm>

namespace pmh {

__device__ __forceinline__ V3 sv(const PmhVec3 &v) { return {v.x, v.y, v.z}; }
__device__ __forceinline__ Q sq(const PmhQuat &q) { return {q.x, q.y, q.z, q.w}; }
__device__ __forceinline__ PmhVec3 pv(V3 v) { return {v.x, v.y, v.z}; }
__device__ __forceinline__ PmhQuat pq(Q q) { return {q.x, q.y, q.z, q.w}; }
__device__ __forceinline__ V3 v3(float4 f) { return {f.x, f.y, f.z}; }
__device__ __forceinline__ float4 f4(V3 v, float w) { return make_float4(v.x, v.y, v.z, w); }
__device__ __forceinline__ V3 sarr(const float *a) { return {a[0], a[1], a[2]}; }
__device__ __forceinline__ V3 transform_point(const PmhRigidBodyState &s, V3 p) {
    return add(sv(s.position), rotate(sq(s.orientation), p));
}

// ---------------------------------------------------------------------
// Predictor + proxies (geometry.slang:524-612, 716-827).
// ---------------------------------------------------------------------
__device__ __forceinline__ float correction_reach(const PmhBodyParameters &p, const ShapeDev &s) {
    if (p.motion != kDynamic) return 0.0f;
    const V3 e = sub(sarr(s.mx), sarr(s.mn));
    return smin(0.5f, 0.25f * smax(0.0f, smin(e.x, smin(e.y, e.z))));
}

__device__ __forceinline__ V3 inverse_inertia_world(const PmhBodyParameters &p, Q o, V3 w) {
    const V3 l = inv_rotate(o, w);
    return rotate(o, {l.x * p.inverse_inertia_local.x, l.y * p.inverse_inertia_local.y,
                      l.z * p.inverse_inertia_local.z});
}

__global__ void k_integrate_proxy(uint32_t n, const PmhBodyParameters *P, const ShapeDev *shapes,
                                  const PmhRigidBodyState *cur, PmhRigidBodyState *prev,
                                  PmhRigidBodyState *pred, float4 *pmn, float4 *pmx, V3 g, float dt,
                                  float4 *inputs, const PmhRigidBodyState *targets, uint32_t *target_flags,
                                  uint32_t remaining, uint32_t first_substep, uint32_t last_substep,
                                  uint32_t *bucket_count, uint32_t buckets) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    // The hash table's counts, which the next kernel adds to.
    for (uint32_t k = i; k < buckets; k += gridDim.x * blockDim.x) bucket_count[k] = 0u;
    if (i >= n) return;
    const PmhBodyParameters b = P[i];
    const PmhRigidBodyState s0 = cur[i];
    prev[i] = s0;
    PmhRigidBodyState s = s0;
    const uint32_t target_active = target_flags[i];
    if (b.motion == kStatic) {
        s.linear_velocity = {0.0f, 0.0f, 0.0f};
        s.angular_velocity = {0.0f, 0.0f, 0.0f};
    } else if (b.motion == kKinematic) {
        if (target_active) {
            // The target moves 1/remaining of the way each substep and is
            // reached in the frame's last.
            const PmhRigidBodyState t = targets[i];
            const float fraction = 1.0f / float(remaining);
            const V3 p0 = sv(s0.position);
            const V3 p1 = add(p0, mul(sub(sv(t.position), p0), fraction));
            const Q o = sq(s0.orientation);
            Q q = sq(t.orientation);
            if (o.x * q.x + o.y * q.y + o.z * q.z + o.w * q.w < 0.0f) q = {-q.x, -q.y, -q.z, -q.w};
            const Q no = qnormalize({o.x + (q.x - o.x) * fraction, o.y + (q.y - o.y) * fraction,
                                     o.z + (q.z - o.z) * fraction, o.w + (q.w - o.w) * fraction});
            s.position = pv(p1);
            s.orientation = pq(no);
            s.linear_velocity = pv(mul(sub(p1, p0), 1.0f / dt));
            s.angular_velocity = pv(quaternion_delta_velocity(o, no, dt));
        } else {
            s.linear_velocity = {0.0f, 0.0f, 0.0f};
            s.angular_velocity = {0.0f, 0.0f, 0.0f};
        }
    } else {
        const V3 force = v3(inputs[4 * i]), torque = v3(inputs[4 * i + 1]);
        const V3 imp = v3(inputs[4 * i + 2]), aimp = v3(inputs[4 * i + 3]);
        V3 v = add(sv(s.linear_velocity), mul(add(g, mul(force, b.inverse_mass)), dt));
        V3 w = add(sv(s.angular_velocity), mul(inverse_inertia_world(b, sq(s.orientation), torque), dt));
        if (first_substep) {
            v = add(v, mul(imp, b.inverse_mass));
            w = add(w, inverse_inertia_world(b, sq(s.orientation), aimp));
        }
        v = mul(v, 1.0f / (1.0f + b.linear_damping * dt));
        w = mul(w, 1.0f / (1.0f + b.angular_damping * dt));
        v = clamp_length(v, b.maximum_linear_speed);
        w = clamp_length(w, b.maximum_angular_speed);
        const V3 p = add(sv(s.position), mul(v, dt));
        const Q o = sq(s.orientation);
        const Q d = qmul({w.x, w.y, w.z, 0.0f}, o);
        const Q no = qnormalize({o.x + 0.5f * d.x * dt, o.y + 0.5f * d.y * dt, o.z + 0.5f * d.z * dt,
                                 o.w + 0.5f * d.w * dt});
        s.position = pv(p);
        s.orientation = pq(no);
        s.linear_velocity = pv(v);
        s.angular_velocity = pv(w);
    }
    // pm_clear_rigid_inputs (geometry.slang:2877-2886) after the frame's
    // last substep: inputs and targets last one frame.
    if (last_substep) {
        const float4 z = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        inputs[4 * i] = z;
        inputs[4 * i + 1] = z;
        inputs[4 * i + 2] = z;
        inputs[4 * i + 3] = z;
        if (target_active) target_flags[i] = 0u;
    }
    pred[i] = s;
    // Proxy: production arguments path_deviation 0, correction_budget 1,
    // epsilon 1e-5 (production_realtime_backend.cu.inc:2663-2684).
    const ShapeDev sh = shapes[b.mesh_index];
    const float eps = 1.0e-5f;
    const float reach = len(sarr(sh.center)) + sh.bradius + b.collision_margin + eps;
    const float cr = correction_reach(b, sh);
    const V3 bc = {smin(1.0f, cr), smin(1.0f, cr), smin(1.0f, cr)};
    const V3 e = add(add(V3{0.0f, 0.0f, 0.0f}, bc), V3{reach, reach, reach});
    const V3 mn = sub(cmin(sv(s0.position), sv(s.position)), e);
    const V3 mx = add(cmax(sv(s0.position), sv(s.position)), e);
    pmn[i] = f4(mn, 0.0f);
    pmx[i] = f4(mx, 0.0f);
}

// ---------------------------------------------------------------------
// Broadphase.
// ---------------------------------------------------------------------
__device__ __forceinline__ uint32_t cell_hash(int x, int y, int z) {
    uint32_t h = uint32_t(x) * 0x8da6b343u ^ uint32_t(y) * 0xd8163841u ^ uint32_t(z) * 0xcb1ab31fu;
    h ^= h >> 15;
    h *= 0x2c1b3c6du;
    h ^= h >> 12;
    return h;
}

constexpr int kLargeCell = 0x7fffffff;

// Proxies no wider than `cell` go into the hash grid under the cell of
// their minimum corner; wider ones (floors, walls, fast movers) into the
// large list.  Any overlapping gridded pair then lies in neighbouring cells.
__global__ void k_bp_cells(uint32_t n, const float4 *pmn, const float4 *pmx, int4 *cell_of, uint32_t *bucket_count,
                           uint32_t table_mask, uint32_t *large, StepCounters *ctr, float cell) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float4 mn = pmn[i], mx = pmx[i];
    const float ext = smax(mx.x - mn.x, smax(mx.y - mn.y, mx.z - mn.z));
    if (!(ext <= cell) || !isfinite(mn.x) || !isfinite(mn.y) || !isfinite(mn.z)) {
        large[atomicAdd(&ctr->large_count, 1u)] = i;
        cell_of[i] = make_int4(kLargeCell, kLargeCell, kLargeCell, 0);
        return;
    }
    const int cx = int(floorf(mn.x / cell)), cy = int(floorf(mn.y / cell)), cz = int(floorf(mn.z / cell));
    const uint32_t b = cell_hash(cx, cy, cz) & table_mask;
    cell_of[i] = make_int4(cx, cy, cz, int(b));
    atomicAdd(&bucket_count[b], 1u);
}

// Places each body in its bucket and copies, in entry order, what a query
// tests of a candidate (cell, dynamic flag, box), so the query reads those
// records by entry index instead of gathering them by body index.
__global__ void k_bp_scatter(uint32_t n, const PmhBodyParameters *P, const float4 *pmn, const float4 *pmx,
                             const int4 *cell_of, const uint32_t *bucket_start, uint32_t *count, int4 *entry_cell,
                             float4 *entry_mn, float4 *entry_mx) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int4 c = cell_of[i];
    if (c.x == kLargeCell) return;
    const uint32_t e = bucket_start[c.w] + atomicSub(&count[c.w], 1u) - 1u;
    const float4 mn = pmn[i];
    entry_cell[e] = make_int4(c.x, c.y, c.z, P[i].motion == kDynamic ? 1 : 0);
    entry_mn[e] = make_float4(mn.x, mn.y, mn.z, __uint_as_float(i));
    entry_mx[e] = pmx[i];
}

__device__ __forceinline__ bool overlap(float4 amn, float4 amx, float4 bmn, float4 bmx) {
    return amn.x <= bmx.x && amx.x >= bmn.x && amn.y <= bmx.y && amx.y >= bmn.y && amn.z <= bmx.z &&
           amx.z >= bmn.z;
}

// Collision exclusions of joints (geometry.slang:494-511, 3108-3136): bodies
// of one weld group never collide, and a pair joined by a joint with
// disable_collisions does not while that joint is alive, enabled and
// unbroken.  A null `weld` or `excl_start` turns that test off.
// A batch of independent scenes adds the scene filter: bodies of
// different scenes never pair (null `scene`: one scene).
struct JointFilter {
    const uint32_t *weld = nullptr;
    const uint32_t *excl_start = nullptr;
    const uint2 *excl_list = nullptr;   // (partner, joint)
    const PmhRigidConstraint *joints = nullptr;
    const uint32_t *scene = nullptr;    // scene of each body
    // Batch: each scene's large bodies (a segment of scene_large per scene)
    // and each scene's body range.
    const uint32_t *scene_large_start = nullptr, *scene_large = nullptr;
    const uint32_t *scene_first = nullptr, *scene_count = nullptr;
};

__device__ __forceinline__ bool joint_excluded(const JointFilter &f, uint32_t a, uint32_t b) {
    if (f.scene && f.scene[a] != f.scene[b]) return true;
    if (f.weld && f.weld[a] == f.weld[b]) return true;
    if (f.excl_start) {
        for (uint32_t e = f.excl_start[a]; e < f.excl_start[a + 1]; ++e) {
            const uint2 x = f.excl_list[e];
            if (x.x == b && f.joints[x.y].state_broken == 0u) return true;
        }
    }
    return false;
}

__device__ uint32_t weld_find(const uint32_t *weld, uint32_t v) {
    uint32_t p = __hip_atomic_load(&weld[v], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    while (p != v) {
        v = p;
        p = __hip_atomic_load(&weld[v], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    return v;
}

__global__ void k_weld_init(uint32_t n, uint32_t *weld) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) weld[i] = i;
}

// Fixed joints that disable collisions join their bodies' weld group; the
// larger root hooks under the smaller, so each group's root is its
// smallest index whatever the order of the hooks.
__global__ void k_weld_hook(uint32_t n, uint32_t nj, const PmhRigidConstraint *joints, uint32_t *weld) {
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= nj) return;
    const PmhRigidConstraint &j = joints[k];
    const PmhRigidConstraintOptions &o = j.options;
    if (j.alive == 0u || o.enabled == 0u || j.state_broken != 0u || o.disable_collisions == 0u ||
        o.type != kJointFixed)
        return;
    if (o.body_a.index >= n || o.body_a.generation != 1u || o.body_b.index >= n || o.body_b.generation != 1u)
        return;
    uint32_t u = weld_find(weld, o.body_a.index), v = weld_find(weld, o.body_b.index);
    while (u != v) {
        if (u > v) { const uint32_t t = u; u = v; v = t; }
        const uint32_t old = atomicCAS(&weld[v], v, u);
        if (old == v) break;
        u = weld_find(weld, u);
        v = weld_find(weld, old);
    }
}

__global__ void k_weld_compress(uint32_t n, uint32_t *weld) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) weld[i] = weld_find(weld, i);
}

// A batch's large bodies by scene: counts, then (after a scan over the
// scenes) placement.  The order within a scene's segment is free: every
// query sorts its candidates.
__global__ void k_scene_large(const StepCounters *ctr, const uint32_t *large, const uint32_t *scene,
                              uint32_t *count, const uint32_t *start, uint32_t *out) {
    const uint32_t nl = ctr->large_count;
    for (uint32_t k = blockIdx.x * blockDim.x + threadIdx.x; k < nl; k += gridDim.x * blockDim.x) {
        const uint32_t b = large[k];
        const uint32_t slot = atomicAdd(&count[scene[b]], 1u);
        if (start) out[start[scene[b]] + slot] = b;
    }
}

// Grid query, a group of 32 lanes per body: the entries of the body's 27
// cells' buckets as one list dealt over the lanes (a bucket has none, a few
// or, in a crowd, dozens, and a lane per cell waited for the longest chain),
// two at a time so that their loads overlap.  Pass 0 gathers what it finds in
// LDS, counts it, and leaves it sorted ascending (identity order = index) in
// the body's segment of `pool`, `segment` candidates for every body; pass 1
// copies it to the body's offset (an exclusive scan of the counts).  A body
// with more candidates walks again in pass 1 and sorts where it writes, so a
// body may own any number of pairs.  Bounded by the latency of bucket, entry
// and box loads.  Counting in pass 0 and walking twice more in pass 1 took
// 217 + 416 us of a step of 32768 bodies (0.52M pairs), now 60 + 9;
// segments reserved from one counter instead of laid out took 330 us, and 405
// over 65538 chain links (by segments 52).
constexpr uint32_t kQueryLanes = 32, kQueryBlock = 256;
constexpr uint32_t kQueryHeld = 128;       // candidates of a body held in LDS

template <int kPass>
__global__ void __launch_bounds__(kQueryBlock) k_bp_query(uint32_t n, const PmhBodyParameters *P, const float4 *pmn,
                                                  const float4 *pmx, const int4 *cell_of, const uint32_t *bucket_start,
                                                  const int4 *entry_cell, const float4 *entry_mn,
                                                  const float4 *entry_mx, uint32_t table_mask, const uint32_t *large,
                                                  uint32_t *cand_count, uint32_t *pool, uint32_t segment,
                                                  const uint32_t *offset, uint32_t *code, uint2 *ab,
                                                  const StepCounters *ctr, JointFilter jf) {
    constexpr uint32_t groups = kQueryBlock / kQueryLanes;
    __shared__ uint32_t s_held[kPass == 0 ? groups : 1][kQueryHeld];
    // Every exit is uniform over the body's group.
    const uint32_t g = threadIdx.x / kQueryLanes, q = threadIdx.x % kQueryLanes;
    const uint32_t a = blockIdx.x * groups + g;
    const uint32_t below = (1u << q) - 1u;
    if (a >= n) return;
    if (P[a].motion != kDynamic) {
        if (kPass == 0 && q == 0) cand_count[a] = 0;
        return;
    }
    if (kPass == 1 && ctr->pairs == 0) return;   // pair pool overflow: nothing is emitted
    const int4 c = cell_of[a];
    if (c.x == kLargeCell) return;   // k_bp_large owns this body
    uint32_t *mine = pool + size_t(a) * segment;
    uint32_t base = 0;
    if (kPass == 1) {
        const uint32_t total = cand_count[a];
        base = offset[a];
        if (total <= segment) {
            for (uint32_t k = q; k < total; k += kQueryLanes) {
                const uint32_t b = mine[k];
                code[base + k] = a * n + b;
                ab[base + k] = make_uint2(a, b);
            }
            return;
        }
    }
    const float4 amn = pmn[a], amx = pmx[a];
    uint32_t first = 0, len = 0;
    if (q < 27u) {
        const uint32_t bk = cell_hash(c.x + int(q % 3u) - 1, c.y + int((q / 3u) % 3u) - 1, c.z + int(q / 9u) - 1) &
                            table_mask;
        first = bucket_start[bk];
        len = bucket_start[bk + 1] - first;
    }
    uint32_t incl = len;
    for (uint32_t d = 1; d < kQueryLanes; d <<= 1) {
        const uint32_t y = __shfl_up(incl, d, kQueryLanes);
        if (q >= d) incl += y;
    }
    const uint32_t entries = __shfl(incl, kQueryLanes - 1, kQueryLanes);
    first -= incl - len;                             // entry f of the list is first + f
    // Calls emit(slot, body) for every candidate, slots in the order found.
    auto walk = [&](auto &&emit) -> uint32_t {
        uint32_t found = 0;
        auto gather = [&](bool hit, uint32_t b) {
            const uint32_t mask = uint32_t(__ballot(hit) >> (threadIdx.x & 32u));
            if (hit) emit(found + uint32_t(__popc(mask & below)), b);
            found += uint32_t(__popc(mask));
        };
        for (uint32_t f0 = 0; f0 < entries; f0 += 2 * kQueryLanes) {
            int4 at[2], cb[2];
            float4 bmn[2], bmx[2];
#pragma unroll
            for (uint32_t u = 0; u < 2; ++u) {
                const uint32_t f = min(f0 + u * kQueryLanes + q, entries - 1u);
                uint32_t k = 0;                          // its cell: as many lists end at or before f
#pragma unroll
                for (uint32_t step = kQueryLanes / 2; step >= 1u; step /= 2)
                    if (__shfl(incl, k + step - 1u, kQueryLanes) <= f) k += step;
                const uint32_t e = f + __shfl(first, k, kQueryLanes);
                at[u] = make_int4(c.x + int(k % 3u) - 1, c.y + int((k / 3u) % 3u) - 1, c.z + int(k / 9u) - 1, 0);
                cb[u] = entry_cell[e];
                bmn[u] = entry_mn[e];
                bmx[u] = entry_mx[e];
            }
#pragma unroll
            for (uint32_t u = 0; u < 2; ++u) {
                const uint32_t b = __float_as_uint(bmn[u].w);
                const bool hit = f0 + u * kQueryLanes + q < entries && cb[u].x == at[u].x && cb[u].y == at[u].y &&
                                 cb[u].z == at[u].z && b != a && (cb[u].w == 0 || a < b) &&
                                 overlap(amn, amx, bmn[u], bmx[u]) && !joint_excluded(jf, a, b);
                gather(hit, b);
            }
        }
        const uint32_t *list = large;
        uint32_t lb = 0, le = ctr->large_count;
        if (jf.scene_large) {
            const uint32_t sc = jf.scene[a];
            list = jf.scene_large;
            lb = jf.scene_large_start[sc];
            le = jf.scene_large_start[sc + 1];
        }
        for (; lb < le; lb += kQueryLanes) {
            const uint32_t b = lb + q < le ? list[lb + q] : a;
            const bool hit = b != a && (P[b].motion != kDynamic || a < b) && overlap(amn, amx, pmn[b], pmx[b]) &&
                             !joint_excluded(jf, a, b);
            gather(hit, b);
        }
        return found;
    };
    if (kPass == 0) {
        const uint32_t total = walk([&](uint32_t slot, uint32_t b) {
            if (slot < kQueryHeld) s_held[g][slot] = b;
        });
        if (q == 0) cand_count[a] = total;
        if (total > segment) return;
        __threadfence_block();
        __builtin_amdgcn_wave_barrier();
        // Rank sort: element k goes to the count of elements below it (a body
        // is found once).
        for (uint32_t k = q; k < total; k += kQueryLanes) {
            const uint32_t v = s_held[g][k];
            uint32_t rank = 0;
            for (uint32_t i = 0; i < total; ++i) rank += s_held[g][i] < v ? 1u : 0u;
            mine[rank] = v;
        }
        return;
    }
    uint32_t *out = code + base;
    const uint32_t total = walk([&](uint32_t slot, uint32_t b) { out[slot] = b; });
    // The segment's writes of every lane are visible to the whole group.
    __threadfence_block();
    __builtin_amdgcn_wave_barrier();
    // The pairs are written first, then the codes from them, since the codes'
    // slots hold the unsorted segment.
    for (uint32_t k = q; k < total; k += kQueryLanes) {
        const uint32_t v = out[k];
        uint32_t rank = 0;
        for (uint32_t i = 0; i < total; ++i) rank += out[i] < v ? 1u : 0u;
        ab[base + rank] = make_uint2(a, v);
    }
    __threadfence_block();
    __builtin_amdgcn_wave_barrier();
    for (uint32_t k = q; k < total; k += kQueryLanes) out[k] = a * n + ab[base + k].y;
}

__global__ void k_set_pairs(StepCounters *ctr, const uint32_t *offset, uint32_t n, uint32_t pair_cap) {
    if (threadIdx.x != 0) return;
    const uint32_t M = offset[n];
    if (M > pair_cap) {
        atomicOr(&ctr->status, kStatusPairOverflow);
        ctr->pairs = 0;
    } else {
        ctr->pairs = M;
    }
}

// Large bodies: one block scans every body in index order; a block-wide
// prefix sum places the hits, so the segment comes out ascending.  Blocks
// beyond the number of large bodies return at once.
// Four chunks of 256 at a time, their boxes loaded together: one chunk took
// 0.36 us for its two loads and barriers (65538 bodies, 93 us a pass, now
// 36).
constexpr uint32_t kLargeBlocks = 1024, kLargeChunks = 4;
template <int kPass>
__global__ void __launch_bounds__(256) k_bp_large(uint32_t n, const PmhBodyParameters *P, const float4 *pmn,
                                                  const float4 *pmx, const uint32_t *large, uint32_t *cand_count,
                                                  const uint32_t *offset, uint32_t *code, uint2 *ab,
                                                  const StepCounters *ctr, JointFilter jf) {
    __shared__ uint32_t warp_tot[kLargeChunks][4];
    const uint32_t nl = ctr->large_count;
    const uint32_t lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    for (uint32_t k = blockIdx.x; k < nl; k += gridDim.x) {
        const uint32_t a = large[k];
        if (P[a].motion != kDynamic) {
            if (kPass == 0 && threadIdx.x == 0) cand_count[a] = 0;
            continue;
        }
        if (kPass == 1 && ctr->pairs == 0) continue;
        const float4 amn = pmn[a], amx = pmx[a];
        uint32_t running = kPass == 1 ? offset[a] : 0u;
        // In a batch only the body's own scene can pair with it.
        const uint32_t first = jf.scene_first ? jf.scene_first[jf.scene[a]] : 0u;
        const uint32_t last = jf.scene_first ? first + jf.scene_count[jf.scene[a]] : n;
        for (uint32_t base = first; base < last; base += 256 * kLargeChunks) {
            float4 bmn[kLargeChunks], bmx[kLargeChunks];
            uint64_t bal[kLargeChunks];
#pragma unroll
            for (uint32_t u = 0; u < kLargeChunks; ++u) {
                const uint32_t b = min(base + u * 256 + threadIdx.x, last - 1u);
                bmn[u] = pmn[b];
                bmx[u] = pmx[b];
            }
#pragma unroll
            for (uint32_t u = 0; u < kLargeChunks; ++u) {
                const uint32_t b = base + u * 256 + threadIdx.x;
                const bool hit = b < last && b != a && overlap(amn, amx, bmn[u], bmx[u]) &&
                                 !(P[b].motion == kDynamic && !(a < b)) && !joint_excluded(jf, a, b);
                bal[u] = __ballot(hit);
                if (lane == 0) warp_tot[u][wid] = __popcll(bal[u]);
            }
            __syncthreads();
#pragma unroll
            for (uint32_t u = 0; u < kLargeChunks; ++u) {
                uint32_t before = 0, total = 0;
                for (uint32_t w = 0; w < 4; ++w) {
                    if (w < wid) before += warp_tot[u][w];
                    total += warp_tot[u][w];
                }
                if (kPass == 1 && ((bal[u] >> lane) & 1ull) != 0ull) {
                    const uint32_t b = base + u * 256 + threadIdx.x;
                    const uint32_t pos = running + before + __popcll(bal[u] & ((1ull << lane) - 1ull));
                    code[pos] = a * n + b;
                    ab[pos] = make_uint2(a, b);
                }
                running += total;
            }
            __syncthreads();
        }
        if (kPass == 0 && threadIdx.x == 0) cand_count[a] = running;
    }
}

// ---------------------------------------------------------------------
// Narrowphase.
// ---------------------------------------------------------------------
struct Contact {
    V3 normal, point;
    float pen, impact_fraction;
};
struct Manifold {
    Contact c[8];
    uint32_t count;
    uint32_t face_patch;
};

struct ShapeView {
    ShapeDev s;
    const V3 *v;
    const uint32_t *idx;
    const float4 *planes;
    const BvhDev *nodes = nullptr;
    const uint32_t *leaves = nullptr;
    const float4 *shell = nullptr;
    __device__ float4 plane(uint32_t f) const { return planes[s.plane_off + f]; }
    __device__ V3 vert(uint32_t k) const { return v[s.vtx_off + k]; }
    __device__ uint32_t index(uint32_t k) const { return idx[s.idx_off + k]; }
    __device__ const BvhDev &node(uint32_t k) const { return nodes[s.node_off + k]; }
    __device__ uint32_t leaf(uint32_t k) const { return leaves[s.leaf_off + k]; }
};

// rigid_add_contact, geometry.slang:1129-1220 (unguided, no swept-witness
// canonicalisation on the convex face path).
__device__ void add_contact(Manifold &m, const Contact &c, float spacing) {
    const float sp2 = spacing * spacing;
    for (uint32_t i = 0; i < m.count; ++i) {
        if (len2(sub(m.c[i].point, c.point)) < sp2) {
            if (c.pen - m.c[i].pen > 0.0f) m.c[i] = c;
            return;
        }
    }
    if (m.count < 8u) { m.c[m.count++] = c; return; }
    uint32_t sh = 0;
    for (uint32_t i = 1; i < m.count; ++i) if (m.c[i].pen < m.c[sh].pen) sh = i;
    if (c.pen > m.c[sh].pen) m.c[sh] = c;
}

// ---- hinge contact frames (joints that shape contacts) ------------------
using HingeFrame = PmhHingeContactFrame;

__device__ __forceinline__ bool guided_pair(const HingeFrame &a, const HingeFrame &b) {   // geometry.slang:373-377
    return (a.axial != 0u && b.static_body != 0u) || (b.axial != 0u && a.static_body != 0u);
}

// rigid_guide_direction, geometry.slang:1118-1127 (`g` is the pair's axial frame).
__device__ __forceinline__ V3 guide_direction(const Contact &c, const HingeFrame &g) {
    return {dot(c.normal, sv(g.axis)) * sqrtf(g.inverse_mass),
            g.axial_rotation != 0u ? dot(sv(g.axis), cross(sub(c.point, sv(g.anchor)), c.normal)) * sqrtf(g.inverse_moment)
                                   : 0.0f,
            0.0f};
}

// rigid_add_contact's guided branch, geometry.slang:1129-1168: the first
// impact keeps its rows (later impacts are dropped, earlier ones replace
// the swept rows), and a contact whose guide direction matches a kept one
// replaces it when it is deeper per unit of direction.  All contacts of a
// pair share its frames, so `g` serves for both.
__device__ void add_contact_guided(Manifold &m, const Contact &c, const HingeFrame &g) {
    const V3 cand_dir = guide_direction(c, g);
    const float cand_len = len(cand_dir);
    if (cand_len * cand_len <= kEpsilon) return;
    if (c.impact_fraction > 0.0f) {
        float first_impact = 1.0f;
        for (uint32_t r = 0; r < m.count; ++r)
            if (m.c[r].impact_fraction > 0.0f) first_impact = smin(first_impact, m.c[r].impact_fraction);
        if (c.impact_fraction > first_impact + 1.0e-4f) return;
        if (c.impact_fraction < first_impact - 1.0e-4f) {
            uint32_t kept = 0;
            for (uint32_t r = 0; r < m.count; ++r)
                if (m.c[r].impact_fraction == 0.0f) m.c[kept++] = m.c[r];
            m.count = kept;
        }
    }
    for (uint32_t i = 0; i < m.count; ++i) {
        const V3 dir = guide_direction(m.c[i], g);
        const float size = len(dir);
        if (dot(cand_dir, dir) > 0.9999f * cand_len * size) {
            if (c.pen / cand_len > m.c[i].pen / size) m.c[i] = c;
            return;
        }
    }
    if (m.count < 8u) { m.c[m.count++] = c; return; }
    uint32_t sh = 0;
    for (uint32_t i = 1; i < m.count; ++i) if (m.c[i].pen < m.c[sh].pen) sh = i;
    if (c.pen > m.c[sh].pen) m.c[sh] = c;
}

// rigid_fixed_hinge_inverse_moment, geometry.slang:384-402.
__device__ float fixed_hinge_inverse_moment(const PmhBodyParameters &p, const PmhRigidBodyState &s,
                                            const HingeFrame &f) {
    if ((f.fixed == 0u && f.axial_rotation == 0u) || p.inverse_mass <= kEpsilon) return 0.0f;
    const V3 la = inv_rotate(sq(s.orientation), sv(f.axis));
    const float center = la.x * la.x / smax(p.inverse_inertia_local.x, kEpsilon) +
                         la.y * la.y / smax(p.inverse_inertia_local.y, kEpsilon) +
                         la.z * la.z / smax(p.inverse_inertia_local.z, kEpsilon);
    const V3 arm = sub(sv(s.position), sv(f.anchor));
    const V3 perpendicular = sub(arm, mul(sv(f.axis), dot(arm, sv(f.axis))));
    const float pivot = center + len2(perpendicular) / p.inverse_mass;
    return pivot > kEpsilon ? 1.0f / pivot : 0.0f;
}

// The world's joints as the narrowphase sees them: the records and each
// body's candidate joints (alive, both ids valid) in descending index.
struct JointView {
    const PmhRigidConstraint *joints = nullptr;
    const uint32_t *list_start = nullptr, *list = nullptr;
};

// rigid_hinge_contact_frame, geometry.slang:404-491: over the body's
// enabled, unbroken joints in ascending index, the first hinge (or slider
// or piston held by a static body with no breaking threshold) gives the
// frame, anchored on the static body when that holds it; a slider or
// piston counts only as the body's single joint; fixed and point members
// are flagged.  `reference` is the anchor of a non-axial frame, else the
// body's position.  Body ids are {dense index, 1}.
__device__ HingeFrame hinge_frame(const JointView &jv, const PmhBodyParameters *P, uint32_t n,
                                  const PmhRigidBodyState *states, uint32_t dense, const PmhRigidBodyState &state,
                                  V3 &reference) {
    HingeFrame r;
    memset(&r, 0, sizeof r);
    const PmhBodyParameters pd = P[dense];
    r.static_body = pd.motion == kStatic ? 1u : 0u;
    if (pd.inverse_mass <= 0.0f || !jv.joints) {
        reference = sv(state.position);
        return r;
    }
    uint32_t incident = 0;
    for (uint32_t e = jv.list_start[dense + 1]; e > jv.list_start[dense]; --e) {
        const PmhRigidConstraint &j = jv.joints[jv.list[e - 1]];
        const PmhRigidConstraintOptions &o = j.options;
        if (j.alive == 0u || o.enabled == 0u || j.state_broken != 0u) continue;
        const bool is_a = o.body_a.index == dense && o.body_a.generation == 1u;
        const bool is_b = o.body_b.index == dense && o.body_b.generation == 1u;
        if (!is_a && !is_b) continue;
        ++incident;
        if (o.type == kJointFixed) r.fixed_member = 1u;
        if (o.type == kJointPoint) r.point_member = 1u;
        const bool axial = o.type == kJointPiston || o.type == kJointSlider;
        const PmhBodyId oid = is_a ? o.body_b : o.body_a;
        const uint32_t other = oid.index < n && oid.generation == 1u ? oid.index : kInvalid;
        const bool static_anchor = other != kInvalid && P[other].motion == kStatic;
        if (r.present != 0u ||
            (o.type != kJointHinge && !(axial && static_anchor && o.breaking_impulse_threshold <= 0.0f)))
            continue;
        const V3 local_axis = axial ? V3{1.0f, 0.0f, 0.0f} : V3{0.0f, 0.0f, 1.0f};
        r.local_anchor = is_a ? o.local_anchor_a : o.local_anchor_b;
        const Q lo = sq(is_a ? o.local_orientation_a : o.local_orientation_b);
        const Q so = sq(state.orientation);
        V3 anchor = add(sv(state.position), rotate(so, sv(r.local_anchor)));
        V3 axis = normalized_or(rotate(qmul(so, lo), local_axis), local_axis);
        r.present = 1u;
        r.fixed = static_anchor && !axial ? 1u : 0u;
        r.axial = static_anchor && axial ? 1u : 0u;
        r.axial_rotation = r.axial != 0u && o.type == kJointPiston ? 1u : 0u;
        if (static_anchor) {
            const PmhRigidBodyState os = states[other];
            const Q oo = sq(os.orientation);
            anchor = add(sv(os.position), rotate(oo, sv(is_a ? o.local_anchor_b : o.local_anchor_a)));
            axis = normalized_or(rotate(qmul(oo, sq(is_a ? o.local_orientation_b : o.local_orientation_a)), local_axis),
                                 axis);
        }
        r.anchor = pv(anchor);
        r.axis = pv(axis);
    }
    if (r.axial != 0u && incident != 1u) {
        r.axial = 0u;
        r.axial_rotation = 0u;
        r.present = 0u;
    }
    if (r.axial != 0u) {
        r.inverse_mass = pd.inverse_mass;
        r.inverse_moment = fixed_hinge_inverse_moment(pd, state, r);
    }
    reference = r.present != 0u && r.axial == 0u ? sv(r.anchor) : sv(state.position);
    return r;
}

// Per body: its frame at the predicted state and its reference point at the
// previous and the predicted state (.xyz of ref[2i], ref[2i + 1]).  Worlds
// without joints skip this: every frame then carries only the static flag.
__global__ void k_hinge_frames(uint32_t n, const PmhBodyParameters *P, const PmhRigidBodyState *prev,
                               const PmhRigidBodyState *pred, JointView jv, HingeFrame *frames, float4 *ref) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    V3 rp, rc;
    (void)hinge_frame(jv, P, n, prev, i, prev[i], rp);
    frames[i] = hinge_frame(jv, P, n, pred, i, pred[i], rc);
    ref[2 * i] = f4(rp, 0.0f);
    ref[2 * i + 1] = f4(rc, 0.0f);
}

// The frames of one pair, and the body's reference points.
struct PairFrames {
    HingeFrame ha, hb;
    V3 ref_prev, ref;
};
__device__ __forceinline__ PairFrames pair_frames(const HingeFrame *frames, const float4 *ref, const PmhBodyParameters &pa,
                                                  const PmhBodyParameters &pb, uint2 p, const PmhRigidBodyState &A0,
                                                  const PmhRigidBodyState &A) {
    PairFrames f;
    if (frames) {
        f.ha = frames[p.x];
        f.hb = frames[p.y];
        f.ref_prev = v3(ref[2 * p.x]);
        f.ref = v3(ref[2 * p.x + 1]);
    } else {
        memset(&f.ha, 0, sizeof f.ha);
        memset(&f.hb, 0, sizeof f.hb);
        f.ha.static_body = pa.motion == kStatic ? 1u : 0u;
        f.hb.static_body = pb.motion == kStatic ? 1u : 0u;
        f.ref_prev = sv(A0.position);
        f.ref = sv(A.position);
    }
    return f;
}

__device__ float rotational_motion_bound(const PmhRigidBodyState &p, const PmhRigidBodyState &c,
                                         const ShapeDev &s) {
    const Q d = relative_quaternion(sq(p.orientation), sq(c.orientation), false);
    const float sh = len({d.x, d.y, d.z});
    const V3 ma = {smax(fabsf(s.mn[0]), fabsf(s.mx[0])), smax(fabsf(s.mn[1]), fabsf(s.mx[1])),
                   smax(fabsf(s.mn[2]), fabsf(s.mx[2]))};
    return 2.0f * len(ma) * sh;
}

__device__ bool requires_swept(const PmhRigidBodyState &pa, const PmhRigidBodyState &a, const ShapeDev &ma,
                               const PmhRigidBodyState &pb, const PmhRigidBodyState &b, const ShapeDev &mb,
                               float threshold) {
    const bool planes_a = ma.kind != kShapeMesh || ma.has_planes;
    const bool planes_b = mb.kind != kShapeMesh || mb.has_planes;
    if (!planes_a || !planes_b) threshold = smin(threshold, 1.0e-3f);
    const V3 rel = sub(sub(sv(a.position), sv(pa.position)), sub(sv(b.position), sv(pb.position)));
    return len(rel) + rotational_motion_bound(pa, a, ma) + rotational_motion_bound(pb, b, mb) > threshold;
}

// Analytic round shapes (no reference counterpart).  The normal points
// from the collider towards the body; the point is the midpoint of the two
// surface points; penetration = rest offset - separation + 1e-5.
__device__ __forceinline__ V3 closest_on_segment(V3 p0, V3 p1, V3 q) {
    const V3 d = sub(p1, p0);
    const float dd = len2(d);
    const float t = dd > 0.0f ? clampf(dot(sub(q, p0), d) / dd, 0.0f, 1.0f) : 0.0f;
    return add(p0, mul(d, t));
}

__device__ bool point_shape_distance(V3 c, const PmhRigidBodyState &ss, const ShapeDev &sh, V3 &normal,
                                     V3 &surface, float &distance) {
    const Q o = sq(ss.orientation);
    const V3 sp = sv(ss.position);
    if (sh.kind == kShapeSphere) {
        const V3 d = sub(c, sp);
        normal = normalized_or(d, {0.0f, 1.0f, 0.0f});
        distance = len(d) - sh.sphere_radius;
        surface = add(sp, mul(normal, sh.sphere_radius));
        return true;
    }
    if (sh.kind == kShapeCapsule) {
        const V3 axis = rotate(o, {0.0f, sh.half_length, 0.0f});
        const V3 p = closest_on_segment(sub(sp, axis), add(sp, axis), c);
        const V3 d = sub(c, p);
        normal = normalized_or(d, rotate(o, {1.0f, 0.0f, 0.0f}));
        distance = len(d) - sh.sphere_radius;
        surface = add(p, mul(normal, sh.sphere_radius));
        return true;
    }
    if (!sh.is_box) return false;
    const V3 half = sarr(sh.box_half);
    const V3 l = inv_rotate(o, sub(c, sp));
    V3 q = {clampf(l.x, -half.x, half.x), clampf(l.y, -half.y, half.y), clampf(l.z, -half.z, half.z)};
    const bool inside = q.x == l.x && q.y == l.y && q.z == l.z;
    V3 ln;
    float dist;
    if (!inside) {
        const V3 d = sub(l, q);
        const float dl = len(d);
        ln = mul(d, 1.0f / dl);
        dist = dl;
    } else {
        const float dx = half.x - fabsf(l.x), dy = half.y - fabsf(l.y), dz = half.z - fabsf(l.z);
        if (dx <= dy && dx <= dz) { ln = {l.x < 0.0f ? -1.0f : 1.0f, 0.0f, 0.0f}; q.x = l.x < 0.0f ? -half.x : half.x; dist = -dx; }
        else if (dy <= dz) { ln = {0.0f, l.y < 0.0f ? -1.0f : 1.0f, 0.0f}; q.y = l.y < 0.0f ? -half.y : half.y; dist = -dy; }
        else { ln = {0.0f, 0.0f, l.z < 0.0f ? -1.0f : 1.0f}; q.z = l.z < 0.0f ? -half.z : half.z; dist = -dz; }
    }
    normal = rotate(o, ln);
    surface = transform_point(ss, q);
    distance = dist;
    return true;
}

__device__ void push_round_contact(Manifold &m, V3 normal, V3 surface_collider, float gap, float margin,
                                   float reach) {
    if (gap > reach) return;
    const float rest = smin(margin, 1.0e-3f);
    Contact c;
    c.normal = normal;
    c.point = add(surface_collider, mul(normal, gap * 0.5f));
    c.pen = rest - gap + 1.0e-5f;
    c.impact_fraction = 1.0f;
    add_contact(m, c, smax(margin * 2.0f, 1.0e-4f));
}

__device__ bool analytic_manifold(const PmhRigidBodyState &as, const ShapeDev &am, const PmhRigidBodyState &bs,
                                  const ShapeDev &bm, float margin, float reach, Manifold &out) {
    out.count = 0;
    out.face_patch = 0;
    const bool a_round = am.kind == kShapeSphere || am.kind == kShapeCapsule;
    const bool b_round = bm.kind == kShapeSphere || bm.kind == kShapeCapsule;
    if (!a_round && !b_round) return false;
    V3 n, s;
    float d;
    if (am.kind == kShapeSphere) {
        if (!point_shape_distance(sv(as.position), bs, bm, n, s, d)) return false;
        push_round_contact(out, n, s, d - am.sphere_radius, margin, reach);
        return true;
    }
    if (bm.kind == kShapeSphere) {
        if (!point_shape_distance(sv(bs.position), as, am, n, s, d)) return false;
        const V3 nb = mul(n, -1.0f);
        const V3 sb = sub(sv(bs.position), mul(n, bm.sphere_radius));
        push_round_contact(out, nb, sb, d - bm.sphere_radius, margin, reach);
        return true;
    }
    const bool a_cap = am.kind == kShapeCapsule;
    const ShapeDev &cap = a_cap ? am : bm;
    const PmhRigidBodyState &cs = a_cap ? as : bs;
    const ShapeDev &other = a_cap ? bm : am;
    const PmhRigidBodyState &os = a_cap ? bs : as;
    const V3 axis = rotate(sq(cs.orientation), {0.0f, cap.half_length, 0.0f});
    V3 ends[3] = {sub(sv(cs.position), axis), add(sv(cs.position), axis), sv(cs.position)};
    uint32_t samples = 2;
    if (other.kind == kShapeCapsule) {
        const V3 oaxis = rotate(sq(os.orientation), {0.0f, other.half_length, 0.0f});
        ends[2] = closest_on_segment(ends[0], ends[1],
                                     closest_on_segment(sub(sv(os.position), oaxis), add(sv(os.position), oaxis),
                                                        sv(cs.position)));
        samples = 3;
    }
    for (uint32_t k = 0; k < samples; ++k) {
        if (!point_shape_distance(ends[k], os, other, n, s, d)) return false;
        const float gap = d - cap.sphere_radius;
        if (a_cap) push_round_contact(out, n, s, gap, margin, reach);
        else push_round_contact(out, mul(n, -1.0f), sub(ends[k], mul(n, cap.sphere_radius)), gap, margin, reach);
    }
    return true;
}

// ---------------------------------------------------------------------
// Triangle-pair narrowphase: mesh pairs the convex face path does not take
// (edge-on-edge contacts of convex meshes, non-convex or large meshes).
// Same steps and float operations as rigid_collide_triangle_ranges and its
// swept variant (geometry.slang:949-1117, 1272-1584, 1855-2154), the
// leaf-pair candidate order of pm_generate_rigid_leaf_pairs (:2303-2492),
// the per-candidate merge of pm_evaluate_rigid_leaf_pairs (:2525-2706)
// and the BVH traversal of rigid_collide_meshes (:2156-2285).
// ---------------------------------------------------------------------
__device__ __forceinline__ float normal_speed(const PmhRigidBodyState &b, const PmhRigidBodyState &c, V3 p, V3 n) {
    const V3 bv = add(sv(b.linear_velocity), cross(sv(b.angular_velocity), sub(p, sv(b.position))));
    const V3 cv = add(sv(c.linear_velocity), cross(sv(c.angular_velocity), sub(p, sv(c.position))));
    return dot(sub(bv, cv), n);
}

__device__ void closest_segments(V3 p0, V3 p1, V3 q0, V3 q1, V3 &on_p, V3 &on_q) {
    const V3 d0 = sub(p1, p0), d1 = sub(q1, q0), r = sub(p0, q0);
    const float a = dot(d0, d0), e = dot(d1, d1);
    float s = 0.0f, t = 0.0f;
    if (a <= 1.0e-12f && e <= 1.0e-12f) { on_p = p0; on_q = q0; return; }
    if (a <= 1.0e-12f) {
        t = clampf(dot(d1, r) / e, 0.0f, 1.0f);
    } else {
        const float c = dot(d0, r);
        if (e <= 1.0e-12f) {
            s = clampf(-c / a, 0.0f, 1.0f);
        } else {
            const float b = dot(d0, d1), f = dot(d1, r);
            const float den = a * e - b * b;
            if (fabsf(den) > kEpsilon * a * e) s = clampf((b * f - c * e) / den, 0.0f, 1.0f);
            t = (b * s + f) / e;
            if (t < 0.0f) { t = 0.0f; s = clampf(-c / a, 0.0f, 1.0f); }
            else if (t > 1.0f) { t = 1.0f; s = clampf((b - c) / a, 0.0f, 1.0f); }
        }
    }
    on_p = add(p0, mul(d0, s));
    on_q = add(q0, mul(d1, t));
}

__device__ V3 closest_on_triangle(V3 p, V3 a, V3 b, V3 c) {
    const V3 ab = sub(b, a), ac = sub(c, a), ap = sub(p, a);
    const float d1 = dot(ab, ap), d2 = dot(ac, ap);
    if (d1 <= 0.0f && d2 <= 0.0f) return a;
    const V3 bp = sub(p, b);
    const float d3 = dot(ab, bp), d4 = dot(ac, bp);
    if (d3 >= 0.0f && d4 <= d3) return b;
    const float vc = d1 * d4 - d3 * d2;
    if (vc <= 0.0f && d1 >= 0.0f && d3 <= 0.0f) return add(a, mul(ab, d1 / (d1 - d3)));
    const V3 cp = sub(p, c);
    const float d5 = dot(ab, cp), d6 = dot(ac, cp);
    if (d6 >= 0.0f && d5 <= d6) return c;
    const float vb = d5 * d2 - d1 * d6;
    if (vb <= 0.0f && d2 >= 0.0f && d6 <= 0.0f) return add(a, mul(ac, d2 / (d2 - d6)));
    const float va = d3 * d6 - d5 * d4;
    if (va <= 0.0f && d4 - d3 >= 0.0f && d5 - d6 >= 0.0f)
        return add(b, mul(sub(c, b), (d4 - d3) / ((d4 - d3) + (d5 - d6))));
    const V3 n = cross(ab, ac);
    return sub(p, mul(n, dot(ap, n) / len2(n)));
}

__device__ bool segment_hits_triangle(V3 p, V3 q, V3 a, V3 b, V3 c, V3 &hit) {
    hit = {0.0f, 0.0f, 0.0f};
    const V3 n = cross(sub(b, a), sub(c, a));
    const V3 dir = sub(q, p);
    const float den = dot(n, dir);
    if (len2(n) <= kEpsilon * kEpsilon || fabsf(den) <= kEpsilon) return false;
    const float amount = dot(n, sub(a, p)) / den;
    if (amount < 0.0f || amount > 1.0f) return false;
    hit = add(p, mul(dir, amount));
    const float tol = -1.0e-5f * len2(n);
    return dot(cross(sub(b, a), sub(hit, a)), n) >= tol && dot(cross(sub(c, b), sub(hit, b)), n) >= tol &&
           dot(cross(sub(a, c), sub(hit, c)), n) >= tol;
}

// A triangle in registers.  Every loop over corners or edges turns it instead
// of indexing it: an index that is not a constant would put it in memory.
struct Triangle {
    V3 p0, p1, p2;
};
__device__ __forceinline__ void turn(Triangle &t) {
    const V3 p = t.p0;
    t.p0 = t.p1;
    t.p1 = t.p2;
    t.p2 = p;
}
__device__ __forceinline__ V3 triangle_cross(const Triangle &t) { return cross(sub(t.p1, t.p0), sub(t.p2, t.p0)); }

// Closest points of two triangles, on four lanes that hold the same two: lane
// e takes edge and corner e of both through the crossing tests, the corners
// against the other face and its edge of A against B's three, and the first of
// the nearest in the serial order wins.  The swept pass calls it up to 32 times
// in a row, and each test is one chain of operations: 21 of them on one lane
// took 10.6 us a round of the swept pass where 8000 bodies fly (1400 pairs, the
// longest 0.39 ms), these 7 and the exchange 6 us (0.25 ms).
struct ClosestPair {
    V3 a, b;
};
constexpr int kQuadFirst = 0x00, kQuadSecond = 0x55, kQuadThird = 0xaa;   // broadcasts within four lanes

template <int kFrom>
__device__ __forceinline__ V3 quad_v3(V3 v) {
    return {dpp_f32<kFrom>(v.x), dpp_f32<kFrom>(v.y), dpp_f32<kFrom>(v.z)};
}
__device__ __forceinline__ Triangle turned(const Triangle &t, uint32_t e) {
    const V3 p0 = e == 0u ? t.p0 : e == 1u ? t.p1 : t.p2, p1 = e == 0u ? t.p1 : e == 1u ? t.p2 : t.p0;
    return {p0, p1, e == 0u ? t.p2 : e == 1u ? t.p0 : t.p1};
}
// The first hit of the lanes in order.
__device__ __forceinline__ bool quad_first_hit(bool hit, V3 at, V3 &first) {
    const uint32_t h = hit ? 1u : 0u;
    const bool h0 = dpp_u32<kQuadFirst>(h) != 0u, h1 = dpp_u32<kQuadSecond>(h) != 0u, h2 = dpp_u32<kQuadThird>(h) != 0u;
    const V3 a0 = quad_v3<kQuadFirst>(at), a1 = quad_v3<kQuadSecond>(at), a2 = quad_v3<kQuadThird>(at);
    first = h0 ? a0 : h1 ? a1 : a2;
    return h0 || h1 || h2;
}
struct NearestPair {
    float d;
    uint32_t order;                       // in the serial search
    ClosestPair at;
};
__device__ __forceinline__ void keep_nearer(NearestPair &best, V3 a, V3 b, uint32_t order) {
    const float d = len2(sub(a, b));
    if (d < best.d) best = {d, order, {a, b}};
}
template <int kFrom>
__device__ __forceinline__ void quad_nearer(NearestPair &best) {
    const NearestPair o{dpp_f32<kFrom>(best.d), dpp_u32<kFrom>(best.order),
                        {quad_v3<kFrom>(best.at.a), quad_v3<kFrom>(best.at.b)}};
    if (o.d < best.d || (o.d == best.d && o.order < best.order)) best = o;
}
__device__ __noinline__ ClosestPair closest_points(float a0, float a1, float a2, float a3, float a4, float a5, float a6,
                                                   float a7, float a8, float b0, float b1, float b2, float b3, float b4,
                                                   float b5, float b6, float b7, float b8) {
    const Triangle A{{a0, a1, a2}, {a3, a4, a5}, {a6, a7, a8}}, B{{b0, b1, b2}, {b3, b4, b5}, {b6, b7, b8}};
    const uint32_t e = min(threadIdx.x & 3u, 2u);       // the fourth lane repeats the third
    const Triangle Ae = turned(A, e);
    Triangle Be = turned(B, e);
    V3 hit, first;
    bool crosses = segment_hits_triangle(Ae.p0, Ae.p1, B.p0, B.p1, B.p2, hit);
    if (quad_first_hit(crosses, hit, first)) return {first, first};
    crosses = segment_hits_triangle(Be.p0, Be.p1, A.p0, A.p1, A.p2, hit);
    if (quad_first_hit(crosses, hit, first)) return {first, first};
    NearestPair best{3.402823466e+38f, ~0u, {{0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f}}};
    keep_nearer(best, Ae.p0, closest_on_triangle(Ae.p0, B.p0, B.p1, B.p2), e);
    keep_nearer(best, closest_on_triangle(Be.p0, A.p0, A.p1, A.p2), Be.p0, 3u + e);
    Be = B;
#pragma unroll 1
    for (uint32_t j = 0; j < 3; ++j) {
        V3 u, w;
        closest_segments(Ae.p0, Ae.p1, Be.p0, Be.p1, u, w);
        keep_nearer(best, u, w, 6u + 3u * e + j);
        turn(Be);
    }
    quad_nearer<kDppXor1>(best);
    quad_nearer<kDppXor2>(best);
    return best.at;
}
__device__ __forceinline__ void closest_triangle_pair(const Triangle &A, const Triangle &B, V3 &pa, V3 &pb) {
    const ClosestPair c = closest_points(A.p0.x, A.p0.y, A.p0.z, A.p1.x, A.p1.y, A.p1.z, A.p2.x, A.p2.y, A.p2.z, B.p0.x,
                                         B.p0.y, B.p0.z, B.p1.x, B.p1.y, B.p1.z, B.p2.x, B.p2.y, B.p2.z);
    pa = c.a;
    pb = c.b;
}

__device__ __forceinline__ bool boxes_touch(V3 amin, V3 amax, V3 bmin, V3 bmax) {
    return amin.x <= bmax.x && amax.x >= bmin.x && amin.y <= bmax.y && amax.y >= bmin.y && amin.z <= bmax.z &&
           amax.z >= bmin.z;
}

__device__ V3 advect_triangle_point(V3 q, const Triangle &from, const Triangle &to) {
    const V3 ab = sub(from.p1, from.p0), ac = sub(from.p2, from.p0);
    const V3 n = cross(ab, ac);
    const float sq2 = len2(n);
    if (sq2 <= 1.0e-20f) return to.p0;
    const V3 rel = sub(q, from.p0);
    const float v = dot(cross(rel, ac), n) / sq2;
    const float w = dot(cross(ab, rel), n) / sq2;
    return add(to.p0, add(mul(sub(to.p1, to.p0), v), mul(sub(to.p2, to.p0), w)));
}

// Certified outward direction of a (possibly swept) world triangle: unit
// for exterior faces, a quarter for two-sided interior features, zero when
// uncertified (rigid_shell_outward, geometry.slang:1308-1322).
__device__ V3 shell_outward(const ShapeView &m, uint32_t t, const Triangle &W) {
    if (!m.s.has_shell) return {0.0f, 0.0f, 0.0f};
    const V3 o = v3(m.shell[m.s.shell_off + t]);
    const float sq2 = len2(o);
    if (sq2 < 0.01f) return {0.0f, 0.0f, 0.0f};
    const V3 la = m.vert(m.index(3 * t)), lb = m.vert(m.index(3 * t + 1)), lc = m.vert(m.index(3 * t + 2));
    const float sign = dot(cross(sub(lb, la), sub(lc, la)), o) >= 0.0f ? 1.0f : -1.0f;
    return mul(normalized_or(triangle_cross(W), {0.0f, 0.0f, 0.0f}),
               sign * (sq2 > 0.5f ? 1.0f : 0.25f));
}

__device__ __forceinline__ bool shell_facing(V3 n, V3 oa, V3 ob) {
    const float sa = len2(oa), sb = len2(ob);
    return (sa < 0.01f || (sa > 0.5f ? dot(n, oa) < -1.0e-3f : fabsf(dot(n, oa)) > 2.5e-4f)) &&
           (sb < 0.01f || (sb > 0.5f ? dot(n, ob) > 1.0e-3f : fabsf(dot(n, ob)) > 2.5e-4f));
}

__device__ bool point_inside_convex(const ShapeView &m, const PmhRigidBodyState &st, V3 world) {
    if (!m.s.has_planes) return false;
    const V3 l = inv_rotate(sq(st.orientation), sub(world, sv(st.position)));
    const uint32_t tris = m.s.idx_count / 3u;
    const uint32_t unique = m.s.unique_planes;
    const uint32_t count = unique != 0u ? unique : tris;
    const uint32_t first = unique != 0u ? tris : 0u;
    for (uint32_t f = 0; f < count; ++f) {
        const float4 pl = m.plane(first + f);
        if (dot(v3(pl), l) > pl.w + 1.0e-5f) return false;
    }
    return true;
}

// One triangle's part of the feature normal: the closest point strictly
// inside it takes its face, the face most along the normal first.
__device__ __forceinline__ void interior_face(const Triangle &T, V3 pt, V3 face, V3 normal, V3 delta, V3 fallback,
                                              float &align_best, V3 &interior_normal) {
    const V3 raw = triangle_cross(T);
    const float tol = 1.0e-5f * len2(raw);
    bool interior = tol > 0.0f;
    interior = interior && dot(cross(sub(T.p1, T.p0), sub(pt, T.p0)), raw) > tol;
    interior = interior && dot(cross(sub(T.p2, T.p1), sub(pt, T.p1)), raw) > tol;
    interior = interior && dot(cross(sub(T.p0, T.p2), sub(pt, T.p2)), raw) > tol;
    const float alignment = fabsf(dot(face, normal));
    if (interior && alignment > align_best) {
        align_best = alignment;
        const float proj = dot(delta, face);
        const float dir = fabsf(proj) > kEpsilon ? proj : dot(fallback, face);
        interior_normal = dir >= 0.0f ? face : mul(face, -1.0f);
    }
}
__device__ __forceinline__ void aligned_face(V3 face, V3 delta, float &best, V3 &normal) {
    const float proj = dot(delta, face);
    const float err = len2(sub(delta, mul(face, proj)));
    if (err < best) {
        best = err;
        normal = proj >= 0.0f ? face : mul(face, -1.0f);
    }
}
__device__ __forceinline__ V3 triangle_feature_normal(const Triangle &A, const Triangle &B, V3 pa, V3 pb, V3 fallback) {
    const V3 delta = sub(pa, pb);
    V3 normal = normalized_or(delta, fallback);
    const V3 face_a = normalized_or(triangle_cross(A), normal), face_b = normalized_or(triangle_cross(B), normal);
    float align_best = -1.0f;
    V3 interior_normal = {0.0f, 0.0f, 0.0f};
    interior_face(A, pa, face_a, normal, delta, fallback, align_best, interior_normal);
    interior_face(B, pb, face_b, normal, delta, fallback, align_best, interior_normal);
    if (align_best >= 0.0f) return interior_normal;
    float best = 4.0f * kEpsilon * kEpsilon;
    if (len2(delta) > kEpsilon * kEpsilon) {
        aligned_face(face_a, delta, best, normal);
        aligned_face(face_b, delta, best, normal);
    }
    return normal;
}

// Inputs of one pair on the triangle path: shapes, previous and predicted
// states, the pair's hinge contact frames and the body's reference points
// (rigid_hinge_contact_frame, geometry.slang:404-491).
struct TrianglePair {
    ShapeView am, bm;
    PmhRigidBodyState ap, a, bp, b;   // previous and predicted states
    PairFrames f;
    float margin, dt;
};

__device__ __forceinline__ Triangle world_triangle(const ShapeView &m, const PmhRigidBodyState &st, uint32_t t) {
    return {transform_point(st, m.vert(m.index(3 * t))), transform_point(st, m.vert(m.index(3 * t + 1))),
            transform_point(st, m.vert(m.index(3 * t + 2)))};
}
// The triangle on its way from one pose to the next.
__device__ __forceinline__ Triangle between(const Triangle &from, const Triangle &to, float time) {
    return {add(from.p0, mul(sub(to.p0, from.p0), time)), add(from.p1, mul(sub(to.p1, from.p1), time)),
            add(from.p2, mul(sub(to.p2, from.p2), time))};
}
__device__ __forceinline__ V3 triangle_min(const Triangle &t) { return cmin(t.p0, cmin(t.p1, t.p2)); }
__device__ __forceinline__ V3 triangle_max(const Triangle &t) { return cmax(t.p0, cmax(t.p1, t.p2)); }

// The box test that begins both passes: the triangles' boxes, of the swept
// pass at both poses (that box holds the discrete pass's, which tests again).
__device__ __forceinline__ bool triangle_boxes_touch(const TrianglePair &P, uint32_t at, uint32_t bt, bool swept) {
    const Triangle A = world_triangle(P.am, P.a, at), B = world_triangle(P.bm, P.b, bt);
    V3 amin = triangle_min(A), amax = triangle_max(A), bmin = triangle_min(B), bmax = triangle_max(B);
    if (swept) {
        const Triangle pA = world_triangle(P.am, P.ap, at), pB = world_triangle(P.bm, P.bp, bt);
        amin = cmin(amin, triangle_min(pA));
        amax = cmax(amax, triangle_max(pA));
        bmin = cmin(bmin, triangle_min(pB));
        bmax = cmax(bmax, triangle_max(pB));
    }
    const V3 e = {P.margin, P.margin, P.margin};
    return boxes_touch(sub(amin, e), add(amax, e), bmin, bmax);
}

// The discrete pass for one triangle pair (the body of the triangle loops
// of rigid_collide_triangle_ranges, geometry.slang:1359-1584): at most one
// contact, independent of every other triangle pair.
__device__ __noinline__ bool triangle_pair_contact(const TrianglePair &P, uint32_t at, uint32_t bt, bool inside_a,
                                                   bool inside_b, Contact &c) {
    const float margin = P.margin;
    const float rest = smin(margin, 1.0e-3f);
    const V3 body_ref = P.f.ref;
    const Triangle A = world_triangle(P.am, P.a, at), B = world_triangle(P.bm, P.b, bt);
    {
        const V3 e = {margin, margin, margin};
        if (!boxes_touch(sub(triangle_min(A), e), add(triangle_max(A), e), triangle_min(B), triangle_max(B))) return false;
    }
    const V3 oa = shell_outward(P.am, at, A), ob = shell_outward(P.bm, bt, B);
    const V3 coa = P.f.ha.static_body != 0u && inside_a ? V3{0.0f, 0.0f, 0.0f} : oa;
    const V3 cob = P.f.hb.static_body != 0u && inside_b ? V3{0.0f, 0.0f, 0.0f} : ob;
    if (dot(oa, ob) > 0.9999f) return false;
    V3 pa, pb;
    closest_triangle_pair(A, B, pa, pb);
    const V3 delta = sub(pa, pb);
    const float sq2 = len2(delta);
    if (sq2 > margin * margin) return false;
    const V3 cn = normalized_or(triangle_cross(B), {0.0f, 1.0f, 0.0f});
    V3 fallback = dot(cn, sub(body_ref, pb)) >= 0.0f ? cn : mul(cn, -1.0f);
    if (len2(cob) > 0.5f) fallback = cob;
    const float distance = sqrtf(smax(sq2, 0.0f));
    const V3 point = mul(add(pa, pb), 0.5f);
    const V3 proj = sub(pa, mul(cn, dot(sub(pa, B.p0), cn)));
    const bool on_face = len2(sub(proj, closest_on_triangle(proj, B.p0, B.p1, B.p2))) <= 1.0e-10f;
    const V3 normal = (distance <= 1.0e-5f || on_face) ? fallback : normalized_or(delta, fallback);
    if (on_face && len2(oa) < 0.01f && len2(ob) > 0.5f && P.bm.s.has_planes) {
        const V3 face_a = normalized_or(triangle_cross(A), {0.0f, 0.0f, 0.0f});
        if (fabsf(dot(face_a, normal)) < 1.0e-3f) {
            const float depth = smax(0.0f, -smin(dot(sub(A.p0, B.p0), normal),
                                                 smin(dot(sub(A.p1, B.p0), normal), dot(sub(A.p2, B.p0), normal))));
            const V3 axis = inv_rotate(sq(P.b.orientation), face_a);
            const float offset = dot(sub(sv(P.b.position), A.p0), face_a);
            float lo = 3.402823466e+38f, hi = -3.402823466e+38f;
            for (uint32_t k = 0; k < P.bm.s.vtx_count; ++k) {
                const float pr = dot(P.bm.vert(k), axis) + offset;
                lo = smin(lo, pr);
                hi = smax(hi, pr);
            }
            const float alternate = smax(0.0f, smin(-lo, hi));
            if (alternate + 1.0e-5f < depth) return false;
        }
    }
    const float separation = on_face && len2(cob) > 0.5f ? dot(delta, normal) : distance;
    // rigid_contact_reaches_rest_offset (:1282-1290)
    if (!(separation <= rest + 1.0e-5f)) {
        const float speed = normal_speed(P.a, P.b, point, normal);
        if (speed > 1.0e-5f || !(-speed * P.dt + rest + 1.0e-5f >= separation)) return false;
    }
    c.normal = normal;
    c.point = point;
    c.pen = rest - separation + 1.0e-5f;
    bool recovered = false;
    if (!P.am.s.has_planes && !P.bm.s.has_planes && distance <= 1.0e-5f) {
        const Triangle oldA = world_triangle(P.am, P.ap, at), oldB = world_triangle(P.bm, P.bp, bt);
        V3 opa, opb;
        closest_triangle_pair(oldA, oldB, opa, opb);
        V3 od = sub(opa, opb);
        if (len2(od) > 1.0e-10f) {
            float lo = 0.0f, hi = 1.0f;
            const float gap = smin(rest, 0.5f * sqrtf(len2(od)));
            for (uint32_t k = 0; k < 10u; ++k) {
                const float time = 0.5f * (lo + hi);
                V3 u, w;
                closest_triangle_pair(between(oldA, A, time), between(oldB, B, time), u, w);
                if (len2(sub(u, w)) > gap * gap) lo = time;
                else hi = time;
            }
            const Triangle IA = between(oldA, A, lo), IB = between(oldB, B, lo);
            closest_triangle_pair(IA, IB, opa, opb);
            od = sub(opa, opb);
            c.normal = triangle_feature_normal(IA, IB, opa, opb, normalized_or(od, fallback));
            const V3 ca = advect_triangle_point(opa, IA, A), cb = advect_triangle_point(opb, IB, B);
            c.point = mul(add(ca, cb), 0.5f);
            c.pen = rest - dot(sub(ca, cb), c.normal) + 1.0e-5f;
            recovered = true;
        }
    }
    if (distance <= 1.0e-5f) {
        if (!recovered && (P.f.ha.fixed_member != 0u || P.f.hb.fixed_member != 0u || on_face)) {
            const float depth = smax(0.0f, -smin(dot(sub(A.p0, pb), normal),
                                                 smin(dot(sub(A.p1, pb), normal), dot(sub(A.p2, pb), normal))));
            c.pen = smin(margin, depth + rest) + 1.0e-5f;
        } else if (!recovered) {
            c.pen = margin + 1.0e-5f;
        }
    }
    if (!shell_facing(c.normal, coa, cob)) return false;
    c.impact_fraction = 1.0f;
    return true;
}

// rigid_triangle_pair_face_contact, geometry.slang:1910-1919.
__device__ __forceinline__ bool triangle_pair_face_contact(const Triangle &A, const Triangle &B, V3 separation) {
    const V3 n = normalized_or(separation, {0.0f, 0.0f, 0.0f});
    const V3 fa = normalized_or(triangle_cross(A), {0.0f, 0.0f, 0.0f});
    const V3 fb = normalized_or(triangle_cross(B), {0.0f, 0.0f, 0.0f});
    return fabsf(dot(n, fa)) > 0.9999f || fabsf(dot(n, fb)) > 0.9999f;
}

// The swept pass for one triangle pair (conservative advancement, the body
// of rigid_collide_triangle_ranges_swept, geometry.slang:1921-2154): at
// most one contact.  A guided pair rests at 0.1 mm, takes edge contacts that
// both slide along and turn about the guide axis at zero offset, and
// advances by the faces' closing speed along the feature normal.
__device__ __noinline__ bool triangle_pair_swept_contact(const TrianglePair &P, uint32_t at, uint32_t bt,
                                                         bool inside_a, bool inside_b, Contact &c) {
    const float margin = P.margin;
    const bool guided = guided_pair(P.f.ha, P.f.hb);
    const float rest = guided ? smin(margin, 1.0e-4f) : smin(margin, 1.0e-3f);
    const Triangle pA = world_triangle(P.am, P.ap, at), cA = world_triangle(P.am, P.a, at);
    const Triangle pB = world_triangle(P.bm, P.bp, bt), cB = world_triangle(P.bm, P.b, bt);
    const V3 e = {margin, margin, margin};
    if (!boxes_touch(sub(cmin(triangle_min(pA), triangle_min(cA)), e), add(cmax(triangle_max(pA), triangle_max(cA)), e),
                     cmin(triangle_min(pB), triangle_min(cB)), cmax(triangle_max(pB), triangle_max(cB))))
        return false;
    const Triangle dA{sub(cA.p0, pA.p0), sub(cA.p1, pA.p1), sub(cA.p2, pA.p2)};
    const Triangle dB{sub(cB.p0, pB.p0), sub(cB.p1, pB.p1), sub(cB.p2, pB.p2)};
    const float speed_abs = smax(smax(smax(0.0f, len(dA.p0)), len(dA.p1)), len(dA.p2)) +
                            smax(smax(smax(0.0f, len(dB.p0)), len(dB.p1)), len(dB.p2));
    const V3 common = dB.p0;
    const float rel_a = smax(smax(smax(0.0f, len(sub(dA.p0, common))), len(sub(dA.p1, common))), len(sub(dA.p2, common)));
    const float rel_b = smax(smax(smax(0.0f, len(sub(dB.p0, common))), len(sub(dB.p1, common))), len(sub(dB.p2, common)));
    const float bound = smin(speed_abs, rel_a + rel_b);
    if (bound <= kEpsilon) return false;
    float time = 0.0f;
    bool starts_near = false;
    // The last step's time and closest points: the normal the triangles were
    // apart along is needed at the contact only (and in guided pairs).
    float sep_time = -1.0f;
    V3 sep_pa = {0.0f, 0.0f, 0.0f}, sep_pb = {0.0f, 0.0f, 0.0f};
    auto at_time = [&](const Triangle &from, const Triangle &d, float time) {
        return Triangle{add(from.p0, mul(d.p0, time)), add(from.p1, mul(d.p1, time)), add(from.p2, mul(d.p2, time))};
    };
    for (uint32_t it = 0; it < 32u; ++it) {
        const Triangle A = at_time(pA, dA, time), B = at_time(pB, dB, time);
        V3 pa, pb;
        closest_triangle_pair(A, B, pa, pb);
        const V3 delta = sub(pa, pb);
        const float distance = sqrtf(smax(0.0f, len2(delta)));
        float offset = rest;
        if (guided && !triangle_pair_face_contact(A, B, delta)) {
            const HingeFrame &guide = P.f.ha.axial != 0u ? P.f.ha : P.f.hb;
            const V3 direction = normalized_or(delta, {0.0f, 0.0f, 0.0f});
            const float axial = dot(direction, sv(guide.axis));
            const float angular = dot(sv(guide.axis), cross(sub(pa, sv(guide.anchor)), direction));
            if (fabsf(axial) > 1.0e-3f && fabsf(angular) > 1.0e-3f) offset = 0.0f;
        }
        if (it == 0u) starts_near = distance <= offset + 5.0e-5f;
        if (distance <= offset + 1.0e-5f) {
            const V3 cn = normalized_or(triangle_cross(B), {0.0f, 1.0f, 0.0f});
            const V3 center = add(sv(P.ap.position), mul(sub(sv(P.a.position), sv(P.ap.position)), time));
            V3 fallback = dot(cn, sub(center, pb)) >= 0.0f ? cn : mul(cn, -1.0f);
            if (P.f.ha.present != 0u) {
                const V3 reference = add(P.f.ref_prev, mul(sub(P.f.ref, P.f.ref_prev), time));
                fallback = dot(cn, sub(reference, pb)) >= 0.0f ? cn : mul(cn, -1.0f);
            }
            const V3 oa = shell_outward(P.am, at, A), ob = shell_outward(P.bm, bt, B);
            const V3 coa = P.f.ha.static_body != 0u && inside_a ? V3{0.0f, 0.0f, 0.0f} : oa;
            const V3 cob = P.f.hb.static_body != 0u && inside_b ? V3{0.0f, 0.0f, 0.0f} : ob;
            if (dot(oa, ob) > 0.9999f) return false;
            if (len2(cob) > 0.5f) fallback = cob;
            else if (len2(coa) > 0.5f) fallback = mul(coa, -1.0f);
            if (sep_time >= 0.0f)
                fallback = triangle_feature_normal(at_time(pA, dA, sep_time), at_time(pB, dB, sep_time), sep_pa, sep_pb,
                                                   normalized_or(sub(sep_pa, sep_pb), {0.0f, 1.0f, 0.0f}));
            const V3 normal = triangle_feature_normal(A, B, pa, pb, fallback);
            if (!shell_facing(normal, coa, cob)) return false;
            const V3 point = mul(add(pa, pb), 0.5f);
            const float vn = normal_speed(P.a, P.b, point, normal);
            if (vn > 1.0e-5f) return false;
            const float remaining = -vn * P.dt * (1.0f - time) - distance;
            c.normal = normal;
            c.point = point;
            c.pen = smax(0.0f, remaining + offset) + 1.0e-5f;
            c.impact_fraction = starts_near ? 0.0f : time;
            return true;
        }
        sep_time = time;
        sep_pa = pa;
        sep_pb = pb;
        float advance = (distance - offset) / (bound + kEpsilon) * 0.9f;
        if (guided) {
            const V3 apart = triangle_feature_normal(A, B, pa, pb, normalized_or(delta, {0.0f, 1.0f, 0.0f}));
            const V3 plane = triangle_feature_normal(A, B, pa, pb, apart);
            const float big = 3.402823466e+38f;
            const float min_a = smin(smin(smin(big, dot(sub(A.p0, pb), plane)), dot(sub(A.p1, pb), plane)),
                                     dot(sub(A.p2, pb), plane));
            const float max_b = smax(smax(smax(-big, dot(sub(B.p0, pb), plane)), dot(sub(B.p1, pb), plane)),
                                     dot(sub(B.p2, pb), plane));
            const float min_speed_a = smin(smin(smin(big, dot(dA.p0, plane)), dot(dA.p1, plane)), dot(dA.p2, plane));
            const float max_speed_b = smax(smax(smax(-big, dot(dB.p0, plane)), dot(dB.p1, plane)), dot(dB.p2, plane));
            const float gap = min_a - max_b - offset;
            const float closing = max_speed_b - min_speed_a;
            if (gap > 1.0e-5f && closing <= 0.0f) return false;
            if (gap > 0.0f && closing > kEpsilon) advance = smax(advance, 0.9f * gap / closing);
        }
        time += smax(advance, 1.0e-5f);
        if (time > 1.0f) return false;
    }
    return false;
}

__device__ __forceinline__ void inside_flags(const TrianglePair &P, bool &inside_a, bool &inside_b) {
    inside_a = P.f.ha.static_body != 0u && point_inside_convex(P.am, P.ap, sv(P.bp.position));
    inside_b = P.f.hb.static_body != 0u && point_inside_convex(P.bm, P.bp, sv(P.ap.position));
}

// The merge rule of the pair: guided pairs merge by guide direction.
__device__ __forceinline__ void merge_contact(const TrianglePair &P, Manifold &m, const Contact &c, float spacing) {
    if (guided_pair(P.f.ha, P.f.hb)) add_contact_guided(m, c, P.f.ha.axial != 0u ? P.f.ha : P.f.hb);
    else add_contact(m, c, spacing);
}

// rigid_collide_triangle_ranges: triangles in order, body-major.  Called on
// the four lanes of a closest-point search, which share the manifold: one of
// them (`writer`) reads and writes it.
__device__ void collide_triangle_ranges(const TrianglePair &P, uint32_t a_first, uint32_t a_count,
                                        uint32_t b_first, uint32_t b_count, Manifold &m, bool writer) {
    if (guided_pair(P.f.ha, P.f.hb)) return;   // geometry.slang:1371
    bool inside_a, inside_b;
    inside_flags(P, inside_a, inside_b);
    const float spacing = smax(2.0f * P.margin, 1.0e-4f);
    for (uint32_t ai = 0; ai < a_count; ++ai) {
        const uint32_t at = a_first + ai;
        if (3u * at + 2u >= P.am.s.idx_count) break;
        for (uint32_t bi = 0; bi < b_count; ++bi) {
            const uint32_t bt = b_first + bi;
            if (3u * bt + 2u >= P.bm.s.idx_count) break;
            Contact c;
            if (triangle_pair_contact(P, at, bt, inside_a, inside_b, c) && writer) add_contact(m, c, spacing);
        }
    }
}

__device__ void collide_triangle_ranges_swept(const TrianglePair &P, uint32_t a_first, uint32_t a_count,
                                              uint32_t b_first, uint32_t b_count, Manifold &m, bool writer) {
    bool inside_a, inside_b;
    inside_flags(P, inside_a, inside_b);
    const float spacing = smax(P.margin * 2.0f, 1.0e-4f);
    for (uint32_t ai = 0; ai < a_count; ++ai) {
        const uint32_t at = a_first + ai;
        if (3u * at + 2u >= P.am.s.idx_count) break;
        for (uint32_t bi = 0; bi < b_count; ++bi) {
            const uint32_t bt = b_first + bi;
            if (3u * bt + 2u >= P.bm.s.idx_count) break;
            Contact c;
            if (triangle_pair_swept_contact(P, at, bt, inside_a, inside_b, c) && writer) merge_contact(P, m, c, spacing);
        }
    }
}

// BoundsTransform and transformed_(motion_)bounds, math.slang:142-190.
struct BoundsFrame {
    V3 position, ax, ay, az;
};
__device__ __forceinline__ BoundsFrame bounds_frame(const PmhRigidBodyState &s) {
    const Q q = sq(s.orientation);
    return {sv(s.position), rotate(q, {1.0f, 0.0f, 0.0f}), rotate(q, {0.0f, 1.0f, 0.0f}), rotate(q, {0.0f, 0.0f, 1.0f})};
}
__device__ __forceinline__ void frame_bounds(V3 lmin, V3 lmax, const BoundsFrame &f, float margin, V3 &mn, V3 &mx) {
    const V3 c = mul(add(lmin, lmax), 0.5f), h = mul(sub(lmax, lmin), 0.5f);
    const V3 wc = add(f.position, add(mul(f.ax, c.x), add(mul(f.ay, c.y), mul(f.az, c.z))));
    const V3 wh = {fabsf(f.ax.x) * h.x + fabsf(f.ay.x) * h.y + fabsf(f.az.x) * h.z,
                   fabsf(f.ax.y) * h.x + fabsf(f.ay.y) * h.y + fabsf(f.az.y) * h.z,
                   fabsf(f.ax.z) * h.x + fabsf(f.ay.z) * h.y + fabsf(f.az.z) * h.z};
    const V3 e = {margin, margin, margin};
    mn = sub(sub(wc, wh), e);
    mx = add(add(wc, wh), e);
}
__device__ __forceinline__ void motion_bounds(V3 lmin, V3 lmax, const BoundsFrame &prev, const BoundsFrame &cur,
                                              bool swept, float margin, V3 &mn, V3 &mx) {
    frame_bounds(lmin, lmax, cur, margin, mn, mx);
    if (!swept) return;
    V3 pmn, pmx;
    frame_bounds(lmin, lmax, prev, margin, pmn, pmx);
    mn = cmin(mn, pmn);
    mx = cmax(mx, pmx);
}
__device__ __forceinline__ void node_bounds(const BvhDev &nd, const BoundsFrame &prev, const BoundsFrame &cur,
                                            bool swept, float margin, V3 &mn, V3 &mx) {
    motion_bounds(sarr(nd.mn), sarr(nd.mx), prev, cur, swept, margin, mn, mx);
}

__device__ __forceinline__ void collide_leaf_ranges(const TrianglePair &P, bool swept, const BvhDev &na,
                                                    const BvhDev &nb, Manifold &m, bool writer) {
    collide_triangle_ranges(P, na.first, na.count, nb.first, nb.count, m, writer);
    if (swept) collide_triangle_ranges_swept(P, na.first, na.count, nb.first, nb.count, m, writer);
}

// rigid_collide_meshes: simultaneous descent with a 64-entry stack, all
// triangles when the stack would overflow.
__device__ __noinline__ void collide_meshes(const TrianglePair &P, bool swept, Manifold &m, bool writer) {
    if (writer) {
        m.count = 0;
        m.face_patch = 0;
    }
    const BoundsFrame fa = bounds_frame(P.a), fb = bounds_frame(P.b);
    const BoundsFrame pfa = swept ? bounds_frame(P.ap) : BoundsFrame{};
    const BoundsFrame pfb = swept ? bounds_frame(P.bp) : BoundsFrame{};
    V3 amn, amx, bmn, bmx;
    motion_bounds(sarr(P.am.s.mn), sarr(P.am.s.mx), pfa, fa, swept, P.margin, amn, amx);
    motion_bounds(sarr(P.bm.s.mn), sarr(P.bm.s.mx), pfb, fb, swept, 0.0f, bmn, bmx);
    if (!boxes_touch(amn, amx, bmn, bmx)) return;
    constexpr uint32_t kStack = 64;
    uint32_t sa[kStack], sb[kStack];
    sa[0] = 0;
    sb[0] = 0;
    uint32_t top = 1;
    bool overflow = P.am.s.node_count == 0u || P.bm.s.node_count == 0u;
    while (top > 0u && !overflow) {
        --top;
        const uint32_t ia = sa[top], ib = sb[top];
        const BvhDev na = P.am.node(ia), nb = P.bm.node(ib);
        node_bounds(na, pfa, fa, swept, P.margin, amn, amx);
        node_bounds(nb, pfb, fb, swept, 0.0f, bmn, bmx);
        if (!boxes_touch(amn, amx, bmn, bmx)) continue;
        const bool la = na.count != 0u, lb = nb.count != 0u;
        if (la && lb) {
            collide_leaf_ranges(P, swept, na, nb, m, writer);
            continue;
        }
        const uint32_t need = la || lb ? 2u : 4u;
        if (top + need > kStack) { overflow = true; break; }
        if (la) {
            sa[top] = ia; sb[top++] = nb.right;
            sa[top] = ia; sb[top++] = nb.left;
        } else if (lb) {
            sa[top] = na.right; sb[top++] = ib;
            sa[top] = na.left; sb[top++] = ib;
        } else {
            sa[top] = na.right; sb[top++] = nb.right;
            sa[top] = na.right; sb[top++] = nb.left;
            sa[top] = na.left; sb[top++] = nb.right;
            sa[top] = na.left; sb[top++] = nb.left;
        }
    }
    if (overflow) {
        if (writer) {
            m.count = 0;
            m.face_patch = 0;
        }
        collide_triangle_ranges(P, 0, P.am.s.idx_count / 3u, 0, P.bm.s.idx_count / 3u, m, writer);
        if (swept) collide_triangle_ranges_swept(P, 0, P.am.s.idx_count / 3u, 0, P.bm.s.idx_count / 3u, m, writer);
    }
}

// Narrowphase outputs: per-pair records and the point arrays, into which
// each non-empty manifold writes a contiguous range.
struct NarrowOut {
    uint32_t *m_count, *m_start, *m_face;
    float4 *m_init_rel;
    float4 *c_np, *c_pt, *c_aa, *c_ab, *c_err, *c_lam, *c_pen, *c_acc, *c_rep;
    uint32_t *c_flags, *c_pair;
    uint32_t point_cap;
    StepCounters *ctr;
};

// Reserves `count` (< 16) consecutive slots of *counter per active lane
// with one atomic per wavefront: each lane's offset is the sum of the
// counts of the active lanes below it, built from one ballot per bit.
// Works in divergent code (ballots and the broadcast see active lanes only).
__device__ __forceinline__ uint32_t wave_reserve(uint32_t *counter, uint32_t count) {
    const uint32_t lane = threadIdx.x & 63;
    const uint64_t active = __ballot(1);
    const uint64_t below = (1ull << lane) - 1ull;
    uint32_t offset = 0, total = 0;
#pragma unroll
    for (uint32_t b = 0; b < 4; ++b) {
        const uint64_t bits = __ballot((count >> b) & 1u);
        offset += uint32_t(__popcll(bits & below)) << b;
        total += uint32_t(__popcll(bits)) << b;
    }
    const uint32_t leader = __builtin_ctzll(active);
    uint32_t base = 0;
    if (lane == leader && total) base = atomicAdd(counter, total);
    base = __shfl(base, leader, 64);
    return base + offset;
}

// pm_finalize_rigid_contact_manifolds (geometry.slang:2805-2873): the
// initial relative position, persistence and the initial normal speed, and
// the point range.  Where the range lies does not affect any result.
// Guided contacts persist; contacts of a hinged or fixed member do not
// (:2855-2862).  Point flags: 2 persistent, 8 guided (the solver's rest
// offset).
constexpr uint32_t kPointGuided = 8u;
__device__ __forceinline__ void write_manifold(const NarrowOut &o, uint32_t m, Manifold &man, uint32_t start,
                                               const PmhRigidBodyState &A, const PmhRigidBodyState &B,
                                               bool persistent_shapes, const HingeFrame &ha, const HingeFrame &hb) {
    const bool guided = guided_pair(ha, hb);
    const bool persistent = guided || (persistent_shapes && ha.present == 0u && hb.present == 0u &&
                                       ha.fixed_member == 0u && hb.fixed_member == 0u);
    if (man.count) {
        if (start + man.count > o.point_cap) {
            atomicOr(&o.ctr->status, kStatusPointOverflow);
            man.count = 0;
        }
    }
    o.m_count[m] = man.count;
    o.m_start[m] = start;
    o.m_face[m] = man.face_patch;
    o.m_init_rel[m] = f4(sub(sv(A.position), sv(B.position)), 0.0f);
    for (uint32_t k = 0; k < man.count; ++k) {
        const Contact &c = man.c[k];
        const float speed = normal_speed(A, B, c.point, c.normal);
        const uint32_t i = start + k;
        const float4 z = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        o.c_np[i] = f4(c.normal, c.pen);
        o.c_pt[i] = f4(c.point, speed);
        o.c_aa[i] = make_float4(0.0f, 0.0f, 0.0f, c.impact_fraction);   // w: impact fraction
        o.c_ab[i] = z;
        o.c_err[i] = z;
        o.c_lam[i] = z;
        o.c_pen[i] = z;
        o.c_acc[i] = z;
        o.c_rep[i] = z;
        o.c_flags[i] = (persistent ? 2u : 0u) | (guided ? kPointGuided : 0u);
        o.c_pair[i] = m;
    }
}

__device__ void emit_manifold(const NarrowOut &o, uint32_t m, Manifold &man, const PmhRigidBodyState &A,
                              const PmhRigidBodyState &B, bool persistent_shapes, const HingeFrame &ha,
                              const HingeFrame &hb) {
    const uint32_t start = wave_reserve(&o.ctr->point_alloc, man.count);
    write_manifold(o, m, man, start, A, B, persistent_shapes, ha, hb);
}

__device__ __forceinline__ bool persistent_pair(const ShapeDev &a, const ShapeDev &b, const PmhBodyParameters &pb) {
    const auto sup = [](const ShapeDev &s) { return s.kind != kShapeMesh || (s.has_planes && s.idx_count <= 96u); };
    return sup(a) && (pb.motion != kDynamic || sup(b));
}

__device__ __forceinline__ uint32_t wave_sum(uint32_t v) {
    for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
    return v;
}

__device__ __forceinline__ uint32_t wave_exclusive_scan(uint32_t v, uint32_t lane) {
    uint32_t x = v;
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t y = __shfl_up(x, d, 64);
        if (lane >= uint32_t(d)) x += y;
    }
    return x - v;
}

// ---- the convex face path on 16 lanes ------------------------------------
// A row of 16 lanes works on one pair, so that a small world's few pairs do
// not each wait for one lane's serial search: the separating axes run over
// the lanes, a clipped polygon has one vertex per lane and a manifold one
// contact per lane.  The results are those of the reference's serial search
// (the same operations on each value, ties decided by the serial order).
constexpr uint32_t kFaceLanes = 16;
constexpr uint32_t kFacePolygon = 36;   // vertices of a clipped polygon (the reference's capacity)
struct FaceShared {
    float v[kFaceLanes][3];     // polygon vertices on their way to the next plane; contact points
    float wide[2][kFacePolygon][3];   // a polygon of more vertices than lanes, before and after a plane
};

__device__ __forceinline__ uint32_t row_bits(bool p) {   // one bit per lane of the row
    return uint32_t(__ballot(p) >> (threadIdx.x & 48u)) & 0xffffu;
}
__device__ __forceinline__ void row_sync() {   // orders the row's LDS accesses (one wavefront: in order already)
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
// Largest value of the row and, among equals, the smallest index.
__device__ __forceinline__ void row_first_max(float &v, uint32_t &i) {
    auto take = [&](float ov, uint32_t oi) {
        if (ov > v || (ov == v && oi < i)) { v = ov; i = oi; }
    };
    take(dpp_f32<kDppRowRor + 8>(v), dpp_u32<kDppRowRor + 8>(i));
    take(dpp_f32<kDppRowRor + 4>(v), dpp_u32<kDppRowRor + 4>(i));
    take(dpp_f32<kDppRowRor + 2>(v), dpp_u32<kDppRowRor + 2>(i));
    take(dpp_f32<kDppRowRor + 1>(v), dpp_u32<kDppRowRor + 1>(i));
}
__device__ __forceinline__ float row_min(float v) {
    v = smin(v, dpp_f32<kDppRowRor + 8>(v));
    v = smin(v, dpp_f32<kDppRowRor + 4>(v));
    v = smin(v, dpp_f32<kDppRowRor + 2>(v));
    return smin(v, dpp_f32<kDppRowRor + 1>(v));
}
__device__ __forceinline__ V3 row_get(V3 v, uint32_t lane) {
    return {__shfl(v.x, int(lane), 16), __shfl(v.y, int(lane), 16), __shfl(v.z, int(lane), 16)};
}

// What the face path needs of one side of a pair, in registers: lanes of one
// row look at different sides at once, so a side is chosen by value.
struct FaceSide {
    V3 pos;
    Q rot;
    uint32_t planes, verts, vert_count, indices, faces;
};
__device__ __forceinline__ FaceSide pick(bool first, const FaceSide &a, const FaceSide &b) {
    FaceSide r;
    r.pos = {first ? a.pos.x : b.pos.x, first ? a.pos.y : b.pos.y, first ? a.pos.z : b.pos.z};
    r.rot = {first ? a.rot.x : b.rot.x, first ? a.rot.y : b.rot.y, first ? a.rot.z : b.rot.z, first ? a.rot.w : b.rot.w};
    r.planes = first ? a.planes : b.planes;
    r.verts = first ? a.verts : b.verts;
    r.vert_count = first ? a.vert_count : b.vert_count;
    r.indices = first ? a.indices : b.indices;
    r.faces = first ? a.faces : b.faces;
    return r;
}
struct FaceGeometry {
    const V3 *verts;
    const uint32_t *idx;
    const float4 *planes;
};

// The support of a shape along an axis of its own frame.
__device__ __forceinline__ float face_support(const FaceGeometry &geo, const FaceSide &m, V3 axis) {
    const V3 *v = geo.verts + m.verts;
    float support = 3.402823466e+38f;
    uint32_t k = 0;
    for (; k + 4 <= m.vert_count; k += 4) {
        const V3 a = v[k], b = v[k + 1], c = v[k + 2], d = v[k + 3];
        support = smin(support, dot(axis, a));
        support = smin(support, dot(axis, b));
        support = smin(support, dot(axis, c));
        support = smin(support, dot(axis, d));
    }
    for (; k < m.vert_count; ++k) support = smin(support, dot(axis, v[k]));
    return support;
}

// A manifold held by a row: contact i in lane i; all share the normal.
struct RowManifold {
    uint32_t count;
    V3 normal, point;
    float pen, impact;
};

// add_contact for a row: the candidate is the same in all lanes.
__device__ __forceinline__ void row_add_contact(RowManifold &m, uint32_t lane, V3 point, float pen, float spacing) {
    const float sp2 = spacing * spacing;
    const uint32_t near = row_bits(lane < m.count && len2(sub(m.point, point)) < sp2);
    uint32_t at;
    bool put;
    if (near != 0u) {
        at = __builtin_ctz(near);
        put = lane == at && pen - m.pen > 0.0f;
    } else if (m.count < 8u) {
        put = lane == m.count;
        ++m.count;
    } else {
        uint32_t sh = 0;
        float low = __shfl(m.pen, 0, 16);
        for (uint32_t i = 1; i < 8u; ++i) {
            const float p = __shfl(m.pen, int(i), 16);
            if (p < low) { low = p; sh = i; }
        }
        put = lane == sh && pen > m.pen;
    }
    if (put) {
        m.point = point;
        m.pen = pen;
    }
}

// rigid_reduce_face_patch (geometry.slang:1228-1270) for a row: the 28 pairs (f, s) of at most 8 contacts are
// shared out over the lanes.
__device__ __forceinline__ void row_reduce_patch(RowManifold &m, uint32_t lane, FaceShared &S, float tol) {
    const float t2 = tol * tol;
    for (uint32_t cand = 0; cand < m.count;) {
        row_sync();
        if (lane < m.count) {
            S.v[lane][0] = m.point.x; S.v[lane][1] = m.point.y; S.v[lane][2] = m.point.z;
        }
        row_sync();
        auto at = [&](uint32_t i) { return V3{S.v[i][0], S.v[i][1], S.v[i][2]}; };
        bool removed = false;
        for (; cand < m.count && !removed;) {
            const V3 p = at(cand);
            bool on = false;
            for (uint32_t q = lane; q < 28u; q += kFaceLanes) {
                // pair q of the 28: f < s < 8
                const uint32_t f = q < 7u ? 0u : q < 13u ? 1u : q < 18u ? 2u : q < 22u ? 3u : q < 25u ? 4u : q < 27u ? 5u : 6u;
                const uint32_t s = q - f * (13u - f) / 2u + 1u;
                if (s >= m.count || f == cand || s == cand) continue;
                const V3 pf = at(f);
                const V3 e = sub(at(s), pf);
                const float e2 = len2(e);
                if (e2 <= t2) continue;
                const float t = dot(sub(p, pf), e) / e2;
                if (t <= 1.0e-4f || t >= 0.9999f) continue;
                const V3 cl = add(pf, mul(e, t));
                if (len2(sub(p, cl)) > t2) continue;
                on = true;
            }
            removed = row_bits(on) != 0u;
            if (!removed) ++cand;
        }
        if (removed) {
            const uint32_t from = lane >= cand && lane < 15u ? lane + 1u : lane;
            m.point = row_get(m.point, from);
            m.pen = __shfl(m.pen, int(from), 16);
            --m.count;
            cand = 0;
        }
    }
}

// The separating-axis search of rigid_convex_face_manifold
// (geometry.slang:1606-1745) for a row: the face of
// the largest separation (the collider's faces first), kFaceApart past reach.
constexpr uint32_t kFaceApart = 0xffffffffu;
__device__ __forceinline__ uint32_t row_axis(const FaceGeometry &geo, const FaceSide &body, const FaceSide &collider,
                                             float reach, uint32_t lane) {
    const uint32_t nc = collider.faces, faces = nc + body.faces;
    float best = -3.402823466e+38f;
    uint32_t best_at = 0xffffu;
    for (uint32_t j = lane; j < faces; j += kFaceLanes) {
        const bool of_c = j < nc;
        const FaceSide rm = pick(of_c, collider, body), im = pick(of_c, body, collider);
        const float4 pl = geo.planes[rm.planes + (of_c ? j : j - nc)];
        const V3 nrm = rotate(rm.rot, v3(pl));
        const V3 inn = inv_rotate(im.rot, nrm);
        const float sep = face_support(geo, im, inn) + dot(nrm, sub(im.pos, rm.pos)) - pl.w;
        if (sep > best) { best = sep; best_at = j; }
    }
    row_first_max(best, best_at);
    if (best > reach) return kFaceApart;
    return best_at == 0xffffu ? 0u : best_at;
}

// Clips the polygon in S.wide[0] by the planes from `pi` on, on one lane;
// returns its vertices and, in `buf`, the buffer they end in.
__device__ __forceinline__ uint32_t clip_wide(const float4 *planes, uint32_t pi, uint32_t count_planes, V3 rn, float reach,
                                              uint32_t count, FaceShared &S, uint32_t &buf) {
    buf = 0;
#pragma unroll 1
    for (; pi < count_planes && count != 0u; ++pi) {
        const float4 pl = planes[pi];
        const V3 pn = v3(pl);
        const float off = pl.w + (dot(pn, rn) > 0.99999f ? reach : 0.0f);
        float (*const from)[3] = S.wide[buf], (*const to)[3] = S.wide[buf ^ 1u];
        uint32_t next = 0;
        V3 prev = {from[count - 1][0], from[count - 1][1], from[count - 1][2]};
        float pd = dot(pn, prev) - off;
        auto put = [&](V3 x) {
            if (next >= kFacePolygon) return;
            to[next][0] = x.x; to[next][1] = x.y; to[next][2] = x.z;
            ++next;
        };
#pragma unroll 1
        for (uint32_t k = 0; k < count; ++k) {
            const V3 cur = {from[k][0], from[k][1], from[k][2]};
            const float d = dot(pn, cur) - off;
            if ((d <= 0.0f) != (pd <= 0.0f)) put(add(prev, mul(sub(cur, prev), pd / (pd - d))));
            if (d <= 0.0f) put(cur);
            prev = cur;
            pd = d;
        }
        count = next;
        buf ^= 1u;
    }
    return count;
}

// The rest of rigid_convex_face_manifold for a row; false where it finds no
// contact.  A polygon that grows past `widest` vertices (at most one per lane)
// goes on in LDS, its planes on one lane.  A plane adds at most one vertex to
// a convex polygon, so that is expected of shapes of more than 13 triangles;
// rounded distances can cut a sliver more than twice in any.
__device__ __forceinline__ bool row_clip(const FaceGeometry &geo, const FaceSide &body, const FaceSide &collider,
                                         float margin, float reach, uint32_t best_at, uint32_t widest,
                                         uint32_t lane, FaceShared &S, RowManifold &out) {
    const float rest = smin(margin, 1.0e-3f);
    const uint32_t nc = collider.faces;
    const bool ref_is_body = best_at >= nc;
    const uint32_t ref_face = ref_is_body ? best_at - nc : best_at;
    const FaceSide rm = pick(ref_is_body, body, collider), im = pick(ref_is_body, collider, body);
    const Q rq = rm.rot;
    const float4 reference = geo.planes[rm.planes + ref_face];
    const V3 rn = v3(reference);
    const V3 outward = rotate(rq, rn);
    const V3 iaxis = inv_rotate(im.rot, outward);
    const uint32_t ni = im.faces, rfaces = rm.faces;
    const float4 *ip = geo.planes + im.planes, *rp = geo.planes + rm.planes;
    // The most opposed face: the smallest alignment below one, negated for
    // the search (the first face when none is below).
    float opposed = -1.0f;
    uint32_t inc_face = 0xffffu;
    for (uint32_t f = lane; f < ni; f += kFaceLanes) {
        const float val = -dot(iaxis, v3(ip[f]));
        if (val > opposed) { opposed = val; inc_face = f; }
    }
    row_first_max(opposed, inc_face);
    if (inc_face == 0xffffu) inc_face = 0u;
    out.normal = mul(outward, ref_is_body ? -1.0f : 1.0f);
    const float4 incident = ip[inc_face];
    for (uint32_t t0 = 0; t0 < ni; t0 += kFaceLanes) {
        // The triangles of the incident face among these 16.
        bool same = t0 + lane < ni;
        if (same) {
            const float4 face = ip[t0 + lane];
            if (dot(v3(face), v3(incident)) < 0.99999f || fabsf(face.w - incident.w) > 1.0e-5f) same = false;
        }
        for (uint32_t todo = row_bits(same); todo != 0u; todo &= todo - 1u) {
            const uint32_t t = t0 + __builtin_ctz(todo);
            uint32_t count = 3, wide = 2u;           // 2: one vertex per lane
            V3 cur = {0.0f, 0.0f, 0.0f};
            if (lane < 3u) {
                const V3 local = geo.verts[im.verts + geo.idx[im.indices + t * 3 + lane]];
                cur = inv_rotate(rq, sub(add(im.pos, rotate(im.rot, local)), rm.pos));
            }
            for (uint32_t pi = 0; pi < rfaces && count != 0u; ++pi) {
                const float4 pl = rp[pi];
                const V3 pn = v3(pl);
                const float off = pl.w + (dot(pn, rn) > 0.99999f ? reach : 0.0f);
                const float d = dot(pn, cur) - off;
                const uint32_t all = (1u << count) - 1u;
                const uint32_t in = row_bits(d <= 0.0f) & all;
                if (in == all) continue;             // every vertex kept
                if (in == 0u) { count = 0; break; }
                // Vertex k follows vertex k - 1 (the first the last); where
                // the two differ, their crossing comes before vertex k.
                const uint32_t before = ((in << 1) | (in >> (count - 1u))) & all;
                const uint32_t cut = in ^ before;
                const uint32_t next = __builtin_popcount(in) + __builtin_popcount(cut);
                if (next > widest) {
                    row_sync();
                    if (lane < count) {
                        S.wide[0][lane][0] = cur.x; S.wide[0][lane][1] = cur.y; S.wide[0][lane][2] = cur.z;
                    }
                    row_sync();
                    if (lane == 0u) count = clip_wide(rp, pi, rfaces, rn, reach, count, S, wide);
                    row_sync();
                    count = uint32_t(__shfl(int(count), 0, 16));
                    wide = uint32_t(__shfl(int(wide), 0, 16));
                    break;
                }
                const uint32_t prev_lane = lane == 0u ? count - 1u : lane - 1u;
                const V3 prev = row_get(cur, prev_lane);
                const float pd = __shfl(d, int(prev_lane), 16);
                const uint32_t below = (1u << lane) - 1u;
                uint32_t at = __builtin_popcount(in & below) + __builtin_popcount(cut & below);
                row_sync();
                if (lane < count && ((cut >> lane) & 1u)) {
                    const V3 x = add(prev, mul(sub(cur, prev), pd / (pd - d)));
                    S.v[at][0] = x.x; S.v[at][1] = x.y; S.v[at][2] = x.z;
                    ++at;
                }
                if (lane < count && ((in >> lane) & 1u)) {
                    S.v[at][0] = cur.x; S.v[at][1] = cur.y; S.v[at][2] = cur.z;
                }
                row_sync();
                count = next;
                cur = {S.v[lane][0], S.v[lane][1], S.v[lane][2]};
            }
#pragma unroll 1
            for (uint32_t k0 = 0; k0 < count; k0 += kFaceLanes) {
                if (wide < 2u) {
                    const float *q = S.wide[wide][min(k0 + lane, kFacePolygon - 1u)];
                    cur = {q[0], q[1], q[2]};
                }
                const float d = dot(rn, cur) - reference.w;
                const V3 point = add(rm.pos, rotate(rq, sub(cur, mul(rn, d * 0.5f))));
                const float pen = rest - d + 1.0e-5f;
                for (uint32_t keep = row_bits(k0 + lane < count && !(d > reach)); keep != 0u; keep &= keep - 1u) {
                    const uint32_t k = __builtin_ctz(keep);
                    row_add_contact(out, lane, row_get(point, k), __shfl(pen, int(k), 16), smax(margin * 2.0f, 1.0e-4f));
                }
            }
        }
    }
    if (out.count == 0u) return false;
    row_reduce_patch(out, lane, S, smax(1.0e-6f, margin * 1.0e-3f));
    return true;
}

// The separating-axis half of rigid_swept_convex_face_manifold
// (geometry.slang:1751-1853) for a row.
enum : uint32_t { kSweptDecline = 0, kSweptEmpty = 1, kSweptTouching = 2, kSweptImpact = 3 };
__device__ __forceinline__ uint32_t row_swept_entry(const FaceGeometry &geo, const FaceSide &pb, const FaceSide &b,
                                                    const FaceSide &pc, const FaceSide &c, float margin, uint32_t lane,
                                                    float &entry, V3 &entry_normal) {
    const Q bd = relative_quaternion(pb.rot, b.rot, false);
    const Q cd = relative_quaternion(pc.rot, c.rot, false);
    if (bd.x != 0.0f || bd.y != 0.0f || bd.z != 0.0f || cd.x != 0.0f || cd.y != 0.0f || cd.z != 0.0f)
        return kSweptDecline;
    const V3 bmo = sub(b.pos, pb.pos), cmo = sub(c.pos, pc.pos);
    const float rest = smin(margin, 1.0e-3f);
    float exit_time = 1.0f;
    entry = 0.0f;
    uint32_t entry_at = 0xffffu;
    bool apart = false;
    const uint32_t nc = pc.faces, faces = nc + pb.faces;
    for (uint32_t j = lane; j < faces; j += kFaceLanes) {
        const bool of_c = j < nc;
        const FaceSide rm = pick(of_c, pc, pb), im = pick(of_c, pb, pc);
        const V3 rel = of_c ? sub(bmo, cmo) : sub(cmo, bmo);
        const float4 pl = geo.planes[rm.planes + (of_c ? j : j - nc)];
        const V3 nrm = rotate(rm.rot, v3(pl));
        const V3 inn = inv_rotate(im.rot, nrm);
        const float gap = face_support(geo, im, inn) + dot(nrm, sub(im.pos, rm.pos)) - pl.w;
        const float speed = dot(nrm, rel);
        if (speed == 0.0f) {
            apart = apart || gap > rest;
        } else {
            const float crossing = (rest - gap) / speed;
            if (speed < 0.0f && crossing > entry) { entry = crossing; entry_at = j; }
            if (speed > 0.0f) exit_time = smin(exit_time, crossing);
        }
    }
    if (row_bits(apart) != 0u) return kSweptEmpty;
    row_first_max(entry, entry_at);
    exit_time = row_min(exit_time);
    if (entry > exit_time || entry > 1.0f || exit_time < 0.0f) return kSweptEmpty;
    if (entry == 0.0f) return kSweptTouching;
    const bool of_c = entry_at < nc;
    const FaceSide rm = pick(of_c, pc, pb);
    entry_normal = mul(rotate(rm.rot, v3(geo.planes[rm.planes + (of_c ? entry_at : entry_at - nc)])), of_c ? 1.0f : -1.0f);
    return kSweptImpact;
}

// One thread per pair: the convex face path (and its swept variant) for
// convex meshes, closed forms for round shapes.  Mesh pairs the face path
// declines are queued for the triangle-pair kernel.
// The narrowphase runs in two kernels so that no wavefront mixes the cheap
// analytic pairs with the convex face path's separating-axis search:
// k_narrowphase solves every pair with an analytic shape and queues the
// pairs of two meshes; k_face_pairs runs the face path over that queue and
// passes what it declines on to the triangle-pair path.  Each pair's output
// sits at its own index, so the queues' order changes nothing.
//
// A block reserves the points and list places of its 256 pairs with one
// atomic each: atomics on one address queue (about 10 ns each), and one per
// wavefront kept this kernel at 121 us on a heap of 32768 bodies (517k pairs),
// now 43 us.
constexpr uint32_t kNarrowBlock = 256;
__global__ void __launch_bounds__(kNarrowBlock) k_narrowphase(const uint32_t *npairs, const PmhBodyParameters *P,
                                                              const ShapeDev *shapes, const PmhRigidBodyState *prev,
                                                              const PmhRigidBodyState *pred, const uint2 *ab,
                                                              NarrowOut o, uint32_t *face_list,
                                                              const HingeFrame *frames, const float4 *frame_ref) {
    __shared__ uint32_t part[2][kNarrowBlock / 64], base[2];
    const uint32_t M = *npairs;
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    uint32_t unsupported = 0;
    for (uint32_t first = blockIdx.x * kNarrowBlock; first < M; first += gridDim.x * kNarrowBlock) {
        const uint32_t m = first + threadIdx.x;
        Manifold man;
        man.count = 0;
        man.face_patch = 0;
        bool mesh = false, persistent = false;
        uint2 p = make_uint2(0u, 0u);
        PmhRigidBodyState A, B;
        HingeFrame ha, hb;
        if (m < M) {
            p = ab[m];
            const PmhBodyParameters pa = P[p.x], pb = P[p.y];
            const ShapeDev sa = shapes[pa.mesh_index], sb = shapes[pb.mesh_index];
            mesh = sa.kind == kShapeMesh && sb.kind == kShapeMesh;
            if (!mesh) {
                A = pred[p.x];
                B = pred[p.y];
                const float margin = pa.collision_margin + pb.collision_margin;
                const float cr = correction_reach(pa, sa) + correction_reach(pb, sb);
                const PairFrames fr = pair_frames(frames, frame_ref, pa, pb, p, prev[p.x], A);
                ha = fr.ha;
                hb = fr.hb;
                persistent = persistent_pair(sa, sb, pb);
                if (!analytic_manifold(A, sa, B, sb, margin, margin + cr, man)) {
                    man.count = 0;
                    man.face_patch = 0;
                    ++unsupported;
                }
            }
        }
        // Places: this thread's within its wavefront, the wavefronts' within
        // the block, the block's from one atomic per counter.
        const uint64_t meshes = __ballot(mesh);
        const uint32_t points_before = wave_exclusive_scan(man.count, lane);
        if (lane == 63u) {
            part[0][wave] = points_before + man.count;
            part[1][wave] = uint32_t(__popcll(meshes));
        }
        __syncthreads();
        if (threadIdx.x < 2u) {
            uint32_t total = 0;
            for (uint32_t w = 0; w < kNarrowBlock / 64; ++w) {
                const uint32_t v = part[threadIdx.x][w];
                part[threadIdx.x][w] = total;
                total += v;
            }
            base[threadIdx.x] =
                total ? atomicAdd(threadIdx.x == 0u ? &o.ctr->point_alloc : &o.ctr->face_pairs, total) : 0u;
        }
        __syncthreads();
        if (mesh) {
            face_list[base[1] + part[1][wave] + uint32_t(__popcll(meshes & ((1ull << lane) - 1ull)))] = m;
        } else if (m < M) {
            write_manifold(o, m, man, base[0] + part[0][wave] + points_before, A, B, persistent, ha, hb);
        }
        __syncthreads();
    }
    if (unsupported) atomicAdd(&o.ctr->unsupported, unsupported);
}

// The queued mesh pairs, one row of 16 lanes each.  The face path runs at
// most twice on the swept side (at the predicted states, then at the previous
// ones, or at the time of impact) and once without; the rows of a wavefront
// may be at different ones of these.
//
// One lane per pair took 213 us on a 55-box pyramid and 716 us on a heap of
// 32768 bodies (one lane's serial search and clipping in scratch memory, too
// few wavefronts in flight to hide it), and 538 us on 1024 scenes; rows take 31,
// 188 and 194 us.
//
// A block first reads its pairs one lane each (bodies, shapes, whether the
// pair is swept) into records in LDS, then its rows take the records one by
// one: read by every lane of a row, that set-up cost more than the search on
// worlds with many pairs that turn out apart.
constexpr uint32_t kFaceBlock = 256, kFaceRows = kFaceBlock / kFaceLanes;
constexpr uint32_t kFaceChunk = 64;     // most pairs of a block's round
struct FaceInput {
    float pose[4][7];                   // body before, after; collider before, after
    uint32_t shape[2][5];               // planes, vertices, vertex count, indices, faces
    float margin, reach;                // reach: the bounded solver correction
};
struct FaceResult {                     // in the place of the input of a pair that is done
    float contact[8][4];                // point and penetration
    float normal[3], impact;
    uint32_t count, face_patch, kind, start;
};
enum : uint32_t { kResultEmit = 0, kResultTriangles = 1 };
struct FaceRecord {
    union {
        FaceInput in;
        FaceResult out;
    };
    uint32_t pair, flags;
    float entry, normal[3];             // swept: time of impact and its axis
    uint32_t at, axis;                  // where the search stands, and the reference face
    uint32_t pad;                       // odd stride: the records of a wavefront's lanes hit different banks
};
static_assert(sizeof(FaceRecord) % 8 == 4, "odd number of words");
enum : uint32_t { kFaceConvex = 1, kFaceSwept = 2, kFaceGuided = 4, kFacePersistent = 8 };

__device__ __forceinline__ FaceSide record_side(const FaceRecord &r, uint32_t pose, uint32_t shape) {
    const float *q = r.in.pose[pose];
    const uint32_t *s = r.in.shape[shape];
    return {{q[0], q[1], q[2]}, {q[3], q[4], q[5], q[6]}, s[0], s[1], s[2], s[3], s[4]};
}

__global__ void __launch_bounds__(kFaceBlock) k_face_pairs(const uint32_t *face_list, const PmhBodyParameters *P,
                                                           const ShapeDev *shapes, FaceGeometry geo,
                                                           const PmhRigidBodyState *prev, const PmhRigidBodyState *pred,
                                                           const uint2 *ab, NarrowOut o, uint32_t *tri_list,
                                                           const HingeFrame *frames, uint32_t widest) {
    __shared__ FaceShared shared_rows[kFaceRows];
    __shared__ FaceRecord records[kFaceChunk];
    __shared__ uint8_t list[kFaceChunk];
    __shared__ uint32_t listed;
    const uint32_t row = threadIdx.x / kFaceLanes, lane = threadIdx.x % kFaceLanes;
    FaceShared &S = shared_rows[row];
    const uint32_t F = o.ctr->face_pairs;
    // One pair per row while blocks are left, then more per block.
    const uint32_t share = (F + gridDim.x - 1) / gridDim.x;
    const uint32_t chunk = min(max((share + kFaceRows - 1) / kFaceRows * kFaceRows, kFaceRows), kFaceChunk);
    enum : uint32_t { kPlain, kAtEnd, kAtStart, kAtImpact, kDone, kListed };
    for (uint32_t base = blockIdx.x * chunk; base < F; base += gridDim.x * chunk) {
        const uint32_t pairs = min(chunk, F - base);
        if (threadIdx.x < pairs) {
            FaceRecord &r = records[threadIdx.x];
            const uint32_t m = face_list[base + threadIdx.x];
            const uint2 p = ab[m];
            const PmhBodyParameters pa = P[p.x], pb = P[p.y];
            const ShapeDev sa = shapes[pa.mesh_index], sb = shapes[pb.mesh_index];
            const PmhRigidBodyState A0 = prev[p.x], A = pred[p.x], B0 = prev[p.y], B = pred[p.y];
            const float margin = pa.collision_margin + pb.collision_margin;
            // Of the bodies' hinge contact frames only flags matter here.
            bool guided = false, persistent = persistent_pair(sa, sb, pb);
            if (frames) {
                const HingeFrame &ha = frames[p.x], &hb = frames[p.y];
                guided = guided_pair(ha, hb);
                persistent = guided || (persistent && ha.present == 0u && hb.present == 0u && ha.fixed_member == 0u &&
                                        hb.fixed_member == 0u);
            }
            auto put = [&](uint32_t k, const PmhRigidBodyState &s) {
                r.in.pose[k][0] = s.position.x; r.in.pose[k][1] = s.position.y; r.in.pose[k][2] = s.position.z;
                r.in.pose[k][3] = s.orientation.x; r.in.pose[k][4] = s.orientation.y; r.in.pose[k][5] = s.orientation.z;
                r.in.pose[k][6] = s.orientation.w;
            };
            put(0, A0);
            put(1, A);
            put(2, B0);
            put(3, B);
            auto shape = [&](uint32_t k, const ShapeDev &s) {
                r.in.shape[k][0] = s.plane_off; r.in.shape[k][1] = s.vtx_off; r.in.shape[k][2] = s.vtx_count;
                r.in.shape[k][3] = s.idx_off; r.in.shape[k][4] = s.idx_count / 3;
            };
            shape(0, sa);
            shape(1, sb);
            r.in.margin = margin;
            r.in.reach = correction_reach(pa, sa) + correction_reach(pb, sb);
            r.pair = m;
            // A guided pair leaves the face path (geometry.slang:2779).
            const bool convex = sa.convex_face && sb.convex_face && !guided;
            r.flags = (convex ? kFaceConvex : 0u) | (guided ? kFaceGuided : 0u) | (persistent ? kFacePersistent : 0u) |
                      (convex && requires_swept(A0, A, sa, B0, B, sb, margin) ? kFaceSwept : 0u);
        }
        if (threadIdx.x == 0) listed = 0;
        __syncthreads();
        // Stage 0 searches the axes; pairs that are apart end there, the
        // others are listed for stage 1, which clips.  A wavefront's four
        // rows run in step: without the list one pair to clip made three
        // that were done wait.
#pragma unroll 1
        for (uint32_t stage = 0; stage < 2u; ++stage) {
            const uint32_t todo = stage == 0u ? pairs : listed;
            for (uint32_t k = row; k < todo; k += kFaceRows) {
                FaceRecord &r = records[stage == 0u ? k : list[k]];
                const uint32_t flags = r.flags;
                const float margin = r.in.margin, rest = smin(margin, 1.0e-3f);
                const bool swept = (flags & kFaceSwept) != 0u;
                RowManifold man;
                man.count = 0;
                man.normal = man.point = {0.0f, 0.0f, 0.0f};
                man.pen = 0.0f;
                man.impact = 1.0f;
                bool face = false;
                uint32_t face_patch = 0, at = (flags & kFaceConvex) != 0u ? kPlain : kDone, axis = 0;
                float entry = 0.0f;
                V3 entry_normal = {0.0f, 0.0f, 0.0f};
                if (stage != 0u) {
                    at = r.at;
                    axis = r.axis;
                    entry = r.entry;
                    entry_normal = {r.normal[0], r.normal[1], r.normal[2]};
                } else if (swept) {
                    const uint32_t kind = row_swept_entry(geo, record_side(r, 0, 0), record_side(r, 1, 0),
                                                          record_side(r, 2, 1), record_side(r, 3, 1), margin, lane, entry,
                                                          entry_normal);
                    if (kind == kSweptEmpty) { at = kDone; face = true; }
                    else if (kind == kSweptTouching) at = kAtEnd;
                    else if (kind == kSweptImpact) at = kAtImpact;
                }
                bool search = stage == 0u;
                while (at < kDone) {
                    const uint32_t end = at == kAtStart || at == kAtImpact ? 0u : 1u;
                    FaceSide a = record_side(r, end, 0), b = record_side(r, 2u + end, 1);
                    if (at == kAtImpact) {
                        a.pos = add(a.pos, mul(sub(record_side(r, 1, 0).pos, a.pos), entry));
                        b.pos = add(b.pos, mul(sub(record_side(r, 3, 1).pos, b.pos), entry));
                    }
                    const float mg = at == kAtImpact ? rest + 1.0e-5f : margin;
                    const float reach = mg + (at == kPlain ? r.in.reach : 0.0f);
                    if (search) axis = row_axis(geo, a, b, reach, lane);
                    search = true;
                    bool ok = true;
                    man.count = 0;
                    man.impact = 1.0f;
                    if (axis != kFaceApart) {
                        if (stage == 0u) {
                            if (lane == 0u) {
                                r.at = at;
                                r.axis = axis;
                                r.entry = entry;
                                r.normal[0] = entry_normal.x;
                                r.normal[1] = entry_normal.y;
                                r.normal[2] = entry_normal.z;
                                list[atomicAdd(&listed, 1u)] = uint8_t(k);
                            }
                            at = kListed;
                            break;
                        }
                        ok = row_clip(geo, a, b, mg, reach, axis, widest, lane, S, man);
                    }
                    face_patch = ok && man.count != 0u ? 1u : 0u;
                    if (at == kPlain) {
                        face = ok && !(swept && man.count == 0u);
                        at = kDone;
                    } else if (!ok || man.count == 0u) {
                        at = at == kAtEnd ? kAtStart : kPlain;
                    } else if (at == kAtEnd) {
                        face = true;
                        at = kDone;
                    } else {
                        const V3 motion = sub(sub(record_side(r, 1, 0).pos, record_side(r, 0, 0).pos),
                                              sub(record_side(r, 3, 1).pos, record_side(r, 2, 1).pos));
                        const float closing = -dot(motion, man.normal);
                        if (at == kAtStart) {
                            face = !(closing <= 0.0f);
                            man.pen += closing;
                            man.impact = 0.0f;
                        } else {
                            face = !(dot(man.normal, entry_normal) < 0.99999f);
                            const float remaining = closing * (1.0f - entry);
                            man.pen = smax(0.0f, remaining + man.pen) + rest + 1.0e-5f;
                            man.impact = entry;
                        }
                        at = face ? kDone : kPlain;
                    }
                }
                if (at == kListed) continue;
                row_sync();
                if (lane < man.count) {
                    r.out.contact[lane][0] = man.point.x; r.out.contact[lane][1] = man.point.y;
                    r.out.contact[lane][2] = man.point.z; r.out.contact[lane][3] = man.pen;
                }
                if (lane == 0u) {
                    r.out.normal[0] = man.normal.x; r.out.normal[1] = man.normal.y; r.out.normal[2] = man.normal.z;
                    r.out.impact = man.impact;
                    r.out.kind = face ? kResultEmit : kResultTriangles;
                    r.out.count = face ? man.count : 0u;
                    r.out.face_patch = face_patch;
                }
            }
            __syncthreads();
        }
        // The block's results go out together: one reservation of points and
        // of list places for all its pairs (atomics on one address queue,
        // about 10 ns each), then one thread per contact.
        if (threadIdx.x < 64u) {
            const bool live = threadIdx.x < pairs;
            FaceRecord &r = records[live ? threadIdx.x : 0u];
            const uint32_t kind = live ? r.out.kind : kResultEmit;
            uint32_t count = live ? r.out.count : 0u;
            const uint64_t tri = __ballot(kind == kResultTriangles);
            const uint32_t before = wave_exclusive_scan(count, threadIdx.x), total = wave_sum(count);
            uint32_t at_point = 0, at_tri = 0;
            if (threadIdx.x == 0u) {
                if (total) at_point = atomicAdd(&o.ctr->point_alloc, total);
                if (tri) at_tri = atomicAdd(&o.ctr->tri_pairs, uint32_t(__popcll(tri)));
            }
            const uint64_t below = (1ull << threadIdx.x) - 1ull;
            const uint32_t start = __shfl(at_point, 0, 64) + before;
            at_tri = __shfl(at_tri, 0, 64) + uint32_t(__popcll(tri & below));
            if (live) {
                const uint32_t m = r.pair;
                if (kind == kResultTriangles) {
                    tri_list[at_tri] = m;
                } else {
                    if (count && start + count > o.point_cap) {
                        atomicOr(&o.ctr->status, kStatusPointOverflow);
                        count = 0;
                    }
                    const uint2 p = ab[m];
                    o.m_count[m] = count;
                    o.m_start[m] = start;
                    o.m_face[m] = r.out.face_patch;
                    o.m_init_rel[m] = f4(sub(sv(pred[p.x].position), sv(pred[p.y].position)), 0.0f);
                }
                r.out.count = count;
                r.out.start = start;
            }
        }
        __syncthreads();
        for (uint32_t k = threadIdx.x; k < 8u * pairs; k += kFaceBlock) {
            const FaceRecord &r = records[k / 8u];
            const uint32_t q = k % 8u;
            if (q >= r.out.count) continue;
            const uint32_t i = r.out.start + q, m = r.pair;
            const uint2 p = ab[m];
            const PmhRigidBodyState A = pred[p.x], B = pred[p.y];
            const float *c = r.out.contact[q];
            const V3 normal = {r.out.normal[0], r.out.normal[1], r.out.normal[2]}, point = {c[0], c[1], c[2]};
            const float4 z = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            o.c_np[i] = f4(normal, c[3]);
            o.c_pt[i] = f4(point, normal_speed(A, B, point, normal));
            o.c_aa[i] = make_float4(0.0f, 0.0f, 0.0f, r.out.impact);   // w: impact fraction
            o.c_ab[i] = z;
            o.c_err[i] = z;
            o.c_lam[i] = z;
            o.c_pen[i] = z;
            o.c_acc[i] = z;
            o.c_rep[i] = z;
            o.c_flags[i] = ((r.flags & kFacePersistent) ? 2u : 0u) | ((r.flags & kFaceGuided) ? kPointGuided : 0u);
            o.c_pair[i] = m;
        }
        __syncthreads();
    }
}

// Scenes of a batch: each body's scene, each scene's body count and the
// index of its first pair (pairs are sorted by body, scenes are contiguous
// body ranges).
struct SceneRules {
    const uint32_t *scene = nullptr;
    const uint32_t *count = nullptr;
    const uint32_t *pair_start = nullptr;
};

// Candidate slots of a world of n bodies: the contact-cache slot rule,
// min(n(n-1)/2, max(4096, 8n)) (resource_plan.hpp:151-164).
__host__ __device__ inline uint32_t leaf_slot_rule(uint64_t n) {
    const uint64_t pairs = n * (n - 1) / 2;
    const uint64_t cap = 8 * n > 4096 ? 8 * n : 4096;
    return uint32_t(pairs < cap ? pairs : cap);
}

__global__ void k_scene_pairs(const uint32_t *npairs, const uint2 *ab, const uint32_t *scene, uint32_t *pair_start) {
    const uint32_t M = *npairs;
    for (uint32_t m = blockIdx.x * blockDim.x + threadIdx.x; m < M; m += gridDim.x * blockDim.x) {
        const uint32_t s = scene[ab[m].x];
        if (m == 0 || scene[ab[m - 1].x] != s) pair_start[s] = m;
    }
}

// ---- triangle-pair kernel: one wavefront per queued pair ----------------
constexpr uint32_t kTriWaves = 4;          // wavefronts per block
constexpr uint32_t kLeafListCap = 512;     // ordered leaf pairs held in LDS per wavefront
constexpr uint32_t kListOverflow = 0xffffffffu;
constexpr uint32_t kTraversalStack = 64;   // the reference's
constexpr uint32_t kTriBatch = 16;         // triangle pairs of a wavefront's batch, four lanes each

struct TriWaveShared {
    uint2 list[kLeafListCap];              // (body leaf node, collider leaf node) in evaluation order
    uint2 stack[kTraversalStack];          // of the BVH traversal
    uint32_t cand[kTriBatch];              // triangle pairs to evaluate: leaf pair << 4 | slot in it
    uint32_t found[2];                     // which of them gave a contact, discrete and swept
    uint32_t held;                         // how many there are
    float4 disc[kTriBatch][2], swept[kTriBatch][2];   // their contacts: normal+pen, point+impact fraction
    Manifold man, local;
    uint32_t count;
    // The wavefront's triangle pair (one per wavefront, read by every lane):
    // held here rather than copied into each lane's private memory.
    alignas(16) unsigned char pair[sizeof(TrianglePair)];
};

__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
    __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ bool leaf_cell_overlaps(const TrianglePair &tp, bool swept, const BoundsFrame &fa,
                                                   const BoundsFrame &fb, const BoundsFrame &pfa,
                                                   const BoundsFrame &pfb, uint64_t f, uint2 &nodes) {
    const uint32_t lb = tp.bm.s.leaf_count;
    nodes = make_uint2(tp.am.leaf(uint32_t(f / lb)), tp.bm.leaf(uint32_t(f % lb)));
    V3 amn, amx, bmn, bmx;
    node_bounds(tp.am.node(nodes.x), pfa, fa, swept, tp.margin, amn, amx);
    node_bounds(tp.bm.node(nodes.y), pfb, fb, swept, 0.0f, bmn, bmx);
    return boxes_touch(amn, amx, bmn, bmx);
}

// The leaf pairs rigid_collide_meshes visits, in visiting order, or
// kListOverflow when its stack would overflow (the reference then runs
// every triangle pair) or the list does not fit.
__device__ uint32_t traversal_list(const TrianglePair &P, bool swept, uint2 *list, uint2 *stack) {
    const BoundsFrame fa = bounds_frame(P.a), fb = bounds_frame(P.b);
    const BoundsFrame pfa = swept ? bounds_frame(P.ap) : BoundsFrame{};
    const BoundsFrame pfb = swept ? bounds_frame(P.bp) : BoundsFrame{};
    V3 amn, amx, bmn, bmx;
    motion_bounds(sarr(P.am.s.mn), sarr(P.am.s.mx), pfa, fa, swept, P.margin, amn, amx);
    motion_bounds(sarr(P.bm.s.mn), sarr(P.bm.s.mx), pfb, fb, swept, 0.0f, bmn, bmx);
    if (!boxes_touch(amn, amx, bmn, bmx)) return 0;
    if (P.am.s.node_count == 0u || P.bm.s.node_count == 0u) return kListOverflow;
    stack[0] = make_uint2(0u, 0u);
    uint32_t top = 1, count = 0;
    while (top > 0u) {
        --top;
        const uint32_t ia = stack[top].x, ib = stack[top].y;
        const BvhDev na = P.am.node(ia), nb = P.bm.node(ib);
        node_bounds(na, pfa, fa, swept, P.margin, amn, amx);
        node_bounds(nb, pfb, fb, swept, 0.0f, bmn, bmx);
        if (!boxes_touch(amn, amx, bmn, bmx)) continue;
        const bool la = na.count != 0u, lb = nb.count != 0u;
        if (la && lb) {
            if (count == kLeafListCap) return kListOverflow;
            list[count++] = make_uint2(ia, ib);
            continue;
        }
        const uint32_t need = la || lb ? 2u : 4u;
        if (top + need > kTraversalStack) return kListOverflow;
        if (la) {
            stack[top++] = make_uint2(ia, nb.right);
            stack[top++] = make_uint2(ia, nb.left);
        } else if (lb) {
            stack[top++] = make_uint2(na.right, ib);
            stack[top++] = make_uint2(na.left, ib);
        } else {
            stack[top++] = make_uint2(na.right, nb.right);
            stack[top++] = make_uint2(na.right, nb.left);
            stack[top++] = make_uint2(na.left, nb.right);
            stack[top++] = make_uint2(na.left, nb.left);
        }
    }
    return count;
}

// Serial evaluation for the rare pairs whose leaf list does not fit in
// LDS: the same candidate order and merge rule, the contacts computed on four
// lanes of the same data (which the closest-point search is laid out for) and
// merged by one of them (`writer`), which alone touches the manifolds.  Leaf
// candidates come from the motion test alone (`swept`); the ranges of a
// guided pair always take the swept pass (`swept_eval`).
__device__ void triangle_pair_serial(const TrianglePair &tp, bool swept, bool swept_eval, bool leaf_mode,
                                     Manifold &man, Manifold &local, bool writer) {
    if (!leaf_mode) {
        collide_meshes(tp, swept_eval, man, writer);
        return;
    }
    if (writer) {
        man.count = 0;
        man.face_patch = 0;
    }
    const BoundsFrame fa = bounds_frame(tp.a), fb = bounds_frame(tp.b);
    const BoundsFrame pfa = swept ? bounds_frame(tp.ap) : BoundsFrame{};
    const BoundsFrame pfb = swept ? bounds_frame(tp.bp) : BoundsFrame{};
    const uint64_t cells = uint64_t(tp.am.s.leaf_count) * tp.bm.s.leaf_count;
    const float spacing = smax(tp.margin * 2.0f, 1.0e-4f);
    for (uint32_t w = 0; w < 128u && w < cells; ++w)
        for (uint64_t f = w; f < cells; f += 128u) {
            uint2 nodes;
            if (!leaf_cell_overlaps(tp, swept, fa, fb, pfa, pfb, f, nodes)) continue;
            if (writer) {
                local.count = 0;
                local.face_patch = 0;
            }
            collide_leaf_ranges(tp, swept_eval, tp.am.node(nodes.x), tp.bm.node(nodes.y), local, writer);
            if (writer)
                for (uint32_t k = 0; k < local.count; ++k) merge_contact(tp, man, local.c[k], spacing);
        }
}

// Slot and limit rules of pair m (in a batch those of its own scene): whether
// it has a candidate slot.
__device__ __forceinline__ bool candidate_slot(const SceneRules &scenes, uint32_t m, uint32_t body, uint32_t slots,
                                               uint32_t &limit) {
    if (!scenes.scene) return m < slots;
    const uint32_t sc = scenes.scene[body];
    const uint64_t ns = scenes.count[sc];
    limit = ns <= 8u ? 4096u : 512u;
    return m - scenes.pair_start[sc] < leaf_slot_rule(ns);
}

// Queued pairs whose leaf bounds all miss each other, one thread per pair:
// most of the queue where bodies fly (their boxes swell with the motion), and
// a wavefront's setup, leaf tests and reservation took 16 us for each of them.
// They get their empty manifold here; the others go on to k_triangle_pairs
// with the overlapping cells as a mask.  Pairs of more than 64 cells pass
// unseen.  So do pairs without a candidate slot whose traversal could run out
// of stack (the reference then tries every triangle pair): a level adds at
// most 3 entries while both sides descend and 1 after that, and a tree has
// fewer levels than leaves.  8000 bodies flying into each
// other: 33500 pairs queued, an eighth of them pass, 1.14 ms for the queue, now
// 0.02 here and 0.39 for the rest.  1024 small scenes: 131000 queued, none
// pass, 0.82 ms, now 0.02.
constexpr uint32_t kScreenCells = 64;
constexpr uint32_t kScreenBlock = 256;
__global__ void __launch_bounds__(kScreenBlock) k_triangle_screen(
    const uint32_t *tri_list, const PmhBodyParameters *P, const ShapeDev *shapes, const BvhDev *nodes,
    const uint32_t *leaves, const PmhRigidBodyState *prev, const PmhRigidBodyState *pred, const uint2 *ab, NarrowOut o,
    uint32_t slots, SceneRules scenes, const HingeFrame *frames, uint32_t *hit_list, unsigned long long *hit_mask) {
    __shared__ uint32_t s_count[kScreenBlock / 64], s_base;
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t T = o.ctr->tri_pairs;
    uint32_t fallback = 0;
    for (uint32_t base = blockIdx.x * kScreenBlock; base < T; base += gridDim.x * kScreenBlock) {
        const uint32_t t = base + threadIdx.x;
        uint32_t m = 0;
        bool hit = false;
        uint64_t mask = 0;
        if (t < T) {
            m = tri_list[t];
            const uint2 p = ab[m];
            const ShapeDev sa = shapes[P[p.x].mesh_index], sb = shapes[P[p.y].mesh_index];
            uint32_t unused = 0;
            const bool slot = candidate_slot(scenes, m, p.x, slots, unused);
            const uint64_t cells = uint64_t(sa.leaf_count) * sb.leaf_count;
            const uint32_t few = min(sa.leaf_count, sb.leaf_count), many = max(sa.leaf_count, sb.leaf_count);
            hit = cells > kScreenCells || (!slot && (cells == 0u || 3u * few + (many - few) > 64u));
            if (!hit) {
                const PmhRigidBodyState A0 = prev[p.x], A = pred[p.x], B0 = prev[p.y], B = pred[p.y];
                const float margin = P[p.x].collision_margin + P[p.y].collision_margin;
                bool swept = requires_swept(A0, A, sa, B0, B, sb, margin);
                if (!slot && frames) swept = swept || guided_pair(frames[p.x], frames[p.y]);
                const BoundsFrame fa = bounds_frame(A), fb = bounds_frame(B);
                const BoundsFrame pfa = swept ? bounds_frame(A0) : BoundsFrame{};
                const BoundsFrame pfb = swept ? bounds_frame(B0) : BoundsFrame{};
                for (uint32_t i = 0; i < sa.leaf_count; ++i) {
                    V3 amn, amx;
                    node_bounds(nodes[sa.node_off + leaves[sa.leaf_off + i]], pfa, fa, swept, margin, amn, amx);
                    for (uint32_t j = 0; j < sb.leaf_count; ++j) {
                        V3 bmn, bmx;
                        node_bounds(nodes[sb.node_off + leaves[sb.leaf_off + j]], pfb, fb, swept, 0.0f, bmn, bmx);
                        if (boxes_touch(amn, amx, bmn, bmx)) mask |= 1ull << (i * sb.leaf_count + j);
                    }
                }
                hit = mask != 0ull;
                if (!hit) {
                    fallback += slot ? 0u : 1u;
                    o.m_count[m] = 0u;
                    o.m_start[m] = 0u;
                    o.m_face[m] = 0u;
                    o.m_init_rel[m] = f4(sub(sv(A.position), sv(B.position)), 0.0f);
                }
            }
        }
        const uint64_t hits = __ballot(hit);
        if (lane == 0) s_count[wave] = uint32_t(__popcll(hits));
        __syncthreads();
        if (threadIdx.x == 0) {
            uint32_t total = 0;
            for (uint32_t w = 0; w < kScreenBlock / 64; ++w) {
                const uint32_t c = s_count[w];
                s_count[w] = total;
                total += c;
            }
            s_base = total ? atomicAdd(&o.ctr->tri_hits, total) : 0u;
        }
        __syncthreads();
        if (hit) {
            const uint32_t at = s_base + s_count[wave] + uint32_t(__popcll(hits & ((1ull << lane) - 1ull)));
            hit_list[at] = m;
            hit_mask[at] = mask;
        }
        __syncthreads();
    }
    fallback = wave_sum(fallback);
    if (lane == 0 && fallback) atomicAdd(&o.ctr->fallback_pairs, fallback);
}

// The triangle-pair path for the queued pairs, one wavefront per pair.
// A pair with a candidate slot (active index below `slots`) and at most
// `limit` overlapping leaf pairs takes its candidates in the order 128
// workers emit them (worker w takes cells w, w + 128, ... of the row-major
// leaf-pair grid) and merges each candidate's own manifold in that order;
// any other pair takes the leaf pairs of the BVH traversal in visiting
// order and merges contacts directly.  Of 4 leaf pairs x 16 triangle pairs at
// a time (leaves hold at most 4 triangles) those whose boxes touch are
// gathered until 16 are there, whole leaf pairs at a time, and evaluated on
// four lanes each: by fours of leaf pairs most lanes held pairs that the box
// test ended (8 or 9 of a mesh pair's are left in the mean).  One lane then
// replays the contacts through the merge rule in order: per leaf pair the
// discrete contacts body-triangle-major, then the swept ones.
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) k_triangle_pairs(const uint32_t *hit_list,
                                                        const unsigned long long *hit_mask, const PmhBodyParameters *P,
                                                        const ShapeDev *shapes, const V3 *verts, const uint32_t *idx,
                                                        const float4 *planes, const BvhDev *nodes,
                                                        const uint32_t *leaves, const float4 *shell,
                                                        const PmhRigidBodyState *prev,
                                                        const PmhRigidBodyState *pred, const uint2 *ab,
                                                        NarrowOut o, uint32_t slots, uint32_t limit, float dt,
                                                        SceneRules scenes, const HingeFrame *frames,
                                                        const float4 *frame_ref) {
    __shared__ TriWaveShared shared_waves[kTriWaves];
    const uint32_t lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    TriWaveShared &S = shared_waves[wv];
    const uint32_t T = o.ctr->tri_hits;
    // A list with no more pairs than blocks gives each pair a whole block: its
    // wavefronts gather the same candidates, each evaluates its turn of the
    // batches, and the first merges.  A pair that needs all 32 advances of the
    // swept pass in several batches otherwise outlasts all others (8000 flying
    // bodies, 1400 pairs: 0.31 ms, so 0.25).  A longer list keeps every
    // wavefront busy by itself (7200 pairs of meshes at rest: 0.21 ms, 0.51 by
    // blocks).
    const bool wide = T <= gridDim.x;
    const uint32_t stride = wide ? gridDim.x : gridDim.x * kTriWaves;
    uint32_t fallback = 0;
    for (uint32_t t = wide ? blockIdx.x : blockIdx.x * kTriWaves + wv; t < T; t += stride) {
        const uint32_t m = hit_list[t];
        const uint64_t mask = hit_mask[t];
        const uint2 p = ab[m];
        const PmhBodyParameters pa = P[p.x], pb = P[p.y];
        TrianglePair &shared_pair = *reinterpret_cast<TrianglePair *>(S.pair);
        wave_sync();   // every lane is done with the previous pair
        if (lane == 0)
            shared_pair = TrianglePair{ShapeView{shapes[pa.mesh_index], verts, idx, planes, nodes, leaves, shell},
                                       ShapeView{shapes[pb.mesh_index], verts, idx, planes, nodes, leaves, shell},
                                       prev[p.x], pred[p.x], prev[p.y], pred[p.y],
                                       pair_frames(frames, frame_ref, pa, pb, p, prev[p.x], pred[p.x]),
                                       pa.collision_margin + pb.collision_margin, dt};
        wave_sync();
        const TrianglePair &tp = shared_pair;
        // Leaf candidates from the motion test alone; the ranges of a guided
        // pair always take the swept pass (geometry.slang:2350, 2574-2579,
        // 2167-2170), and its discrete pass finds nothing (:1371).
        const bool guided = guided_pair(tp.f.ha, tp.f.hb);
        const bool swept = requires_swept(tp.ap, tp.a, tp.am.s, tp.bp, tp.b, tp.bm.s, tp.margin);
        const bool swept_eval = guided || swept;
        const BoundsFrame fa = bounds_frame(tp.a), fb = bounds_frame(tp.b);
        const BoundsFrame pfa = swept ? bounds_frame(tp.ap) : BoundsFrame{};
        const BoundsFrame pfb = swept ? bounds_frame(tp.bp) : BoundsFrame{};
        bool inside_a, inside_b;
        inside_flags(tp, inside_a, inside_b);
        const uint64_t cells = uint64_t(tp.am.s.leaf_count) * tp.bm.s.leaf_count;
        // 1. Leaf pairs in evaluation order.
        bool leaf_mode = candidate_slot(scenes, m, p.x, slots, limit);
        const bool known = leaf_mode && mask != 0ull;   // (then there are at most 64 cells, in the grid's order)
        // Each lane counts the cells f = lane (mod 128) and f = lane + 64
        // (mod 128) apart, so the same counts give the total and the list
        // offsets.
        uint32_t total = 0, c0 = 0, c1 = 0;
        if (leaf_mode && !known) {
            uint2 nd;
            for (uint64_t f = lane; f < cells; f += 128u) c0 += leaf_cell_overlaps(tp, swept, fa, fb, pfa, pfb, f, nd) ? 1u : 0u;
            for (uint64_t f = lane + 64u; f < cells; f += 128u) c1 += leaf_cell_overlaps(tp, swept, fa, fb, pfa, pfb, f, nd) ? 1u : 0u;
            total = wave_sum(c0 + c1);
            leaf_mode = total <= limit;
        }
        uint32_t nlist = 0;
        if (known) {
            const uint32_t lb = tp.bm.s.leaf_count;
            if ((mask >> lane) & 1ull)
                S.list[__popcll(mask & ((1ull << lane) - 1ull))] = make_uint2(tp.am.leaf(lane / lb), tp.bm.leaf(lane % lb));
            nlist = uint32_t(__popcll(mask));
        } else if (leaf_mode) {
            if (total > kLeafListCap) {
                nlist = kListOverflow;
            } else {
                uint2 nd;
                uint32_t at0 = wave_exclusive_scan(c0, lane);
                uint32_t at1 = wave_sum(c0) + wave_exclusive_scan(c1, lane);
                for (uint64_t f = lane; f < cells; f += 128u)
                    if (leaf_cell_overlaps(tp, swept, fa, fb, pfa, pfb, f, nd)) S.list[at0++] = nd;
                for (uint64_t f = lane + 64u; f < cells; f += 128u)
                    if (leaf_cell_overlaps(tp, swept, fa, fb, pfa, pfb, f, nd)) S.list[at1++] = nd;
                nlist = total;
            }
        } else {
            if (lane == 0) {
                fallback += wide && wv != 0 ? 0u : 1u;
                S.count = traversal_list(tp, swept_eval, S.list, S.stack);
            }
            wave_sync();
            nlist = S.count;
        }
        wave_sync();
        // 2. Contacts.
        if (nlist == kListOverflow) {
            if (lane < 4u && !(wide && wv != 0)) triangle_pair_serial(tp, swept, swept_eval, leaf_mode, S.man, S.local, lane == 0);
        } else {
            if (lane == 0) {
                S.man.count = 0;
                S.man.face_patch = 0;
            }
            const float spacing = smax(tp.margin * 2.0f, 1.0e-4f);
            uint32_t held = 0, batch = 0;
            // Merges the batches evaluated since the last merge.
            auto merge = [&](uint32_t batches) {
                if (wide) __syncthreads();
                else wave_sync();
                for (uint32_t w = 0; w < batches; ++w) {
                    if (lane != 0 || (wide && wv != 0)) continue;
                    TriWaveShared &R = wide ? shared_waves[w] : S;
                    const uint32_t md = R.found[0], ms = R.found[1];
                    Manifold &dst = leaf_mode ? S.local : S.man;
                    for (uint32_t left = md | ms; left;) {
                        // the candidates of the next leaf pair with contacts
                        const uint32_t k0 = uint32_t(__builtin_ctz(left)), leaf = R.cand[k0] >> 4;
                        uint32_t k1 = k0 + 1;
                        while (k1 < R.held && R.cand[k1] >> 4 == leaf) ++k1;
                        const uint32_t group = (1u << k1) - (1u << k0);
                        left &= ~group;
                        if (leaf_mode) {
                            S.local.count = 0;
                            S.local.face_patch = 0;
                        }
                        for (uint32_t b = md & group; b; b &= b - 1u) {
                            const uint32_t k = uint32_t(__builtin_ctz(b));
                            const Contact c{v3(R.disc[k][0]), v3(R.disc[k][1]), R.disc[k][0].w, R.disc[k][1].w};
                            merge_contact(tp, dst, c, spacing);
                        }
                        for (uint32_t b = ms & group; b; b &= b - 1u) {
                            const uint32_t k = uint32_t(__builtin_ctz(b));
                            const Contact c{v3(R.swept[k][0]), v3(R.swept[k][1]), R.swept[k][0].w, R.swept[k][1].w};
                            merge_contact(tp, dst, c, spacing);
                        }
                        if (leaf_mode)
                            for (uint32_t k = 0; k < S.local.count; ++k) merge_contact(tp, S.man, S.local.c[k], spacing);
                    }
                }
                if (wide) __syncthreads();
                else wave_sync();
                batch = 0;
            };
            // Evaluates the candidates held, as this wavefront's batch or
            // another's.
            auto evaluate = [&]() {
                wave_sync();
                bool hd = false, hs = false;
                Contact cd, cs;
                const bool mine = !wide || batch == wv;
                const uint32_t k = lane / 4u;
                if (mine && k < held) {
                    const uint32_t cand = S.cand[k];
                    const uint2 e = S.list[cand >> 4];
                    const uint32_t at = tp.am.node(e.x).first + (cand >> 2 & 3u);
                    const uint32_t bt = tp.bm.node(e.y).first + (cand & 3u);
                    hd = !guided && triangle_pair_contact(tp, at, bt, inside_a, inside_b, cd);
                    if (swept_eval) hs = triangle_pair_swept_contact(tp, at, bt, inside_a, inside_b, cs);
                }
                if (hd && lane % 4u == 0u) {
                    S.disc[k][0] = f4(cd.normal, cd.pen);
                    S.disc[k][1] = f4(cd.point, cd.impact_fraction);
                }
                if (hs && lane % 4u == 0u) {
                    S.swept[k][0] = f4(cs.normal, cs.pen);
                    S.swept[k][1] = f4(cs.point, cs.impact_fraction);
                }
                if (mine && lane == 0) S.found[0] = S.found[1] = 0u;
                if (hd && lane % 4u == 0u) atomicOr(&S.found[0], 1u << k);
                if (hs && lane % 4u == 0u) atomicOr(&S.found[1], 1u << k);
                if (mine && lane == 0) S.held = held;
                held = 0;
                ++batch;
            };
            for (uint32_t first = 0;; first += 4u) {
                const bool end = first >= nlist;
                const uint32_t j = first + lane / 16u, ai = lane / 4u % 4u, bi = lane % 4u;
                bool near = false;
                if (j < nlist) {
                    const uint2 e = S.list[j];
                    const BvhDev na = tp.am.node(e.x), nb = tp.bm.node(e.y);
                    const uint32_t at = na.first + ai, bt = nb.first + bi;
                    near = ai < na.count && bi < nb.count && 3u * at + 2u < tp.am.s.idx_count &&
                           3u * bt + 2u < tp.bm.s.idx_count && triangle_boxes_touch(tp, at, bt, swept_eval);
                }
                const uint64_t found = __ballot(near);
#pragma unroll 1
                for (uint32_t g = 0; g < 4u; ++g) {
                    const uint32_t bits = uint32_t(found >> (16u * g)) & 0xffffu, count = uint32_t(__popc(bits));
                    if (held + count > kTriBatch || (end && held)) evaluate();
                    if (batch == (wide ? kTriWaves : 1u) || (end && batch)) merge(batch);
                    if (lane / 16u == g && near && (!wide || batch == wv))
                        S.cand[held + __popc(bits & ((1u << (lane % 16u)) - 1u))] = j << 4 | lane % 16u;
                    held += count;
                }
                if (end) break;
            }
        }
        wave_sync();
        // 3. Emit.
        if (lane == 0 && !(wide && wv != 0)) {
            Manifold man = S.man;
            emit_manifold(o, m, man, tp.a, tp.b, persistent_pair(tp.am.s, tp.bm.s, pb), tp.f.ha, tp.f.hb);
        }
        wave_sync();
    }
    if (lane == 0 && fallback) atomicAdd(&o.ctr->fallback_pairs, fallback);
}

__global__ void k_nonempty(const uint32_t *npairs, const uint32_t *m_count, uint32_t *flag) {
    const uint32_t M = *npairs;
    for (uint32_t m = blockIdx.x * blockDim.x + threadIdx.x; m < M; m += gridDim.x * blockDim.x)
        flag[m] = m_count[m] != 0u ? 1u : 0u;
}

// An overflowing step solves nothing (its manifolds are incomplete) and is
// reported as PM_ERROR_CAPACITY_EXCEEDED.
__global__ void k_guard_points(StepCounters *ctr, uint32_t point_cap) {
    if (threadIdx.x != 0) return;
    const uint32_t P = ctr->point_alloc;
    if (P > point_cap) {
        atomicOr(&ctr->status, kStatusPointOverflow);
        ctr->points = 0;
        ctr->pairs = 0;
    } else {
        ctr->points = P;
    }
}

// pm_load_rigid_contact_cache (geometry.slang:2941-3009) against the
// previous step's saved pairs, found by binary search on their sorted codes.
// Cache key of a pair: (a, b) as one 64-bit number, ordered like the
// reference's pair code a*n+b (ascending a, then b) for any body count.
__device__ __forceinline__ unsigned long long pair_key(uint2 p) {
    return ((unsigned long long)p.x << 32) | p.y;
}

__global__ void k_cache_load(const uint32_t *npairs, const uint32_t *code, const uint2 *ab, const uint32_t *m_count,
                             const uint32_t *m_start, const PmhRigidBodyState *pred, const unsigned long long *saved_code,
                             const uint32_t *saved_count, const float4 *saved, const uint32_t *n_saved_ptr,
                             float4 *c_np, float4 *c_pt, float4 *c_aa, float4 *c_ab, float4 *c_lam,
                             float4 *c_pen, float4 *c_acc, uint32_t *c_flags, float dt, StepCounters *ctr) {
    const uint32_t M = *npairs;
    const uint32_t ns = *n_saved_ptr;
    uint32_t hits = 0;
    for (uint32_t m = blockIdx.x * blockDim.x + threadIdx.x; m < M; m += gridDim.x * blockDim.x) {
        if (m_count[m] == 0) continue;
        const unsigned long long key = pair_key(ab[m]);
        uint32_t lo = 0, hi = ns;
        while (lo < hi) {
            const uint32_t mid = (lo + hi) >> 1;
            if (saved_code[mid] < key) lo = mid + 1; else hi = mid;
        }
        if (lo >= ns || saved_code[lo] != key) continue;
        const uint32_t sc = saved_count[lo];
        const float4 *rec = saved + (size_t)lo * 8 * kCacheFloat4PerPoint;
        const PmhRigidBodyState body = pred[ab[m].x];
        uint32_t used = 0;
        for (uint32_t k = 0; k < m_count[m]; ++k) {
            const uint32_t c = m_start[m] + k;
            const V3 n = v3(c_np[c]), point = v3(c_pt[c]);
            const V3 local = inv_rotate(sq(body.orientation), sub(point, sv(body.position)));
            float nearest = 0.02f * 0.02f;
            uint32_t match = 8;
            for (uint32_t q = 0; q < sc; ++q) {
                const float4 *r = rec + q * kCacheFloat4PerPoint;
                if ((used & (1u << q)) != 0u || dot(n, v3(r[1])) < 0.99f) continue;
                const float d = len2(sub(local, v3(r[0])));
                if (d < nearest) { nearest = d; match = q; }
            }
            if (match == 8u) continue;
            used |= 1u << match;
            const float4 *r = rec + match * kCacheFloat4PerPoint;
            // r0: local point, normal impulse; r1: normal; r2: friction
            // impulse; r3: lambdas; r4: penalties; r5: anchor a; anchor b in
            // r1.w/r2.w/r4.w
            V3 t0, t1;
            contact_basis(n, t0, t1);
            const V3 fi = v3(r[2]);
            const float4 lam = r[3], pen = r[4];
            c_lam[c] = make_float4(lam.x, dot(fi, t0) / dt, dot(fi, t1) / dt, 0.0f);
            c_pen[c] = make_float4(pen.x, pen.y, pen.z, 0.0f);
            c_aa[c] = f4(v3(r[5]), c_aa[c].w);
            c_ab[c] = make_float4(r[1].w, r[2].w, r[4].w, 0.0f);
            c_flags[c] |= 1u;
            const V3 af = sub(fi, mul(n, dot(fi, n)));
            c_acc[c] = make_float4(r[0].w, af.x, af.y, af.z);
            ++hits;
        }
    }
    // One atomic per wavefront (one per thread queued ~10^5 atomics on one
    // address).
    hits = wave_sum(hits);
    if ((threadIdx.x & 63) == 0 && hits) atomicAdd(&ctr->cache_hits, hits);
}

// pm_save_rigid_contact_cache (geometry.slang:3011-3070): the pair of
// response slot s (its rank among non-empty manifolds) is saved at s.
__global__ void k_cache_save(const uint32_t *npairs, const uint32_t *code, const uint2 *ab, const uint32_t *m_count,
                             const uint32_t *m_start, const uint32_t *m_slot, const PmhRigidBodyState *states,
                             const float4 *c_np, const float4 *c_pt, const float4 *c_aa, const float4 *c_ab,
                             const float4 *c_lam, const float4 *c_pen, const float4 *c_acc, unsigned long long *saved_code,
                             uint32_t *saved_count, float4 *saved, uint32_t *n_saved, uint32_t cap,
                             const StepCounters *ctr) {
    const uint32_t M = *npairs;
    for (uint32_t m = blockIdx.x * blockDim.x + threadIdx.x; m < M; m += gridDim.x * blockDim.x) {
        if (m_count[m] == 0) continue;
        const uint32_t s = m_slot[m];
        if (s >= cap) continue;
        saved_code[s] = pair_key(ab[m]);
        saved_count[s] = m_count[m];
        const PmhRigidBodyState body = states[ab[m].x];
        float4 *rec = saved + (size_t)s * 8 * kCacheFloat4PerPoint;
        for (uint32_t k = 0; k < m_count[m]; ++k) {
            const uint32_t c = m_start[m] + k;
            const V3 local = inv_rotate(sq(body.orientation), sub(v3(c_pt[c]), sv(body.position)));
            const float4 acc = c_acc[c], bb = c_ab[c];
            float4 *r = rec + k * kCacheFloat4PerPoint;
            r[0] = f4(local, acc.x);
            r[1] = f4(v3(c_np[c]), bb.x);
            r[2] = make_float4(acc.y, acc.z, acc.w, bb.y);
            r[3] = c_lam[c];
            r[4] = make_float4(c_pen[c].x, c_pen[c].y, c_pen[c].z, bb.z);
            r[5] = f4(v3(c_aa[c]), 0.0f);
        }
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) *n_saved = std::min(ctr->manifolds, cap);
}

// A step whose dataflow sweep failed keeps its states: the pre-step
// states replace the result.
__global__ void k_clamp_speeds(uint32_t n, const PmhBodyParameters *P, PmhRigidBodyState *s,
                               const PmhRigidBodyState *before, const StepCounters *ctr) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    if (ctr->color_abort != 0u) {
        s[i] = before[i];
        return;
    }
    if (P[i].motion != kDynamic) return;
    s[i].linear_velocity = pv(clamp_length(sv(s[i].linear_velocity), P[i].maximum_linear_speed));
    s[i].angular_velocity = pv(clamp_length(sv(s[i].angular_velocity), P[i].maximum_angular_speed));
}

__global__ void k_step_begin(StepCounters *ctr) {
    if (threadIdx.x != 0) return;
    ctr->status = 0;   // per substep: the host checks it before the solve and after the last substep
    ctr->color_abort = 0;
    ctr->pairs = 0;
    ctr->points = 0;
    ctr->manifolds = 0;
    ctr->colors = 0;
    ctr->islands = 0;
    ctr->impact = 0;
    ctr->unsupported = 0;
    ctr->cache_hits = 0;
    ctr->large_count = 0;
    ctr->color_ticket = 0;
    ctr->point_alloc = 0;
    ctr->tri_pairs = 0;
    ctr->tri_hits = 0;
    ctr->face_pairs = 0;
    ctr->fallback_pairs = 0;
    ctr->cell_size_bits = 0.0f;
}

static uint32_t blocks_for(uint32_t items, uint32_t block = 256, uint32_t cap = 4096) {
    uint32_t g = (items + block - 1) / block;
    return std::max<uint32_t>(1, std::min(g, cap));
}

PmhResult World::step_once(uint32_t k_step, bool warm_infer) {
    hipStream_t s = stream;
    const uint32_t n = body_count;
    Solver &v = solver;
    StepCounters *ctr = v.counters.p;
    // Grids of one thread per body or joint are never capped: those kernels
    // take one item per thread.
    const uint32_t bg = blocks_for(n, 256, 0xffffffffu);
    const uint32_t pg = blocks_for(v.pair_cap, 256, 2048);
    auto mark = [&](int k) { if (timing_enabled) (void)hipEventRecord(events[k], s); };
    mark(0);
    k_step_begin<<<1, 64, 0, s>>>(ctr);
    PmhRigidBodyState *cur = state_cur.p, *prev = state_prev.p, *pred = state_next.p;
    k_integrate_proxy<<<bg, 256, 0, s>>>(n, params.p, shapes_dev.p, cur, prev, pred, proxy_mn.p, proxy_mx.p,
                                         gravity, dt, inputs_dev.p, targets_dev.p, target_flags_dev.p,
                                         substeps - substep, substep == 0 ? 1u : 0u,
                                         substep + 1 == substeps ? 1u : 0u, bucket_count.p, table_size + 1);
    mark(1);
    JointFilter jf;
    SceneRules rules;
    if (scene_first.size() > 1) {
        jf.scene = scene_of.p;
        rules.scene = scene_of.p;
        rules.count = scene_count.p;
        rules.pair_start = scene_pair_start.p;
    }
    if (solver.nj && weld_joints) {
        k_weld_init<<<bg, 256, 0, s>>>(n, weld.p);
        k_weld_hook<<<blocks_for(solver.nj, 256, 0xffffffffu), 256, 0, s>>>(n, solver.nj, joints_dev.p, weld.p);
        k_weld_compress<<<bg, 256, 0, s>>>(n, weld.p);
        jf.weld = weld.p;
    }
    if (solver.nj && excl_count) {
        jf.excl_start = excl_start.p;
        jf.excl_list = excl_list.p;
        jf.joints = joints_dev.p;
    }
    // Broadphase.
    k_bp_cells<<<bg, 256, 0, s>>>(n, proxy_mn.p, proxy_mx.p, cell_of.p, bucket_count.p, table_size - 1,
                                  large.p, ctr, grid_cell);
    PmhResult r = exclusive_scan(s, bucket_count.p, bucket_start.p, table_size, nullptr, nullptr, v.scan_tmp);
    if (r != PMH_SUCCESS) return r;
    k_bp_scatter<<<bg, 256, 0, s>>>(n, params.p, proxy_mn.p, proxy_mx.p, cell_of.p, bucket_start.p, bucket_count.p,
                                    entry_cell.p, entry_mn.p, entry_mx.p);
    if (jf.scene) {
        const uint32_t ns = uint32_t(scene_first.size());
        PMH_CHECK(hipMemsetAsync(scene_large_count.p, 0, sizeof(uint32_t) * (ns + 1), s));
        k_scene_large<<<64, 256, 0, s>>>(ctr, large.p, scene_of.p, scene_large_count.p, nullptr, nullptr);
        r = exclusive_scan(s, scene_large_count.p, scene_large_start.p, ns, nullptr, nullptr, v.scan_tmp);
        if (r != PMH_SUCCESS) return r;
        PMH_CHECK(hipMemsetAsync(scene_large_count.p, 0, sizeof(uint32_t) * (ns + 1), s));
        k_scene_large<<<64, 256, 0, s>>>(ctr, large.p, scene_of.p, scene_large_count.p, scene_large_start.p,
                                         scene_large.p);
        jf.scene_large_start = scene_large_start.p;
        jf.scene_large = scene_large.p;
        jf.scene_first = scene_first_dev.p;
        jf.scene_count = scene_count.p;
    }
    const uint32_t query_blocks = uint32_t((uint64_t(n) * kQueryLanes + kQueryBlock - 1) / kQueryBlock);
    // The triangle list is not in use yet: the pool of the candidates.
    const uint32_t segment = std::min(v.pair_cap / std::max<uint32_t>(1, n), kQueryHeld);
    k_bp_query<0><<<query_blocks, kQueryBlock, 0, s>>>(
        n, params.p, proxy_mn.p, proxy_mx.p, cell_of.p, bucket_start.p, entry_cell.p, entry_mn.p, entry_mx.p,
        table_size - 1, large.p, cand_count.p, v.tri_list.p, segment, nullptr, nullptr, nullptr, ctr, jf);
    k_bp_large<0><<<kLargeBlocks, 256, 0, s>>>(n, params.p, proxy_mn.p, proxy_mx.p, large.p, cand_count.p, nullptr, nullptr,
                                     nullptr, ctr, jf);
    r = exclusive_scan(s, cand_count.p, cand_offset.p, n, nullptr, nullptr, v.scan_tmp);
    if (r != PMH_SUCCESS) return r;
    k_set_pairs<<<1, 64, 0, s>>>(ctr, cand_offset.p, n, v.pair_cap);
    k_bp_large<1><<<kLargeBlocks, 256, 0, s>>>(n, params.p, proxy_mn.p, proxy_mx.p, large.p, cand_count.p, cand_offset.p,
                                     v.code.p, v.ab.p, ctr, jf);
    k_bp_query<1><<<query_blocks, kQueryBlock, 0, s>>>(
        n, params.p, proxy_mn.p, proxy_mx.p, cell_of.p, bucket_start.p, entry_cell.p, entry_mn.p, entry_mx.p,
        table_size - 1, large.p, cand_count.p, v.tri_list.p, segment, cand_offset.p, v.code.p, v.ab.p, ctr, jf);
    mark(2);
    if (rules.scene) k_scene_pairs<<<pg, 256, 0, s>>>(&ctr->pairs, v.ab.p, scene_of.p, scene_pair_start.p);
    // Narrowphase + point compaction.
    const NarrowOut out{v.m_count.p, v.m_start.p, v.m_face.p, v.m_init_rel.p, v.c_np.p, v.c_pt.p, v.c_aa.p,
                        v.c_ab.p, v.c_err.p, v.c_lam.p, v.c_pen.p, v.c_acc.p, v.c_rep.p, v.c_flags.p,
                        v.c_pair.p, v.point_cap, ctr};
    // Hinge contact frames of every body (worlds with joints only).
    HingeFrame *frames = nullptr;
    float4 *frame_ref = nullptr;
    if (v.nj) {
        if ((r = hinge_frames.reserve(n)) != PMH_SUCCESS || (r = hinge_ref.reserve(2 * size_t(n))) != PMH_SUCCESS)
            return r;
        frames = hinge_frames.p;
        frame_ref = hinge_ref.p;
        JointView jv;
        jv.joints = v.joints;
        jv.list_start = v.jlist_start;
        jv.list = v.jlist;
        k_hinge_frames<<<bg, 256, 0, s>>>(n, params.p, prev, pred, jv, frames, frame_ref);
    }
    k_narrowphase<<<blocks_for(v.pair_cap, kNarrowBlock, 2048), kNarrowBlock, 0, s>>>(&ctr->pairs, params.p, shapes_dev.p, prev, pred,
                                                                    v.ab.p, out, v.face_list.p, frames, frame_ref);
    const FaceGeometry geo{verts_dev.p, idx_dev.p, planes_dev.p};
    k_face_pairs<<<blocks_for(v.pair_cap, kFaceRows, 4096), kFaceBlock, 0, s>>>(
        v.face_list.p, params.p, shapes_dev.p, geo, prev, pred, v.ab.p, out, v.tri_list.p, frames,
        std::min(face_row_limit, kFaceLanes));
    // The face list is free by now, the adjacency not yet in use.
    auto *hit_mask = reinterpret_cast<unsigned long long *>(v.adj.p);
    k_triangle_screen<<<blocks_for(v.pair_cap, kScreenBlock, 1024), kScreenBlock, 0, s>>>(
        v.tri_list.p, params.p, shapes_dev.p, nodes_dev.p, leaves_dev.p, prev, pred, v.ab.p, out, leaf_slots, rules, frames,
        v.face_list.p, hit_mask);
    k_triangle_pairs<<<2048, 256, 0, s>>>(
        v.face_list.p, hit_mask, params.p, shapes_dev.p, verts_dev.p, idx_dev.p, planes_dev.p, nodes_dev.p, leaves_dev.p,
        shell_dev.p, prev, pred, v.ab.p, out, leaf_slots, leaf_limit, dt, rules, frames, frame_ref);
    k_guard_points<<<1, 64, 0, s>>>(ctr, v.point_cap);
    mark(3);
    // Response slots and the contact cache.
    k_nonempty<<<pg, 256, 0, s>>>(&ctr->pairs, v.m_count.p, v.m_impact.p);
    r = exclusive_scan(s, v.m_impact.p, v.m_slot.p, v.pair_cap, &ctr->pairs, nullptr, v.scan_tmp);
    if (r != PMH_SUCCESS) return r;
    const int rd = cache_parity, wr = cache_parity ^ 1;
    k_cache_load<<<pg, 256, 0, s>>>(&ctr->pairs, v.code.p, v.ab.p, v.m_count.p, v.m_start.p, pred,
                                    cache_code[rd].p, cache_count[rd].p, cache_data[rd].p, &cache_n.p[rd],
                                    v.c_np.p, v.c_pt.p, v.c_aa.p, v.c_ab.p, v.c_lam.p, v.c_pen.p, v.c_acc.p,
                                    v.c_flags.p, dt, ctr);
    mark(4);
    SolveParams sp{dt, gravity, base_iterations, requested_iterations, profile, cooperative ? 1u : 0u, solve_lanes,
                   residual_tolerance, warm_infer && warm_enabled, color_wait_limit};
    sp.sweep_wait_limit = sweep_wait_limit;
    sp.dataflow = !per_color_sweep;
    SolveTiming st;
    st.kernels = &kernel_timer;
    if (timing_enabled) {
        st.start = solve_events[2 * k_step];
        st.stop = solve_events[2 * k_step + 1];
    }
    r = avbd_prepare_solve(s, v, params.p, prev, pred, sp, timing_enabled ? &st : nullptr);
    solve_timing.launches += st.launches;
    if (r != PMH_SUCCESS) return r;
    mark(5);
    k_clamp_speeds<<<bg, 256, 0, s>>>(n, params.p, pred, cur, ctr);
    k_cache_save<<<pg, 256, 0, s>>>(&ctr->pairs, v.code.p, v.ab.p, v.m_count.p, v.m_start.p, v.m_slot.p, pred,
                                    v.c_np.p, v.c_pt.p, v.c_aa.p, v.c_ab.p, v.c_lam.p, v.c_pen.p, v.c_acc.p,
                                    cache_code[wr].p, cache_count[wr].p, cache_data[wr].p, &cache_n.p[wr],
                                    cache_capacity, ctr);
    mark(6);
    cache_parity = wr;
    std::swap(state_cur.p, state_next.p);
    substep = (substep + 1) % substeps;
    PMH_CHECK(hipGetLastError());
    return PMH_SUCCESS;
}

}  // namespace pmh
