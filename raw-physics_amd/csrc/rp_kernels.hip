// rp_kernels.hip — CDNA4 kernels of the batched step.
//
// One frame of every scene (pbd_simulate_with_constraints, pbd.cpp:468-747):
//   k_frame_begin   body lanes:  external force / torque of the frame
//   k_broad         wave/scene:  all-pairs bounding-sphere test, ordered compaction
//   k_islands       wave/scene:  union-find islands, sleeping, live-pair list
//   k_scan_live     one block:   prefix over scenes' live-pair counts
//   k_scatter_live  wave/scene:  global live-pair list
//   then num_substeps times:
//   k_integrate     body lanes:  integration + model matrix
//   k_transform     element lanes: hull vertices / face normals to world
//   k_narrow        pair lanes:  GJK -> EPA -> manifold -> collision constraints
//   k_solve         wave/scene:  dependency-levelled Gauss-Seidel position solve,
//                                velocity update, velocity solve
//
// The Gauss-Seidel order of the reference is kept exactly: constraints are
// assigned levels so that two constraints on the same non-fixed body keep
// their relative order, and constraints of one level (which touch disjoint
// writable bodies) run on different lanes. Fixed bodies are never written by
// any solve (pbd_base_constraints.cpp:103-133, pbd.cpp:702-711), so sharing
// one does not order two constraints. Every body therefore sees the same
// sequence of updates as in the sequential loop and results are bit-identical.
#include <algorithm>
#include <mutex>
#include <vector>

#include "rp_device.h"
#include "rp_pairsolve.h"

namespace rp {

// ---------------------------------------------------------------------------
__global__ void k_frame_begin(DevWorld w, double gravity) {
    int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= w.nb) return;
    b += w.body_base;
    Body& e = w.body[b];
    // Caller pattern (stack.cpp:93-96) and force / torque sums over its one
    // force (physics_util.cpp:5-23).
    V3 pos = v3(0.0, 0.0, 0.0);
    V3 force = v3(0.0, -gravity * 1.0 / e.inv_mass, 0.0);
    e.F = add(v3(0.0, 0.0, 0.0), force);
    e.T = add(v3(0.0, 0.0, 0.0), cross(sub(pos, v3(0.0, 0.0, 0.0)), force));
}

// broad_get_collision_pairs (broad.cpp:6-29): pairs (i<j) in i-major order.
__global__ void k_broad(DevWorld w) {
    int s = blockIdx.x;
    if (w.scene_big[s]) return;
    int lane = threadIdx.x;
    int b0 = w.scene_body_off[s], n = w.scene_body_off[s + 1] - b0;
    int base = w.scene_pair_base[s];
    int count = 0;
    for (int i = lane; i < n; i += 64) w.need[b0 + i] = 0;
    for (int i = 0; i < n; ++i) {
        const Body& e1 = w.body[b0 + i];
        for (int j0 = i + 1; j0 < n; j0 += 64) {
            int j = j0 + lane;
            bool hit = false;
            if (j < n) hit = broad_hit(e1, w.body[b0 + j]);
            int total;
            int slot = wave_compact(hit, &total);
            if (hit) w.pairs[base + count + slot] = make_int2(i, j);
            count += total;
        }
    }
    if (lane == 0) w.pair_count[s] = count;
}

// Islands and sleeping (broad.cpp:31-116, pbd.cpp:476-506), then the list of
// pairs the narrow phase visits (pbd.cpp:593-596). The reference joins the
// islands one pair after another (uf_union, broad.cpp:55-59); the wave's
// lanes join them at once with the lock-free union-find, which gives the same
// partition, and a body is active unless every body of its island has slept
// for a second, which depends on the partition only.
__global__ void k_islands(DevWorld w, double dt) {
    int s = blockIdx.x;
    if (w.scene_big[s]) return;
    int lane = threadIdx.x;
    int b0 = w.scene_body_off[s], n = w.scene_body_off[s + 1] - b0;
    int base = w.scene_pair_base[s];
    int np = w.pair_count[s];
    int* parent = w.uf_parent + b0;  // scene-local indices
    int* alli = w.uf_flag + b0;
    for (int i = lane; i < n; i += 64) { parent[i] = i; alli[i] = 1; }
    __syncthreads();
    for (int k = lane; k < np; k += 64) {
        int2 p = w.pairs[base + k];
        if (!w.body[b0 + p.x].fixed && !w.body[b0 + p.y].fixed) uf_link(parent, p.x, p.y);
    }
    for (int k = w.scene_ext_off[s] + lane; k < w.scene_ext_off[s + 1]; k += 64) {
        int i = w.ext[k].b1 - b0, j = w.ext[k].b2 - b0;
        if (!w.body[b0 + i].fixed && !w.body[b0 + j].fixed) uf_link(parent, i, j);
    }
    __syncthreads();
    for (int i = lane; i < n; i += 64) {
        Body& e = w.body[b0 + i];
        if (e.fixed) continue;
        double lv = len(e.v), av = len(e.w);
        if (lv < 0.10 && av < 0.10) e.deact += dt;
        else e.deact = 0.0;
        if (e.deact < 1.0) alli[uf_root(parent, i)] = 0;
    }
    __syncthreads();
    for (int i = lane; i < n; i += 64) {
        Body& e = w.body[b0 + i];
        if (e.fixed) continue;
        e.active = !alli[uf_root(parent, i)];
    }
    __syncthreads();
    // live pairs, in pair order
    int count = 0;
    uint32_t err = 0;
    for (int k0 = 0; k0 < np; k0 += 64) {
        int k = k0 + lane;
        bool live = false;
        if (k < np) {
            int2 p = w.pairs[base + k];
            const Body& e1 = w.body[b0 + p.x];
            const Body& e2 = w.body[b0 + p.y];
            if (!e1.fixed && !e2.fixed && !((e1.active && e2.active) || (!e1.active && !e2.active))) err |= ERR_ACTIVITY;
            live = !((e1.fixed || !e1.active) && (e2.fixed || !e2.active));
        }
        int total;
        int slot = wave_compact(live, &total);
        if (live) w.live_local[base + count + slot] = k;
        count += total;
    }
    if (err) atomicOr(&w.scene_err[s], err);
    if (lane == 0) w.live_count[s] = count;
}

// Exclusive prefix sum of live_count over scenes -> live_prefix[0..ns].
__global__ void k_scan_live(DevWorld w) {
    __shared__ int part[1024];
    int t = threadIdx.x, nt = blockDim.x;
    if (t == 0) {  // the size-class lists of this frame start empty
        w.counters[CNT_SMALL] = 0;
        w.counters[CNT_BIG] = 0;
    }
    int ns = w.ns;
    int chunk = (ns + nt - 1) / nt;
    int lo = min(ns, t * chunk), hi = min(ns, lo + chunk);
    int sum = 0;
    for (int i = lo; i < hi; ++i) sum += w.live_count[i];
    part[t] = sum;
    __syncthreads();
    for (int off = 1; off < nt; off <<= 1) {
        int v = (t >= off) ? part[t - off] : 0;
        __syncthreads();
        part[t] += v;
        __syncthreads();
    }
    int run = part[t] - sum;
    for (int i = lo; i < hi; ++i) {
        w.live_prefix[i] = run;
        run += w.live_count[i];
    }
    if (t == nt - 1) w.live_prefix[ns] = part[t];
}

__global__ void k_scatter_live(DevWorld w) {
    int s = blockIdx.x;
    if (w.scene_big[s]) return;
    int base = w.scene_pair_base[s];
    int g0 = w.live_prefix[s], n = w.live_count[s];
    int b0 = w.scene_body_off[s];
    for (int m0 = 0; m0 < n; m0 += blockDim.x) {
        int m = m0 + threadIdx.x;
        bool valid = m < n;
        int b1 = 0, b2 = 0;
        if (valid) {
            int slot = base + w.live_local[base + m];
            w.live_global[g0 + m] = make_int2(s, slot);
            int2 p = w.pairs[slot];
            b1 = b0 + p.x;
            b2 = b0 + p.y;
            write_live_records(w, g0 + m, b1, b2);
            w.need[b1] = 1;  // same value from every writer
            w.need[b2] = 1;
        }
        if (w.small_nv > 0) classify_pair(w, valid, g0 + m, b1, b2);
    }
}

// ---------------------------------------------------------------------------
// Integration of body b (pbd.cpp:565-596), held at e, and its model matrix;
// in a recorded frame the state it starts from is kept.
__device__ __forceinline__ void integrate_body(const DevWorld& w, int b, Body& e, double h) {
    if (w.rec_state && !e.fixed) {
        double* r = w.rec_state + (size_t)b * REC_STATE;
        r[0] = e.x.x; r[1] = e.x.y; r[2] = e.x.z;
        r[3] = e.q.x; r[4] = e.q.y; r[5] = e.q.z; r[6] = e.q.w;
        r[7] = e.v.x; r[8] = e.v.y; r[9] = e.v.z;
        r[10] = e.w.x; r[11] = e.w.y; r[12] = e.w.z;
        r[13] = e.active ? 1.0 : 0.0;
    }
    integrate(e, h);
    w.model[b] = model_matrix(e.x, e.q);
}

__global__ void k_integrate(DevWorld w, double h) {
    int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b == 0) w.counters[CNT_MANIFOLD] = 0;  // the substep's manifold queue starts empty
    if (b >= w.nb) return;
    b += w.body_base;
    Body e = w.body[b];
    integrate_body(w, b, e, h);
    w.body[b].x = e.x;
    w.body[b].q = e.q;
    w.body[b].v = e.v;
    w.body[b].w = e.w;
    w.body[b].px = e.px;
    w.body[b].pq = e.pq;
}

// The pose every body has when the substep's collision pass reads it
// (colliders_update at pbd.cpp:598-599 runs after integration): launched
// after the last substep's integration when the caller wants the colliders'
// transformed geometry of that pose written back.
__global__ void k_keep_pose(DevWorld w) {
    int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= w.nb) return;
    b += w.body_base;
    const Body& e = w.body[b];
    double* p = w.pose + 7 * (size_t)b;
    p[0] = e.x.x; p[1] = e.x.y; p[2] = e.x.z;
    p[3] = e.q.x; p[4] = e.q.y; p[5] = e.q.z; p[6] = e.q.w;
}

// The bodies' states as the flat arrays of rp_state, one after another
// (StateSection), and back: of the arrays in `mask` only.
__global__ void k_state_out(DevWorld w, double* out) {
    int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= w.nb) return;
    const double* e = (const double*)&w.body[b];  // the state leads the record
    double v[STATE_DOUBLES];
#pragma unroll
    for (int c = 0; c < STATE_DOUBLES; ++c) v[c] = e[c];
#pragma unroll
    for (int s = 0; s < STATE_SECTIONS; ++s)
#pragma unroll
        for (int c = state_section(s); c < state_section(s + 1); ++c)
            out[(size_t)state_section(s) * w.nb + (size_t)b * (state_section(s + 1) - state_section(s)) +
                (c - state_section(s))] = v[c];
    ((int32_t*)(out + (size_t)STATE_DOUBLES * w.nb))[b] = w.body[b].active;
}
__global__ void k_state_in(DevWorld w, const double* in, unsigned mask) {
    int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= w.nb) return;
    double* e = (double*)&w.body[b];
#pragma unroll
    for (int s = 0; s < STATE_SECTIONS; ++s)
        if (mask >> s & 1)
#pragma unroll
            for (int c = state_section(s); c < state_section(s + 1); ++c)
                e[c] = in[(size_t)state_section(s) * w.nb + (size_t)b * (state_section(s + 1) - state_section(s)) +
                          (c - state_section(s))];
    if (mask >> STATE_SECTIONS & 1) w.body[b].active = ((const int32_t*)(in + (size_t)STATE_DOUBLES * w.nb))[b];
}

// entity_get_model_matrix of every body, row-major 4x4, as double or as the
// float array util_matrix_to_r32_array (util.cpp:77-94) hands to the renderer.
template <class F>
__global__ void k_model_out(DevWorld w, F* out) {
    int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= w.nb) return;
    const Body& e = w.body[b];
    M4 M = entity_model_matrix(e.x, e.q, w.body_scale[b]);
    F* o = out + 16 * (size_t)b;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) o[4 * i + j] = (F)M.m[i][j];
}

// Transformed vertices of the bodies that take part in a live pair this
// frame (lane-per-pair narrow phase and the inspection path).
__global__ void k_transform(DevWorld w, int all) {
    int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= w.n_xf) return;
    int4 el = w.xf[t];  // (body, hull instance, vertex, tv slot)
    int b = el.x;
    if (!all && !w.need[b]) return;
    w.tv[el.w] = transform_vertex(w.model[b], w.hull_v[w.hull_v_off[el.y] + el.z]);
}

// View of hull instance `hid` of body b whose transformed vertices start at tv_off.
__device__ __forceinline__ HullView hull_view_of(const DevWorld& w, int b, int hid, int tv_off) {
    HullView hv;
    hv.tv = w.tv + tv_off;
    hv.nv = w.hull_nv[hid];
    hv.hid = hid;
    hv.body = b;
    return hv;
}
// The hull of a body with one hull collider (the fast narrow path).
__device__ __forceinline__ HullView hull_view(const DevWorld& w, int b) {
    return hull_view_of(w, b, w.body_hull[b], w.body_tv_off[b]);
}
// Collider c (global index) of body b.
__device__ __forceinline__ ColView col_view(const DevWorld& w, int b, int c) {
    ColView v;
    v.type = w.col_type[c];
    v.radius = w.col_radius[c];
    v.center = w.body[b].x;  // colliders_update: the sphere follows the entity (collider.cpp:431-433)
    if (v.type == COL_HULL) v.h = hull_view_of(w, b, w.col_hull[c], w.col_tv_off[c]);
    else memset(&v.h, 0, sizeof(v.h));
    return v;
}

// Narrow phase over the live pairs of all scenes (pbd.cpp:583-612), in two
// kernels: GJK + EPA for every live pair, then the contact manifold for the
// pairs whose EPA converged (collider.cpp:523-558). Both take G lanes per
// pair: G = 1 is one lane per pair over the pre-transformed vertices
// (k_transform); G = 4, 8, 16 put 64/G pairs in a wave, transform both
// hulls' vertices into LDS and split every support search across the group
// (support_index<G>); the rest runs identically on the group's lanes and
// lane 0 of the group writes the results. Results go to the pair's slot g in
// the live list (scene, then pair order), so the queue order between the
// kernels does not matter.
__device__ __forceinline__ void group_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// Scene and global body indices of live pair g (both loads depend on g
// only: the bodies come from the frame's live-pair record).
__device__ __forceinline__ void pair_bodies(const DevWorld& w, int g, int& s, int& b1, int& b2) {
    s = w.live_global[g].x;
    int4 r = w.live_rec[g];
    b1 = r.x;
    b2 = r.y;
}
// Pairs with a sphere or a multi-collider body take the general path.
__device__ __forceinline__ bool general_pair(const DevWorld& w, int b1, int b2) {
    return w.has_general && (w.body_general[b1] | w.body_general[b2]);
}

// Two hulls of bodies b1 and b2, transformed by the group's lanes into the
// group's LDS slice `st`, one after the other. hv: first local vertices and
// vertex counts.
template <int G>
__device__ __forceinline__ void stage_pair(const DevWorld& w, int b1, int b2, int4 hv, V3* st, int gl) {
    const V3* lv1 = w.hull_v + hv.x;
    const V3* lv2 = w.hull_v + hv.y;
    int nv1 = hv.z, nv2 = hv.w;
    const M4 M1 = w.model[b1], M2 = w.model[b2];
    // both hulls together, two vertices of each per lane and batch, all
    // loaded before any is transformed
    int n = nv1 > nv2 ? nv1 : nv2;
    for (int i = gl; i < n; i += 2 * G) {
        V3 va[2], vb[2];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            int j = i + k * G;
            if (j < nv1) va[k] = lv1[j];
            if (j < nv2) vb[k] = lv2[j];
        }
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            int j = i + k * G;
            if (j < nv1) st[j] = transform_vertex(M1, va[k]);
            if (j < nv2) st[nv1 + j] = transform_vertex(M2, vb[k]);
        }
    }
    group_lds_sync();
}
// Hull views of live pair g, staged in `st` for G > 1 (vertex offsets and
// counts from the pair's record: the vertex loads depend on that one load
// only).
template <int G>
__device__ __forceinline__ void pair_views(const DevWorld& w, int g, V3* st, int gl, int& s, int& b1, int& b2,
                                           HullView& h1, HullView& h2) {
    s = w.live_global[g].x;
    int4 r = w.live_rec[g];  // bodies and hull instances: no pair-slot and scene-offset loads first
    b1 = r.x;
    b2 = r.y;
    if constexpr (G == 1) {
        h1 = hull_view_of(w, b1, r.z, w.body_tv_off[b1]);
        h2 = hull_view_of(w, b2, r.w, w.body_tv_off[b2]);
    } else {
        int4 hv = w.live_hull[g];
        stage_pair<G>(w, b1, b2, hv, st, gl);
        h1 = HullView{st, hv.z, r.z, b1};
        h2 = HullView{st + hv.z, hv.w, r.w, b2};
    }
}

// The contact manifold of live pair g with EPA normal n: its contacts become
// collision constraints as they are made. Returns their count.
template <int G>
__device__ __forceinline__ int pair_manifold(const DevWorld& w, int g, const HullView& h1, const HullView& h2, V3 n,
                                             uint32_t& err, char* work, V3* spare, int spare_n) {
    const Body& e1 = w.body[h1.body];
    const Body& e2 = w.body[h2.body];
    Contact* out = w.contacts + (size_t)g * MAXC;
    auto emit = [&](int k, const ContactPt& c) { contact_to_constraint(e1, e2, c, out[k]); };
    if constexpr (G == 1) return manifold_lane(w.hulls, h1, h2, n, emit, err, work);
    else return manifold_group<G>(w.hulls, h1, h2, n, emit, err, work, spare, spare_n);
}

// kManifold: the contact manifold of a converged pair is built here too, on
// the same staged hulls, and its contacts written (no manifold queue).
// list / count: visit the pairs of a size-class list, or (list null) every live
// pair. LDS slices of `stage` vertices per pair: both hulls and what EPA and
// clipping use beside them (stage_slice).
template <int G, bool kManifold>
__device__ __forceinline__ void gjk_epa_pairs(DevWorld& w, const int32_t* list, const int32_t* count, int stage) {
    extern __shared__ V3 rp_stage[];
    constexpr int NG = 64 / G;
    alignas(16) char own[G == 1 ? (kManifold ? GROUP_WORK_BYTES : EPA_BYTES) : 1];  // a lone lane's working memory
    int grp = threadIdx.x / G, gl = threadIdx.x & (G - 1);
    V3* st = rp_stage + grp * stage;
    int total = list ? *count : w.live_prefix[w.ns];
    for (int k = blockIdx.x * NG + grp; k < total; k += gridDim.x * NG) {
        int g = list ? list[k] : k;
        int s, b1, b2;
        pair_bodies(w, g, s, b1, b2);
        if (general_pair(w, b1, b2)) continue;  // k_narrow_general (uniform per group)
        HullView h1, h2;
        pair_views<G>(w, g, st, gl, s, b1, b2, h1, h2);
        uint32_t err = 0;
        bool cycled = false;
        Simplex sx;
        V3 n = v3(0.0, 0.0, 0.0);
        double pen;
        int r = 0;
        char* work = G > 1 ? w.group_work + (size_t)(blockIdx.x * NG + grp) * GROUP_WORK_BYTES : own;
        bool hit = gjk<G>(h1, h2, sx, err, cycled);
        const int used = h1.nv + h2.nv;  // the rest of the pair's LDS slice is free
        if (hit) r = epa<G>(h1, h2, sx, n, pen, err, work, st + used, stage - used);
        if constexpr (kManifold) {
            int nc = 0;
            if (r == 1) nc = pair_manifold<G>(w, g, h1, h2, n, err, work, st + used, stage - used);
            if (gl == 0) w.ncontact[g] = nc;
        }
        if (gl == 0) {
            if constexpr (!kManifold) {
                if (r == 1) {
                    w.pair_normal[g] = n;
                    w.mlist[atomicAdd(&w.counters[CNT_MANIFOLD], 1)] = g;
                } else {
                    w.ncontact[g] = 0;
                }
            }
            if (err) atomicOr(&w.scene_err[s], err);
            if (hit && r != 1) atomicAdd(&w.stats[STAT_EPA_FAIL], 1ull);  // epa.cpp:233-236
            if (cycled) atomicAdd(&w.stats[STAT_GJK_CYCLE], 1ull);
        }
        if constexpr (G > 1) group_lds_sync();
    }
}

// Lane groups (G = 4, 8, 16) at two waves per SIMD; one lane per pair (G = 1).
template <int G, bool kManifold>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2)))
k_gjk_epa(DevWorld w, const int32_t* list, const int32_t* count, int stage) {
    static_assert(G > 1, "lane groups");
    gjk_epa_pairs<G, kManifold>(w, list, count, stage);
}
template <bool kManifold>
__global__ void __launch_bounds__(64) k_gjk_epa_lane(DevWorld w) {
    gjk_epa_pairs<1, kManifold>(w, nullptr, nullptr, 0);
}

template <int G>
__global__ void __launch_bounds__(64) k_manifold(DevWorld w, int stage) {
    extern __shared__ V3 rp_stage[];
    constexpr int NG = 64 / G;
    int grp = threadIdx.x / G, gl = threadIdx.x & (G - 1);
    V3* st = rp_stage + grp * stage;
    alignas(16) char own[G == 1 ? CLIP_BYTES : 1];
    int total = w.counters[CNT_MANIFOLD];
    for (int k = blockIdx.x * NG + grp; k < total; k += gridDim.x * NG) {
        int g = w.mlist[k];
        int s, b1, b2;
        HullView h1, h2;
        pair_views<G>(w, g, st, gl, s, b1, b2, h1, h2);
        uint32_t err = 0;
        char* work = G > 1 ? w.group_work + (size_t)(blockIdx.x * NG + grp) * GROUP_WORK_BYTES : own;
        int used = h1.nv + h2.nv;
        int nc = pair_manifold<G>(w, g, h1, h2, w.pair_normal[g], err, work, st + used, stage - used);
        if (gl == 0) {
            w.ncontact[g] = nc;
            if (err) atomicOr(&w.scene_err[s], err);
        }
        if constexpr (G > 1) group_lds_sync();
    }
}

// Live pairs with a sphere collider or a multi-collider body:
// colliders_get_contacts (collider.cpp:560-572) over every collider pair in
// order, each by collider_get_contacts (collider.cpp:523-558), at most MAXC
// contacts of the pair kept. One lane group per pair, each collider pair's
// hulls staged in its LDS slice (G = 8 or 16), as the fast path (256 scenes of
// spheres, boxes and dumbbells: 170 -> 97 us per launch, and the world may be
// stepped in concurrent views, 4.9 -> 2.8 ms per frame); in worlds whose hulls
// leave no room for that, one lane per pair over the pre-transformed vertices
// with private arrays (G = 1).
template <int G>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2)))
k_narrow_general(DevWorld w, int stage) {
    extern __shared__ V3 rp_stage[];
    constexpr int NG = 64 / G;
    const int grp = threadIdx.x / G, gl = threadIdx.x & (G - 1);
    V3* st = rp_stage + grp * stage;
    alignas(16) char own[G == 1 ? GROUP_WORK_BYTES : 1];
    char* work = G > 1 ? w.group_work + (size_t)(blockIdx.x * NG + grp) * GROUP_WORK_BYTES : own;
    int total = w.live_prefix[w.ns];
    for (int g = blockIdx.x * NG + grp; g < total; g += gridDim.x * NG) {
        int s, b1, b2;
        pair_bodies(w, g, s, b1, b2);
        if (!general_pair(w, b1, b2)) continue;
        uint32_t err = 0;
        int flags = 0, nc = 0;
        const Body& e1 = w.body[b1];
        const Body& e2 = w.body[b2];
        Contact* out = w.contacts + (size_t)g * MAXC;
        const int c1e = w.body_col_off[b1 + 1], c2e = w.body_col_off[b2 + 1];
        for (int c1 = w.body_col_off[b1]; c1 < c1e; ++c1)
            for (int c2 = w.body_col_off[b2]; c2 < c2e; ++c2) {
                ColView v1 = col_view(w, b1, c1), v2 = col_view(w, b2, c2);
                int used = v1.h.nv + v2.h.nv;
                if constexpr (G > 1) {
                    if (used > 0) {
                        int4 hv = make_int4(v1.h.nv ? w.hull_v_off[v1.h.hid] : 0, v2.h.nv ? w.hull_v_off[v2.h.hid] : 0,
                                            v1.h.nv, v2.h.nv);
                        stage_pair<G>(w, b1, b2, hv, st, gl);
                    }
                    v1.h.tv = st;
                    v2.h.tv = st + v1.h.nv;
                }
                auto emit = [&](int k, const ContactPt& c) {
                    if (nc + k < MAXC) contact_to_constraint(e1, e2, c, out[nc + k]);
                };
                int n = collider_contacts<G>(w.hulls, v1, v2, emit, err, flags, work, st + used, stage - used);
                if (nc + n > MAXC) err |= ERR_CONTACT_CAPACITY;
                nc = min(nc + n, MAXC);
                if constexpr (G > 1) group_lds_sync();
            }
        if (gl == 0) {
            w.ncontact[g] = nc;
            if (err) atomicOr(&w.scene_err[s], err);
            if (flags & PAIR_EPA_FAIL) atomicAdd(&w.stats[STAT_EPA_FAIL], 1ull);
            if (flags & PAIR_GJK_CYCLE) atomicAdd(&w.stats[STAT_GJK_CYCLE], 1ull);
        }
    }
}

// Dependency levels of one frame's solve items (wave/scene). An item is one
// external constraint or the contacts of one live pair (solved in order by
// two lanes, rp_pairsolve.h). The reference's sequence is: external constraints, then the
// contacts of each pair in pair order (pbd.cpp:580-620). An item's level is
// one above the last level of either of its non-fixed bodies, so items that
// share a writable body keep their order and items of one level touch
// disjoint writable bodies. Pairs are fixed for the frame (the broad phase
// and activity run once per frame, pbd.cpp:474-506), so levels are too.
constexpr int LEV_CHUNK = 512;
constexpr int LEV_LDS_BODIES = 1024;

__global__ void __launch_bounds__(64) k_levels(DevWorld w, int collisions, int pipelined) {
    int s = blockIdx.x;
    if (w.scene_big[s]) return;
    int lane = threadIdx.x;
    int b0 = w.scene_body_off[s], n = w.scene_body_off[s + 1] - b0;
    int e0 = w.scene_ext_off[s], next = w.scene_ext_off[s + 1] - e0;
    int g0 = w.live_prefix[s];
    int np = collisions ? w.live_count[s] : 0;
    int K = next + np;
    int ib = w.scene_item_base[s];
    int* lev = w.item_level + ib;
    int* order = w.item_order + ib;
    int* ls = w.item_lstart + ib + s;
    __shared__ int sb1[LEV_CHUNK], sb2[LEV_CHUNK], slev[LEV_CHUNK];
    __shared__ int slast[LEV_LDS_BODIES], sfirst[LEV_LDS_BODIES], stouch[LEV_LDS_BODIES];
    __shared__ int sL;
    bool in_lds = n <= LEV_LDS_BODIES;
    // per body: one above its last item's level, its first item's level, its
    // first contact item's level
    int* last = in_lds ? slast : (w.body_last + 2 * (size_t)b0);
    int* first = in_lds ? sfirst : (w.body_last + 2 * (size_t)b0 + n);
    int* touch = in_lds ? stouch : (w.body_touch + b0);
    for (int i = lane; i < n; i += 64) {
        last[i] = 0;
        first[i] = touch[i] = INT_MAX;
    }
    if (lane == 0) sL = 0;
    __syncthreads();
    for (int c0 = 0; c0 < K; c0 += LEV_CHUNK) {
        int cn = min(LEV_CHUNK, K - c0);
        for (int k = lane; k < cn; k += 64) {
            int t = c0 + k, i1, i2;
            if (t < next) {
                i1 = w.ext[e0 + t].b1 - b0;
                i2 = w.ext[e0 + t].b2 - b0;
            } else {
                int2 p = w.pairs[w.live_global[g0 + t - next].y];
                i1 = p.x;
                i2 = p.y;
            }
            sb1[k] = w.body[b0 + i1].fixed ? -1 : i1;  // fixed bodies never order items
            sb2[k] = w.body[b0 + i2].fixed ? -1 : i2;
        }
        __syncthreads();
        if (lane == 0) {
            int L = sL;
            for (int k = 0; k < cn; ++k) {
                int i1 = sb1[k], i2 = sb2[k];
                int lv = 0;
                if (i1 >= 0) lv = last[i1];
                if (i2 >= 0) lv = max(lv, last[i2]);
                ++lv;
                if (i1 >= 0) last[i1] = lv;
                if (i2 >= 0) last[i2] = lv;
                slev[k] = lv - 1;
                L = max(L, lv);
            }
            sL = L;
        }
        __syncthreads();
        for (int k = lane; k < cn; k += 64) {
            int lv = slev[k];
            lev[c0 + k] = lv;
            if (!pipelined) continue;
            for (int i : {sb1[k], sb2[k]}) {
                if (i < 0) continue;
                atomicMin(&first[i], lv);
                if (c0 + k >= next) atomicMin(&touch[i], lv);
            }
        }
        __syncthreads();
    }
    // The period: the fewest levels by which a sweep may start after the one
    // before it so that no body's item runs before its last item of that
    // sweep (at least 2: k_solve reads multipliers one level ahead).
    int period = 2;
    for (int i = lane; pipelined && i < n; i += 64)
        if (last[i] > 0) period = max(period, last[i] - first[i]);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) period = max(period, __shfl_xor(period, off));
    int L = sL;
    // counting sort by level; the order inside a level does not matter (its
    // items touch disjoint writable bodies)
    int* cur = w.item_cursor + ib + s;
    for (int l = lane; l <= L; l += 64) ls[l] = 0;
    __syncthreads();
    for (int t = lane; t < K; t += 64) atomicAdd(&ls[lev[t] + 1], 1);
    __syncthreads();
    if (lane == 0) {
        for (int l = 0; l < L; ++l) ls[l + 1] += ls[l];
        w.scene_nlevels[s] = L;
        w.scene_period[s] = period;
    }
    __syncthreads();
    for (int l = lane; l <= L; l += 64) cur[l] = ls[l];
    __syncthreads();
    int2* bodies = w.item_bodies + ib;
    for (int t = lane; t < K; t += 64) {
        int pos = atomicAdd(&cur[lev[t]], 1);
        int code = (t < next) ? ~(e0 + t) : (g0 + t - next);
        order[pos] = code;
        int2 bb = item_body_pair(w, code, b0);
        if (pipelined && t >= next) {
            if (touch[bb.x - b0] == lev[t]) bb.x |= FIRST_CONTACT;
            if (touch[bb.y - b0] == lev[t]) bb.y |= FIRST_CONTACT;
        }
        bodies[pos] = bb;
    }
    if (!pipelined) return;
    __syncthreads();
    for (int i = lane; i < n; i += 64) w.body_touch[b0 + i] = touch[i] == INT_MAX ? 0 : 1;
}

// Solve of one scene and substep: position Gauss-Seidel (pbd.cpp:615-620),
// velocity update (pbd.cpp:623-643), velocity solve (pbd.cpp:646-711), level
// by level over the frame's items. LPS lanes serve one scene, two per item, so
// a wave solves 64/LPS scenes side by side (small scenes leave most of a
// 64-lane wave idle otherwise).
//
// kLds: the scenes' bodies are held in LDS (`cap` records per scene) from the
// first level to the next substep's integration, and only poses and
// velocities (the first STATE_VECS 16-byte words of a record) go back. A level
// then costs its items' arithmetic and an LDS round trip instead of two
// trips to L2. The items' codes are read two levels ahead and, without
// joints, their first contacts one level ahead, both independent of the
// bodies. What is left is the instructions of one item at a time (about 780
// FP64 operations per contact in both sweeps): a call on a stack of 10 boxes
// went from 3.07 to 2.81 ms, a scene of 16 bodies from 25 to 20 us per launch.
constexpr int BODY_VECS = sizeof(Body) / sizeof(int4);
constexpr int STATE_VECS = offsetof(Body, deact) / sizeof(int4);  // x, q, v, w, px, pq, pv, pw
static_assert(sizeof(Body) % sizeof(int4) == 0 && offsetof(Body, deact) % sizeof(int4) == 0, "copied as 16-byte words");

// In worlds with joints, and for scenes on several waves, sweeps are pipelined
// by the period P of the scene's order (k_levels): level l of position
// iteration i runs at step l + iP, beside the levels of earlier iterations that
// are still due, and level l of the velocity sweep at step l + iters P. Items of one step share no body that they write, and every body
// sees its items in the list's order, so the bits are those of one sweep after
// another. With several waves per scene (kSplit) the velocity sweep has waves
// of its own: they follow the position sweep P levels behind instead of waiting
// for its end. Against one sweep after another on one wave (64 lanes) or four:
// 10 frames of 500 chains of 6 links (4 iterations) 80.5 -> 65.3 ms, 4 frames
// of 150 scenes of 4 to 256 bodies with chains 25.3 -> 23.1. Scenes without
// joints on one wave or less keep one sweep after another: their floor is in a
// pair with every body at level 0, so P is about their whole depth, and the
// steps' bookkeeping cost scenes of up to 64 bodies 0.5 to 2 %.
template <bool kExt, int LPS, bool kLds>
__global__ void __launch_bounds__(LPS > 64 ? 2 * LPS : 64) __attribute__((amdgpu_waves_per_eu(2)))
k_solve(DevWorld w, double h, int iters, int collisions, int integrate_next, int cap) {
    extern __shared__ int4 rp_solve_lds[];
    constexpr bool kSplit = LPS > 64, kPipe = kExt || kSplit;
    constexpr int TPS = kSplit ? 2 * LPS : LPS;   // threads that serve one scene
    constexpr int SPB = LPS < 64 ? 64 / LPS : 1;  // scenes per block
    constexpr int LPW = LPS < 64 ? LPS : 64;      // lanes of a wave that serve one scene
    int s = blockIdx.x * SPB + (int)threadIdx.x / TPS;
    int thread = (int)threadIdx.x % TPS;
    int lane = thread % LPS;  // in its sweep
    bool valid = s < w.ns && !w.scene_big[s];  // large scenes: coloured solve (rp_large.hip)
    int b0 = 0, n = 0, e0 = 0, e1x = 0, L = 0, P = 2, g0 = 0, np = 0;
    const int* order = nullptr;
    const int2* bodies = nullptr;
    const int* ls = nullptr;
    if (valid) {
        b0 = w.scene_body_off[s];
        n = w.scene_body_off[s + 1] - b0;
        e0 = w.scene_ext_off[s];
        e1x = w.scene_ext_off[s + 1];
        int ib = w.scene_item_base[s];
        order = w.item_order + ib;
        bodies = w.item_bodies + ib;
        ls = w.item_lstart + ib + s;
        L = w.scene_nlevels[s];
        P = w.scene_period[s];
        g0 = w.live_prefix[s];
        np = collisions ? w.live_count[s] : 0;
    }
    // whether some live pair of the scene has contacts (its pairs are
    // contiguous in the live list): without, and without external
    // constraints, there is nothing to sweep
    int touching = 0;
    for (int k = thread; k < np; k += TPS) touching |= w.ncontact[g0 + k];
    Body* body = w.body + b0;
    if constexpr (kLds) {
        int4* own = rp_solve_lds + (size_t)((int)threadIdx.x / TPS) * cap * BODY_VECS;
        const int4* src = (const int4*)body;
        for (int i = thread; i < n * BODY_VECS; i += TPS) own[i] = src[i];
        body = (Body*)own;
    }
    if constexpr (kSplit) {
        touching = __syncthreads_or(touching);
    } else {
        unsigned long long m = __ballot(touching != 0);
        if constexpr (LPS < 64) m &= ((1ull << LPS) - 1ull) << ((int)threadIdx.x & ~(LPS - 1));
        touching = m != 0;
    }
    // levels and steps of both sweeps
    if (!touching && !(kExt && e1x > e0)) L = 0;
    const int pos_levels = !kPipe || iters > 0 ? L : 0;
    const int vel_levels = touching ? L : 0;
    int pos_steps = kPipe && pos_levels > 0 ? (iters - 1) * P + L : pos_levels;
    int vel_steps = kSplit && touching ? iters * P + L : vel_levels;
    // level starts ls[0..L] in the lanes' registers (lane l of the wave's
    // lanes of a scene holds ls[l]) when every scene of the block fits, read
    // back by lane exchange instead of a global load per level (the branch is
    // uniform per block)
    int Lmax = L;
    if constexpr (kSplit) {
        pos_steps = vel_steps = max(pos_steps, vel_steps);
    } else if constexpr (SPB > 1) {  // every lane joins every barrier
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            Lmax = max(Lmax, __shfl_xor(Lmax, off));
            if constexpr (kPipe) pos_steps = max(pos_steps, __shfl_xor(pos_steps, off));
        }
        if constexpr (!kPipe) pos_steps = Lmax;
        vel_steps = Lmax;
    }
    const bool ls_in_lanes = Lmax + 1 <= LPW;
    const int my_ls = (valid && lane % LPW <= L) ? ls[lane % LPW] : 0;
    auto level_start = [&](int l) -> int {
        if (!ls_in_lanes) return valid ? ls[l] : 0;
        if constexpr (kSplit) return __builtin_amdgcn_readlane(my_ls, l);
        else return __shfl(my_ls, l, LPW);
    };
    uint32_t err = 0;

    // multipliers of the external constraints start at zero (pbd.cpp:426-462)
    if constexpr (kExt) {
        for (int k = e0 + thread; k < e1x; k += TPS) {
            w.ext_lambda[3 * k] = 0.0;
            w.ext_lambda[3 * k + 1] = 0.0;
            w.ext_lambda[3 * k + 2] = 0.0;
        }
    }
    __syncthreads();
    auto position = [&](const PairItem& t) { solve_item_pos<kExt>(w, body, b0, t, h, err); };
    auto velocity = [&](const PairItem& t) { solve_item_vel<kPipe>(w, body, b0, t, h); };
    if constexpr (kPipe) {
        // What a sweep solves at one step: level `l` of its sweep `it`, and the
        // levels l + P, l + 2P, ... of the sweeps before it.
        struct Step { int it, l; };
        // Item `slot` of a step or -1, and the number of its items (all lanes of
        // a scene take the same turns: the exchanges need their partners).
        auto locate = [&](Step st, int levels, int slot, int& count) -> int {
            int idx = -1;
            count = 0;
            if (st.l < 0) return -1;
            for (int l = st.l, it = st.it; l < levels && it >= 0; l += P, --it) {
                int a = level_start(l), m = level_start(l + 1) - a;
                if (idx < 0 && slot - count < m) idx = a + slot - count;
                count += m;
            }
            return idx;
        };
        // `sweeps` sweeps from step `begin` on, up to step `steps`. `here` is this
        // pair's first item of a step with its contact, `next` that of the step
        // after it (its code, then its contact), `after` the one two steps ahead.
        auto sweep = [&](int sweeps, int begin, int levels, int steps, auto solve) {
            auto advance = [&](Step st) -> Step {
                ++st.l;
                if (st.l >= P && st.it + 1 < sweeps) {
                    st.l -= P;
                    ++st.it;
                }
                return st;
            };
            // the items of a step go round the sweep's waves: fewer per wave, and
            // fewer different branches one after another on one
            constexpr int WAVES = LPS < 64 ? 1 : LPS / 64;
            const int slot = (lane % LPW / 2) * WAVES + lane / LPW;
            Step s0 = {0, -begin}, s1 = advance(s0), s2 = advance(s1);
            int c0, c1, c2, i0 = locate(s0, levels, slot, c0), i1 = locate(s1, levels, slot, c1);
            PairItem here, next;
            if (i0 >= 0) {
                load_item(here, order, bodies, i0);
                if (!kExt) load_item_contact<kExt>(here, w);
            }
            if (i1 >= 0) load_item(next, order, bodies, i1);
            for (int g = 0; g < steps; ++g) {
                int i2 = locate(s2, levels, slot, c2);
                PairItem after;
                // (with joints the registers go to the joint solve)
                if (!kExt && i1 >= 0) load_item_contact<kExt>(next, w);
                if (i2 >= 0) load_item(after, order, bodies, i2);
                if (kExt && i0 >= 0) load_item_contact<kExt>(here, w);
                for (int base = 0;;) {
                    if (i0 >= 0) solve(here);
                    base += LPS / 2;
                    if (base >= c0) break;
                    int c;
                    i0 = locate(s0, levels, base + slot, c);
                    if (i0 >= 0) {
                        load_item(here, order, bodies, i0);
                        load_item_contact<kExt>(here, w);
                    }
                }
                __syncthreads();
                here = next;
                next = after;
                i0 = i1;
                i1 = i2;
                c0 = c1;
                c1 = c2;
                s0 = s1;
                s1 = s2;
                s2 = advance(s2);
            }
        };
        // (both branches pass the same number of barriers)
        if (!kSplit || thread < LPS) sweep(iters, 0, pos_levels, pos_steps, position);
        if (!kSplit || thread >= LPS) sweep(1, kSplit ? iters * P : 0, vel_levels, vel_steps, velocity);
    } else {
        // One sweep over the levels. `here` is this pair's first item of level l
        // with its contact, `next` that of level l + 1 (its code only).
        auto sweep = [&](int levels, int steps, auto solve) {
            auto start = [&](int l) { return level_start(min(l, levels)); };
            int i0 = start(0), i1 = start(1), i2 = start(2);
            PairItem here, next;
            bool has = 0 < levels && i0 + lane / 2 < i1, has_next = 1 < levels && i1 + lane / 2 < i2;
            if (has) {
                load_item(here, order, bodies, i0 + lane / 2);
                load_item_contact<kExt>(here, w);
            }
            if (has_next) load_item(next, order, bodies, i1 + lane / 2);
            for (int l = 0; l < steps; ++l) {
                int i3 = start(l + 3);
                bool has_after = l + 2 < levels && i2 + lane / 2 < i3;
                PairItem after;
                if (has_next) load_item_contact<kExt>(next, w);
                if (has_after) load_item(after, order, bodies, i2 + lane / 2);
                if (has) {
                    for (int idx = i0 + lane / 2;;) {
                        solve(here);
                        idx += LPS / 2;
                        if (idx >= i1) break;
                        load_item(here, order, bodies, idx);
                        load_item_contact<kExt>(here, w);
                    }
                }
                __syncthreads();
                here = next;
                next = after;
                has = has_next;
                has_next = has_after;
                i0 = i1;
                i1 = i2;
                i2 = i3;
            }
        };
        for (int it = 0; it < iters; ++it) sweep(pos_levels, pos_steps, position);
        // velocity update
        for (int i = lane; i < n; i += LPS) velocity_update_body(body[i], h);
        __syncthreads();
        // velocity solve over the collision items, in the same levels
        sweep(vel_levels, vel_steps, velocity);
    }
    if (err && valid) atomicOr(&w.scene_err[s], err);
    // the velocity update of the bodies without contact items (pipelined), and
    // the next substep's integration of the scene's bodies (worlds without
    // large scenes), in place of a k_integrate launch
    if (kPipe || integrate_next)
        for (int i = thread; i < n; i += TPS) {
            if (kPipe && (!touching || !w.body_touch[b0 + i])) velocity_update_body(body[i], h);
            if (integrate_next) integrate_body(w, b0 + i, body[i], h);
        }
    if (integrate_next && blockIdx.x == 0 && threadIdx.x == 0) w.counters[CNT_MANIFOLD] = 0;
    if constexpr (kLds) {
        __syncthreads();
        int4* dst = (int4*)(w.body + b0);
        const int4* src = (const int4*)body;
        for (int i = thread; i < n * STATE_VECS; i += TPS) {
            int b = i / STATE_VECS, k = i - b * STATE_VECS;
            dst[b * BODY_VECS + k] = src[b * BODY_VECS + k];
        }
    }
}

// LDS bytes of the solve's body records per block, or 0 to leave them in
// global memory: the records may not cost the launch waves that the
// registers (two waves per SIMD, eight per CU) would allow it to hold.
static size_t solve_lds_bytes(const DevWorld& w, int lanes, int blocks) {
    int scenes = std::max(1, 64 / lanes), waves = lanes > 64 ? 2 * lanes / 64 : 1;
    size_t bytes = (size_t)scenes * w.small_bodies * sizeof(Body);
    if (bytes == 0 || bytes > (size_t)(lanes == 256 ? w.solve_lds : std::min(w.solve_lds, SOLVE_LDS_LIMIT))) return 0;
    size_t per_cu = std::min<size_t>(8 / waves, 160 * 1024 / bytes);
    return per_cu * waves == 8 || (size_t)blocks <= 256 * per_cu ? bytes : 0;
}

template <bool kExt, int LPS>
static void launch_solve_lanes(const DevWorld& w, const FrameParams& fp, hipStream_t st, int integrate_next) {
    constexpr int SPB = LPS < 64 ? 64 / LPS : 1;
    dim3 grid((w.ns + SPB - 1) / SPB), block(LPS > 64 ? 2 * LPS : 64);
    int it = (int)fp.iters, co = fp.collisions ? 1 : 0;
    size_t lds = solve_lds_bytes(w, LPS, (int)grid.x);
    if (lds > 0)
        hipLaunchKernelGGL((k_solve<kExt, LPS, true>), grid, block, lds, st, w, fp.h, it, co, integrate_next,
                           w.small_bodies);
    else
        hipLaunchKernelGGL((k_solve<kExt, LPS, false>), grid, block, 0, st, w, fp.h, it, co, integrate_next, 0);
}
// Lanes per sweep and scene where whole waves serve a scene (solve_lanes 64).
// One width serves every scene of the world, so it also follows how many there
// are: with one wave per SIMD slot taken by a small scene's idle waves, the
// others wait. ms per frame of worlds of n scenes at 64 / 128 / 256 lanes:
//   above 64 bodies, whose steps have many items: four waves per sweep while
//   their blocks fit one to a CU, two up to four times as many
//     150 of 4 to 256 bodies     7.3 /  6.3 /  6.0   256 of them      7.7 /  6.5 /  6.2
//     600 of them                9.7 /  8.6 /  9.3   1500 of them    15.9 / 17.4 / 20.0
//     512 of 66 bodies           2.8 /  2.6 /  3.3   3000 of them    11.1 / 13.3 / 18.0
//     256 of 16 and one of 66    1.9 /  1.7 /  1.8   1500 and one     2.3 /  2.3 /  3.4
//   with joints: two (a wave solves a joint and a contact one after the other)
//   up to three scenes per CU
//     500 chains of 6 links      7.3 /  6.5          600 of them      7.3 /  6.6
//     800 of them                7.4 /  7.6          1200 of them     7.7 /  9.6
//   others: one (one scene of 16 bodies 0.89 / 0.95 / 1.08, 1000 scenes 1.7 /
//   1.9 / 2.7).
static int solve_width(const DevWorld& w) {
    if (w.solve_lanes < 64) return w.solve_lanes;
    if (w.small_bodies > 64) return w.all_scenes <= 256 ? 256 : w.all_scenes <= 1024 ? 128 : 64;
    return w.n_ext > 0 && w.all_scenes <= 768 ? 128 : 64;
}
static bool solve_pipelined(const DevWorld& w) {  // kPipe of the kernel that launch_solve takes
    return w.n_ext > 0 || solve_width(w) > 64;
}
template <bool kExt>
static void launch_solve(const DevWorld& w, const FrameParams& fp, hipStream_t st, int integrate_next) {
    switch (solve_width(w)) {
    case 16: launch_solve_lanes<kExt, 16>(w, fp, st, integrate_next); break;
    case 32: launch_solve_lanes<kExt, 32>(w, fp, st, integrate_next); break;
    case 64: launch_solve_lanes<kExt, 64>(w, fp, st, integrate_next); break;
    case 128: launch_solve_lanes<kExt, 128>(w, fp, st, integrate_next); break;
    default: launch_solve_lanes<kExt, 256>(w, fp, st, integrate_next); break;
    }
}

// Contacts of one body pair at the current transformed poses (debug / parity).
// One lane group of 8 over the pre-transformed hulls, its polytope and
// polygons in lane-group working memory slot 0 (no large private arrays).
__global__ void __launch_bounds__(64) k_pair_contacts(DevWorld w, int b1, int b2, double* out, int* count,
                                                     uint32_t* err_out) {
    if (blockIdx.x != 0 || threadIdx.x >= 8) return;
    HullView h1 = hull_view(w, b1), h2 = hull_view(w, b2);
    uint32_t err = 0;
    int flags = 0;
    auto emit = [&](int k, const ContactPt& c) {
        double* o = out + 9 * k;
        o[0] = c.p1.x; o[1] = c.p1.y; o[2] = c.p1.z;
        o[3] = c.p2.x; o[4] = c.p2.y; o[5] = c.p2.z;
        o[6] = c.n.x; o[7] = c.n.y; o[8] = c.n.z;
    };
    int nc = pair_contacts<8>(w.hulls, h1, h2, emit, err, flags, w.group_work);
    if (threadIdx.x != 0) return;
    *count = nc;
    *err_out = err;
}

// Model matrices of all bodies at their current pose (no integration).
__global__ void k_model(DevWorld w) {
    int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= w.nb) return;
    w.model[b] = model_matrix(w.body[b].x, w.body[b].q);
}

// Elementwise FP64 primitives the step relies on: sqrt and division must be
// correctly rounded for bit-exactness; asin/sin/cos feed the joint limits.
__global__ void k_fp64_selftest(const double* a, const double* b, double* out, int64_t n) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double x = a[i], y = b[i];
    out[5 * i + 0] = sqrt(x);
    out[5 * i + 1] = x / y;
    out[5 * i + 2] = asin(y / (fabs(y) + 1.0));
    out[5 * i + 3] = sin(y);
    out[5 * i + 4] = cos(y);
}

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------
static inline int cdiv(int a, int b) { return (a + b - 1) / b; }

// LDS vertices of a pair's slice in the lane-group kernels: both hulls (`base`
// vertices at most) and room beside them for the EPA polytope and then the
// clipping polygons, which otherwise go through the group's working memory
// (the polygons on one lane: a pair of the world's largest hulls, or any pair
// of a world of boxes, had no room and took 45 000 to 62 000 cycles per
// manifold instead of 21 000). 8 points per polygon always, up to 96 vertices
// (40 faces) while eight blocks (two waves per SIMD) still share a CU's
// 160 KiB, and never beyond the world's LDS limit.
static int stage_slice(const DevWorld& w, int group, int base) {
    if (group <= 1) return 0;
    int per = 64 / group * (int)sizeof(V3);
    int extra = std::max(16, std::min(96, 20 * 1024 / per - base));
    return std::max(base, std::min(base + extra, w.lds_limit / per));
}
static size_t stage_bytes(int group, int stage) {
    return group > 1 ? (size_t)(64 / group) * stage * sizeof(V3) : 0;
}

static void launch_frame_begin(const DevWorld& w, const FrameParams& fp, hipStream_t st, KernelTimer& t,
                               const BigScene* bigs, int nbig) {
    t.begin(KC_FRAME, st);
    if (!fp.forces_given) hipLaunchKernelGGL(k_frame_begin, dim3(cdiv(w.nb, 256)), dim3(256), 0, st, w, fp.gravity);
    hipLaunchKernelGGL(k_broad, dim3(w.ns), dim3(64), 0, st, w);
    for (int k = 0; k < nbig; ++k) big_broad(w, bigs[k], st);
    hipLaunchKernelGGL(k_islands, dim3(w.ns), dim3(64), 0, st, w, fp.dt);
    for (int k = 0; k < nbig; ++k) big_islands(w, bigs[k], fp.dt, st);
    hipLaunchKernelGGL(k_scan_live, dim3(1), dim3(1024), 0, st, w);
    hipLaunchKernelGGL(k_scatter_live, dim3(w.ns), dim3(64), 0, st, w);
    for (int k = 0; k < nbig; ++k) big_scatter(w, bigs[k], st);
    hipLaunchKernelGGL(k_levels, dim3(w.ns), dim3(64), 0, st, w, fp.collisions ? 1 : 0, solve_pipelined(w) ? 1 : 0);
    for (int k = 0; k < nbig; ++k) big_colour(w, bigs[k], fp.collisions, st);
    t.end(st);
}

hipError_t launch_frame(const DevWorld& world, const FrameParams& fp, hipStream_t st, KernelTimer* kt,
                        const BigScene* bigs, int nbig, const Recorder* rec, FramePart part) {
    if (world.nb == 0) return hipSuccess;
    DevWorld w = world;
    KernelTimer none;
    KernelTimer& t = kt ? *kt : none;
    if (part != FRAME_SUBSTEPS) launch_frame_begin(w, fp, st, t, bigs, nbig);
    if (part == FRAME_BEGIN) return hipGetLastError();
    // without large scenes, the solve kernel integrates its scenes' bodies for
    // the next substep
    bool fuse_integrate = nbig == 0;
    // a recorded frame keeps each substep's contacts and start states in its
    // slice of the record: the kernels work in place, nothing is copied
    auto record_state = [&](unsigned sub) { return rec->state + (size_t)sub * rec->nb * REC_STATE; };
    for (unsigned sub = 0; sub < fp.substeps; ++sub) {
        if (rec) {
            size_t slot = (size_t)sub * rec->pair_cap + rec->p0;
            w.contacts = rec->contacts + slot * MAXC;
            w.ncontact = rec->ncontact + slot;
            w.rec_state = record_state(sub);
        }
        if (sub == 0 || !fuse_integrate) {
            t.begin(KC_INTEGRATE, st);
            hipLaunchKernelGGL(k_integrate, dim3(cdiv(w.nb, 128)), dim3(128), 0, st, w, fp.h);
            t.end(st);
        }
        if (fp.keep_pose && sub + 1 == fp.substeps)
            hipLaunchKernelGGL(k_keep_pose, dim3(cdiv(w.nb, 256)), dim3(256), 0, st, w);
        if (fp.collisions) {
            bool fused = w.manifold_group == 0;
            if (w.narrow_group == 1 || w.manifold_group == 1) {
                t.begin(KC_TRANSFORM, st);
                hipLaunchKernelGGL(k_transform, dim3(cdiv(w.n_xf, 256)), dim3(256), 0, st, w, 0);
                t.end(st);
            }
            t.begin(KC_NARROW, st);
            int stage = stage_slice(w, w.narrow_group, w.stage_cap);
            size_t lds = stage_bytes(w.narrow_group, stage);
            dim3 nb(w.narrow_blocks), t64(64);
            if (fused && w.small_nv > 0 && w.narrow_group > 1) {
                // two size classes: small-hull pairs with small LDS slices on the
                // narrow schedule, the others on the schedule with the fewest
                // groups per block that fits
                const int32_t* small = w.pair_lists;
                const int32_t* big = w.pair_lists + w.list_stride;
                int stage_s = stage_slice(w, w.narrow_group, w.stage_small), stage_b = stage_slice(w, 16, w.stage_cap);
                size_t lds_s = stage_bytes(w.narrow_group, stage_s), lds_b = stage_bytes(16, stage_b);
                switch (w.narrow_group) {
                case 4: hipLaunchKernelGGL((k_gjk_epa<4, true>), nb, t64, lds_s, st, w, small, w.counters + CNT_SMALL, stage_s); break;
                case 8: hipLaunchKernelGGL((k_gjk_epa<8, true>), nb, t64, lds_s, st, w, small, w.counters + CNT_SMALL, stage_s); break;
                default: hipLaunchKernelGGL((k_gjk_epa<16, true>), nb, t64, lds_s, st, w, small, w.counters + CNT_SMALL, stage_s); break;
                }
                hipLaunchKernelGGL((k_gjk_epa<16, true>), nb, t64, lds_b, st, w, big, w.counters + CNT_BIG, stage_b);
            } else if (fused) {
                switch (w.narrow_group) {
                case 4: hipLaunchKernelGGL((k_gjk_epa<4, true>), nb, t64, lds, st, w, nullptr, nullptr, stage); break;
                case 8: hipLaunchKernelGGL((k_gjk_epa<8, true>), nb, t64, lds, st, w, nullptr, nullptr, stage); break;
                case 16: hipLaunchKernelGGL((k_gjk_epa<16, true>), nb, t64, lds, st, w, nullptr, nullptr, stage); break;
                default: hipLaunchKernelGGL(k_gjk_epa_lane<true>, nb, t64, 0, st, w); break;
                }
            } else {
                switch (w.narrow_group) {
                case 4: hipLaunchKernelGGL((k_gjk_epa<4, false>), nb, t64, lds, st, w, nullptr, nullptr, stage); break;
                case 8: hipLaunchKernelGGL((k_gjk_epa<8, false>), nb, t64, lds, st, w, nullptr, nullptr, stage); break;
                case 16: hipLaunchKernelGGL((k_gjk_epa<16, false>), nb, t64, lds, st, w, nullptr, nullptr, stage); break;
                default: hipLaunchKernelGGL(k_gjk_epa_lane<false>, nb, t64, 0, st, w); break;
                }
            }
            if (w.has_general) {
                // (at least 8 lanes per pair: the working memory is sized for
                // the narrow schedule's groups)
                int gg = w.narrow_group == 4 ? 8 : w.narrow_group;
                int gs = stage_slice(w, gg, w.stage_cap);
                switch (gg) {
                case 8: hipLaunchKernelGGL(k_narrow_general<8>, nb, t64, stage_bytes(8, gs), st, w, gs); break;
                case 16: hipLaunchKernelGGL(k_narrow_general<16>, nb, t64, stage_bytes(16, gs), st, w, gs); break;
                default: hipLaunchKernelGGL(k_narrow_general<1>, dim3(1024), t64, 0, st, w, 0); break;
                }
            }
            t.end(st);
            if (!fused) {
                t.begin(KC_MANIFOLD, st);
                stage = stage_slice(w, w.manifold_group, w.stage_cap);
                lds = stage_bytes(w.manifold_group, stage);
                dim3 mb(w.manifold_blocks);
                switch (w.manifold_group) {
                case 4: hipLaunchKernelGGL(k_manifold<4>, mb, t64, lds, st, w, stage); break;
                case 8: hipLaunchKernelGGL(k_manifold<8>, mb, t64, lds, st, w, stage); break;
                case 16: hipLaunchKernelGGL(k_manifold<16>, mb, t64, lds, st, w, stage); break;
                default: hipLaunchKernelGGL(k_manifold<1>, mb, t64, 0, st, w, 0); break;
                }
                t.end(st);
            }
        }
        t.begin(KC_SOLVE, st);
        int next = fuse_integrate && sub + 1 < fp.substeps ? 1 : 0;
        if (rec && next) w.rec_state = record_state(sub + 1);
        if (w.n_ext > 0) launch_solve<true>(w, fp, st, next);
        else launch_solve<false>(w, fp, st, next);
        for (int k = 0; k < nbig; ++k) big_solve(w, bigs[k], fp, st);
        t.end(st);
    }
    return hipGetLastError();
}

hipError_t launch_pair_contacts(const DevWorld& w, int b1, int b2, double* out, int* count, uint32_t* err,
                                hipStream_t st) {
    hipLaunchKernelGGL(k_model, dim3(cdiv(w.nb, 128)), dim3(128), 0, st, w);
    hipLaunchKernelGGL(k_transform, dim3(cdiv(w.n_xf, 256)), dim3(256), 0, st, w, 1);
    hipLaunchKernelGGL(k_pair_contacts, dim3(1), dim3(64), 0, st, w, b1, b2, out, count, err);
    return hipGetLastError();
}

hipError_t launch_state_out(const DevWorld& w, double* out, hipStream_t st) {
    hipLaunchKernelGGL(k_state_out, dim3(cdiv(w.nb, 256)), dim3(256), 0, st, w, out);
    return hipGetLastError();
}
hipError_t launch_state_in(const DevWorld& w, const double* in, unsigned mask, hipStream_t st) {
    hipLaunchKernelGGL(k_state_in, dim3(cdiv(w.nb, 256)), dim3(256), 0, st, w, in, mask);
    return hipGetLastError();
}

hipError_t launch_model_matrices(const DevWorld& w, void* out, bool f32, hipStream_t st) {
    if (w.nb == 0) return hipSuccess;
    if (f32) hipLaunchKernelGGL(k_model_out<float>, dim3(cdiv(w.nb, 256)), dim3(256), 0, st, w, (float*)out);
    else hipLaunchKernelGGL(k_model_out<double>, dim3(cdiv(w.nb, 256)), dim3(256), 0, st, w, (double*)out);
    return hipGetLastError();
}

hipError_t launch_fp64_selftest(const double* a, const double* b, double* out, int64_t n, hipStream_t st) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_fp64_selftest, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, a, b, out, n);
    return hipGetLastError();
}

// Lane-group working memory of rp_world_step_noalloc: a file-scope device
// array instead of a hipMalloc'd buffer. Each device that runs the library
// holds its own copy until the process ends. Host code never passes the
// array's name to a kernel (it is a host-side stand-in there): it takes the
// device address from noalloc_scratch(), which looks it up once per device.
static __device__ __align__(256) unsigned char scratch[NOALLOC_SCRATCH_BYTES];

unsigned char* noalloc_scratch() {
    static std::mutex mu;
    static std::vector<unsigned char*> ptr;  // per device, null until looked up
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0) return nullptr;
    std::lock_guard<std::mutex> lock(mu);
    if ((size_t)dev >= ptr.size()) ptr.resize(dev + 1, nullptr);
    if (!ptr[dev]) {
        void* p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess) return nullptr;
        ptr[dev] = (unsigned char*)p;
    }
    return ptr[dev];
}

int64_t group_work_slots_needed(const DevWorld& w) {
    int64_t n = 1;  // k_pair_contacts
    if (w.narrow_group > 1) n = std::max<int64_t>(n, (int64_t)w.narrow_blocks * (64 / w.narrow_group));
    if (w.manifold_group > 1) n = std::max<int64_t>(n, (int64_t)w.manifold_blocks * (64 / w.manifold_group));
    return n;
}

bool narrow_group_supported(const DevWorld& w, int g) {
    if (g == 1) return true;
    if (g != 4 && g != 8 && g != 16) return false;
    return (size_t)(64 / g) * w.stage_cap * sizeof(V3) <= (size_t)w.lds_limit;
}

hipError_t allow_narrow_lds(int bytes) {
    const void* k[] = {(const void*)k_gjk_epa<4, true>, (const void*)k_gjk_epa<8, true>,
                       (const void*)k_gjk_epa<16, true>, (const void*)k_gjk_epa<4, false>,
                       (const void*)k_gjk_epa<8, false>, (const void*)k_gjk_epa<16, false>,
                       (const void*)k_manifold<4>, (const void*)k_manifold<8>, (const void*)k_manifold<16>,
                       (const void*)k_narrow_general<8>, (const void*)k_narrow_general<16>};
    for (const void* f : k) {
        hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t allow_solve_lds(int bytes) {
    for (const void* f : {(const void*)k_solve<false, 256, true>, (const void*)k_solve<true, 256, true>}) {
        hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

// Blocks of the narrow-phase kernels: one lane group per pair slot, up to
// 8192 one-wave blocks (32 per CU). Live pairs beyond the groups are taken in
// grid-stride order; frames with more live pairs than 4096 blocks hold ran
// 5 % faster with the larger cap (batched 4096-scene workload, 600 frames).
int narrow_blocks_for(const DevWorld& w, int g, int64_t pcap) {
    int64_t per_block = 64 / g;
    int64_t blocks = (pcap + per_block - 1) / per_block;
    int64_t cap = w.narrow_block_cap > 0 ? w.narrow_block_cap : 256 * 32;
    return (int)std::max<int64_t>(1, std::min<int64_t>(blocks, cap));
}

hipError_t launch_broad(const DevWorld& w, hipStream_t st, const BigScene* bigs, int nbig) {
    hipLaunchKernelGGL(k_broad, dim3(w.ns), dim3(64), 0, st, w);
    for (int k = 0; k < nbig; ++k) big_broad(w, bigs[k], st);
    return hipGetLastError();
}

}  // namespace rp
