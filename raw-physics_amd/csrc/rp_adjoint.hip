// rp_adjoint.hip — reverse-mode gradients of the step over a recorded run.
//
// Scope: scenes with one dynamic body (any number of fixed bodies), as in a
// body thrown onto static geometry. The contact set is frozen: the contacts
// the forward pass generated in each substep (r1_lc, r2_lc, n) are constants
// of the backward pass, so the gradient is that of the step with those
// contacts (the discrete collision decisions and the contact geometry carry
// no derivative).
//
// Per substep the state is (x, q, v, w) of the dynamic body: integration
// overwrites the previous pose at the substep start and the velocity update
// overwrites the previous velocities before the velocity solve reads them.
// The parameters are the body's mass (through 1/m, the inertia tensor and
// its inverse, and the gravity force m g), static and dynamic friction.
//
// The forward pass records every substep's start state and contacts as it
// runs. A substep's Jacobian depends on that record only, so the backward
// pass evaluates the Jacobians of all recorded substeps at once: for each
// substep, lane k of a 16-lane group re-evaluates it from its start state
// with a dual number seeded on input k, which gives column k of J. A second
// kernel then walks the substeps in reverse, one 16-lane group per scene:
// lane k forms (J^T abar)_k; lanes 0-12 produce the new state adjoint, lanes
// 13-15 accumulate the parameter gradients. (Evaluating a frame's substeps
// one after another left 16 lanes per scene busy, a wave per two SIMDs at 2048
// scenes, and each frame was stepped again first: 1024 scenes of 30 frames
// took 50 ms backward, now 5.0 ms; forward and backward together 71.3 -> 29.4
// ms, 37 scenes of 12 frames 15.3 -> 4.8 ms.) The dual value parts repeat the primal operations, so each
// re-evaluation reproduces the recorded next state bit for bit; a mismatch is
// counted (STAT_ADJ_MISMATCH).
#include <algorithm>

#include "rp_device.h"
#include "rp_dual.h"

namespace rp {

using D1 = ad::Dual<1>;
constexpr int ADJ_LANES = 16;       // 13 state inputs + mass, static and dynamic friction
constexpr int ADJ_MAX_CONTACTS = 32;  // contacts of one scene in one substep

template <class S> RP_HD V3T<S> lift(V3 a) { return v3<S>(S(a.x), S(a.y), S(a.z)); }
template <class S> RP_HD Q4T<S> lift(Q4 a) { Q4T<S> r = {S(a.x), S(a.y), S(a.z), S(a.w)}; return r; }
template <class S> RP_HD M3T<S> lift(const M3& a) {
    M3T<S> r;
    for (int i = 0; i < 3; ++i)
        for (int j = 0; j < 3; ++j) r.m[i][j] = S(a.m[i][j]);
    return r;
}
RP_HD V3T<D1> sub(V3T<D1> a, V3 b) { return v3<D1>(a.x - b.x, a.y - b.y, a.z - b.z); }
RP_HD V3T<D1> sub(V3 a, V3T<D1> b) { return v3<D1>(a.x - b.x, a.y - b.y, a.z - b.z); }
RP_HD D1 dot(V3T<D1> a, V3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }

// State component k of (x, q, v, w).
__device__ __forceinline__ D1& state_comp(BodyT<D1>& e, int k) {
    switch (k) {
    case 0: return e.x.x; case 1: return e.x.y; case 2: return e.x.z;
    case 3: return e.q.x; case 4: return e.q.y; case 5: return e.q.z; case 6: return e.q.w;
    case 7: return e.v.x; case 8: return e.v.y; case 9: return e.v.z;
    case 10: return e.w.x; case 11: return e.w.y; default: return e.w.z;
    }
}

// The dynamic body against one fixed body. Only the dynamic body's side
// carries derivatives; a fixed body has no inverse mass and no inverse
// inertia, so its generalized inverse mass is zero and it is never moved.
struct AdjContactState { D1 lambda_n, lambda_t; };

// d(between the bodies' points): first body's minus second's.
__device__ __forceinline__ V3T<D1> adj_diff(bool first, V3T<D1> own, V3 other) {
    return first ? sub(own, other) : sub(other, own);
}
__device__ __forceinline__ D1 adj_dlambda(D1 w, D1 c, double tc, D1 lambda, uint32_t& err) {
    if (w == 0.0) err |= ERR_ZERO_MASS;
    return (-c - tc * lambda) / (w + tc);
}
__device__ __forceinline__ D1 adj_mass(const BodyT<D1>& e, V3T<D1> r, const M3T<D1>& I, V3T<D1> n) {
    return e.inv_mass + dot(cross(r, n), m3_mulv(I, cross(r, n)));
}
__device__ __forceinline__ void adj_apply(BodyT<D1>& e, bool first, V3T<D1> r, const M3T<D1>& I, D1 dl, V3T<D1> n) {
    V3T<D1> imp = scl(dl, n);
    e.x = add(e.x, scl(first ? e.inv_mass : -e.inv_mass, imp));
    rot_update(e, m3_mulv(I, cross(r, imp)), first);
}
// collision_constraint_solve (pbd.cpp:107-154), as pair_collision: the world
// inverse inertia is computed once per change of the rotation.
__device__ __forceinline__ void adj_collision(const AdjContact& c, bool first, AdjContactState& st, BodyT<D1>& e,
                                              M3T<D1>& I, bool& fresh, const Body& f, double h, uint32_t& err) {
    const V3T<D1> r_lc = lift<D1>(first ? c.r1 : c.r2);
    const V3 rf = q_rot(f.q, first ? c.r2 : c.r1), pf = add(f.x, rf);
    V3T<D1> r = q_rot(e.q, r_lc);
    D1 d = dot(adj_diff(first, add(e.x, r), pf), c.n);
    if (!(d > 0.0)) return;
    if (!fresh) I = world_tensor(e.q, e.Iinv);
    V3T<D1> dx = scl(d, lift<D1>(c.n));
    D1 cl = len(dx);
    double tc = 0.0 / (h * h);
    bool any = !(cl <= 1e-50);
    V3T<D1> n = v3<D1>(dx.x / cl, dx.y / cl, dx.z / cl);
    D1 dl(0.0);
    if (any) {
        dl = adj_dlambda(adj_mass(e, r, I, n), cl, tc, st.lambda_n, err);
        adj_apply(e, first, r, I, dl, n);
    }
    st.lambda_n += dl;
    r = q_rot(e.q, r_lc);
    I = world_tensor(e.q, e.Iinv);
    fresh = true;
    V3T<D1> p = add(e.x, r);
    dl = D1(0.0);
    if (any) dl = adj_dlambda(adj_mass(e, r, I, n), cl, tc, st.lambda_t, err);
    const D1 mu_s = (e.mu_s + f.mu_s) / 2.0f;
    if (st.lambda_t + dl > mu_s * st.lambda_n) {
        V3T<D1> dp_own = sub(p, add(e.px, q_rot(e.pq, r_lc)));
        V3 dp_f = sub(pf, add(f.px, q_rot(f.pq, first ? c.r2 : c.r1)));
        V3T<D1> dp = adj_diff(first, dp_own, dp_f);
        V3T<D1> dp_t = sub(dp, scl(dot(dp, c.n), lift<D1>(c.n)));
        D1 ct = len(dp_t);
        if (!(ct <= 1e-50)) {
            adj_apply(e, first, r, I, dl, v3<D1>(dp_t.x / ct, dp_t.y / ct, dp_t.z / ct));
            fresh = false;
        }
        st.lambda_t += dl;
    }
}
// Velocity solve of one contact (pbd.cpp:646-711), as pair_velocity.
__device__ __forceinline__ void adj_velocity(const AdjContact& c, bool first, D1 lambda_n, BodyT<D1>& e,
                                             const M3T<D1>& I, const Body& f, double h) {
    V3T<D1> r = q_rot(e.q, lift<D1>(first ? c.r1 : c.r2));
    const V3 rf = q_rot(f.q, first ? c.r2 : c.r1);
    V3T<D1> v = adj_diff(first, add(e.v, cross(e.w, r)), add(f.v, cross(f.w, rf)));
    D1 vn = dot(v, c.n);
    V3T<D1> vt = sub(v, scl(vn, lift<D1>(c.n)));
    V3T<D1> dv = v3<D1>(D1(0.0), D1(0.0), D1(0.0));
    const D1 mu_d = (e.mu_d + f.mu_d) / 2.0f;
    D1 fn = lambda_n / h;
    D1 fact = RP_MIN(mu_d * fabs(fn), len(vt));
    dv = add(dv, scl(-fact, nrm(vt)));
    D1 vn_til = dot(adj_diff(first, add(e.pv, cross(e.pw, r)), add(f.pv, cross(f.pw, rf))), c.n);
    D1 rest = e.e * f.e;
    fact = -vn + RP_MIN(-rest * vn_til, D1(0.0));
    dv = add(dv, scl(fact, lift<D1>(c.n)));
    D1 w = adj_mass(e, r, I, lift<D1>(c.n));
    V3T<D1> pimp = scl(1.0 / w, dv);
    V3T<D1> jv = scl(e.inv_mass, pimp), jw = m3_mulv(I, cross(r, pimp));
    e.v = add(e.v, first ? jv : inv3(jv));
    e.w = add(e.w, first ? jw : inv3(jw));
}

// One substep of scene s from its recorded start (pbd.cpp:537-711 for this
// scene: integration, contact position solve in pair order, velocity update,
// velocity solve).
__device__ void adj_substep(const AdjRecord& r, int t, int s, int bd, BodyT<D1>& e, const FrameParams& fp,
                            uint32_t& err) {
    // the frame's gravity force (stack.cpp:93-96, physics_util.cpp:5-23)
    V3T<D1> force = v3<D1>(D1(0.0), -fp.gravity * 1.0 / e.inv_mass, D1(0.0));
    e.F = add(v3<D1>(D1(0.0), D1(0.0), D1(0.0)), force);
    e.T = add(v3<D1>(D1(0.0), D1(0.0), D1(0.0)),
              cross(sub(v3<D1>(D1(0.0), D1(0.0), D1(0.0)), v3<D1>(D1(0.0), D1(0.0), D1(0.0))), force));
    integrate(e, fp.h);
    const int f = t / (int)fp.substeps;
    const int g0 = r.g0[(size_t)f * r.ns + s], g1 = g0 + r.np[(size_t)f * r.ns + s];
    const int2* pair = r.pair + (size_t)f * r.pair_cap;
    const int32_t* ncs = r.ncontact + (size_t)t * r.pair_cap;
    const AdjContact* cs = r.contacts + (size_t)t * r.pair_cap * MAXC;
    AdjContactState st[ADJ_MAX_CONTACTS];
    M3T<D1> I;
    bool fresh = false;
    for (unsigned it = 0; it < fp.iters; ++it) {
        int k = 0;
        for (int g = g0; g < g1; ++g) {
            int2 bb = pair[g];
            bool first = bb.x == bd;
            const Body& other = r.end_state[first ? bb.y : bb.x];
            for (int c = 0; c < ncs[g]; ++c, ++k) {
                if (k >= ADJ_MAX_CONTACTS) { err |= ERR_SOLVER_CAPACITY; break; }
                AdjContactState cst = it == 0 ? AdjContactState{D1(0.0), D1(0.0)} : st[k];
                adj_collision(cs[(size_t)g * MAXC + c], first, cst, e, I, fresh, other, fp.h, err);
                st[k] = cst;
            }
        }
    }
    velocity_update(e, fp.h);
    if (!fresh) I = world_tensor(e.q, e.Iinv);
    int k = 0;
    for (int g = g0; g < g1; ++g) {
        int2 bb = pair[g];
        bool first = bb.x == bd;
        const Body& other = r.end_state[first ? bb.y : bb.x];
        for (int c = 0; c < ncs[g]; ++c, ++k) {
            if (k >= ADJ_MAX_CONTACTS) { err |= ERR_SOLVER_CAPACITY; break; }
            adj_velocity(cs[(size_t)g * MAXC + c], first, fp.iters ? st[k].lambda_n : D1(0.0), e, I, other, fp.h);
        }
    }
}

// Jacobians of substeps t0 .. t0 + nt - 1 (of the record) of every scene: a
// 16-lane group per (substep, scene), lane k the derivatives of the 13 state
// components in input k.
__global__ void __launch_bounds__(64) k_adjoint_jacobian(AdjRecord r, const int32_t* scene_dyn, int t0, int nt,
                                                         double* jac, FrameParams fp, unsigned long long* stats,
                                                         uint32_t* scene_err) {
    constexpr int GPB = 64 / ADJ_LANES;
    int64_t u = (int64_t)blockIdx.x * GPB + (int)threadIdx.x / ADJ_LANES;
    int k = (int)threadIdx.x % ADJ_LANES;
    if (u >= (int64_t)nt * r.ns) return;
    int t = t0 + (int)(u / r.ns), s = (int)(u % r.ns);
    int bd = scene_dyn[s];
    if (bd < 0) return;
    const Body& b = r.end_state[bd];  // the run's constants: mass, inertia, friction, restitution
    const double* start = r.state + ((size_t)t * r.nb + bd) * REC_STATE;
    BodyT<D1> e;
    e.inv_mass = D1(b.inv_mass);
    e.I = lift<D1>(b.I);
    e.Iinv = lift<D1>(b.Iinv);
    e.mu_s = D1(b.mu_s);
    e.mu_d = D1(b.mu_d);
    e.e = D1(b.e);
    e.pv = lift<D1>(b.pv);
    e.pw = lift<D1>(b.pw);
    for (int j = 0; j < 13; ++j) state_comp(e, j) = D1(start[j]);
    e.fixed = 0;
    e.active = start[13] != 0.0;
    if (k < 13) {
        for (int j = 0; j < 13; ++j) state_comp(e, j).d[0] = j == k ? 1.0 : 0.0;
    } else if (k == 13) {  // mass m: 1/m, I = m C, I^-1 = C^-1 / m
        double im = b.inv_mass;
        e.inv_mass.d[0] = -im * im;
        for (int i = 0; i < 3; ++i)
            for (int j = 0; j < 3; ++j) {
                e.I.m[i][j].d[0] = b.I.m[i][j] * im;
                e.Iinv.m[i][j].d[0] = -b.Iinv.m[i][j] * im;
            }
    } else if (k == 14) {
        e.mu_s.d[0] = 1.0;
    } else {
        e.mu_d.d[0] = 1.0;
    }
    uint32_t err = 0;
    adj_substep(r, t, s, bd, e, fp, err);
    const double* next = t + 1 < r.steps ? start + (size_t)r.nb * REC_STATE : (const double*)&r.next_state[bd];
    double* out = jac + ((size_t)(t - t0) * r.ns + s) * (13 * ADJ_LANES) + 13 * k;
    bool mismatch = false;
    for (int j = 0; j < 13; ++j) {
        const D1& o = state_comp(e, j);
        out[j] = o.d[0];
        mismatch |= __double_as_longlong(o.v) != __double_as_longlong(next[j]);
    }
    // (the group's lanes have the same values: a substep counts once)
    if (mismatch && k == 0) atomicAdd(&stats[STAT_ADJ_MISMATCH], 1ull);
    if (err && k == 0) atomicOr(&scene_err[s], err);
}

// abar <- J^T abar over substeps t0 + nt - 1 down to t0, in order.
__global__ void __launch_bounds__(64) k_adjoint_chain(AdjRecord r, const int32_t* scene_dyn, int t0, int nt,
                                                      const double* jac, double* abar, double* gparam, double* amax,
                                                      int substeps) {
    constexpr int SPB = 64 / ADJ_LANES;
    int s = blockIdx.x * SPB + (int)threadIdx.x / ADJ_LANES;
    int k = (int)threadIdx.x % ADJ_LANES;
    int slot = (int)threadIdx.x / ADJ_LANES;
    __shared__ double a[SPB][13];
    int bd = (s < r.ns) ? scene_dyn[s] : -1;
    if (bd >= 0 && k < 13) a[slot][k] = abar[13 * bd + k];
    double gp = bd >= 0 && k >= 13 ? gparam[3 * bd + (k - 13)] : 0.0;
    double top = bd >= 0 && k == 0 ? amax[bd] : 0.0;
    const double* row = jac + (size_t)std::max(s < r.ns ? s : 0, 0) * (13 * ADJ_LANES) + 13 * k;
    const size_t stride = (size_t)r.ns * (13 * ADJ_LANES);
    double next[13];
    if (bd >= 0)
        for (int j = 0; j < 13; ++j) next[j] = row[(nt - 1) * stride + j];
    __syncthreads();
    for (int t = nt - 1; t >= 0; --t) {
        double cur[13], acc = 0.0;
        if (bd >= 0) {
            for (int j = 0; j < 13; ++j) cur[j] = next[j];
            if (t > 0)  // the next substep's row does not depend on abar
                for (int j = 0; j < 13; ++j) next[j] = row[(size_t)(t - 1) * stride + j];
            for (int j = 0; j < 13; ++j) acc += a[slot][j] * cur[j];
        }
        __syncthreads();
        if (bd >= 0) {
            if (k < 13) a[slot][k] = acc;
            else gp += acc;
        }
        __syncthreads();
        if (bd >= 0 && k == 0 && (t0 + t) % substeps == 0)  // largest state adjoint at a frame start so far
            for (int j = 0; j < 13; ++j) top = fmax(top, std::fabs(a[slot][j]));
    }
    if (bd < 0) return;
    if (k < 13) abar[13 * bd + k] = a[slot][k];
    else gparam[3 * bd + (k - 13)] = gp;
    if (k == 0) amax[bd] = top;
}

int adjoint_steps_per_chunk(int ns, size_t bytes) {
    size_t per = (size_t)std::max(ns, 1) * 13 * ADJ_LANES * sizeof(double);
    return (int)std::max<size_t>(1, std::min<size_t>(bytes / per, 1 << 20));
}
size_t adjoint_jacobian_bytes(int ns, int steps) { return (size_t)std::max(ns, 1) * steps * 13 * ADJ_LANES * sizeof(double); }

hipError_t launch_adjoint(const AdjRecord& r, const int32_t* scene_dyn, int chunk, double* jac, double* abar,
                          double* gparam, double* amax, unsigned long long* stats, uint32_t* scene_err,
                          const FrameParams& fp, hipStream_t st) {
    constexpr int GPB = 64 / ADJ_LANES;
    for (int t1 = r.steps; t1 > 0; t1 -= chunk) {
        int t0 = std::max(0, t1 - chunk), nt = t1 - t0;
        int64_t groups = (int64_t)nt * r.ns;
        hipLaunchKernelGGL(k_adjoint_jacobian, dim3((unsigned)((groups + GPB - 1) / GPB)), dim3(64), 0, st, r, scene_dyn,
                           t0, nt, jac, fp, stats, scene_err);
        hipLaunchKernelGGL(k_adjoint_chain, dim3((r.ns + GPB - 1) / GPB), dim3(64), 0, st, r, scene_dyn, t0, nt, jac,
                           abar, gparam, amax, (int)fp.substeps);
    }
    return hipGetLastError();
}

// One frame's staged record (contacts and states written by the step's own
// kernels) into frame f of the run's record. `w` is a view of the world whose
// scenes start at s0 and whose live pairs at p0; `all` marks the one view
// that copies the bodies' states.
__global__ void __launch_bounds__(256) k_adjoint_pack(DevWorld w, Recorder st, AdjRecord r, int f, int s0, int64_t p0,
                                                      int substeps, int all) {
    int64_t stride = (int64_t)gridDim.x * blockDim.x, i0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int total = w.live_prefix[w.ns];
    for (int64_t i = i0; i < w.ns; i += stride) {
        const_cast<int32_t*>(r.g0)[(size_t)f * r.ns + s0 + i] = (int32_t)(p0 + w.live_prefix[i]);
        const_cast<int32_t*>(r.np)[(size_t)f * r.ns + s0 + i] = w.live_count[i];
    }
    for (int64_t g = i0; g < total; g += stride) {
        int4 rec = w.live_rec[g];
        const_cast<int2*>(r.pair)[(size_t)f * r.pair_cap + p0 + g] = make_int2(rec.x, rec.y);
    }
    for (int64_t i = i0; i < (int64_t)total * substeps; i += stride) {
        int k = (int)(i / total);
        int64_t g = p0 + i % total, from = (int64_t)k * r.pair_cap + g, to = ((int64_t)f * substeps + k) * r.pair_cap + g;
        int nc = st.ncontact[from];
        const_cast<int32_t*>(r.ncontact)[to] = nc;
        for (int c = 0; c < nc; ++c) {
            const Contact& a = st.contacts[from * MAXC + c];
            AdjContact& o = const_cast<AdjContact*>(r.contacts)[to * MAXC + c];
            o.r1 = a.r1;
            o.r2 = a.r2;
            o.n = a.n;
        }
    }
    if (!all) return;
    int64_t n = (int64_t)substeps * r.nb * REC_STATE;
    double* dst = const_cast<double*>(r.state) + (size_t)f * n;
    for (int64_t i = i0; i < n; i += stride) dst[i] = st.state[i];
}

hipError_t launch_adjoint_pack(const DevWorld& w, const Recorder& st, const AdjRecord& r, int f, int s0, int64_t p0,
                               int substeps, bool all, hipStream_t s) {
    hipLaunchKernelGGL(k_adjoint_pack, dim3(512), dim3(256), 0, s, w, st, r, f, s0, p0, substeps, all ? 1 : 0);
    return hipGetLastError();
}

}  // namespace rp
