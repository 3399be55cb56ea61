// rp_pairsolve.h — one solve item on two adjacent lanes.
//
// The even lane of a pair holds the item's first body, the odd lane its
// second. What depends on one body (the lever arm, the world inverse inertia,
// the generalized mass, the applied impulse) is computed by that body's lane;
// what depends on both is exchanged by DPP moves inside the quad and computed
// on both lanes with the same operands in the reference's order, so every
// branch below is uniform over a pair and the results are the reference's bit
// for bit (pbd_base_constraints.cpp:6-227, pbd.cpp:81-379, 646-711).
//
// Why two lanes: an item is one chain of dependent FP64 operations, and a
// level of a scene has few items, so the solve is bound by the instructions of
// one item, not by lanes. One lane per item issued both bodies' halves one
// after another and held both bodies' records (246 VGPRs; 256 + 14 with
// joints).
#pragma once
#include "rp_kernels.h"

namespace rp {

// The even lane's, the odd lane's value on both lanes of a pair, and the
// partner's (quad permutations 0022, 1133, 1032).
enum : int { DPP_PAIR_EVEN = 0xA0, DPP_PAIR_ODD = 0xF5 };
__device__ __forceinline__ double pair_first(double v) { return dpp_double<DPP_PAIR_EVEN>(v); }
__device__ __forceinline__ double pair_second(double v) { return dpp_double<DPP_PAIR_ODD>(v); }
__device__ __forceinline__ double pair_other(double v) { return dpp_double<DPP_XOR1>(v); }
__device__ __forceinline__ V3 pair_first(V3 v) { return v3(pair_first(v.x), pair_first(v.y), pair_first(v.z)); }
__device__ __forceinline__ V3 pair_second(V3 v) { return v3(pair_second(v.x), pair_second(v.y), pair_second(v.z)); }
__device__ __forceinline__ bool second_lane() { return __lane_id() & 1; }

// This lane's body in the position solve.
struct HalfPos {
    V3 x; Q4 q; V3 px; Q4 pq;
    double im;   // inverse mass; negated on the second lane (its impulses are)
    M3 Iinv;
    double mu_s;
    bool fixed;
};
struct HalfVel {
    Q4 q; V3 v, w, pv, pw;
    double im;
    M3 Iinv;
    double mu_d, e;
    bool fixed;
};

// A body's generalized inverse mass for an impulse along n at r
// (pbd_base_constraints.cpp:62-66); `im` is the inverse mass itself.
__device__ __forceinline__ double half_mass(double im, V3 r, const M3& I, V3 n) {
    return im + dot(cross(r, n), m3_mulv(I, cross(r, n)));
}
// calculate_positional_constraint_delta_lambda after the direction: w is this
// lane's generalized inverse mass.
__device__ __forceinline__ double pair_dlambda(double w, double c, double tc, double lambda, uint32_t& err) {
    double ws = w + pair_other(w);  // w1 + w2 on both lanes
    if (ws == 0.0) err |= ERR_ZERO_MASS;
    return (-c - tc * lambda) / (ws + tc);
}
// The rotation by `a`, added on the first lane and subtracted on the second.
__device__ __forceinline__ void half_rotate(HalfPos& e, V3 a) {
    double s = second_lane() ? -0.5 : 0.5;
    Q4 aq = {a.x, a.y, a.z, 0.0};
    Q4 qq = q_mul(aq, e.q);
    Q4 q = {e.q.x + s * qq.x, e.q.y + s * qq.y, e.q.z + s * qq.z, e.q.w + s * qq.w};
    q = q_nrm(q);
    if (!e.fixed) e.q = q;
}
// positional_constraint_apply: impulse dl along the unit direction n at r.
__device__ __forceinline__ void half_apply(HalfPos& e, V3 r, const M3& I, double dl, V3 n) {
    V3 imp = scl(dl, n);
    if (!e.fixed) e.x = add(e.x, scl(e.im, imp));
    half_rotate(e, m3_mulv(I, cross(r, imp)));
}
__device__ __forceinline__ double abs_mass(const HalfPos& e) { return second_lane() ? -e.im : e.im; }

// One positional correction dx between the bodies' points at r, with the
// world inverse inertia I (pos_dlambda, pos_apply); returns delta lambda.
__device__ __forceinline__ double pair_position(HalfPos& e, V3 r, const M3& I, double h, double compliance, double lambda,
                                                V3 dx, uint32_t& err) {
    double c = len(dx);
    if (c <= 1e-50) return 0.0;
    V3 n = v3(dx.x / c, dx.y / c, dx.z / c);
    double dl = pair_dlambda(half_mass(abs_mass(e), r, I, n), c, compliance / (h * h), lambda, err);
    half_apply(e, r, I, dl, n);
    return dl;
}
// One angular correction dq (ang_dlambda, ang_apply).
__device__ __forceinline__ double pair_angular(HalfPos& e, const M3& I, double h, double compliance, double lambda, V3 dq,
                                               uint32_t& err) {
    double theta = len(dq);
    if (theta <= 1e-50) return 0.0;
    V3 n = v3(dq.x / theta, dq.y / theta, dq.z / theta);
    double dl = pair_dlambda(dot(n, m3_mulv(I, n)), theta, compliance / (h * h), lambda, err);
    half_rotate(e, m3_mulv(I, scl(-dl, n)));
    return dl;
}

// collision_constraint_solve (pbd.cpp:107-154). `I` is the world inverse
// inertia at e.q when `fresh`: it is computed once per change of the rotation
// (the second preparation's value serves the item's next contact unless
// friction moved the body), and not at all for a separated contact.
__device__ __forceinline__ void pair_collision(V3 r_lc, V3 n, double& lambda_n, double& lambda_t, HalfPos& e, M3& I,
                                               bool& fresh, double mu_s, double h, uint32_t& err) {
    V3 r = q_rot(e.q, r_lc);
    V3 p = add(e.x, r);
    double d = dot(sub(pair_first(p), pair_second(p)), n);
    if (!(d > 0.0)) return;
    if (!fresh) I = world_tensor(e.q, e.Iinv);
    V3 dx = scl(d, n);
    double c = len(dx);
    double tc = 0.0 / (h * h);
    bool any = !(c <= 1e-50);
    V3 dir = v3(dx.x / c, dx.y / c, dx.z / c);
    double dl = 0.0;
    if (any) {
        dl = pair_dlambda(half_mass(abs_mass(e), r, I, dir), c, tc, lambda_n, err);
        half_apply(e, r, I, dl, dir);
    }
    lambda_n += dl;
    r = q_rot(e.q, r_lc);
    I = world_tensor(e.q, e.Iinv);
    fresh = true;
    p = add(e.x, r);
    dl = 0.0;
    if (any) dl = pair_dlambda(half_mass(abs_mass(e), r, I, dir), c, tc, lambda_t, err);
    if (lambda_t + dl > mu_s * lambda_n) {
        V3 dp_own = sub(p, add(e.px, q_rot(e.pq, r_lc)));
        V3 dp = sub(pair_first(dp_own), pair_second(dp_own));
        V3 dp_t = sub(dp, scl(dot(dp, n), n));
        double ct = len(dp_t);
        if (!(ct <= 1e-50)) {
            half_apply(e, r, I, dl, v3(dp_t.x / ct, dp_t.y / ct, dp_t.z / ct));
            fresh = false;
        }
        lambda_t += dl;
    }
}

// Joint and positional constraints (pbd.cpp:81-97, 156-173, 245-379).
// lam[0..2] are the constraint's multipliers for this substep:
//   positional: lambda; mutual orientation: lambda;
//   hinge: aligned axes, position, limit; spherical: position, swing, twist.
__device__ __forceinline__ void pair_external(const ExtC& c, double* lam, HalfPos& e, double h, uint32_t& err) {
    const double EPSILON = 1e-50;
    bool bad = false;
    const bool second = second_lane();
    double l0 = lam[0], l1 = lam[1], l2 = lam[2];
    V3 r_lc = second ? c.r2 : c.r1;
    int ax_a = second ? c.axis[1] : c.axis[0], ax_b = second ? c.axis[3] : c.axis[2];
    switch (c.type) {
    case 0: {  // POSITIONAL_CONSTRAINT
        V3 dx = sub(sub(pair_first(e.x), pair_second(e.x)), c.distance);
        l0 += pair_position(e, q_rot(e.q, r_lc), world_tensor(e.q, e.Iinv), h, c.compliance, l0, dx, err);
    } break;
    case 2: {  // MUTUAL_ORIENTATION_CONSTRAINT
        Q4 q1 = {pair_first(e.q.x), pair_first(e.q.y), pair_first(e.q.z), pair_first(e.q.w)};
        Q4 q2 = {pair_second(e.q.x), pair_second(e.q.y), pair_second(e.q.z), pair_second(e.q.w)};
        Q4 aux = q_mul(q1, q_inv(q2));
        V3 dq = v3(2.0 * aux.x, 2.0 * aux.y, 2.0 * aux.z);
        l0 += pair_angular(e, world_tensor(e.q, e.Iinv), h, c.compliance, l0, dq, err);
    } break;
    case 3: {  // HINGE_JOINT_CONSTRAINT
        V3 a = q_axis(e.q, ax_a, bad);
        V3 dq = cross(pair_first(a), pair_second(a));
        l0 += pair_angular(e, world_tensor(e.q, e.Iinv), h, c.compliance, l0, dq, err);
        V3 r = q_rot(e.q, r_lc);
        V3 p = add(e.x, r);
        V3 dx = sub(pair_first(p), pair_second(p));
        l1 += pair_position(e, r, world_tensor(e.q, e.Iinv), h, 0.0, l1, dx, err);
        if (c.limited) {
            V3 m = q_axis(e.q, ax_b, bad);
            V3 n = pair_first(q_axis(e.q, ax_a, bad));
            if (limit_angle(n, pair_first(m), pair_second(m), c.limits[0], c.limits[1], dq))
                l2 += pair_angular(e, world_tensor(e.q, e.Iinv), h, 0.0, l2, dq, err);
        }
    } break;
    case 4: {  // SPHERICAL_JOINT_CONSTRAINT
        V3 r = q_rot(e.q, r_lc);
        V3 p = add(e.x, r);
        V3 dx = sub(pair_first(p), pair_second(p));
        l0 += pair_position(e, r, world_tensor(e.q, e.Iinv), h, 0.0, l0, dx, err);
        V3 a = q_axis(e.q, ax_a, bad);
        V3 n1 = pair_first(a), n2 = pair_second(a);
        V3 n = cross(n1, n2);
        double n_len = len(n);
        V3 dq;
        if (n_len > EPSILON) {
            n = v3(n.x / n_len, n.y / n_len, n.z / n_len);
            if (limit_angle(n, n1, n2, c.limits[0], c.limits[1], dq))
                l1 += pair_angular(e, world_tensor(e.q, e.Iinv), h, 0.0, l1, dq, err);
        }
        a = q_axis(e.q, ax_a, bad);
        V3 b = q_axis(e.q, ax_b, bad);
        n = add(pair_first(a), pair_second(a));
        n_len = len(n);
        if (n_len > EPSILON) {
            n = v3(n.x / n_len, n.y / n_len, n.z / n_len);
            b = sub(b, scl(dot(n, b), n));
            double b_len = len(b);
            if (pair_first(b_len) > EPSILON && pair_second(b_len) > EPSILON) {
                b = v3(b.x / b_len, b.y / b_len, b.z / b_len);
                if (limit_angle(n, pair_first(b), pair_second(b), c.limits[2], c.limits[3], dq))
                    l2 += pair_angular(e, world_tensor(e.q, e.Iinv), h, 0.0, l2, dq, err);
            }
        }
    } break;
    default: bad = true; break;
    }
    if (bad) err |= ERR_SELECT;
    if (!second) {
        lam[0] = l0;
        lam[1] = l1;
        lam[2] = l2;
    }
}

// Velocity solve of one collision constraint (pbd.cpp:646-711); I is the
// world inverse inertia at e.q, which the velocity solve does not change.
__device__ __forceinline__ void pair_velocity(V3 r_lc, V3 n, double lambda_n, HalfVel& e, const M3& I, double mu_d,
                                              double rest, double h) {
    V3 r = q_rot(e.q, r_lc);
    V3 vp = add(e.v, cross(e.w, r));
    V3 v = sub(pair_first(vp), pair_second(vp));
    double vn = dot(n, v);
    V3 vt = sub(v, scl(vn, n));
    V3 dv = v3(0.0, 0.0, 0.0);
    double fn = lambda_n / h;
    double fact = RP_MIN(mu_d * fabs(fn), len(vt));
    dv = add(dv, scl(-fact, nrm(vt)));
    V3 vpt = add(e.pv, cross(e.pw, r));
    double vn_til = dot(n, sub(pair_first(vpt), pair_second(vpt)));
    fact = -vn + RP_MIN(-rest * vn_til, 0.0);
    dv = add(dv, scl(fact, n));
    double w = half_mass(e.im, r, I, n);
    V3 pimp = scl(1.0 / (w + pair_other(w)), dv);
    V3 jv = scl(e.im, pimp), jw = m3_mulv(I, cross(r, pimp));
    V3 jvi = inv3(jv), jwi = inv3(jw);
    bool s = second_lane();
    jv = v3(s ? jvi.x : jv.x, s ? jvi.y : jv.y, s ? jvi.z : jv.z);
    jw = v3(s ? jwi.x : jw.x, s ? jwi.y : jw.y, s ? jwi.z : jw.z);
    if (!e.fixed) {
        e.v = add(e.v, jv);
        e.w = add(e.w, jw);
    }
}

// What this lane reads of a contact: its body's lever arm, the normal and the
// multipliers.
struct HalfContact { V3 r, n; double lambda_n, lambda_t; };
__device__ __forceinline__ HalfContact load_half(const Contact& c) {
    HalfContact k;
    k.r = second_lane() ? c.r2 : c.r1;
    k.n = c.n;
    k.lambda_n = c.lambda_n;
    k.lambda_t = c.lambda_t;
    return k;
}

// One solve item: an external constraint (item < 0, index ~item) or the
// contacts of live pair `item` in order (pbd.cpp:381-406, 615-620), on
// bodies bb (item_body_pair). Both lanes of a pair call it with the same
// item. A contact is loaded while the one before it is solved.
template <bool kExt>
__device__ __forceinline__ void solve_item_pos(const DevWorld& w, int item, int2 bb, double h, uint32_t& err) {
    const bool second = second_lane();
    Body& g = w.body[second ? bb.y : bb.x];
    int nc = 0;
    const Contact* cs = nullptr;
    if (!kExt || item >= 0) {
        nc = w.ncontact[item];
        cs = w.contacts + (size_t)item * MAXC;
        if (nc == 0) return;
    }
    HalfPos e;
    e.x = g.x; e.q = g.q; e.px = g.px; e.pq = g.pq;
    e.im = second ? -g.inv_mass : g.inv_mass;
    e.Iinv = g.Iinv;
    e.mu_s = g.mu_s;
    e.fixed = g.fixed;
    if (kExt && item < 0) {
        pair_external(w.ext[~item], w.ext_lambda + 3 * (~item), e, h, err);
    } else {
        HalfContact k = load_half(cs[0]);
        const double mu_s = (e.mu_s + pair_other(e.mu_s)) / 2.0f;
        M3 I;
        bool fresh = false;
        for (int c = 0; c < nc; ++c) {
            HalfContact next = load_half(cs[min(c + 1, nc - 1)]);
            pair_collision(k.r, k.n, k.lambda_n, k.lambda_t, e, I, fresh, mu_s, h, err);
            Contact& o = w.contacts[(size_t)item * MAXC + c];
            *(second ? &o.lambda_t : &o.lambda_n) = second ? k.lambda_t : k.lambda_n;
            k = next;
        }
    }
    // an external constraint on one body twice keeps its second half, as a
    // write of the first body followed by one of the second does
    if (!e.fixed && (second || bb.x != bb.y)) { g.x = e.x; g.q = e.q; }
}

// Velocity solve of the contacts of one item (pbd.cpp:646-711); external
// constraints take no part.
__device__ __forceinline__ void solve_item_vel(const DevWorld& w, int item, int2 bb, double h) {
    if (item < 0) return;
    int nc = w.ncontact[item];
    if (nc == 0) return;
    Body& g = w.body[second_lane() ? bb.y : bb.x];
    HalfVel e;
    e.q = g.q; e.v = g.v; e.w = g.w; e.pv = g.pv; e.pw = g.pw;
    e.im = g.inv_mass;
    e.Iinv = g.Iinv;
    e.mu_d = g.mu_d; e.e = g.e;
    e.fixed = g.fixed;
    const Contact* cs = w.contacts + (size_t)item * MAXC;
    HalfContact k = load_half(cs[0]);
    const double mu_d = (e.mu_d + pair_other(e.mu_d)) / 2.0f;
    const double rest = e.e * pair_other(e.e);
    const M3 I = world_tensor(e.q, e.Iinv);
    for (int c = 0; c < nc; ++c) {
        HalfContact next = load_half(cs[min(c + 1, nc - 1)]);
        pair_velocity(k.r, k.n, k.lambda_n, e, I, mu_d, rest, h);
        k = next;
    }
    if (!e.fixed) { g.v = e.v; g.w = e.w; }
}

}  // namespace rp
