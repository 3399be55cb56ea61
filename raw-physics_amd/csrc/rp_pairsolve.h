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
    double iinv_max;  // bound on Iinv's eigenvalues; infinite unless the rotation is a unit quaternion
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

// collision_constraint_solve (pbd.cpp:107-154). `I` is the world inverse
// inertia at e.q when `fresh`: it is computed once per change of the rotation
// and not at all for a separated contact.
//
// Static friction needs the generalized masses after the normal correction,
// whose values matter only if lambda_t + dl > mu_s lambda_n, that is, with
// lambda_t <= 0, only if the masses' sum W' grew to c / (mu_s |lambda_n|), about
// W / mu_s. It hardly changes: in the body's frame the lever arm is fixed and
// the normal turns by at most the angle |a| of the correction, so by the
// triangle inequality in the tensor's norm
//     sqrt(w' - im) <= sqrt(w - im) + sqrt(iinv_max) |r| |a|,
// hence w' <= im + 1.1 (w - im) + 11 iinv_max |r|^2 |a|^2. Where that bound
// decides, the second preparation, a fifth of the contact's operations, is left
// out; its result would not be used. The margin of 1e-9 lies far above rounding
// and above what a rotation that is no unit quaternion can change: such a
// rotation moves w' by four times its norm's error, at most 4e-12 where the
// bound is used at all (solve_item_pos; normalized rotations have 1e-16).
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
    double dl = 0.0, im = abs_mass(e);
    if (any) {
        V3 u = cross(r, dir);
        double wu = dot(u, m3_mulv(I, u));
        dl = pair_dlambda(im + wu, c, tc, lambda_n, err);
        V3 imp = scl(dl, dir);
        V3 a = m3_mulv(I, cross(r, imp));
        if (!e.fixed) e.x = add(e.x, scl(e.im, imp));
        half_rotate(e, a);
        fresh = false;
        double top = im + 1.1 * wu + 11.0 * e.iinv_max * dot(r, r) * dot(a, a);
        top += pair_other(top);
        lambda_n += dl;
        if (tc == 0.0 && lambda_t <= 0.0 && lambda_n < 0.0 && top > 0.0 && mu_s >= 0.0 &&
            mu_s * -lambda_n * top <= c * (1.0 - 1e-9))
            return;
    } else {
        lambda_n += dl;
    }
    r = q_rot(e.q, r_lc);
    I = world_tensor(e.q, e.Iinv);
    fresh = true;
    p = add(e.x, r);
    dl = 0.0;
    if (any) dl = pair_dlambda(half_mass(im, r, I, dir), c, tc, lambda_t, err);
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
// Every constraint is up to three corrections in a row, each positional (along
// the difference d of the bodies' points at r) or angular (about d), so one copy
// of that code runs in a loop: written
// out per constraint type it is 130 KB of instructions, which do not fit the
// instruction cache, and a lone wave that misses it waits for every line.
__device__ __forceinline__ void pair_external(const ExtC& c, double* lam, HalfPos& e, double h, uint32_t& err) {
    const double EPSILON = 1e-50;
    bool bad = false;
    const bool second = second_lane();
    const V3 r_lc = second ? c.r2 : c.r1;
    const int ax_a = second ? c.axis[1] : c.axis[0], ax_b = second ? c.axis[3] : c.axis[2];
    const bool hinge = c.type == 3, spherical = c.type == 4;
    if (c.type < 0 || c.type == 1 || c.type > 4) bad = true;
    const int steps = bad ? 0 : spherical || (hinge && c.limited) ? 3 : hinge ? 2 : 1;
    for (int step = 0; step < steps; ++step) {
        const bool angular = hinge ? step != 1 : spherical ? step != 0 : c.type == 2;
        const double compliance = step == 0 && !spherical ? c.compliance : 0.0;
        bool apply = true;
        V3 d, r = v3(0.0, 0.0, 0.0);
        if (!angular) {
            r = q_rot(e.q, r_lc);
            V3 p = c.type == 0 ? e.x : add(e.x, r);
            d = sub(pair_first(p), pair_second(p));
            if (c.type == 0) d = sub(d, c.distance);  // POSITIONAL_CONSTRAINT
        } else if (c.type == 2) {                      // MUTUAL_ORIENTATION_CONSTRAINT
            Q4 q1 = {pair_first(e.q.x), pair_first(e.q.y), pair_first(e.q.z), pair_first(e.q.w)};
            Q4 q2 = {pair_second(e.q.x), pair_second(e.q.y), pair_second(e.q.z), pair_second(e.q.w)};
            Q4 aux = q_mul(q1, q_inv(q2));
            d = v3(2.0 * aux.x, 2.0 * aux.y, 2.0 * aux.z);
        } else {
            V3 a = q_axis(e.q, ax_a, bad);
            V3 a1 = pair_first(a), a2 = pair_second(a);
            if (step == 0) {
                d = cross(a1, a2);  // hinge: the aligned axes
            } else {
                // hinge limit: limit axes about the first body's hinge axis;
                // swing: swing axes about their normal; twist: twist axes
                // about the mean swing axis, with their parts along it removed
                const bool swing = spherical && step == 1, twist = spherical && step == 2;
                V3 n = a1, m = a;
                if (!swing) m = q_axis(e.q, ax_b, bad);
                if (spherical) {
                    n = swing ? cross(a1, a2) : add(a1, a2);
                    double n_len = len(n);
                    apply = n_len > EPSILON;
                    n = v3(n.x / n_len, n.y / n_len, n.z / n_len);
                }
                if (twist) {
                    m = sub(m, scl(dot(n, m), n));
                    double m_len = len(m);
                    apply = apply & (pair_first(m_len) > EPSILON) & (pair_second(m_len) > EPSILON);
                    m = v3(m.x / m_len, m.y / m_len, m.z / m_len);
                }
                int lim = twist ? 2 : 0;
                V3 m1 = pair_first(m), m2 = pair_second(m);
                apply = apply && limit_angle(n, m1, m2, c.limits[lim], c.limits[lim + 1], d);
            }
        }
        if (!apply) continue;
        double lambda = lam[step];
        double dl = 0.0;
        M3 I = world_tensor(e.q, e.Iinv);
        double size = len(d);
        if (!(size <= 1e-50)) {
            V3 n = v3(d.x / size, d.y / size, d.z / size);
            V3 u = cross(r, n);
            u = v3(angular ? n.x : u.x, angular ? n.y : u.y, angular ? n.z : u.z);
            double wu = dot(u, m3_mulv(I, u));
            double w = angular ? wu : abs_mass(e) + wu;
            dl = pair_dlambda(w, size, compliance / (h * h), lambda, err);
            V3 imp = scl(angular ? -dl : dl, n);
            if (!angular && !e.fixed) e.x = add(e.x, scl(e.im, imp));
            V3 t = cross(r, imp);
            half_rotate(e, m3_mulv(I, v3(angular ? imp.x : t.x, angular ? imp.y : t.y, angular ? imp.z : t.z)));
        }
        if (!second) lam[step] = lambda + dl;
    }
    if (bad) err |= ERR_SELECT;
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

// One solve item on its pair of lanes: an external constraint (code < 0,
// index ~code) or the contacts of live pair `code`, its two global bodies,
// and the first contact, loaded ahead of the solve.
struct PairItem {
    int code;
    int2 bb;
    int first;  // negative: this lane's body's first contact item
    int nc;
    HalfContact k;
};
__device__ __forceinline__ void load_item(PairItem& t, const int* order, const int2* bodies, int idx) {
    t.code = order[idx];
    int2 bb = bodies[idx];
    t.first = second_lane() ? bb.y : bb.x;
    t.bb = make_int2(bb.x & ~FIRST_CONTACT, bb.y & ~FIRST_CONTACT);
}
// The contact count and the first contact of a live pair (its slots are
// always allocated, so both loads are issued together and what an empty
// pair's slot holds is not used).
template <bool kExt>
__device__ __forceinline__ void load_item_contact(PairItem& t, const DevWorld& w) {
    t.nc = 0;
    if (kExt && t.code < 0) return;
    t.nc = w.ncontact[t.code];
    t.k = load_half(w.contacts[(size_t)t.code * MAXC]);
}

// Position solve of item t (pbd.cpp:381-406, 615-620) on the bodies at `body`
// (indexed by global body less b0). Both lanes of a pair call it with the
// same item. A contact is loaded while the one before it is solved.
template <bool kExt>
__device__ __forceinline__ void solve_item_pos(const DevWorld& w, Body* body, int b0, const PairItem& t, double h,
                                               uint32_t& err) {
    const bool second = second_lane();
    if (!(kExt && t.code < 0) && t.nc == 0) return;
    Body& g = body[(second ? t.bb.y : t.bb.x) - b0];
    HalfPos e;
    e.x = g.x; e.q = g.q; e.px = g.px; e.pq = g.pq;
    e.im = second ? -g.inv_mass : g.inv_mass;
    e.Iinv = g.Iinv;
    e.mu_s = g.mu_s;
    e.fixed = g.fixed;
    if (kExt && t.code < 0) {
        pair_external(w.ext[~t.code], w.ext_lambda + 3 * (~t.code), e, h, err);
    } else {
        const double qq = e.q.x * e.q.x + e.q.y * e.q.y + e.q.z * e.q.z + e.q.w * e.q.w;
        e.iinv_max = fabs(qq - 1.0) <= 1e-12 ? g.iinv_max : HUGE_VAL;
        HalfContact k = t.k;
        Contact* cs = w.contacts + (size_t)t.code * MAXC;
        const double mu_s = (e.mu_s + pair_other(e.mu_s)) / 2.0f;
        M3 I;
        bool fresh = false;
        for (int c = 0; c < t.nc; ++c) {
            HalfContact next = load_half(cs[min(c + 1, t.nc - 1)]);
            pair_collision(k.r, k.n, k.lambda_n, k.lambda_t, e, I, fresh, mu_s, h, err);
            *(second ? &cs[c].lambda_t : &cs[c].lambda_n) = second ? k.lambda_t : k.lambda_n;
            k = next;
        }
    }
    // an external constraint on one body twice keeps its second half, as a
    // write of the first body followed by one of the second does
    if (!e.fixed && (second || t.bb.x != t.bb.y)) { g.x = e.x; g.q = e.q; }
}

// Velocity solve of item t's contacts (pbd.cpp:646-711); external constraints
// take no part. kUpdate: a body's velocity update (pbd.cpp:623-643) goes before
// its first item's solve, whether or not that has contacts.
template <bool kUpdate>
__device__ __forceinline__ void solve_item_vel(const DevWorld& w, Body* body, int b0, const PairItem& t, double h) {
    Body& g = body[(second_lane() ? t.bb.y : t.bb.x) - b0];
    if (kUpdate && t.first < 0) velocity_update_body(g, h);
    if (t.nc == 0) return;
    HalfVel e;
    e.q = g.q; e.v = g.v; e.w = g.w; e.pv = g.pv; e.pw = g.pw;
    e.im = g.inv_mass;
    e.Iinv = g.Iinv;
    e.mu_d = g.mu_d; e.e = g.e;
    e.fixed = g.fixed;
    const Contact* cs = w.contacts + (size_t)t.code * MAXC;
    HalfContact k = t.k;
    const double mu_d = (e.mu_d + pair_other(e.mu_d)) / 2.0f;
    const double rest = e.e * pair_other(e.e);
    const M3 I = world_tensor(e.q, e.Iinv);
    for (int c = 0; c < t.nc; ++c) {
        HalfContact next = load_half(cs[min(c + 1, t.nc - 1)]);
        pair_velocity(k.r, k.n, k.lambda_n, e, I, mu_d, rest, h);
        k = next;
    }
    if (!e.fixed) { g.v = e.v; g.w = e.w; }
}

// One item of a class or list in global memory, bodies in global memory.
template <bool kExt, bool kVel>
__device__ __forceinline__ void solve_item_at(const DevWorld& w, const int* order, const int2* bodies, int idx, double h,
                                              uint32_t& err) {
    PairItem t;
    load_item(t, order, bodies, idx);
    load_item_contact<true>(t, w);
    if (kVel) solve_item_vel<false>(w, w.body, 0, t, h);
    else solve_item_pos<kExt>(w, w.body, 0, t, h, err);
}

}  // namespace rp
