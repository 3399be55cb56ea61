// rp_step.h — per-pair and per-constraint device functions of the step.
//
// Each function restates one reference routine (file:line given) with the
// same floating-point evaluation order, so that results are bit-identical
// to the reference's CPU step. Memory is bounded: where the reference grows
// heap arrays, these functions use fixed-capacity per-thread arrays and set
// an error bit if a capacity would be exceeded.
#pragma once
#include <float.h>
#include <math.h>
#include "rp_math.h"

namespace rp {

// ---------------------------------------------------------------------------
// Device data layout
// ---------------------------------------------------------------------------
template <class S> struct alignas(16) BodyT {  // one record per body (464 bytes for S = double, copied as 16-byte words)
    V3T<S> x; Q4T<S> q; V3T<S> v; V3T<S> w;      // world_position, world_rotation, velocities
    V3T<S> px; Q4T<S> pq; V3T<S> pv; V3T<S> pw;  // previous_* (entity.h:43-46)
    S deact;                                     // deactivation_time
    S inv_mass;
    M3T<S> I, Iinv;                              // local inertia tensor and its inverse
    S mu_s, mu_d, e, radius;
    V3T<S> F, T;                                 // external force / torque of the frame
    int32_t fixed, active;
    S iinv_max;                                  // bound on the eigenvalues of Iinv (inverse_inertia_bound)
};
using Body = BodyT<double>;

// A bound on the eigenvalues of an inverse inertia tensor (its largest
// absolute row sum), or infinity where it is not symmetric positive
// definite or zero, so that nothing is concluded from it.
inline double inverse_inertia_bound(const M3& A) {
    double top = 0.0;
    bool zero = true;
    for (int i = 0; i < 3; ++i) {
        double row = 0.0;
        for (int j = 0; j < 3; ++j) {
            row += fabs(A.m[i][j]);
            zero &= A.m[i][j] == 0.0;
        }
        top = row > top ? row : top;
    }
    if (zero) return 0.0;
    bool symmetric = true;
    for (int i = 0; i < 3; ++i)
        for (int j = 0; j < i; ++j) symmetric &= fabs(A.m[i][j] - A.m[j][i]) <= 1e-12 * top;
    double m2 = A.m[0][0] * A.m[1][1] - A.m[0][1] * A.m[1][0];
    double det = A.m[0][0] * (A.m[1][1] * A.m[2][2] - A.m[1][2] * A.m[2][1]) -
                 A.m[0][1] * (A.m[1][0] * A.m[2][2] - A.m[1][2] * A.m[2][0]) +
                 A.m[0][2] * (A.m[1][0] * A.m[2][1] - A.m[1][1] * A.m[2][0]);
    // (margins above the rounding of the minors)
    bool definite = A.m[0][0] > 0.0 && m2 > 1e-9 * top * top && det > 1e-9 * top * top * top;
    return symmetric && definite && top < DBL_MAX ? top : HUGE_VAL;
}

// A collision constraint as built by clipping_contact_to_collision_constraint
// (pbd.cpp:408-424) plus its multipliers.
template <class S> struct ContactT {
    V3T<S> r1, r2, n;
    S lambda_n, lambda_t;
};
using Contact = ContactT<double>;

// External constraint (Constraint, pbd.h:22-91); b1/b2 are global body indices.
struct ExtC {
    int32_t type, b1, b2, limited;
    int32_t axis[4];
    V3 r1, r2, distance;
    double compliance;
    double limits[4];
};

// Hull geometry tables, shared by all hull instances. A hull instance's
// record holds its first vertex record, first face record and first local
// face normal; a vertex record the start and count of its faces and of its
// neighbours in `list`; a face record the start and count of its elements in
// `list` and of its neighbour faces in `nbr` (face, first element).
struct HullTables {
    const int4* hull;   // (vertex records, face records, normals, first local vertex)
    const int4* rec;
    const int32_t* list;
    const int2* nbr;
    const V3* fn;       // local face normals
    const M4* model;    // model matrices of the bodies
};

// One hull at the current substep: its transformed vertices, its instance and
// its body. Face normals are transformed when first needed, with the
// reference's arithmetic (collider.cpp:426-428), so that only the few faces
// the manifold visits are computed.
struct HullView {
    const V3* tv;
    int nv, hid, body;
};
// What the contact manifold reads of a hull beside its vertices.
struct HullFaces {
    const V3* fn;
    const int4 *vrec, *frec;
    M3 R;  // upper-left 3x3 of the model matrix T*R (util.cpp:60-74)
};
RP_HD M3 model_rotation(const HullTables& T, int body) {
    M3 R;
    const M4& M = T.model[body];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) R.m[i][j] = M.m[i][j];
    return R;
}
RP_HD HullFaces hull_faces(const HullTables& T, const HullView& h) {
    HullFaces f;
    int4 r = T.hull[h.hid];
    f.vrec = T.rec + r.x;
    f.frec = T.rec + r.y;
    f.fn = T.fn + r.z;
    f.R = model_rotation(T, h.body);
    return f;
}

// A collider of a body with more than one collider or a sphere (the general
// narrow-phase path): a hull view, or a sphere whose center is the body
// position (collider.cpp:431-433) with an r32 radius (collider.h:29).
enum { COL_HULL = 0, COL_SPHERE = 1 };
struct ColView {
    int type;
    HullView h;
    V3 center;
    float radius;
};

// gm_mat4_multiply_vec3(M, n, false) then normalize (collider.cpp:426-428)
RP_HD V3 face_normal_world(const M3& M, V3 n) {
    V3 r = v3(M.m[0][0] * n.x + M.m[0][1] * n.y + M.m[0][2] * n.z, M.m[1][0] * n.x + M.m[1][1] * n.y + M.m[1][2] * n.z,
              M.m[2][0] * n.x + M.m[2][1] * n.y + M.m[2][2] * n.z);
    return nrm(r);
}

enum : uint32_t {
    ERR_GJK_SIMPLEX = 1u << 0,
    ERR_EPA_DEGENERATE = 1u << 1,
    ERR_SUPPORT_NAN = 1u << 2,
    ERR_SKEW_LINES = 1u << 3,
    ERR_ACTIVITY = 1u << 4,
    ERR_HULL = 1u << 5,
    ERR_ZERO_MASS = 1u << 6,
    ERR_SELECT = 1u << 7,
    ERR_EPA_CAPACITY = 1u << 8,
    ERR_CLIP_CAPACITY = 1u << 9,
    ERR_CONTACT_CAPACITY = 1u << 10,
    ERR_SOLVER_CAPACITY = 1u << 11,
    ERR_PAIR_CAPACITY = 1u << 12,
    ERR_ADJOINT_SCOPE = 1u << 13,
};

constexpr int EPA_MAXV = 104;  // 4 simplex points + at most 100 expansions (epa.cpp:149)
constexpr int EPA_MAXF = 256;
constexpr int EPA_MAXE = 128;
constexpr int CLIP_MAX = 64;
constexpr int MAXC = 16;       // contacts kept per body pair
// Index of a first-maximum / first-minimum search that has found nothing:
// larger than every real index, so "ties to the lower index" also prefers
// a lane that found something (its value is then strictly better, since
// the search starts from the most extreme finite value).
constexpr int NO_SEL = 0x7fffffff;

// t ? a : b by component (selects of values, not of addresses).
RP_HD V3 pick(bool t, V3 a, V3 b) { return v3(t ? a.x : b.x, t ? a.y : b.y, t ? a.z : b.z); }

// ---------------------------------------------------------------------------
// Support mapping (support.cpp:5-39): first index wins on ties
// ---------------------------------------------------------------------------
// G = 1: one lane searches all vertices; they are loaded eight at a time so
// that their memory latencies overlap, and compared in index order.
// G > 1: the G lanes of an aligned group (one body pair per group) each scan
// every G-th vertex, then reduce (larger dot wins, ties to the lower index),
// which selects exactly the first maximum of the sequential scan; every lane
// of the group returns the same index.

// Lane exchanges inside a row of 16 lanes (DPP): partner = lane ^ 1, lane ^ 2
// (quad permutations), 7 - lane within 8 (half mirror), 15 - lane (mirror).
enum : int { DPP_XOR1 = 0xB1, DPP_XOR2 = 0x4E, DPP_HALF_MIRROR = 0x141, DPP_MIRROR = 0x140 };
template <int CTRL> __device__ __forceinline__ int dpp_int(int v) {
    return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xF, 0xF, true);
}
template <int CTRL> __device__ __forceinline__ double dpp_double(double v) {
    long long b = __double_as_longlong(v);
    int lo = dpp_int<CTRL>((int)b), hi = dpp_int<CTRL>((int)(b >> 32));
    return __longlong_as_double((long long)(unsigned)lo | ((long long)hi << 32));
}
// First maximum / minimum over the G lanes of the group (G = 4, 8 or 16) of
// (value, index): the larger (smaller) value, ties to the lower index. The
// values are reduced first, then the lowest index among the lanes that hold
// the result: 15 + 5 instructions for 8 lanes where carrying the index
// through every step took 33. A lane that has found nothing holds the most
// extreme finite value and NO_SEL; a lane that has found something holds a
// strictly better value.
// Written as selects, so that it compiles to compares and v_cndmask.
template <int CTRL, bool kMax> __device__ __forceinline__ void extreme_step(double& m) {
    double om = dpp_double<CTRL>(m);
    bool take = kMax ? om > m : om < m;
    m = take ? om : m;
}
template <int G> __device__ __forceinline__ int group_min(int v);
template <int G, bool kMax> __device__ __forceinline__ void group_extreme(double& m) {
    static_assert(G == 4 || G == 8 || G == 16, "lane groups of 4, 8 or 16");
    extreme_step<DPP_XOR1, kMax>(m);
    extreme_step<DPP_XOR2, kMax>(m);
    if constexpr (G >= 8) extreme_step<DPP_HALF_MIRROR, kMax>(m);
    if constexpr (G >= 16) extreme_step<DPP_MIRROR, kMax>(m);
}
template <int G> __device__ __forceinline__ void group_argmax(double& m, int& sel) {
    double own = m;
    group_extreme<G, true>(m);
    sel = group_min<G>(own == m ? sel : NO_SEL);
}
template <int G> __device__ __forceinline__ void group_argmin(double& m, int& sel) {
    double own = m;
    group_extreme<G, false>(m);
    sel = group_min<G>(own == m ? sel : NO_SEL);
}
// Two independent first maxima, their steps interleaved so that the two
// dependency chains overlap.
template <int G> __device__ __forceinline__ void group_argmax2(double& m1, int& s1, double& m2, int& s2) {
    double o1 = m1, o2 = m2;
    extreme_step<DPP_XOR1, true>(m1);
    extreme_step<DPP_XOR1, true>(m2);
    extreme_step<DPP_XOR2, true>(m1);
    extreme_step<DPP_XOR2, true>(m2);
    if constexpr (G >= 8) {
        extreme_step<DPP_HALF_MIRROR, true>(m1);
        extreme_step<DPP_HALF_MIRROR, true>(m2);
    }
    if constexpr (G >= 16) {
        extreme_step<DPP_MIRROR, true>(m1);
        extreme_step<DPP_MIRROR, true>(m2);
    }
    s1 = group_min<G>(o1 == m1 ? s1 : NO_SEL);
    s2 = group_min<G>(o2 == m2 ? s2 : NO_SEL);
}

// A lane's share of a hull in a support scan over G lanes: vertices gl,
// gl + G, ... of `steps`. The last step of a lane past the hull's end reads
// vertex 0 instead, whose dot lane 0 holds too under the lower index, so no
// step needs a mask. (Scanning both hulls in one loop of masked batches of
// four cost a box against a 42-vertex hull 16 evaluations instead of 7: GJK
// took 34 900 cycles per pair, now 26 600, and the narrow launch of 4096
// scenes of 16 bodies 156 -> 135 us.)
constexpr int SCAN_BATCH = 5;  // vertices loaded before any is compared
template <int G> struct ScanShare {
    const V3 *first, *last;
    int full;  // steps before the last
};
template <int G> RP_HD ScanShare<G> scan_share(const HullView& h) {
    int gl = (int)(__lane_id() & (G - 1));
    ScanShare<G> s;
    s.full = (h.nv - 1) / G;
    int j = gl + s.full * G;
    s.first = h.tv + gl;
    s.last = h.tv + (j < h.nv ? j : 0);
    return s;
}
template <int G> RP_HD void scan_full(const ScanShare<G>& s, V3 d, double& m, int& sel) {
    const V3* p = s.first;
    int k = 0;
    for (; k + SCAN_BATCH <= s.full; k += SCAN_BATCH, p += SCAN_BATCH * G) {
        V3 v[SCAN_BATCH];
#pragma unroll
        for (int i = 0; i < SCAN_BATCH; ++i) v[i] = p[i * G];
#pragma unroll
        for (int i = 0; i < SCAN_BATCH; ++i) {
            double dd = dot(v[i], d);
            bool t = dd > m;
            m = t ? dd : m;
            sel = t ? k + i : sel;
        }
    }
    for (; k < s.full; ++k, p += G) {
        double dd = dot(*p, d);
        bool t = dd > m;
        m = t ? dd : m;
        sel = t ? k : sel;
    }
}
// The lane's best (dot, vertex index); NO_SEL where no dot exceeds -DBL_MAX.
template <int G> RP_HD void scan_lane(const ScanShare<G>& s, V3 last, V3 d, double& m, int& sel) {
    m = -DBL_MAX;
    sel = NO_SEL;
    scan_full<G>(s, d, m, sel);
    double dd = dot(last, d);
    bool t = dd > m;
    m = t ? dd : m;
    sel = t ? s.full : sel;
    int gl = (int)(__lane_id() & (G - 1));
    sel = sel == NO_SEL ? NO_SEL : sel * G + gl;
}

template <int G = 1>
RP_HD int support_index(const HullView& h, V3 d, uint32_t& err) {
    int sel = NO_SEL;
    double max_dot = -DBL_MAX;
    if constexpr (G == 1) {
        int i = 0;
        for (; i + 8 <= h.nv; i += 8) {
            V3 v[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) v[k] = h.tv[i + k];
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                double dd = dot(v[k], d);
                if (dd > max_dot) { sel = i + k; max_dot = dd; }
            }
        }
        for (; i < h.nv; ++i) {
            double dd = dot(h.tv[i], d);
            if (dd > max_dot) { sel = i; max_dot = dd; }
        }
    } else {
        ScanShare<G> s = scan_share<G>(h);
        scan_lane<G>(s, *s.last, d, max_dot, sel);
        group_argmax<G>(max_dot, sel);
    }
    if (sel == NO_SEL) { err |= ERR_SUPPORT_NAN; sel = 0; }
    return sel;
}
// Support indices of two hulls in directions d1 and d2 at once: the two
// scans advance together (eight vertices of each hull per batch for G = 1,
// one vertex of each per lane and step for G > 1) so that their memory
// latencies overlap; each scan keeps its own first-maximum order, and for
// G > 1 the two group reductions run side by side.
template <int G = 1>
RP_HD void support_index2(const HullView& a, V3 d1, const HullView& b, V3 d2, int& i1, int& i2, uint32_t& err) {
    int s1 = NO_SEL, s2 = NO_SEL;
    double m1 = -DBL_MAX, m2 = -DBL_MAX;
    if constexpr (G == 1) {
        int n = a.nv > b.nv ? a.nv : b.nv;
        for (int i = 0; i < n; i += 8) {
            V3 va[8], vb[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                if (i + k < a.nv) va[k] = a.tv[i + k];
                if (i + k < b.nv) vb[k] = b.tv[i + k];
            }
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                if (i + k < a.nv) {
                    double dd = dot(va[k], d1);
                    if (dd > m1) { s1 = i + k; m1 = dd; }
                }
                if (i + k < b.nv) {
                    double dd = dot(vb[k], d2);
                    if (dd > m2) { s2 = i + k; m2 = dd; }
                }
            }
        }
    } else {
        // a lane visits its vertices gl, gl + G, ... in order, each hull as
        // many as it has (a box against a large hull costs the box one step)
        ScanShare<G> sa = scan_share<G>(a), sb = scan_share<G>(b);
        V3 la = *sa.last, lb = *sb.last;
        scan_lane<G>(sa, la, d1, m1, s1);
        scan_lane<G>(sb, lb, d2, m2, s2);
        group_argmax2<G>(m1, s1, m2, s2);
    }
    if (s1 == NO_SEL) { err |= ERR_SUPPORT_NAN; s1 = 0; }
    if (s2 == NO_SEL) { err |= ERR_SUPPORT_NAN; s2 = 0; }
    i1 = s1;
    i2 = s2;
}

template <int G = 1>
RP_HD V3 support_md(const HullView& a, const HullView& b, V3 d, uint32_t& err) {
    int i1, i2;
    support_index2<G>(a, d, b, scl(-1.0, d), i1, i2, err);
    return sub(a.tv[i1], b.tv[i2]);
}

// support_point of one collider (support.cpp:19-31).
template <int G = 1>
RP_HD V3 support_point(const ColView& c, V3 d, uint32_t& err) {
    if (c.type == COL_SPHERE) return add(c.center, scl((double)c.radius, nrm(d)));
    return c.h.tv[support_index<G>(c.h, d, err)];
}
// support_point_of_minkowski_difference (support.cpp:34-39)
template <int G = 1>
RP_HD V3 support_md(const ColView& a, const ColView& b, V3 d, uint32_t& err) {
    V3 s1 = support_point<G>(a, d, err);
    V3 s2 = support_point<G>(b, scl(-1.0, d), err);
    return sub(s1, s2);
}

// ---------------------------------------------------------------------------
// GJK (gjk.cpp:7-379)
// ---------------------------------------------------------------------------
struct Simplex { V3 a, b, c, d; int num; };

RP_HD V3 triple_cross(V3 a, V3 b, V3 c) { return cross(cross(a, b), c); }

// gjk.cpp:36-55
RP_HD void do_simplex_2(Simplex& s, V3& dir) {
    V3 a = s.a, b = s.b;
    V3 ao = inv3(a), ab = sub(b, a);
    if (dot(ab, ao) >= 0.0) { s.a = a; s.b = b; s.num = 2; dir = triple_cross(ab, ao, ab); }
    else { s.a = a; s.num = 1; dir = ao; }
}
// gjk.cpp:57-120 ("A region" keeps num, gjk.cpp:81-85,95-98)
RP_HD void do_simplex_3(Simplex& s, V3& dir) {
    V3 a = s.a, b = s.b, c = s.c;
    V3 ao = inv3(a), ab = sub(b, a), ac = sub(c, a), abc = cross(ab, ac);
    if (dot(cross(abc, ac), ao) >= 0.0) {
        if (dot(ac, ao) >= 0.0) { s.a = a; s.b = c; s.num = 2; dir = triple_cross(ac, ao, ac); }
        else if (dot(ab, ao) >= 0.0) { s.a = a; s.b = b; s.num = 2; dir = triple_cross(ab, ao, ab); }
        else { s.a = a; dir = ao; }
    } else {
        if (dot(cross(ab, abc), ao) >= 0.0) {
            if (dot(ab, ao) >= 0.0) { s.a = a; s.b = b; s.num = 2; dir = triple_cross(ab, ao, ab); }
            else { s.a = a; dir = ao; }
        } else if (dot(abc, ao) >= 0.0) { s.a = a; s.b = b; s.c = c; s.num = 3; dir = abc; }
        else { s.a = a; s.b = c; s.c = b; s.num = 3; dir = inv3(abc); }
    }
}
// gjk.cpp:122-337 (the ACD/AC branch uses ab, gjk.cpp:213)
RP_HD bool do_simplex_4(Simplex& s, V3& dir) {
    V3 a = s.a, b = s.b, c = s.c, d = s.d;
    V3 ao = inv3(a), ab = sub(b, a), ac = sub(c, a), ad = sub(d, a);
    V3 abc = cross(ab, ac), acd = cross(ac, ad), adb = cross(ad, ab);
    unsigned pi = 0;
    if (dot(abc, ao) >= 0.0) pi |= 1;
    if (dot(acd, ao) >= 0.0) pi |= 2;
    if (dot(adb, ao) >= 0.0) pi |= 4;
    switch (pi) {
    case 0: return true;
    case 1:
        if (dot(cross(abc, ac), ao) >= 0.0) {
            if (dot(ac, ao) >= 0.0) { s.a = a; s.b = c; s.num = 2; dir = triple_cross(ac, ao, ac); }
            else if (dot(ab, ao) >= 0.0) { s.a = a; s.b = b; s.num = 2; dir = triple_cross(ab, ao, ab); }
            else { s.a = a; dir = ao; }
        } else {
            if (dot(cross(ab, abc), ao) >= 0.0) {
                if (dot(ab, ao) >= 0.0) { s.a = a; s.b = b; s.num = 2; dir = triple_cross(ab, ao, ab); }
                else { s.a = a; dir = ao; }
            } else { s.a = a; s.b = b; s.c = c; s.num = 3; dir = abc; }
        }
        break;
    case 2:
        if (dot(cross(acd, ad), ao) >= 0.0) {
            if (dot(ad, ao) >= 0.0) { s.a = a; s.b = d; s.num = 2; dir = triple_cross(ad, ao, ad); }
            else if (dot(ac, ao) >= 0.0) { s.a = a; s.b = c; s.num = 2; dir = triple_cross(ab, ao, ab); }
            else { s.a = a; dir = ao; }
        } else {
            if (dot(cross(ac, acd), ao) >= 0.0) {
                if (dot(ac, ao) >= 0.0) { s.a = a; s.b = c; s.num = 2; dir = triple_cross(ac, ao, ac); }
                else { s.a = a; dir = ao; }
            } else { s.a = a; s.b = c; s.c = d; s.num = 3; dir = acd; }
        }
        break;
    case 3:
        if (dot(ac, ao) >= 0.0) { s.a = a; s.b = c; s.num = 2; dir = triple_cross(ac, ao, ac); }
        else { s.a = a; s.num = 1; dir = ao; }
        break;
    case 4:
        if (dot(cross(adb, ab), ao) >= 0.0) {
            if (dot(ab, ao) >= 0.0) { s.a = a; s.b = b; s.num = 2; dir = triple_cross(ab, ao, ab); }
            else if (dot(ad, ao) >= 0.0) { s.a = a; s.b = d; s.num = 2; dir = triple_cross(ad, ao, ad); }
            else { s.a = a; dir = ao; }
        } else {
            if (dot(cross(ad, adb), ao) >= 0.0) {
                if (dot(ad, ao) >= 0.0) { s.a = a; s.b = d; s.num = 2; dir = triple_cross(ad, ao, ad); }
                else { s.a = a; dir = ao; }
            } else { s.a = a; s.b = d; s.c = b; s.num = 3; dir = adb; }
        }
        break;
    case 5:
        if (dot(ab, ao) >= 0.0) { s.a = a; s.b = b; s.num = 2; dir = triple_cross(ab, ao, ab); }
        else { s.a = a; s.num = 1; dir = ao; }
        break;
    case 6:
        if (dot(ad, ao) >= 0.0) { s.a = a; s.b = d; s.num = 2; dir = triple_cross(ad, ao, ad); }
        else { s.a = a; s.num = 1; dir = ao; }
        break;
    case 7: s.a = a; s.num = 1; dir = ao; break;
    }
    return false;
}

RP_HD bool same_bits(V3 a, V3 b) {
    return __double_as_longlong(a.x) == __double_as_longlong(b.x) &&
           __double_as_longlong(a.y) == __double_as_longlong(b.y) &&
           __double_as_longlong(a.z) == __double_as_longlong(b.z);
}
RP_HD bool same_state(const Simplex& s, V3 dir, const Simplex& t, V3 tdir) {
    // most runs differ in the direction's first component alone
    if (__double_as_longlong(dir.x) != __double_as_longlong(tdir.x)) return false;
    return s.num == t.num && same_bits(dir, tdir) && same_bits(s.a, t.a) && same_bits(s.b, t.b) &&
           same_bits(s.c, t.c) && same_bits(s.d, t.d);
}

// gjk_collides (gjk.cpp:350-379).
// Early exit on a repeated state, with the same result as the full loop: the
// loop state (simplex, its count and the search direction) determines the
// rest of the loop, and it takes values in a finite set (support points are
// differences of hull vertices, the direction a function of the simplex). A
// run that neither separates nor encloses the origin therefore cycles until
// its 100th iteration and returns false. Brent's method finds the cycle: the
// state is saved at iterations 1, 2, 4, 8, ... and compared bit for bit with
// every later state; a match means the iterations since the save returned
// nothing and would repeat until the limit (their error bits are already
// set), so false is returned at once. `cycled` is set when this happens.
template <int G = 1, class View = HullView>
RP_HD bool gjk(const View& h1, const View& h2, Simplex& s, uint32_t& err, bool& cycled) {
    s.a = support_md<G>(h1, h2, v3(0.0, 0.0, 1.0), err);
    s.b = s.c = s.d = v3(0.0, 0.0, 0.0);
    s.num = 1;
    V3 dir = scl(-1.0, s.a);
    Simplex saved = s;
    V3 saved_dir = dir;
    int power = 1, lam = 0;
    for (int i = 0; i < 100; ++i) {
        if (lam == power) {
            saved = s;
            saved_dir = dir;
            power <<= 1;
            lam = 0;
        }
        ++lam;
        if (i > 0 && same_state(s, dir, saved, saved_dir) && lam > 1) {
            cycled = true;
            return false;
        }
        V3 p = support_md<G>(h1, h2, dir, err);
        if (dot(p, dir) < 0.0) return false;
        // add_to_simplex (gjk.cpp:7-30); num == 4 is an assert in the reference
        switch (s.num) {
        case 1: s.b = s.a; s.a = p; break;
        case 2: s.c = s.b; s.b = s.a; s.a = p; break;
        case 3: s.d = s.c; s.c = s.b; s.b = s.a; s.a = p; break;
        default: err |= ERR_GJK_SIMPLEX; return false;
        }
        ++s.num;
        bool hit = false;
        if (s.num == 2) do_simplex_2(s, dir);
        else if (s.num == 3) do_simplex_3(s, dir);
        else hit = do_simplex_4(s, dir);
        if (hit) return true;
    }
    return false;
}

// ---------------------------------------------------------------------------
// EPA (epa.cpp:8-237)
// ---------------------------------------------------------------------------
struct I3 { int32_t x, y, z; };

// get_face_normal_and_distance_to_origin (epa.cpp:32-77) of the triangle
// a, b, c; `point(i)` is point i of the polytope's np.
template <class Point>
RP_HD bool epa_face(V3 a, V3 b, V3 c, Point point, int np, V3& n_out, double& d_out) {
    V3 n = nrm(cross(sub(b, a), sub(c, a)));
    if (is_zero(n)) return false;
    const double TOL = 0.0;
    double d = dot(n, a);
    if (d < -TOL) {
        n = inv3(n);
        d = -d;
    } else if (d >= -TOL && d <= TOL) {
        bool found = false;
        for (int i = 0; i < np; ++i) {
            double ad = dot(n, point(i));
            if (ad < -TOL || ad > TOL) {
                n = ad < -TOL ? n : inv3(n);
                found = true;
                break;
            }
        }
        if (!found) return false;
    }
    n_out = n;
    d_out = d;
    return true;
}
RP_HD bool epa_face(I3 f, const V3* poly, int np, V3& n_out, double& d_out) {
    return epa_face(poly[f.x], poly[f.y], poly[f.z], [&](int i) { return poly[i]; }, np, n_out, d_out);
}

// The EPA polytope (epa.cpp:118-237) over caller-owned arrays (separate
// locals, so that the compiler can overlap their scratch with later phases).
struct EpaPoly {
    V3* poly;      // [EPA_MAXV]
    I3* faces;     // [EPA_MAXF]
    V3* normals;   // [EPA_MAXF]
    double* dist;  // [EPA_MAXF]
    int2* edges;   // [EPA_MAXE]
    int np, nf, ne;
    V3 min_n;
    double min_d;

    // The simplex's four faces and the closest one; false on a degenerate face.
    RP_HD bool init(const Simplex& s, uint32_t& err) {
        np = 4; nf = 4; ne = 0;
        poly[0] = s.a; poly[1] = s.b; poly[2] = s.c; poly[3] = s.d;
        faces[0] = {0, 1, 2}; faces[1] = {0, 2, 3}; faces[2] = {0, 3, 1}; faces[3] = {1, 2, 3};
        min_n = v3(0.0, 0.0, 0.0);
        min_d = DBL_MAX;
        for (int i = 0; i < nf; ++i) {
            V3 n; double d;
            if (!epa_face(faces[i], poly, np, n, d)) { err |= ERR_EPA_DEGENERATE; return false; }
            normals[i] = n;
            dist[i] = d;
            if (d < min_d) { min_d = d; min_n = n; }
        }
        return true;
    }
    // add_edge (epa.cpp:79-110): an edge equal to a listed one, by index or
    // by position, cancels it (swap-remove), else it is appended; false when
    // the list is full.
    RP_HD bool add_edge(int2 e, uint32_t& err) {
        for (int j = 0; j < ne; ++j) {
            int2 cur = edges[j];
            bool hit = (e.x == cur.x && e.y == cur.y) || (e.x == cur.y && e.y == cur.x);
            if (!hit) {
                V3 c1 = poly[cur.x], c2 = poly[cur.y], e1 = poly[e.x], e2 = poly[e.y];
                hit = (veq(c1, e1) && veq(c2, e2)) || (veq(c1, e2) && veq(c2, e1));
            }
            if (hit) {
                --ne;
                edges[j] = edges[ne];
                return true;
            }
        }
        if (ne == EPA_MAXE) { err |= ERR_EPA_CAPACITY; return false; }
        edges[ne++] = e;
        return true;
    }
    // One iteration with the support point sp in direction min_n:
    // 1 = converged (n_out, pen_out set), 2 = expanded, -1 = error.
    RP_HD int step(V3 sp, V3& n_out, double& pen_out, uint32_t& err) {
        double d = dot(min_n, sp);
        if (fabs(d - min_d) < 0.0001) {
            n_out = min_n;
            pen_out = min_d;
            return 1;
        }
        int new_idx = np;
        poly[np++] = sp;
        for (int i = 0; i < nf; ++i) {
            V3 n = normals[i];
            I3 f = faces[i];
            // triangle_centroid (epa.cpp:112-116)
            V3 c = scl(1.0 / 3.0, add(add(poly[f.y], poly[f.z]), poly[f.x]));
            if (dot(n, sub(sp, c)) > 0.0) {
                if (!add_edge(make_int2(f.x, f.y), err) || !add_edge(make_int2(f.y, f.z), err) ||
                    !add_edge(make_int2(f.z, f.x), err))
                    return -1;
                // swap-remove faces / distances / normals together (epa.cpp:191-195)
                --nf;
                faces[i] = faces[nf];
                dist[i] = dist[nf];
                normals[i] = normals[nf];
                --i;
            }
        }
        for (int i = 0; i < ne; ++i) {
            if (nf == EPA_MAXF) { err |= ERR_EPA_CAPACITY; return -1; }
            I3 f = {edges[i].x, edges[i].y, new_idx};
            faces[nf] = f;
            V3 n; double fd;
            if (!epa_face(f, poly, np, n, fd)) { err |= ERR_EPA_DEGENERATE; return -1; }
            normals[nf] = n;
            dist[nf] = fd;
            ++nf;
        }
        // first minimum: selects over the distances, then one normal load
        min_d = DBL_MAX;
        int mi = -1;
        for (int i = 0; i < nf; ++i) {
            double di = dist[i];
            bool t = di < min_d;
            min_d = t ? di : min_d;
            mi = t ? i : mi;
        }
        if (mi >= 0) min_n = normals[mi];
        ne = 0;
        return 2;
    }
};

// Orders the memory accesses of a lane group (one wave): writes before the
// call are seen by the group's reads after it.
__device__ __forceinline__ void group_mem_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// Lane exchanges of a lane group by DPP moves (register to register, no LDS
// round trip): the group's lanes all take part (control flow is uniform per
// group), and a group of 4, 8 or 16 lanes never spans two 16-lane rows.
enum : int { DPP_QUAD_BCAST0 = 0x00, DPP_QUAD_BCAST3 = 0xFF, DPP_ROW_SHR0 = 0x110 };
// Value of lane 0 of the caller's aligned group of G lanes: each quad takes
// its first lane's value, then the upper quad (and the upper half of a
// 16-lane group) takes the mirrored lane's, which holds lane 0's by then.
template <int G> __device__ __forceinline__ int group_bcast(int v) {
    static_assert(G == 4 || G == 8 || G == 16, "lane groups of 4, 8 or 16");
    int gl = (int)(__lane_id() & (G - 1));
    v = dpp_int<DPP_QUAD_BCAST0>(v);
    if constexpr (G >= 8) { int m = dpp_int<DPP_HALF_MIRROR>(v); v = (gl & 4) ? m : v; }
    if constexpr (G >= 16) { int m = dpp_int<DPP_MIRROR>(v); v = (gl & 8) ? m : v; }
    return v;
}
// Value of the last lane (G - 1) of the caller's group, the same way.
template <int G> __device__ __forceinline__ int group_bcast_last(int v) {
    static_assert(G == 4 || G == 8 || G == 16, "lane groups of 4, 8 or 16");
    int gl = (int)(__lane_id() & (G - 1));
    v = dpp_int<DPP_QUAD_BCAST3>(v);
    if constexpr (G >= 8) { int m = dpp_int<DPP_HALF_MIRROR>(v); v = (gl & 4) ? v : m; }
    if constexpr (G >= 16) { int m = dpp_int<DPP_MIRROR>(v); v = (gl & 8) ? v : m; }
    return v;
}
// Minimum over the group's lanes (every lane gets it).
template <int G> __device__ __forceinline__ int group_min(int v) {
    static_assert(G == 4 || G == 8 || G == 16, "lane groups of 4, 8 or 16");
    v = min(v, dpp_int<DPP_XOR1>(v));
    v = min(v, dpp_int<DPP_XOR2>(v));
    if constexpr (G >= 8) v = min(v, dpp_int<DPP_HALF_MIRROR>(v));
    if constexpr (G >= 16) v = min(v, dpp_int<DPP_MIRROR>(v));
    return v;
}

// Working memory of the first lane of a lane group (G > 1): the EPA polytope,
// then (reusing it) the clipping polygons. A slice of
// a device buffer, one per group, so that one lane's arrays are contiguous
// (private arrays are interleaved across the 64 lanes of a wave, and a lane
// that works alone would touch a cache line per element).
constexpr size_t EPA_BYTES = sizeof(V3) * EPA_MAXV + sizeof(V3) * EPA_MAXF + sizeof(double) * EPA_MAXF +
                             sizeof(int2) * EPA_MAXE + sizeof(I3) * EPA_MAXF;
constexpr size_t CLIP_BYTES = 2 * sizeof(V3) * CLIP_MAX;
constexpr size_t GROUP_WORK_BYTES = ((EPA_BYTES > CLIP_BYTES ? EPA_BYTES : CLIP_BYTES) + 255) / 256 * 256;
RP_HD void epa_bind(EpaPoly& P, char* m) {
    P.poly = (V3*)m;
    m += sizeof(V3) * EPA_MAXV;
    P.normals = (V3*)m;
    m += sizeof(V3) * EPA_MAXF;
    P.dist = (double*)m;
    m += sizeof(double) * EPA_MAXF;
    P.edges = (int2*)m;
    m += sizeof(int2) * EPA_MAXE;
    P.faces = (I3*)m;
}

// Visibility flags of up to EPA_MAXF = 256 faces in four words.
struct FaceBits {
    unsigned long long w0 = 0, w1 = 0, w2 = 0, w3 = 0;
    __device__ bool get(int i) const {
        unsigned long long w = i < 64 ? w0 : i < 128 ? w1 : i < 192 ? w2 : w3;
        return (w >> (i & 63)) & 1ull;
    }
    __device__ void put(int i, bool v) {
        unsigned long long b = 1ull << (i & 63);
        int k = i >> 6;
        if (k == 0) w0 = v ? (w0 | b) : (w0 & ~b);
        else if (k == 1) w1 = v ? (w1 | b) : (w1 & ~b);
        else if (k == 2) w2 = v ? (w2 | b) : (w2 & ~b);
        else w3 = v ? (w3 | b) : (w3 & ~b);
    }
    __device__ void or_bits(int c0, unsigned long long m) {  // c0 a multiple of the group size
        unsigned long long b = m << (c0 & 63);
        int k = c0 >> 6;
        w0 |= k == 0 ? b : 0ull;
        w1 |= k == 1 ? b : 0ull;
        w2 |= k == 2 ? b : 0ull;
        w3 |= k == 3 ? b : 0ull;
    }
    // lowest set flag (EPA_MAXF if none)
    __device__ int first() const {
        return w0 ? __ffsll((long long)w0) - 1 : w1 ? 63 + __ffsll((long long)w1) : w2 ? 127 + __ffsll((long long)w2)
                 : w3 ? 191 + __ffsll((long long)w3) : EPA_MAXF;
    }
};

// The polytope of a lane group: in the free end of the pair's LDS slice, or
// in the group's working memory (the pointers are generic: one copy of the
// code serves both). Faces and edges hold their point indices in bytes.
struct GroupPoly {
    V3 *poly, *normals;
    double* dist;
    uint32_t *faces, *edges;
    int max_v, max_f, max_e;
    __device__ void bind(char* m, int v, int f, int e) {
        max_v = v; max_f = f; max_e = e;
        poly = (V3*)m;
        normals = poly + v;
        dist = (double*)(normals + f);
        faces = (uint32_t*)(dist + f);
        edges = faces + f;
    }
};
constexpr int GROUP_POLY_FACE_BYTES = sizeof(V3) / 2 + sizeof(V3) + sizeof(double) + 2 * sizeof(uint32_t);

// epa for a lane group (G > 1), with the results of EpaPoly::step. The
// simplex's four faces are computed side by side, one per lane, in
// registers: nine of ten resting contacts converge on the first support
// point (a pile of 16 bodies: 90 % without an expansion, 99 % with one), and
// these touch no memory but the staged hulls. (Lane 0 used to build the four
// faces one after another in the group's working memory, about 20 000 cycles
// per pair; now 3 700. Narrow launch: 4096 scenes of 16 bodies 200 -> 193 us,
// 150 uneven scenes 243 -> 214, 500 chains of 6 links 181 -> 143.)
//
// At the first expansion the polytope moves to memory: to `spare` (LDS) while
// it fits there, then to `work`. The lanes test which faces see the support
// point, look an edge up in the edge list, compute the new faces' normals and
// distances, and search the closest face (first minimum); faces are removed
// and edges listed in the sequential order (epa.cpp:165-195). Links that
// overlap deeply take 2 to 6 expansions, a sphere more. (Lane 0 used to keep
// the edge and face lists in the working memory alone, comparing positions
// with every edge: 500 chains of 6 links 131 -> 85 us per narrow launch, 150
// uneven scenes 193 -> 163.) Every lane returns
// the status and the result; the EPA error bits are lane 0's.
template <int G, class View>
__device__ int epa_group(const View& h1, const View& h2, const Simplex& s, V3& n_out, double& pen_out, uint32_t& err,
                         char* work, V3* spare, int spare_n) {
    const int gl = (int)(__lane_id() & (G - 1));
    const bool leader = gl == 0;
    const int gbase = (int)__lane_id() & ~(G - 1);
    auto group_ballot = [&](bool v) { return (__ballot(v) >> gbase) & ((1ull << G) - 1ull); };
    // lane i (and i + 4, ...): face i of 012, 023, 031, 123
    const int fi = gl & 3;
    const I3 f0 = {fi == 3 ? 1 : 0, fi == 0 ? 1 : fi == 2 ? 3 : 2, fi == 0 ? 2 : fi == 2 ? 1 : 3};
    const V3 sa = s.a, sb = s.b, sc = s.c, sd = s.d;
    auto corner = [=](int i) { return pick(i == 3, sd, pick(i == 2, sc, pick(i == 1, sb, sa))); };
    V3 n0 = v3(0.0, 0.0, 0.0);
    double d0 = 0.0;
    bool ok0 = epa_face(corner(f0.x), corner(f0.y), corner(f0.z), corner, 4, n0, d0);
    if (group_ballot(!ok0) & 0xFull) {
        if (leader) err |= ERR_EPA_DEGENERATE;
        return -1;
    }
    bool below = gl < 4 && d0 < DBL_MAX;
    double min_d = below ? d0 : DBL_MAX;
    int mi0 = below ? gl : NO_SEL;
    group_argmin<G>(min_d, mi0);
    V3 min_n = v3(__shfl(n0.x, mi0 & 3, G), __shfl(n0.y, mi0 & 3, G), __shfl(n0.z, mi0 & 3, G));
    if (mi0 == NO_SEL) min_n = v3(0.0, 0.0, 0.0);
    int np = 4, nf = 4;
    bool dup = false;  // equal points in the polytope
    GroupPoly P;
    P.bind(work, EPA_MAXV, EPA_MAXF, EPA_MAXE);
    bool lds = false;
    for (int it = 0; it < 100; ++it) {
        V3 sp = support_md<G>(h1, h2, min_n, err);
        double d = dot(min_n, sp);
        if (fabs(d - min_d) < 0.0001) {
            n_out = min_n;
            pen_out = min_d;
            return 1;
        }
        int ne = 0;
        // the polytope to the working memory, if it is not there
        auto grow = [&] {
            if (!lds) return;
            lds = false;
            GroupPoly Q = P;
            P.bind(work, EPA_MAXV, EPA_MAXF, EPA_MAXE);
            group_mem_sync();
            for (int i = gl; i < np; i += G) P.poly[i] = Q.poly[i];
            for (int i = gl; i < nf; i += G) {
                P.normals[i] = Q.normals[i];
                P.dist[i] = Q.dist[i];
                P.faces[i] = Q.faces[i];
            }
            for (int i = gl; i < ne; i += G) P.edges[i] = Q.edges[i];
            group_mem_sync();
        };
        if (it == 0) {
            // half as many points as faces and a few more, as many edges
            int f = (spare_n * (int)sizeof(V3) - 6 * (int)sizeof(V3)) / GROUP_POLY_FACE_BYTES;
            f = f < EPA_MAXE ? f : EPA_MAXE;
            if (f >= 8) {
                lds = true;
                P.bind((char*)spare, f / 2 + 6, f & ~1, f & ~1);
            }
            if (gl < 4) {
                P.poly[gl] = corner(gl);
                P.faces[gl] = (uint32_t)(f0.x | f0.y << 8 | f0.z << 16);
                P.normals[gl] = n0;
                P.dist[gl] = d0;
            }
            dup = veq(sa, sb) | veq(sa, sc) | veq(sa, sd) | veq(sb, sc) | veq(sb, sd) | veq(sc, sd);
            group_mem_sync();
        }
        if (np == P.max_v) grow();
        bool same = false;
        for (int i = gl; i < np; i += G) same |= veq(P.poly[i], sp);
        dup |= group_ballot(same) != 0;
        const int new_idx = np;
        if (leader) P.poly[np] = sp;
        ++np;
        // which faces see sp (triangle_centroid, epa.cpp:112-116; a property
        // of each face: computed up front)
        FaceBits vis;
        for (int c0 = 0; c0 < nf; c0 += G) {
            int i = c0 + gl;
            bool v = false;
            if (i < nf) {
                uint32_t f = P.faces[i];
                V3 c = scl(1.0 / 3.0, add(add(P.poly[f >> 8 & 255], P.poly[f >> 16]), P.poly[f & 255]));
                v = dot(P.normals[i], sub(sp, c)) > 0.0;
            }
            vis.or_bits(c0, group_ballot(v));
        }
        // add_edge (epa.cpp:79-110): an edge equal to a listed one, by index
        // or (only where points are equal) by position, cancels it
        // (swap-remove), else it is appended; false when the list is full
        auto add_edge = [&](uint32_t x, uint32_t y) {
            for (int c0 = 0; c0 < ne; c0 += G) {
                int j = c0 + gl;
                bool hit = false;
                if (j < ne) {
                    uint32_t cur = P.edges[j], cx = cur & 255, cy = cur >> 8;
                    hit = (x == cx && y == cy) || (x == cy && y == cx);
                    if (dup && !hit) {
                        V3 c1 = P.poly[cx], c2 = P.poly[cy], e1 = P.poly[x], e2 = P.poly[y];
                        hit = (veq(c1, e1) && veq(c2, e2)) || (veq(c1, e2) && veq(c2, e1));
                    }
                }
                unsigned long long m = group_ballot(hit);
                if (m) {
                    --ne;
                    if (leader) P.edges[c0 + __ffsll((long long)m) - 1] = P.edges[ne];
                    group_mem_sync();
                    return true;
                }
            }
            if (ne == P.max_e) grow();
            if (ne == P.max_e) return false;
            if (leader) P.edges[ne] = x | y << 8;
            ++ne;
            group_mem_sync();
            return true;
        };
        group_mem_sync();
        // the visible faces' edges and the swap-removes, in order
        // (epa.cpp:191-195: faces, distances and normals together)
        for (int i = vis.first(); i < nf; i = vis.first()) {
            uint32_t f = P.faces[i], fx = f & 255, fy = f >> 8 & 255, fz = f >> 16;
            if (!add_edge(fx, fy) || !add_edge(fy, fz) || !add_edge(fz, fx)) {
                if (leader) err |= ERR_EPA_CAPACITY;
                return -1;
            }
            --nf;
            if (gl < 3) ((double*)&P.normals[i])[gl] = ((double*)&P.normals[nf])[gl];
            if (gl == 3) {
                P.dist[i] = P.dist[nf];
                P.faces[i] = P.faces[nf];
            }
            vis.put(i, vis.get(nf) && i < nf);
            vis.put(nf, false);
            group_mem_sync();
        }
        if (nf + ne > P.max_f) grow();
        // the new faces (edge i, new point) at nf + i; the sequential loop
        // stops at the first full list or degenerate face, in that order
        int room = EPA_MAXF - nf;
        int nnew = ne < room ? ne : room;
        int first_bad = nnew;
        for (int i = gl; i < nnew; i += G) {
            uint32_t e = P.edges[i];
            V3 n;
            double fd;
            bool ok = epa_face(P.poly[e & 255], P.poly[e >> 8], sp, [&](int k) { return P.poly[k]; }, np, n, fd);
            P.faces[nf + i] = e | (uint32_t)new_idx << 16;
            P.normals[nf + i] = n;
            P.dist[nf + i] = fd;
            if (!ok && i < first_bad) first_bad = i;
        }
        first_bad = group_min<G>(first_bad);
        if (first_bad < nnew) {
            if (leader) err |= ERR_EPA_DEGENERATE;
            return -1;
        }
        if (ne > room) {
            if (leader) err |= ERR_EPA_CAPACITY;
            return -1;
        }
        nf += ne;
        group_mem_sync();
        // the closest face: first minimum of the distances
        double md = DBL_MAX;
        int mi = NO_SEL;
        for (int i = gl; i < nf; i += G) {
            double di = P.dist[i];
            bool t = di < md;
            md = t ? di : md;
            mi = t ? i : mi;
        }
        group_argmin<G>(md, mi);
        min_d = md;
        if (mi != NO_SEL) min_n = P.normals[mi];
    }
    return 0;
}

// epa (epa.cpp:118-237): 0 = no convergence, 1 = converged, -1 = error.
// On one lane (G = 1) with its working memory, or on a lane group (epa_group).
template <int G = 1, class View = HullView>
RP_HD int epa(const View& h1, const View& h2, const Simplex& s, V3& n_out, double& pen_out, uint32_t& err,
              char* work, V3* spare = nullptr, int spare_n = 0) {
    if constexpr (G == 1) {
        EpaPoly P;
        epa_bind(P, work);
        if (!P.init(s, err)) return -1;
        for (int it = 0; it < 100; ++it) {
            V3 sp = support_md<G>(h1, h2, P.min_n, err);
            int st = P.step(sp, n_out, pen_out, err);
            if (st != 2) return st;
        }
        return 0;
    } else {
        return epa_group<G>(h1, h2, s, n_out, pen_out, err, work, spare, spare_n);
    }
}

// ---------------------------------------------------------------------------
// Contact manifold (clipping.cpp:7-371)
// ---------------------------------------------------------------------------
struct Plane { V3 normal, point; };

// The plane offset is truncated to float (clipping.cpp:14, 27).
RP_HD float plane_offset(const Plane& p) { return (float)-dot(p.normal, p.point); }
// is_point_in_plane (clipping.cpp:12-19)
RP_HD bool point_in_plane(V3 normal, float distance, V3 pos) {
    if (dot(pos, normal) + distance < 0.0) return false;
    return true;
}
// plane_edge_intersection (clipping.cpp:21-47), with its float truncations
RP_HD bool plane_edge(V3 normal, float distance, V3 start, V3 end, V3& out) {
    const double EPSILON = 0.000001;
    V3 ab = sub(end, start);
    float ab_p = dot(normal, ab);
    if (fabs((double)ab_p) > EPSILON) {
        V3 p_co = scl(-distance, normal);
        float fac = -dot(normal, sub(start, p_co)) / ab_p;
        fac = RP_MIN(RP_MAX(fac, 0.0), 1.0);
        out = add(start, scl(fac, ab));
        return true;
    }
    return false;
}

// One Sutherland-Hodgman pass against one plane (clipping.cpp:62-108).
RP_HD int clip_pass(const V3* in, int n, const Plane& p, V3* out, bool remove, uint32_t& err) {
    int m = 0;
    if (n == 0) return 0;
    const float off = plane_offset(p);
    V3 tmp, start = in[n - 1];
    for (int j = 0; j < n; ++j) {
        V3 end = in[j];
        bool s_in = point_in_plane(p.normal, off, start);
        bool e_in = point_in_plane(p.normal, off, end);
        if (remove) {
            if (e_in) { if (m < CLIP_MAX) out[m++] = end; else err |= ERR_CLIP_CAPACITY; }
        } else if (s_in && e_in) {
            if (m < CLIP_MAX) out[m++] = end; else err |= ERR_CLIP_CAPACITY;
        } else if (s_in && !e_in) {
            if (plane_edge(p.normal, off, start, end, tmp)) { if (m < CLIP_MAX) out[m++] = tmp; else err |= ERR_CLIP_CAPACITY; }
        } else if (!s_in && e_in) {
            if (plane_edge(p.normal, off, start, end, tmp)) { if (m < CLIP_MAX) out[m++] = tmp; else err |= ERR_CLIP_CAPACITY; }
            if (m < CLIP_MAX) out[m++] = end; else err |= ERR_CLIP_CAPACITY;
        }
        start = end;
    }
    return m;
}

// Lane-group clipping (G > 1): the polygons live in LDS, and each pass gives
// every lane one edge (start = in[j - 1], end = in[j]); a lane's 0-2 output
// points go to their place in the sequential output order by a prefix sum
// over the group, so the polygon equals clip_pass's point for point.
template <int G> __device__ __forceinline__ int group_inclusive_sum(int v) {
    int gl = (int)(__lane_id() & (G - 1));
    // row_shr:d reads lane - d of the same 16-lane row; every lane moves its
    // value before the group's first d lanes drop what they received
    int o = dpp_int<DPP_ROW_SHR0 + 1>(v);
    v += gl >= 1 ? o : 0;
    o = dpp_int<DPP_ROW_SHR0 + 2>(v);
    v += gl >= 2 ? o : 0;
    if constexpr (G >= 8) {
        o = dpp_int<DPP_ROW_SHR0 + 4>(v);
        v += gl >= 4 ? o : 0;
    }
    if constexpr (G >= 16) {
        o = dpp_int<DPP_ROW_SHR0 + 8>(v);
        v += gl >= 8 ? o : 0;
    }
    return v;
}
// One pass (clip_pass's rules, keeping the points inside) over `in` (n
// points) into `out` (cap points). Returns the output count; more than cap
// sets `ovf` (no point is lost: the caller redoes the clipping in CLIP_MAX
// buffers). `same` is set, and nothing written, when every point is inside:
// the polygon is unchanged.
template <int G>
__device__ __forceinline__ int clip_pass_group(const V3* in, int n, V3 normal, float off, V3* out, int cap, bool& ovf,
                                               bool& same) {
    int gl = (int)(__lane_id() & (G - 1));
    int gbase = (int)__lane_id() & ~(G - 1);
    int m = 0;
    same = false;
    for (int c0 = 0; c0 < n; c0 += G) {
        int j = c0 + gl;
        int cnt = 0;
        V3 o0 = v3(0.0, 0.0, 0.0), o1 = o0;
        V3 start = o0, end = o0;
        bool s_in = true, e_in = true;
        if (j < n) {
            start = in[j == 0 ? n - 1 : j - 1];
            end = in[j];
            s_in = point_in_plane(normal, off, start);
            e_in = point_in_plane(normal, off, end);
        }
        if (n <= G && ((__ballot(!e_in) >> gbase) & ((1ull << G) - 1ull)) == 0) {
            same = true;
            return n;
        }
        if (j < n) {
            V3 t;
            if (s_in && e_in) {
                o0 = end; cnt = 1;
            } else if (s_in != e_in) {
                bool cut = plane_edge(normal, off, start, end, t);
                o0 = cut ? t : end;
                o1 = end;
                cnt = (cut ? 1 : 0) + (e_in ? 1 : 0);
            }
        }
        int incl = group_inclusive_sum<G>(cnt);
        int total = group_bcast_last<G>(incl);
        int pos = m + incl - cnt;
        if (cnt >= 1 && pos < cap) out[pos] = o0;
        if (cnt == 2 && pos + 1 < cap) out[pos + 1] = o1;
        m += total;
    }
    if (m > cap) ovf = true;
    group_mem_sync();
    return m;
}

// get_face_with_most_fitting_normal (clipping.cpp:136-152)
RP_HD int best_face(const HullTables& T, int4 v, const HullFaces& h, V3 n, uint32_t& err) {
    double max_proj = -DBL_MAX;
    int sel = -1;
    for (int i = v.x; i < v.x + v.y; ++i) {
        double proj = dot(face_normal_world(h.R, h.fn[T.list[i]]), n);
        if (proj > max_proj) { max_proj = proj; sel = T.list[i]; }
    }
    if (sel < 0) { err |= ERR_SELECT; sel = 0; }
    return sel;
}

// collision_distance_between_skew_lines (clipping.cpp:210-239)
RP_HD bool skew_lines(V3 p1, V3 d1, V3 p2, V3 d2, V3& l1, V3& l2) {
    double n1 = d1.x * d2.x + d1.y * d2.y + d1.z * d2.z;
    double n2 = d2.x * d2.x + d2.y * d2.y + d2.z * d2.z;
    double m1 = -d1.x * d1.x - d1.y * d1.y - d1.z * d1.z;
    double m2 = -d2.x * d1.x - d2.y * d1.y - d2.z * d1.z;
    double r1 = -d1.x * p2.x + d1.x * p1.x - d1.y * p2.y + d1.y * p1.y - d1.z * p2.z + d1.z * p1.z;
    double r2 = -d2.x * p2.x + d2.x * p1.x - d2.y * p2.y + d2.y * p1.y - d2.z * p2.z + d2.z * p1.z;
    if ((n1 * m2) - (n2 * m1) == 0) return false;
    double n = ((r1 * m2) - (r2 * m1)) / ((n1 * m2) - (n2 * m1));
    double m = ((n1 * r2) - (n2 * r1)) / ((n1 * m2) - (n2 * m1));
    l1 = add(p1, scl(m, d1));
    l2 = add(p2, scl(n, d2));
    return true;
}

struct ContactPt { V3 p1, p2, n; };

// The incident face clipped against the reference face's boundary planes
// (clipping.cpp:121-134, 294) and the points above the reference plane
// removed (clipping.cpp:296-302), by one lane, in two caller-owned buffers
// of CLIP_MAX points; `res` is set to the one holding the result. rtv / itv:
// the two hulls' vertices, rf / inf: the faces' records.
RP_HD int clip_serial(const HullTables& T, const V3* rtv, const V3* rfn, const M3& rR, int4 rf, const V3* itv, int4 inf,
                      const Plane& rp, V3* bufA, V3* bufB, const V3*& res, uint32_t& err) {
    int n = 0;
    for (int i = inf.x; i < inf.x + inf.y; ++i) {
        if (n < CLIP_MAX) bufA[n++] = itv[T.list[i]]; else err |= ERR_CLIP_CAPACITY;
    }
    V3* in = bufA;
    V3* outp = bufB;
    for (int k = rf.z; k < rf.z + rf.w; ++k) {
        if (n == 0) break;
        int2 nb = T.nbr[k];
        Plane p;
        p.point = rtv[nb.y];
        p.normal = inv3(face_normal_world(rR, rfn[nb.x]));
        n = clip_pass(in, n, p, outp, false, err);
        V3* t = in; in = outp; outp = t;
    }
    n = clip_pass(in, n, rp, outp, true, err);
    res = outp;
    return n;
}

// get_closest_point_polygon (clipping.cpp:115-119) and the contact point
// (clipping.cpp:304-329) of one point of the clipped polygon; whether it is
// kept (negative penetration). pd = -normal . point of the reference plane.
RP_HD bool contact_point(V3 pt, const Plane& rp, double pd, V3 normal, bool ref1, ContactPt& c) {
    V3 cp = sub(pt, scl(dot(rp.normal, pt) + pd, rp.normal));
    V3 diff = sub(pt, cp);
    double pen;
    if (ref1) {
        pen = dot(diff, normal);
        c.p1 = sub(pt, scl(pen, normal));
        c.p2 = pt;
    } else {
        pen = -dot(diff, normal);
        c.p1 = pt;
        c.p2 = add(pt, scl(pen, normal));
    }
    c.n = normal;
    return pen < 0.0;
}
// The contacts of the clipped polygon, at most MAXC, handed to emit(k, contact).
template <class Emit>
RP_HD int contacts_from_clip(const V3* pts, int n, const Plane& rp, V3 normal, bool ref1, Emit emit, uint32_t& err) {
    int nc = 0;
    double pd = dot(scl(-1.0, rp.normal), rp.point);
    for (int i = 0; i < n; ++i) {
        ContactPt c;
        if (!contact_point(pts[i], rp, pd, normal, ref1, c)) continue;
        if (nc < MAXC) emit(nc++, c); else err |= ERR_CONTACT_CAPACITY;
    }
    return nc;
}
// The same on the group's lanes, with the removal of the points above the
// reference plane (clipping.cpp:296-302) folded in (both keep the points'
// order): lane j takes point j; the kept points are numbered in point order
// by a prefix sum, and each lane emits its own (more than MAXC set
// ERR_CONTACT_CAPACITY). Returns the count on every lane of the group.
template <int G, class Emit>
__device__ __forceinline__ int contacts_from_clip_group(const V3* pts, int n, const Plane& rp, V3 normal, bool ref1,
                                                        Emit emit, uint32_t& err) {
    int gl = (int)(__lane_id() & (G - 1));
    int nc = 0;
    double pd = dot(scl(-1.0, rp.normal), rp.point);
    const float off = plane_offset(rp);
    for (int c0 = 0; c0 < n; c0 += G) {
        int i = c0 + gl;
        bool keep = false;
        ContactPt c;
        if (i < n) {
            V3 pt = pts[i];
            keep = point_in_plane(rp.normal, off, pt) && contact_point(pt, rp, pd, normal, ref1, c);
        }
        int k = keep ? 1 : 0;
        int incl = group_inclusive_sum<G>(k);
        int total = group_bcast_last<G>(incl);
        int pos = nc + incl - k;
        if (keep && pos < MAXC) emit(pos, c);
        nc += total;
    }
    if (nc > MAXC) {
        if (gl == 0) err |= ERR_CONTACT_CAPACITY;
        nc = MAXC;
    }
    return nc;
}

// convex_convex_contact_manifold (clipping.cpp:249-341), one lane per pair,
// with working memory `work`. Returns the number of contacts handed to emit(k, contact) (at most MAXC).
template <class Emit>
RP_HD int manifold_lane(const HullTables& T, const HullView& h1, const HullView& h2, V3 normal, Emit emit, uint32_t& err,
                        char* work) {
    const double EPSILON = 0.0001;
    V3 inormal = inv3(normal);
    HullFaces hf1 = hull_faces(T, h1), hf2 = hull_faces(T, h2);
    int s1, s2;
    support_index2<1>(h1, normal, h2, inormal, s1, s2, err);
    int4 r1 = hf1.vrec[s1], r2 = hf2.vrec[s2];
    int f1 = best_face(T, r1, hf1, normal, err);
    int f2 = best_face(T, r2, hf2, inormal, err);
    // get_edge_with_most_fitting_normal (clipping.cpp:154-200)
    V3 edge_n = v3(0.0, 0.0, 0.0);
    int e1a = 0, e1b = 0, e2a = 0, e2b = 0;
    V3 sp1 = h1.tv[s1], sp2 = h2.tv[s2];
    double max_dot = -DBL_MAX;
    bool found = false;
    for (int i = r1.z; i < r1.z + r1.w; ++i) {
        int v1 = T.list[i];
        V3 ed1 = sub(sp1, h1.tv[v1]);
        for (int j = r2.z; j < r2.z + r2.w; ++j) {
            int v2 = T.list[j];
            V3 ed2 = sub(sp2, h2.tv[v2]);
            V3 cn = nrm(cross(ed1, ed2));
            V3 cni = inv3(cn);
            double dd = dot(cn, normal);
            if (dd > max_dot) { max_dot = dd; e1a = s1; e1b = v1; e2a = s2; e2b = v2; edge_n = cn; found = true; }
            dd = dot(cni, normal);
            if (dd > max_dot) { max_dot = dd; e1a = s1; e1b = v1; e2a = s2; e2b = v2; edge_n = cni; found = true; }
        }
    }
    if (!found) err |= ERR_SELECT;
    V3 n1 = face_normal_world(hf1.R, hf1.fn[f1]), n2 = face_normal_world(hf2.R, hf2.fn[f2]);
    double d1 = dot(n1, normal);
    double d2 = dot(n2, inormal);
    double de = dot(edge_n, normal);
    if (de > d1 + EPSILON && de > d2 + EPSILON) {
        ContactPt c;
        V3 p1 = h1.tv[e1a], p2 = h2.tv[e2a];
        if (!skew_lines(p1, sub(h1.tv[e1b], p1), p2, sub(h2.tv[e2b], p2), c.p1, c.p2)) { err |= ERR_SKEW_LINES; return 0; }
        c.n = normal;
        emit(0, c);
        return 1;
    }
    bool ref1 = d1 > d2;
    int4 rf = ref1 ? hf1.frec[f1] : hf2.frec[f2], inf = ref1 ? hf2.frec[f2] : hf1.frec[f1];
    const V3* rtv = ref1 ? h1.tv : h2.tv;
    Plane rp;  // the points above it are removed (clipping.cpp:296-302)
    rp.normal = inv3(ref1 ? n1 : n2);
    rp.point = rtv[T.list[rf.x]];
    const V3* res = nullptr;
    int n = clip_serial(T, rtv, ref1 ? hf1.fn : hf2.fn, ref1 ? hf1.R : hf2.R, rf, ref1 ? h2.tv : h1.tv, inf, rp, (V3*)work,
                        (V3*)work + CLIP_MAX, res, err);
    return contacts_from_clip(res, n, rp, normal, ref1, emit, err);
}

// The same on a lane group: the lanes find the support points, the best faces
// and the best edge pair together (split scans, first-maximum reductions),
// each lane prepares one boundary plane of the reference face, and the group
// clips in `spare` (spare_n points of LDS beside the staged hulls) when both
// polygons fit there, else lane 0 clips in `work`. Each lane emits the
// contacts it made; every lane returns their count.
//
// The chain of dependent loads is what this costs: a hull's record, a
// vertex's or face's record, the list entries, then geometry, each side by
// side for both hulls and for all planes. The selections' values are kept
// from the scans (a face's normal stays with the lane that scored it), and
// the edge pairs are scored only where an edge could win: a unit edge normal's
// product with the unit contact normal does not exceed 1, so with either
// face within EPSILON of that the comparison below is decided. Narrow launch:
// 4096 scenes of 16 bodies 193 -> 156 us, one stack of 10 boxes 43 -> 31, one
// scene of 20000 bodies 119 -> 98.
template <int G, class Emit>
__device__ __forceinline__ int manifold_group(const HullTables& T, const HullView& h1, const HullView& h2, V3 normal,
                                              Emit emit, uint32_t& err, char* work, V3* spare, int spare_n) {
    const double EPSILON = 0.0001, EDGE_MAX = 1.0 + 1e-9;
    const int gl = (int)(__lane_id() & (G - 1));
    V3 inormal = inv3(normal);
    int4 hr1 = T.hull[h1.hid], hr2 = T.hull[h2.hid];
    int s1, s2;
    support_index2<G>(h1, normal, h2, inormal, s1, s2, err);
    int4 r1 = T.rec[hr1.x + s1], r2 = T.rec[hr2.x + s2];
    // get_face_with_most_fitting_normal (clipping.cpp:136-152) of both hulls:
    // lane k scores the entries k, k + G, ... of the vertices' face lists
    double d1 = -DBL_MAX, d2 = -DBL_MAX;
    int pos1 = NO_SEL, pos2 = NO_SEL, f1 = 0, f2 = 0;
    V3 n1 = v3(0.0, 0.0, 0.0), n2 = n1;
    {
        const M3 R1 = model_rotation(T, h1.body), R2 = model_rotation(T, h2.body);
        int most = r1.y > r2.y ? r1.y : r2.y;
        for (int k = gl; k < most; k += G) {
            bool in1 = k < r1.y, in2 = k < r2.y;
            int a = T.list[r1.x + (in1 ? k : 0)], b = T.list[r2.x + (in2 ? k : 0)];
            V3 na = face_normal_world(R1, T.fn[hr1.z + a]), nb = face_normal_world(R2, T.fn[hr2.z + b]);
            double pa = dot(na, normal), pb = dot(nb, inormal);
            bool ta = in1 & (pa > d1), tb = in2 & (pb > d2);
            d1 = ta ? pa : d1;
            pos1 = ta ? k : pos1;
            f1 = ta ? a : f1;
            n1 = pick(ta, na, n1);
            d2 = tb ? pb : d2;
            pos2 = tb ? k : pos2;
            f2 = tb ? b : f2;
            n2 = pick(tb, nb, n2);
        }
    }
    group_argmax2<G>(d1, pos1, d2, pos2);
    // the winning lanes' faces (the first face where nothing was selected)
    const int l1 = pos1 & (G - 1), l2 = pos2 & (G - 1);
    f1 = __shfl(f1, l1, G);
    f2 = __shfl(f2, l2, G);
    if (pos1 == NO_SEL || pos2 == NO_SEL) {
        err |= ERR_SELECT;
        if (pos1 == NO_SEL) {
            f1 = 0;
            n1 = face_normal_world(model_rotation(T, h1.body), T.fn[hr1.z]);
            d1 = dot(n1, normal);
        }
        if (pos2 == NO_SEL) {
            f2 = 0;
            n2 = face_normal_world(model_rotation(T, h2.body), T.fn[hr2.z]);
            d2 = dot(n2, inormal);
        }
    }
    // get_edge_with_most_fitting_normal (clipping.cpp:154-200)
    const int pairs = r1.w * r2.w;
    if (pairs == 0 || !(d1 + EPSILON >= EDGE_MAX || d2 + EPSILON >= EDGE_MAX)) {
        // candidates in the sequential order (neighbour i of s1, neighbour j
        // of s2, then n before -n) are numbered 2 (i n2 + j) + variant; lane k
        // scores the pairs k, k + G, ... and the group keeps the first maximum
        V3 sp1 = h1.tv[s1], sp2 = h2.tv[s2];
        const int* nb1 = T.list + r1.z;
        const int* nb2 = T.list + r2.z;
        const float inv = 1.0f / (float)r2.w;
        double de = -DBL_MAX;
        int best = NO_SEL;
        for (int k = gl; k < pairs; k += G) {
            int a = (int)(((float)k + 0.5f) * inv), b = k - a * r2.w;
            V3 ed1 = sub(sp1, h1.tv[nb1[a]]);
            V3 ed2 = sub(sp2, h2.tv[nb2[b]]);
            V3 cn = nrm(cross(ed1, ed2));
            V3 cni = inv3(cn);
            double dd = dot(cn, normal);
            bool t = dd > de;
            de = t ? dd : de;
            best = t ? 2 * k : best;
            dd = dot(cni, normal);
            t = dd > de;
            de = t ? dd : de;
            best = t ? 2 * k + 1 : best;
        }
        group_argmax<G>(de, best);
        if (best == NO_SEL) {  // (a zero edge normal)
            err |= ERR_SELECT;
            de = dot(v3(0.0, 0.0, 0.0), normal);
        }
        if (de > d1 + EPSILON && de > d2 + EPSILON) {
            if (best == NO_SEL) {
                err |= ERR_SKEW_LINES;
                return 0;
            }
            int k = best >> 1, a = (int)(((float)k + 0.5f) * inv), b = k - a * r2.w;
            ContactPt c;
            if (!skew_lines(sp1, sub(h1.tv[nb1[a]], sp1), sp2, sub(h2.tv[nb2[b]], sp2), c.p1, c.p2)) {
                err |= ERR_SKEW_LINES;
                return 0;
            }
            c.n = normal;
            if (gl == 0) emit(0, c);
            return 1;
        }
    }
    const bool ref1 = d1 > d2;
    const int rbody = ref1 ? h1.body : h2.body, rfn = ref1 ? hr1.z : hr2.z;
    const V3* rtv = ref1 ? h1.tv : h2.tv;
    const V3* itv = ref1 ? h2.tv : h1.tv;
    int4 rf = T.rec[ref1 ? hr1.y + f1 : hr2.y + f2], inf = T.rec[ref1 ? hr2.y + f2 : hr1.y + f1];
    const M3 R = model_rotation(T, rbody);
    Plane rp;
    {
        V3 m = pick(ref1, n1, n2);
        int l = ref1 ? l1 : l2;
        rp.normal = inv3(v3(__shfl(m.x, l, G), __shfl(m.y, l, G), __shfl(m.z, l, G)));
    }
    rp.point = rtv[T.list[rf.x]];
    const int cap = spare_n / 2 < CLIP_MAX ? spare_n / 2 : CLIP_MAX;
    if (cap >= 8 && inf.y <= cap) {
        V3* in = spare;
        V3* outp = spare + cap;
        int n = inf.y;
        for (int i = gl; i < n; i += G) in[i] = itv[T.list[inf.x + i]];
        bool ovf = false;
        for (int k0 = 0; k0 < rf.w && n > 0 && !ovf; k0 += G) {
            // lane k: boundary plane k0 + k
            int2 nb = T.nbr[rf.z + (k0 + gl < rf.w ? k0 + gl : 0)];
            Plane mine;
            mine.point = rtv[nb.y];
            mine.normal = inv3(face_normal_world(R, T.fn[rfn + nb.x]));
            float my_off = plane_offset(mine);
            group_mem_sync();
            int planes = rf.w - k0 < G ? rf.w - k0 : G;
            for (int k = 0; k < planes && n > 0; ++k) {
                V3 pn = v3(__shfl(mine.normal.x, k, G), __shfl(mine.normal.y, k, G), __shfl(mine.normal.z, k, G));
                bool same;
                n = clip_pass_group<G>(in, n, pn, __shfl(my_off, k, G), outp, cap, ovf, same);
                if (ovf) break;
                if (!same) { V3* t = in; in = outp; outp = t; }
            }
        }
        if (!ovf) {
            group_mem_sync();
            return contacts_from_clip_group<G>(in, n, rp, normal, ref1, emit, err);
        }
    }
    // lane 0 clips in the group's working memory
    int nc = 0;
    if (gl == 0) {
        const V3* res = nullptr;
        int m = clip_serial(T, rtv, T.fn + rfn, R, rf, itv, inf, rp, (V3*)work, (V3*)work + CLIP_MAX, res, err);
        nc = contacts_from_clip(res, m, rp, normal, ref1, emit, err);
    }
    return group_bcast<G>(nc);
}

// collider_get_contacts for two hulls (collider.cpp:523-558): GJK, EPA,
// manifold, on a lane group with working memory `work`. `flags` gets
// PAIR_EPA_FAIL for an EPA run that did not converge (the reference prints
// and drops the pair's contacts, epa.cpp:233-236, collider.cpp:549-551) and
// PAIR_GJK_CYCLE for a cycle exit of gjk.
enum { PAIR_EPA_FAIL = 1, PAIR_GJK_CYCLE = 2 };
template <int G, class Emit>
__device__ __forceinline__ int pair_contacts(const HullTables& T, const HullView& h1, const HullView& h2, Emit emit,
                                             uint32_t& err, int& flags, char* work) {
    Simplex s;
    bool cycled = false;
    if (!gjk<G>(h1, h2, s, err, cycled)) {
        if (cycled) flags |= PAIR_GJK_CYCLE;
        return 0;
    }
    V3 n; double pen;
    int r = epa<G>(h1, h2, s, n, pen, err, work);
    if (r != 1) { flags |= PAIR_EPA_FAIL; return 0; }
    return manifold_group<G>(T, h1, h2, n, emit, err, work, nullptr, 0);
}

// clipping_get_contact_manifold (clipping.cpp:343-371) where a collider is a
// sphere: one contact at its support point along the normal.
template <int G>
RP_HD ContactPt sphere_contact(const ColView& c1, const ColView& c2, V3 normal, double penetration, uint32_t& err) {
    ContactPt c;
    c.n = normal;
    if (c1.type == COL_SPHERE) {
        c.p1 = support_point<G>(c1, normal, err);
        c.p2 = sub(c.p1, scl(penetration, normal));
    } else {
        c.p2 = support_point<G>(c2, inv3(normal), err);
        c.p1 = add(c.p2, scl(penetration, normal));
    }
    return c;
}

// collider_get_contacts (collider.cpp:523-558) for any two colliders, on one
// lane (G = 1) or on a lane group, whose lanes emit the contacts they made
// (emit(k, contact)). Two spheres are resolved with the reference's float
// arithmetic; the float square root is taken in double and rounded once,
// which is the correctly rounded result (a 53-bit square root of a 24-bit
// value). `spare` as for manifold_group.
template <int G, class Emit>
RP_HD int collider_contacts(const HullTables& T, const ColView& c1, const ColView& c2, Emit emit, uint32_t& err, int& flags,
                            char* work = nullptr, V3* spare = nullptr, int spare_n = 0) {
    V3 n;
    double pen;
    if (c1.type == COL_SPHERE && c2.type == COL_SPHERE) {
        V3 dv = sub(c1.center, c2.center);
        float dsq = (float)dot(dv, dv);
        float mind = c1.radius + c2.radius;
        if (!(dsq < (mind * mind))) return 0;
        n = nrm(sub(c2.center, c1.center));
        float root = (float)sqrt((double)dsq);
        pen = (double)(mind - root);
    } else {
        Simplex s;
        bool cycled = false;
        if (!gjk<G>(c1, c2, s, err, cycled)) {
            if (cycled) flags |= PAIR_GJK_CYCLE;
            return 0;
        }
        if (epa<G>(c1, c2, s, n, pen, err, work, spare, spare_n) != 1) {
            flags |= PAIR_EPA_FAIL;
            return 0;
        }
    }
    if (c1.type == COL_SPHERE || c2.type == COL_SPHERE) {
        ContactPt c = sphere_contact<G>(c1, c2, n, pen, err);
        if (G == 1 || (__lane_id() & (G - 1)) == 0) emit(0, c);
        return 1;
    }
    if constexpr (G == 1) return manifold_lane(T, c1.h, c2.h, n, emit, err, work);
    else return manifold_group<G>(T, c1.h, c2.h, n, emit, err, work, spare, spare_n);
}

// ---------------------------------------------------------------------------
// XPBD base constraints (pbd_base_constraints.cpp:6-227)
// ---------------------------------------------------------------------------
template <class S>
RP_HD void rot_update(BodyT<S>& e, V3T<S> a, bool plus) {
    Q4T<S> aq = {a.x, a.y, a.z, S(0.0)};
    Q4T<S> qq = q_mul(aq, e.q);
    if (plus) {
        e.q.x = e.q.x + 0.5 * qq.x; e.q.y = e.q.y + 0.5 * qq.y; e.q.z = e.q.z + 0.5 * qq.z; e.q.w = e.q.w + 0.5 * qq.w;
    } else {
        e.q.x = e.q.x - 0.5 * qq.x; e.q.y = e.q.y - 0.5 * qq.y; e.q.z = e.q.z - 0.5 * qq.z; e.q.w = e.q.w - 0.5 * qq.w;
    }
    e.q = q_nrm(e.q);
}

// limit_angle (pbd.cpp:175-217)
RP_HD bool limit_angle(V3 n, V3 n1, V3 n2, double alpha, double beta, V3& dq) {
    double phi = asin(dot(cross(n1, n2), n));
    if (dot(n1, n2) < 0.0) phi = RP_PI_F - phi;
    if (phi > RP_PI_F) phi = phi - 2.0 * RP_PI_F;
    if (phi < -RP_PI_F) phi = phi + 2.0 * RP_PI_F;
    if (phi < alpha || phi > beta) {
        phi = RP_CLAMP(phi, alpha, beta);
        Q4 rot = q_from_axis_radians(n, phi);
        n1 = q_rot(rot, n1);
        dq = cross(n1, n2);
        return true;
    }
    return false;
}

// Integration of one body (pbd.cpp:537-577)
template <class S>
RP_HD void integrate(BodyT<S>& e, double h) {
    e.px = e.x;
    e.pq = e.q;
    if (e.fixed || !e.active) return;
    e.v = add(e.v, scl(h * e.inv_mass, e.F));
    e.x = add(e.x, scl(h, e.v));
    M3T<S> Iinv = world_tensor(e.q, e.Iinv);
    M3T<S> I = world_tensor(e.q, e.I);
    e.w = add(e.w, scl(h, m3_mulv(Iinv, sub(e.T, cross(e.w, m3_mulv(I, e.w))))));
    Q4T<S> aux = {e.w.x, e.w.y, e.w.z, S(0.0)};
    Q4T<S> q = q_mul(aux, e.q);
    e.q.x = e.q.x + h * 0.5 * q.x;
    e.q.y = e.q.y + h * 0.5 * q.y;
    e.q.z = e.q.z + h * 0.5 * q.z;
    e.q.w = e.q.w + h * 0.5 * q.w;
    e.q = q_nrm(e.q);
}

// Velocity update of one body (pbd.cpp:623-643)
template <class S>
RP_HD void velocity_update(BodyT<S>& e, double h) {
    if (e.fixed || !e.active) return;
    e.pv = e.v;
    e.pw = e.w;
    e.v = scl(1.0 / h, sub(e.x, e.px));
    Q4T<S> dq = q_mul(e.q, q_inv(e.pq));
    if (dq.w >= 0.0) e.w = scl(2.0 / h, v3<S>(dq.x, dq.y, dq.z));
    else e.w = scl(-2.0 / h, v3<S>(dq.x, dq.y, dq.z));
}

// clipping_contact_to_collision_constraint (pbd.cpp:408-424)
RP_HD void contact_to_constraint(const Body& e1, const Body& e2, const ContactPt& ct, Contact& c) {
    c.n = ct.n;
    c.lambda_n = 0.0;
    c.lambda_t = 0.0;
    V3 r1w = sub(ct.p1, e1.x);
    V3 r2w = sub(ct.p2, e2.x);
    c.r1 = q_rot(q_inv(e1.q), r1w);
    c.r2 = q_rot(q_inv(e2.q), r2w);
}

}  // namespace rp
