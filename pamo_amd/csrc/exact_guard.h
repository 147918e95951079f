// Exact triangle-intersection decisions for the guard's exact mode (device
// code for gfx950).  No counterpart in the reference, whose guard uses a
// mixed FP32/FP64 predicate with skip rules (self_intersect.cuh:229-378,
// tri_tri_3d.cuh:99-276); this mode flags exactly the pairs that intersect.
//
// Predicates on float32 coordinates:
//   * filtered: differences in FP64 (exact when no rounding tail appears),
//     products and sums checked against the error bounds of J. R. Shewchuk,
//     "Adaptive Precision Floating-Point Arithmetic and Fast Robust Geometric
//     Predicates" (Discrete Comput. Geom. 18, 1997); a sign that the bound
//     cannot certify is reported as undecided;
//   * exact: where the differences are exact in FP64, the determinant of the
//     differences, its 24 (4 in 2D) partial products split by two-product and
//     summed into an expansion that stays in registers (the same paper's
//     grow-expansion, of fixed length); otherwise orient3d as the 4x4
//     determinant [p 1] of the raw coordinates, 24 signed triple products; a
//     product of two float32 values is exact in FP64 and two-product makes the
//     third factor exact, so each term is a two-double expansion and their
//     sum, grown term by term with two-sum, is exact.  orient2d likewise from
//     6 exact products.
// Decisions (mesh semantics): faces with no common vertex index must not
// meet; faces sharing one vertex may meet only there; faces sharing an edge
// may meet only along it (a flat fold, both opposite corners on one side of
// the edge in a common plane, is an intersection); repeated faces intersect;
// a degenerate face (collinear corners) is not tested.
#pragma once
#include "hip_common.h"

namespace pamo {
namespace {

struct XP3 {
    float x, y, z;
};
struct XP2 {
    float x, y;
};

__device__ __forceinline__ void x_two_sum(double a, double b, double& x, double& y) {
    x = a + b;
    const double bv = x - a, av = x - bv, br = b - bv, ar = a - av;
    y = ar + br;
}
__device__ __forceinline__ void x_two_diff(double a, double b, double& x, double& y) {
    x = a - b;
    const double bv = a - x, av = x + bv, br = bv - b, ar = a - av;
    y = ar + br;
}
__device__ __forceinline__ void x_split(double a, double& hi, double& lo) {
    const double c = 134217729.0 * a;  // 2^27 + 1
    const double abig = c - a;
    hi = c - abig;
    lo = a - hi;
}
__device__ __forceinline__ void x_two_product(double a, double b, double& x, double& y) {
    x = a * b;
    double ah, al, bh, bl;
    x_split(a, ah, al);
    x_split(b, bh, bl);
    const double e1 = x - ah * bh, e2 = e1 - al * bh, e3 = e2 - ah * bl;
    y = al * bl - e3;
}

constexpr double kXEps = 1.1102230246251565e-16;  // 2^-53
constexpr double kXO3d = (7.0 + 56.0 * kXEps) * kXEps;
constexpr double kXCcw = (3.0 + 16.0 * kXEps) * kXEps;
constexpr int kUndecided = 2;

// Differences of float32 coordinates, and whether FP64 holds them exactly.
struct XD9 {
    double adx, ady, adz, bdx, bdy, bdz, cdx, cdy, cdz;
    bool exact;
};
struct XD4 {
    double acx, acy, bcx, bcy;
    bool exact;
};

__device__ __forceinline__ XD9 x_diff(const XP3& a, const XP3& b, const XP3& c, const XP3& d) {
    XD9 q;
    double t, tails = 0.0;
    x_two_diff(a.x, d.x, q.adx, t); tails += fabs(t);
    x_two_diff(a.y, d.y, q.ady, t); tails += fabs(t);
    x_two_diff(a.z, d.z, q.adz, t); tails += fabs(t);
    x_two_diff(b.x, d.x, q.bdx, t); tails += fabs(t);
    x_two_diff(b.y, d.y, q.bdy, t); tails += fabs(t);
    x_two_diff(b.z, d.z, q.bdz, t); tails += fabs(t);
    x_two_diff(c.x, d.x, q.cdx, t); tails += fabs(t);
    x_two_diff(c.y, d.y, q.cdy, t); tails += fabs(t);
    x_two_diff(c.z, d.z, q.cdz, t); tails += fabs(t);
    q.exact = tails == 0.0;
    return q;
}

__device__ __forceinline__ XD4 x_diff(const XP2& a, const XP2& b, const XP2& c) {
    XD4 q;
    double t, tails = 0.0;
    x_two_diff(a.x, c.x, q.acx, t); tails += fabs(t);
    x_two_diff(a.y, c.y, q.acy, t); tails += fabs(t);
    x_two_diff(b.x, c.x, q.bcx, t); tails += fabs(t);
    x_two_diff(b.y, c.y, q.bcy, t); tails += fabs(t);
    q.exact = tails == 0.0;
    return q;
}

__device__ __forceinline__ int o3_filter(const XD9& q) {
    if (!q.exact) return kUndecided;
    const double bc = q.bdx * q.cdy, cb = q.cdx * q.bdy, ca = q.cdx * q.ady, ac = q.adx * q.cdy,
                 ab = q.adx * q.bdy, ba = q.bdx * q.ady;
    const double det = q.adz * (bc - cb) + q.bdz * (ca - ac) + q.cdz * (ab - ba);
    const double perm = (fabs(bc) + fabs(cb)) * fabs(q.adz) + (fabs(ca) + fabs(ac)) * fabs(q.bdz) +
                        (fabs(ab) + fabs(ba)) * fabs(q.cdz);
    const double bound = kXO3d * perm;
    if (det > bound) return 1;
    if (-det > bound) return -1;
    if (perm == 0.0) return 0;
    return kUndecided;
}

__device__ __forceinline__ int o2_filter(const XD4& q) {
    if (!q.exact) return kUndecided;
    const double l = q.acx * q.bcy, r = q.acy * q.bcx;
    const double det = l - r, bound = kXCcw * (fabs(l) + fabs(r));
    if (det > bound) return 1;
    if (-det > bound) return -1;
    if (l == 0.0 && r == 0.0) return 0;
    return kUndecided;
}

// Sign of the exact sum of kN doubles: each is grown into an expansion of
// fixed length (zero components stay), so that all of it is in registers; the
// largest component that is not zero has the sum's sign.
template <int kN>
__device__ __forceinline__ int x_sum_sign(const double* v) {
    double h[kN];
#pragma unroll
    for (int k = 0; k < kN; ++k) {
        double q = v[k];
#pragma unroll
        for (int i = 0; i < k; ++i) {
            double s, hh;
            x_two_sum(q, h[i], s, hh);
            h[i] = hh;
            q = s;
        }
        h[k] = q;
    }
    int sign = 0;
#pragma unroll
    for (int i = 0; i < kN; ++i) sign = h[i] > 0.0 ? 1 : (h[i] < 0.0 ? -1 : sign);
    return sign;
}

// The determinant of exact differences, exactly.  A difference of float32
// values is below 2^129 and a multiple of 2^-149, so no product here
// overflows or loses bits to underflow.
__device__ __forceinline__ void x_add_minor(double z, double a, double b, double c, double d, double* out) {
    double m[4];  // a b - c d
    x_two_product(a, b, m[0], m[1]);
    x_two_product(-c, d, m[2], m[3]);
#pragma unroll
    for (int i = 0; i < 4; ++i) x_two_product(m[i], z, out[2 * i], out[2 * i + 1]);
}
__device__ __forceinline__ int o3_sum(const XD9& q) {
    double t[24];
    x_add_minor(q.adz, q.bdx, q.cdy, q.cdx, q.bdy, t);
    x_add_minor(q.bdz, q.cdx, q.ady, q.adx, q.cdy, t + 8);
    x_add_minor(q.cdz, q.adx, q.bdy, q.bdx, q.ady, t + 16);
    return x_sum_sign<24>(t);
}
__device__ __forceinline__ int o2_sum(const XD4& q) {
    double t[4];
    x_two_product(q.acx, q.bcy, t[0], t[1]);
    x_two_product(-q.acy, q.bcx, t[2], t[3]);
    return x_sum_sign<4>(t);
}

// Nonoverlapping expansion in increasing magnitude, zero components removed.
struct XExp {
    double h[50];
    int n = 0;
};

__device__ void x_grow(XExp& e, double b) {
    double q = b;
    int k = 0;
    for (int i = 0; i < e.n; ++i) {
        double s, hh;
        x_two_sum(q, e.h[i], s, hh);
        q = s;
        if (hh != 0.0) e.h[k++] = hh;
    }
    if (q != 0.0 || k == 0) e.h[k++] = q;
    e.n = k;
}

__device__ __forceinline__ int x_sign(const XExp& e) {
    const double top = e.h[e.n - 1];
    return top > 0.0 ? 1 : (top < 0.0 ? -1 : 0);
}

// s * u * v * w added exactly (u * v is exact in FP64 for float32 factors)
__device__ __forceinline__ void x_add_triple(XExp& e, float s, float u, float v, float w) {
    double hi, lo;
    x_two_product((double)s * ((double)u * (double)v), (double)w, hi, lo);
    x_grow(e, lo);
    x_grow(e, hi);
}

__device__ void x_add_det3(XExp& e, float s, const XP3& p, const XP3& q, const XP3& r) {
    x_add_triple(e, s, p.x, q.y, r.z);
    x_add_triple(e, -s, p.x, q.z, r.y);
    x_add_triple(e, -s, p.y, q.x, r.z);
    x_add_triple(e, s, p.y, q.z, r.x);
    x_add_triple(e, s, p.z, q.x, r.y);
    x_add_triple(e, -s, p.z, q.y, r.x);
}

// det[a-d; b-d; c-d] = det3(a,b,c) - det3(a,b,d) + det3(a,c,d) - det3(b,c,d)
__device__ __noinline__ int o3_raw(XP3 a, XP3 b, XP3 c, XP3 d) {
    XExp e;
    x_add_det3(e, 1.0f, a, b, c);
    x_add_det3(e, -1.0f, a, b, d);
    x_add_det3(e, 1.0f, a, c, d);
    x_add_det3(e, -1.0f, b, c, d);
    return x_sign(e);
}

// (a - c) x (b - c) = a.x b.y - a.y b.x - a.x c.y + a.y c.x + b.x c.y - b.y c.x
__device__ __noinline__ int o2_raw(XP2 a, XP2 b, XP2 c) {
    XExp e;
    const float s[6] = {1.f, -1.f, -1.f, 1.f, 1.f, -1.f};
    const float u[6] = {a.x, a.y, a.x, a.y, b.x, b.y}, v[6] = {b.y, b.x, c.y, c.x, c.y, c.x};
#pragma unroll
    for (int k = 0; k < 6; ++k) x_grow(e, (double)s[k] * ((double)u[k] * (double)v[k]));
    return x_sign(e);
}

// Exact signs: filtered first.  Called functions: the decisions below use them
// in some thirty places.
__device__ __noinline__ int o3_exact(XP3 a, XP3 b, XP3 c, XP3 d) {
    const XD9 q = x_diff(a, b, c, d);
    const int s = o3_filter(q);
    if (s != kUndecided) return s;
    return q.exact ? o3_sum(q) : o3_raw(a, b, c, d);
}
__device__ __noinline__ int o2_exact(XP2 a, XP2 b, XP2 c) {
    const XD4 q = x_diff(a, b, c);
    const int s = o2_filter(q);
    if (s != kUndecided) return s;
    return q.exact ? o2_sum(q) : o2_raw(a, b, c);
}

__device__ __forceinline__ XP2 x_proj(const XP3& p, int drop) {
    return drop == 0 ? XP2{p.y, p.z} : (drop == 1 ? XP2{p.z, p.x} : XP2{p.x, p.y});
}

__device__ int x_proj_axis(const XP3& a, const XP3& b, const XP3& c) {
    for (int d = 0; d < 3; ++d)
        if (o2_exact(x_proj(a, d), x_proj(b, d), x_proj(c, d)) != 0) return d;
    return -1;
}

__device__ __forceinline__ bool x_on_segment(const XP2& p, const XP2& q, const XP2& r) {
    return fminf(p.x, q.x) <= r.x && r.x <= fmaxf(p.x, q.x) && fminf(p.y, q.y) <= r.y && r.y <= fmaxf(p.y, q.y);
}

__device__ bool x_seg_seg_2d(const XP2& p1, const XP2& p2, const XP2& q1, const XP2& q2) {
    const int o1 = o2_exact(p1, p2, q1), o2 = o2_exact(p1, p2, q2);
    const int o3 = o2_exact(q1, q2, p1), o4 = o2_exact(q1, q2, p2);
    if (o1 * o2 < 0 && o3 * o4 < 0) return true;
    if (o1 == 0 && x_on_segment(p1, p2, q1)) return true;
    if (o2 == 0 && x_on_segment(p1, p2, q2)) return true;
    if (o3 == 0 && x_on_segment(q1, q2, p1)) return true;
    if (o4 == 0 && x_on_segment(q1, q2, p2)) return true;
    return false;
}

__device__ bool x_point_in_tri_2d(const XP2& p, const XP2& a, const XP2& b, const XP2& c) {
    const int s1 = o2_exact(a, b, p), s2 = o2_exact(b, c, p), s3 = o2_exact(c, a, p);
    const bool has_neg = s1 < 0 || s2 < 0 || s3 < 0, has_pos = s1 > 0 || s2 > 0 || s3 > 0;
    return !(has_neg && has_pos);
}

// Closed segment pq against closed non-degenerate triangle abc.
__device__ bool x_seg_tri(const XP3& p, const XP3& q, const XP3& a, const XP3& b, const XP3& c) {
    const int o1 = o3_exact(a, b, c, p), o2 = o3_exact(a, b, c, q);
    if ((o1 > 0 && o2 > 0) || (o1 < 0 && o2 < 0)) return false;
    if (o1 == 0 && o2 == 0) {
        const int d = x_proj_axis(a, b, c);
        if (d < 0) return false;
        const XP2 P2 = x_proj(p, d), Q2 = x_proj(q, d), A = x_proj(a, d), B = x_proj(b, d), C = x_proj(c, d);
        return x_point_in_tri_2d(P2, A, B, C) || x_point_in_tri_2d(Q2, A, B, C) ||
               x_seg_seg_2d(P2, Q2, A, B) || x_seg_seg_2d(P2, Q2, B, C) || x_seg_seg_2d(P2, Q2, C, A);
    }
    const int s1 = o3_exact(p, q, a, b), s2 = o3_exact(p, q, b, c), s3 = o3_exact(p, q, c, a);
    return (s1 >= 0 && s2 >= 0 && s3 >= 0) || (s1 <= 0 && s2 <= 0 && s3 <= 0);
}

__device__ bool x_tri_tri(const XP3* t, const XP3* u) {
    const int s0 = o3_exact(t[0], t[1], t[2], u[0]), s1 = o3_exact(t[0], t[1], t[2], u[1]),
              s2 = o3_exact(t[0], t[1], t[2], u[2]);
    if ((s0 > 0 && s1 > 0 && s2 > 0) || (s0 < 0 && s1 < 0 && s2 < 0)) return false;
    if (s0 == 0 && s1 == 0 && s2 == 0) {
        const int d = x_proj_axis(t[0], t[1], t[2]);
        if (d < 0) return false;
        XP2 a[3], b[3];
        for (int i = 0; i < 3; ++i) {
            a[i] = x_proj(t[i], d);
            b[i] = x_proj(u[i], d);
        }
        for (int i = 0; i < 3; ++i)
            for (int j = 0; j < 3; ++j)
                if (x_seg_seg_2d(a[i], a[(i + 1) % 3], b[j], b[(j + 1) % 3])) return true;
        return x_point_in_tri_2d(a[0], b[0], b[1], b[2]) || x_point_in_tri_2d(b[0], a[0], a[1], a[2]);
    }
    for (int i = 0; i < 3; ++i)
        if (x_seg_tri(t[i], t[(i + 1) % 3], u[0], u[1], u[2]) ||
            x_seg_tri(u[i], u[(i + 1) % 3], t[0], t[1], t[2]))
            return true;
    return false;
}

// x coplanar with non-degenerate (v, a, b) and v -> x entering the closed
// angle of the triangle at v (x != v).
__device__ bool x_in_sector(const XP3& v, const XP3& a, const XP3& b, const XP3& x) {
    if (o3_exact(v, a, b, x) != 0) return false;
    if (x.x == v.x && x.y == v.y && x.z == v.z) return false;
    const int d = x_proj_axis(v, a, b);
    if (d < 0) return false;
    const XP2 V = x_proj(v, d), A = x_proj(a, d), B = x_proj(b, d), X = x_proj(x, d);
    const int o = o2_exact(V, A, B);
    const int s1 = o2_exact(V, A, X), s2 = o2_exact(V, X, B);
    if (s1 * o < 0 || s2 * o < 0) return false;
    auto sg = [](float p, float q) { return (p > q) - (p < q); };
    if (s1 == 0 && !(sg(A.x, V.x) == sg(X.x, V.x) && sg(A.y, V.y) == sg(X.y, V.y))) return false;
    if (s2 == 0 && !(sg(B.x, V.x) == sg(X.x, V.x) && sg(B.y, V.y) == sg(X.y, V.y))) return false;
    return true;
}

// Faces (ids ia, corners pa) and (ib, pb): do they intersect beyond what
// their shared vertices allow?  Degenerate faces are not tested.
__device__ bool x_faces_intersect(const int* ia, const XP3* pa, const int* ib, const XP3* pb) {
    if (x_proj_axis(pa[0], pa[1], pa[2]) < 0 || x_proj_axis(pb[0], pb[1], pb[2]) < 0) return false;
    int share = 0, sa[3] = {-1, -1, -1}, sb[3] = {-1, -1, -1};
    for (int i = 0; i < 3; ++i)
        for (int j = 0; j < 3; ++j)
            if (ia[i] == ib[j] && share < 3) {
                sa[share] = i;
                sb[share] = j;
                ++share;
            }
    if (share == 0) return x_tri_tri(pa, pb);
    if (share >= 3) return true;
    if (share == 1) {
        const int i = sa[0], j = sb[0];
        const XP3 v = pa[i], a = pa[(i + 1) % 3], b = pa[(i + 2) % 3];
        const XP3 c = pb[(j + 1) % 3], d = pb[(j + 2) % 3];
        return x_seg_tri(a, b, pb[0], pb[1], pb[2]) || x_seg_tri(c, d, pa[0], pa[1], pa[2]) ||
               x_in_sector(v, a, b, c) || x_in_sector(v, a, b, d) || x_in_sector(v, c, d, a) ||
               x_in_sector(v, c, d, b);
    }
    const int oa = 3 - sa[0] - sa[1], ob = 3 - sb[0] - sb[1];
    const XP3 u = pa[sa[0]], w = pa[sa[1]], a = pa[oa], b = pb[ob];
    if (o3_exact(u, w, a, b) != 0) return false;
    const int d = x_proj_axis(u, w, a);
    if (d < 0) return false;
    return o2_exact(x_proj(u, d), x_proj(w, d), x_proj(a, d)) == o2_exact(x_proj(u, d), x_proj(w, d), x_proj(b, d));
}

// The decision where filtered signs suffice, without arrays that are indexed
// at run time: kApart or kMeet, or kUnsure for x_faces_intersect.  Orientations
// change sign with every exchange of two points, which the signs below use.
// Most candidates share a vertex or an edge and end here after one to five
// determinants, in a query kernel of 84 registers and no scratch memory; with
// the whole decision in that kernel it took 248 registers and 208 B of scratch a
// lane.  A run on 200k faces with slivers: 118 us a query launch (336 before), 42
// us for the open pairs (115 before, with every expansion in scratch memory;
// now those of o3_raw and o2_raw alone are).
enum { kApart = 0, kMeet = 1, kUnsure = 2 };

__device__ __forceinline__ int x_o3(const XP3& a, const XP3& b, const XP3& c, const XP3& d) {
    return o3_filter(x_diff(a, b, c, d));
}
__device__ __forceinline__ bool x_strict(int s) { return s == 1 || s == -1; }
// Corner i of a face, by selection.
struct XFace {
    XP3 p0, p1, p2;
    int i0, i1, i2;
};
__device__ __forceinline__ float x_sel(int i, float a, float b, float c) { return i == 0 ? a : (i == 1 ? b : c); }
__device__ __forceinline__ XP3 x_pick(const XFace& f, int i) {
    return XP3{x_sel(i, f.p0.x, f.p1.x, f.p2.x), x_sel(i, f.p0.y, f.p1.y, f.p2.y), x_sel(i, f.p0.z, f.p1.z, f.p2.z)};
}
__device__ __forceinline__ int x_next(int i) { return i == 2 ? 0 : i + 1; }

__device__ __forceinline__ int x_faces_quick(XFace A, XFace B) {
    int rows = 0, cols = 0, share = 0;
    auto same = [&](int i, int j, bool eq) {
        share += eq;
        rows |= eq ? 1 << i : 0;
        cols |= eq ? 1 << j : 0;
    };
    same(0, 0, A.i0 == B.i0); same(0, 1, A.i0 == B.i1); same(0, 2, A.i0 == B.i2);
    same(1, 0, A.i1 == B.i0); same(1, 1, A.i1 == B.i1); same(1, 2, A.i1 == B.i2);
    same(2, 0, A.i2 == B.i0); same(2, 1, A.i2 == B.i1); same(2, 2, A.i2 == B.i2);
    if (share == 0) {
        // all corners of one face strictly on one side of the other's plane
        const int a0 = x_o3(B.p0, B.p1, B.p2, A.p0), a1 = x_o3(B.p0, B.p1, B.p2, A.p1),
                  a2 = x_o3(B.p0, B.p1, B.p2, A.p2);
        if (x_strict(a0) && a0 == a1 && a0 == a2) return kApart;
        const int b0 = x_o3(A.p0, A.p1, A.p2, B.p0), b1 = x_o3(A.p0, A.p1, A.p2, B.p1),
                  b2 = x_o3(A.p0, A.p1, A.p2, B.p2);
        if (x_strict(b0) && b0 == b1 && b0 == b2) return kApart;
        return kUnsure;
    }
    if (share == 2 && __popc(rows) == 2 && __popc(cols) == 2) {
        // not in one plane: they meet in the shared edge alone
        const int oa = rows == 6 ? 0 : (rows == 5 ? 1 : 2), ob = cols == 6 ? 0 : (cols == 5 ? 1 : 2);
        const int i1 = x_next(oa);
        const int s = x_o3(x_pick(A, i1), x_pick(A, x_next(i1)), x_pick(A, oa), x_pick(B, ob));
        return x_strict(s) ? kApart : kUnsure;
    }
    if (share != 1) return kUnsure;
    // v a b and v c d: with a and b strictly on one side of the plane of v c d
    // the first face touches that plane in v alone; else, with both pairs
    // strictly on two sides, a b meets v c d (c d meets v a b) if the line
    // passes the third side like the other two, whose signs are sc (sa)
    const int i = rows == 1 ? 0 : (rows == 2 ? 1 : 2), j = cols == 1 ? 0 : (cols == 2 ? 1 : 2);
    const XP3 v = x_pick(A, i), a = x_pick(A, x_next(i)), b = x_pick(A, x_next(x_next(i)));
    const XP3 c = x_pick(B, x_next(j)), d = x_pick(B, x_next(x_next(j)));
    const int sa = x_o3(v, c, d, a), sb = x_o3(v, c, d, b);
    if (x_strict(sa) && sa == sb) return kApart;
    const int sc = x_o3(v, a, b, c), sd = x_o3(v, a, b, d);
    if (x_strict(sc) && sc == sd) return kApart;
    if (!x_strict(sa) || !x_strict(sb) || !x_strict(sc) || !x_strict(sd)) return kUnsure;
    const int s = x_o3(a, b, c, d);
    if (!x_strict(s)) return kUnsure;
    return s == sc || s == sa ? kMeet : kApart;
}

}  // namespace
}  // namespace pamo
