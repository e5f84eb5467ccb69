// Face intersection, normals, aperture shapes and Zernike distortions (FP64).
//
// Each routine solves the equation of the reference face it stands in for, whose
// line is cited beside it, and takes its decisions (root choice, range and
// aperture tests, when a root search gives up) as it does; the arithmetic is its
// own, equal to a few ulp.  rpx_faces_ref.h has the intersections with the
// reference's roundings.  `is_base` is the reference's is_base_ray flag:
// parabasal rays skip most aperture tests.
#pragma once
#include "rpx_internal.h"

namespace rpx {

// --------------------------------------------------------------- shapes
// PolygonShape.point_inside_c (cshapes.pyx:150-168)
RPX_DEV bool polygon_shape_inside(const double *pts, int size, double X, double Y) {
    bool ct = false;
    double y1 = pts[2 * (size - 1) + 1], x1 = pts[2 * (size - 1)];
    for (int i = 0; i < size; ++i) {
        double y2 = pts[2 * i + 1], x2 = pts[2 * i];
        if ((y1 <= Y && Y < y2) || (y2 <= Y && Y < y1)) {
            if ((x1 + ((Y - y1) * (x2 - x1)) / (y2 - y1)) > X) ct = !ct;
        }
        y1 = y2;
        x1 = x2;
    }
    return ct;
}

// point_in_polygon_c used by PolygonFace (cfaces.pyx:1050-1068)
RPX_DEV bool polygon_face_inside(const double *pts, int size, double X, double Y) {
    bool ct = false;
    double y1 = pts[2 * (size - 1) + 1], x1 = pts[2 * (size - 1)];
    for (int i = 0; i < size; ++i) {
        double y2 = pts[2 * i + 1], x2 = pts[2 * i];
        double h = (Y - y1) / (y2 - y1);
        if (0.0 < h && h <= 1.0) {
            double x = x1 + h * (x2 - x1);
            if (x > X) ct = !ct;
        }
        y1 = y2;
        x1 = x2;
    }
    return ct;
}

// Shape tree (cshapes.pyx:34-168) evaluated as a postfix program.
RPX_DEV bool shape_inside(const SceneView &S, int root, double x, double y) {
    if (root < 0) return true;
    uint32_t stack = 0;
    int sp = 0;
    int begin = S.shape_ops[root].begin;
    for (int i = begin; i <= root; ++i) {
        const rpx_shape_op_t &op = S.shape_ops[i];
        uint32_t v = 0;
        switch (op.op) {
        case RPX_SHAPE_TRUE:
            v = 1;
            break;
        case RPX_SHAPE_CIRCLE: {
            double dx = x - op.p[0], dy = y - op.p[1];
            v = ((dx * dx) + (dy * dy) < (op.p[2] * op.p[2])) ? 1u : 0u;
        } break;
        case RPX_SHAPE_RECT: {
            double dx = x - op.p[0], dy = y - op.p[1];
            v = ((2 * fabs(dx) < op.p[2]) && (2 * fabs(dy)) < op.p[3]) ? 1u : 0u;
        } break;
        case RPX_SHAPE_POLYGON:
            v = polygon_shape_inside(S.vertices + 2 * op.a, op.b, x, y) ? 1u : 0u;
            break;
        case RPX_SHAPE_NOT:
            --sp;
            v = ((stack >> sp) & 1u) ^ 1u;
            stack &= ~(1u << sp);
            break;
        default: {  // AND / OR / XOR
            --sp;
            uint32_t b = (stack >> sp) & 1u;
            stack &= ~(1u << sp);
            --sp;
            uint32_t a = (stack >> sp) & 1u;
            stack &= ~(1u << sp);
            v = op.op == RPX_SHAPE_AND ? (a & b) : op.op == RPX_SHAPE_OR ? (a | b) : (a ^ b);
        } break;
        }
        stack |= (v << sp);
        ++sp;
    }
    return ((stack >> (sp - 1)) & 1u) != 0;
}

// ------------------------------------------------------------- Zernike
// The memoised radial recursion of cdistortions.pyx:149-316 is expanded at
// scene build into integer polynomials in r (rpx_zernike_coef_t.poly, the
// exact values of the compiled recursion, slot sharing included).  Scene
// creation sums N * polynomial over the coefficients of one |m| and parity
// (ZGroup), so a distortion is evaluated as one Horner chain in r^2 per
// group and quantity, with cos and sin(m theta) advanced from group to group
// by the angle-addition recurrence.  Noll 4-15 (twelve coefficients, five
// groups of three terms): about 160 float64 instructions per gradient and 70
// per sag, against 670 and 330 with a chain in r over all ten powers, and a
// fresh recurrence, per coefficient; the Michelson trace of 65,536 rays to
// depth 12 went from 23.3 to 16.0 ms on MI355X.
//
// When every active lane evaluates the same distortion the tables are read
// through the constant address space, i.e. with scalar loads into SGPRs;
// otherwise (per-lane faces: normals, parabasal rays) with vector loads.
// The scene tables are not written while kernels run.
typedef __attribute__((address_space(4))) const ZTable ZTableK;
typedef __attribute__((address_space(4))) const ZGroup ZGroupK;

// sum of p[i] u^i over the first T coefficients
template <int T, class PT>
RPX_DEV double zhorner(PT &p, double u) {
    double v = p[T - 1];
#pragma unroll
    for (int i = T - 2; i >= 0; --i) v = fma(v, u, p[i]);
    return v;
}

// Normalised polar position of (x, y): r, u = r^2, cos and sin of theta =
// atan2(y, x) (at r = 0 those of atan2's branch values 0 and pi).
struct ZPolar {
    double r, u, ct, st;
};

template <class ZT>
RPX_DEV ZPolar zpolar(ZT &Z, double x, double y) {
    ZPolar q;
    x *= Z.inv_radius;
    y *= Z.inv_radius;
    q.u = fma(x, x, y * y);
    const double rs = rsq_third(q.u);
    q.r = q.u * rs;
    q.ct = x * rs;
    q.st = y * rs;
    if (!(q.u > 1e-280)) {      // 0 (or NaN), and where the estimate would overflow
        const bool zero = q.u == 0.0;
        q.r = sqrt(q.u);
        q.ct = zero ? copysign(1.0, x) : x / q.r;
        q.st = zero ? copysign(signbit(x) ? 1.2246467991473532e-16 : 0.0, y) : y / q.r;
    }
    return q;
}

// cos and sin(m theta), advanced in m
struct ZHarmonic {
    double c = 1.0, s = 0.0;
    int m = 0;
    RPX_DEV void to(int target, const ZPolar &q) {
        for (; m < target; ++m) {
            const double cn = fma(c, q.ct, -(s * q.st));
            s = fma(s, q.ct, c * q.st);
            c = cn;
        }
    }
};

// ZernikeDistortion.z_offset_c (cdistortions.pyx:416-450): the sum over
// groups of (SC(u) cos(m theta) + SS(u) sin(m theta)) r^odd, where SC collects the
// coefficients with m >= 0 and SS those with m < 0 (-sin(m theta) = sin(|m|
// theta)).
template <int T, class ZT, class GT>
RPX_DEV double zernike_sag_t(ZT &Z, GT *groups, double x, double y) {
    const ZPolar q = zpolar(Z, x, y);
    ZHarmonic h;
    double z = 0.0;
    for (int i = 0; i < Z.n; ++i) {
        GT &g = groups[Z.first + i];
        h.to(g.m, q);
        const double v = fma(zhorner<T>(g.p[ZG_SAG_C], q.u), h.c, zhorner<T>(g.p[ZG_SAG_S], q.u) * h.s);
        z = fma(v, g.odd ? q.r : 1.0, z);
    }
    return z;
}

RPX_DEV double zernike_sag(const SceneView &S, int zi, double x, double y) {
    const int z0 = __builtin_amdgcn_readfirstlane(zi);
    if (__ballot(zi != z0) == 0) {
        ZTableK &Z = ((ZTableK *)S.ztables)[z0];
        if (Z.terms <= 3) return zernike_sag_t<3>(Z, (ZGroupK *)S.zgroups, x, y);
        return zernike_sag_t<ZG_TERMS>(Z, (ZGroupK *)S.zgroups, x, y);
    }
    return zernike_sag_t<ZG_TERMS>(S.ztables[zi], S.zgroups, x, y);
}

// ZernikeDistortion.z_offset_and_gradient_c (cdistortions.pyx:456-514):
// returns (dz/dx, dz/dy, z).  With P = sum R'_C cos + R'_S sin and Q = sum m
// ((R/r)_S cos - (R/r)_C sin), the gradient is (ct P - st Q, st P + ct Q) / Ru.
template <int T, class ZT, class GT>
RPX_DEV V3 zernike_grad_t(ZT &Z, GT *groups, double x, double y) {
    const ZPolar q = zpolar(Z, x, y);
    ZHarmonic h;
    double z = 0.0, P = 0.0, Q = 0.0;
    for (int i = 0; i < Z.n; ++i) {
        GT &g = groups[Z.first + i];
        h.to(g.m, q);
        const double vz = fma(zhorner<T>(g.p[ZG_R_C], q.u), h.c, zhorner<T>(g.p[ZG_R_S], q.u) * h.s);
        const double vp = fma(zhorner<T>(g.p[ZG_RP_C], q.u), h.c, zhorner<T>(g.p[ZG_RP_S], q.u) * h.s);
        const double vq = fma(zhorner<T>(g.p[ZG_ROR_S], q.u), h.c, -(zhorner<T>(g.p[ZG_ROR_C], q.u) * h.s));
        const double fz = g.odd ? q.r : 1.0, fd = g.odd ? 1.0 : q.r;
        z = fma(vz, fz, z);
        P = fma(vp, fd, P);
        Q = fma(vq * (double)g.m, fd, Q);
    }
    return v3(fma(q.ct, P, -(q.st * Q)) * Z.inv_radius, fma(q.st, P, q.ct * Q) * Z.inv_radius, z);
}

RPX_DEV V3 zernike_grad(const SceneView &S, int zi, double x, double y) {
    const int z0 = __builtin_amdgcn_readfirstlane(zi);
    if (__ballot(zi != z0) == 0) {
        ZTableK &Z = ((ZTableK *)S.ztables)[z0];
        if (Z.terms <= 3) return zernike_grad_t<3>(Z, (ZGroupK *)S.zgroups, x, y);
        return zernike_grad_t<ZG_TERMS>(Z, (ZGroupK *)S.zgroups, x, y);
    }
    return zernike_grad_t<ZG_TERMS>(S.ztables[zi], S.zgroups, x, y);
}

// -------------------------------------------------------------- segments
// A ray segment in a face list's frame: from p1 along the unit vector u for
// slen.  The reference parametrises a segment by the fraction h of p2 - p1 and
// scales the root it accepts by |p2 - p1|, for every face (cfaces.pyx); here a
// face's test gives the distance itself, so that the length, the reciprocals
// and the unit vector are formed once per face list (once for all lists that
// share the global frame) and a plane costs a multiplication.  Roots agree
// with the reference's to a few ulp of the segment.
struct Seg {
    V3 p1, u;
    double slen, inv_uz;
};

RPX_DEV Seg make_seg(V3 p1, V3 p2) {
    Seg g;
    const V3 s = sub(p2, p1);
    g.p1 = p1;
    g.slen = sqrt(fma(s.x, s.x, fma(s.y, s.y, s.z * s.z)));
    g.u = mul(s, 1.0 / g.slen);
    g.inv_uz = 1.0 / g.u.z;
    return g;
}

RPX_DEV V3 seg_at(const Seg &g, double t) {
    return v3(fma(g.u.x, t, g.p1.x), fma(g.u.y, t, g.p1.y), fma(g.u.z, t, g.p1.z));
}

// Face list flags, set at scene creation in rpx_face_list_t.pad[0].
enum : int { FL_INV_IDENTITY = 1, FL_TRANS_IDENTITY = 2 };

RPX_DEV V3 to_local(const rpx_face_list_t &fl, V3 p) {
    if (fl.pad[0] & FL_INV_IDENTITY) return p;
    return transform(fl.inv_trans, p);
}
RPX_DEV V3 to_global_dir(const rpx_face_list_t &fl, V3 d) {
    if (fl.pad[0] & FL_TRANS_IDENTITY) return d;
    return rotate(fl.trans, d);
}

// ----------------------------------------------------------- conic / asphere
// intersect_conic (cfaces.pyx:1695-1747) for a unit direction d: the distance
// t, or false where the ray misses the conic.
RPX_DEV bool intersect_conic(V3 a, V3 d, double curvature, double conic_const, double &t) {
    const double beta = 1 + conic_const;
    const double R = -curvature;
    const double b2 = beta * beta;
    const double dt = fma(d.x, d.x, d.y * d.y), at = fma(a.x, a.x, a.y * a.y), ad = fma(a.x, d.x, a.y * d.y);
    const double A = fma(b2, d.z * d.z, beta * dt);
    // half of the reference's B
    const double B = fma(beta, fma(-R, d.z, ad), b2 * (a.z * d.z));
    const double C = fma(beta, fma(-2 * R, a.z, at), b2 * (a.z * a.z));
    double D = fma(B, B, -(A * C));
    if (D < 0) return false;
    D = sqrt(D);
    t = (R * beta * d.z <= 0 ? -B + D : -B - D) / A;
    return true;
}

// x = r^2 polynomial A4 x^2 + .. + A16 x^8 and its derivative, by Horner's rule
// (p[3..9] of an aspheric face).
RPX_DEV double asph_poly(const rpx_face_t &f, double x) {
    double v = f.p[9];
#pragma unroll
    for (int i = 8; i >= 3; --i) v = fma(v, x, f.p[i]);
    return v * (x * x);
}
RPX_DEV double asph_dpoly(const rpx_face_t &f, double x) {
    double v = 8 * f.p[9];
#pragma unroll
    for (int i = 8; i >= 3; --i) v = fma(v, x, (i - 1) * f.p[i]);
    return v * x;
}

// A base-ray hit on an aspheric face is accepted only inside the aperture,
// where the surface lies within z_height +/- p[12]; the converged root
// satisfies the sag equation to within the Newton tolerance.  A segment whose
// z-range misses that band cannot be accepted.
RPX_DEV bool asph_outside_band(const rpx_face_t &f, const Seg &g, int is_base) {
    if (!is_base || f.p[12] < 0.0) return false;
    const double m = f.p[12] + 1e-9 * (1.0 + fabs(f.p[1]) + f.p[12]) + 10.0 * f.p[10] * g.slen * (1.0 + f.p[13]);
    const double z2 = fma(g.u.z, g.slen, g.p1.z);
    return fmax(g.p1.z, z2) < f.p[1] - m || fmin(g.p1.z, z2) > f.p[1] + m;
}

// A base ray's nearest-face search only accepts a face's hit closer than
// the nearest one so far.  p[14]..p[15] of a face record hold a z band (in
// its face list's frame, widened for rounding on the host; NaN when not
// bounded) containing every point at which the face can accept a base-ray
// hit; an aspheric face's Newton tolerance widens it by a multiple of the
// segment length, as in asph_outside_band.  If the part of the segment
// closer than the current nearest hit -- z from z1 over zspan -- misses the
// band, the face cannot give a nearer hit and its exact test is skipped.
// Skipping removes only candidates the exact test would reject, so the
// nearest face, its distance and the tie rule are unchanged.
RPX_DEV bool face_out_of_reach(const rpx_face_t &f, double z1, double zspan, double slen) {
    const double m = f.type == RPX_FACE_ASPHERIC ? 10.0 * f.p[10] * slen * (1.0 + f.p[13]) : 0.0;
    const double z2 = z1 + zspan;
    return fmax(z1, z2) < f.p[14] - m || fmin(z1, z2) > f.p[15] + m;
}

// ------------------------------------------------------------- intersect
// Face record k of a table in global memory, for an index that is the same
// in every lane: read through the constant address space, i.e. with scalar
// loads into SGPRs (word by word, so that the host pass of the compiler,
// which cannot copy-construct from that address space, accepts it).  Scene
// tables are not written while kernels run.
RPX_DEV rpx_face_t face_uniform(const rpx_face_t *faces, int k) {
    typedef __attribute__((address_space(4))) const uint64_t WordK;
    static_assert(sizeof(rpx_face_t) % 8 == 0, "face records are copied as 64-bit words");
    const WordK *w = (const WordK *)(faces + k);
    rpx_face_t f;
    uint64_t *d = (uint64_t *)&f;
#pragma unroll
    for (int i = 0; i < (int)(sizeof(rpx_face_t) / 8); ++i) d[i] = w[i];
    return f;
}

// Whether a root at distance t passes the reference's range test on h = t /
// slen (tol <= h <= 1); false for NaN.
RPX_DEV bool in_segment(const Seg &g, double t, double tol) { return t >= tol * g.slen && t <= g.slen; }

// Base-face intersection, also used by DistortionFace (no recursion into a
// second distortion level: the host refuses nested distortions).  Returns the
// distance, or -1.
template <uint32_t F>
RPX_DEV double plain_intersect(const SceneView &S, const rpx_face_t &f, const Seg &g, int is_base) {
    const double tol = f.tolerance;
    switch (f.type) {
    case RPX_FACE_CIRCULAR: {
        if constexpr ((F & F_PLANE) == 0) return -1;  // cfaces.pyx:151-178
        const double t = (f.p[2] - g.p1.z) * g.inv_uz, d = f.p[0];
        if (!in_segment(g, t, tol)) return -1;
        const double X = fma(g.u.x, t, g.p1.x) - f.p[1], Y = fma(g.u.y, t, g.p1.y);
        if (is_base && fma(X, X, Y * Y) > (d * d / 4)) return -1;
        return t;
    }
    case RPX_FACE_SHAPED_PLANAR: {
        if constexpr ((F & F_PLANE) == 0) return -1;  // cfaces.pyx:201-226
        const double t = (f.p[0] - g.p1.z) * g.inv_uz;
        if (!in_segment(g, t, tol)) return -1;
        if (is_base && !shape_inside(S, f.shape, fma(g.u.x, t, g.p1.x), fma(g.u.y, t, g.p1.y))) return -1;
        return t;
    }
    case RPX_FACE_RECTANGULAR: {
        if constexpr ((F & F_PLANE) == 0) return -1;  // cfaces.pyx:365-397
        const double t = (f.p[3] - g.p1.z) * g.inv_uz;
        if (!in_segment(g, t, tol)) return -1;
        if (is_base) {
            const double X = fma(g.u.x, t, g.p1.x) - f.p[2], Y = fma(g.u.y, t, g.p1.y);
            if (X * X > f.p[0] * f.p[0] / 4) return -1;
            if (Y * Y > f.p[1] * f.p[1] / 4) return -1;
        }
        return t;
    }
    case RPX_FACE_POLYGON: {
        if constexpr ((F & F_PLANE) == 0) return -1;  // cfaces.pyx:1093-1108
        const double t = (f.p[0] - g.p1.z) * g.inv_uz;
        if (!is_base || !in_segment(g, t, tol)) return -1;
        return polygon_face_inside(S.vertices + 2 * f.aux0, f.aux1, fma(g.u.x, t, g.p1.x), fma(g.u.y, t, g.p1.y))
                   ? t : -1;
    }
    case RPX_FACE_SPHERICAL:
    case RPX_FACE_SHAPED_SPHERICAL: {
        if constexpr ((F & F_SPHERE) == 0) return -1;  // cfaces.pyx:421-486 / 513-576
        const bool shaped = f.type == RPX_FACE_SHAPED_SPHERICAL;
        const double curvature = shaped ? f.p[0] : f.p[1];
        const double z_height = shaped ? f.p[1] : f.p[2];
        const double cz = z_height - curvature;
        V3 d = g.p1;
        d.z -= cz;
        // half of the reference's B, over |s|
        const double B = fma(g.u.x, d.x, fma(g.u.y, d.y, g.u.z * d.z));
        const double C = fma(d.x, d.x, fma(d.y, d.y, d.z * d.z)) - curvature * curvature;
        double D = fma(B, B, -C);
        if (D < 0) return -1;
        D = sqrt(D);
        double a1 = D - B, a2 = -B - D;
        const V3 pt1 = seg_at(g, a1), pt2 = seg_at(g, a2);
        if (curvature >= 0) {
            if (pt1.z < cz) a1 = RPX_INF;
            if (pt2.z < cz) a2 = RPX_INF;
        } else {
            if (pt1.z > cz) a1 = RPX_INF;
            if (pt2.z > cz) a2 = RPX_INF;
        }
        if (is_base) {
            if (shaped) {
                if (!shape_inside(S, f.shape, pt1.x, pt1.y)) a1 = RPX_INF;
                if (!shape_inside(S, f.shape, pt2.x, pt2.y)) a2 = RPX_INF;
            } else {
                const double DD = f.p[0] * f.p[0] / 4.;
                if (fma(pt1.x, pt1.x, pt1.y * pt1.y) > DD) a1 = RPX_INF;
                if (fma(pt2.x, pt2.x, pt2.y * pt2.y) > DD) a2 = RPX_INF;
            }
        }
        if (a2 < a1) a1 = a2;
        return in_segment(g, a1, tol) ? a1 : -1;
    }
    case RPX_FACE_EXTRUDED_PLANAR: {
        if constexpr ((F & F_PLANE) == 0) return -1;  // cfaces.pyx:665-699
        const double ux = f.p[0], uy = f.p[1];
        const double vx = f.p[2] - ux, vy = f.p[3] - uy;
        const double den = fma(g.u.x, vy, -(g.u.y * vx));
        const double ax = g.p1.x - ux, ay = g.p1.y - uy;
        if (is_base) {
            // the position along the edge, num / den, must lie in 0..1
            const double num = fma(g.u.x, ay, -(g.u.y * ax));
            const double q = den < 0 ? -num : num;
            if (q < 0 || q > fabs(den)) return -1;
        }
        const double num = fma(vx, ay, -(vy * ax));
        // behind the start: no division, where the caller would reject it
        if (is_base && tol >= 0 && (den < 0 ? num > 0 : num < 0)) return -1;
        const double t = num / den;
        if (is_base) {
            const double zz = fma(g.u.z, t, g.p1.z);
            return f.p[4] < zz && zz < f.p[5] ? t : -1;
        }
        return t;
    }
    case RPX_FACE_CONIC: {
        if constexpr ((F & F_CONIC) == 0) return -1;  // cfaces.pyx:1767-1798
        V3 a = g.p1;
        a.z -= f.p[1];
        double t;
        if (!intersect_conic(a, g.u, f.p[0], f.p[2], t)) return -1;
        if (is_base && !shape_inside(S, f.shape, fma(g.u.x, t, a.x), fma(g.u.y, t, a.y))) return -1;
        return in_segment(g, t, tol) ? t : -1;
    }
    case RPX_FACE_ASPHERIC: {
        if constexpr ((F & F_ASPHERE) == 0) return -1;  // cfaces.pyx:1909-1976
        if (asph_outside_band(f, g, is_base)) return -1;
        // Newton from the conic's root on f(t) = r^2 / (R (1 + w)) + P(r^2) -
        // (a.z + t u.z), w = sqrt(1 - beta r^2 / R^2); the conic term's
        // derivative in r^2 is 1 / (2 R w) (the reference's two fractions,
        // cfaces.pyx:1866-1882, added up), so a step takes one square root and
        // one division.  A ray that misses the conic starts at h = -1 as in the
        // reference, a whole segment behind p1: from nearer by, the iteration
        // finds roots that the reference does not accept.
        const double atol = f.p[10] * g.slen;
        const double tl = atol * atol;
        V3 a = g.p1;
        a.z -= f.p[1];
        const double R = -f.p[0], k2 = (1 + f.p[2]) / (R * R);
        double t;
        if (!intersect_conic(a, g.u, f.p[0], f.p[2], t)) t = -g.slen;
        double f_last = RPX_INF, dt = RPX_INF;
        bool converged = false;
        for (int i = 0; i <= 100; ++i) {
            const double tx = fma(t, g.u.x, a.x), ty = fma(t, g.u.y, a.y);
            const double r2 = fma(tx, tx, ty * ty);
            const double w = sqrt(fma(-k2, r2, 1.0)), w1 = 1 + w;
            const double inv = 1.0 / (R * w * w1);
            const double fv = fma(r2 * w, inv, asph_poly(f, r2)) - fma(t, g.u.z, a.z);
            // growing, or no number (outside the conic's domain), which no later
            // step can mend: the reference runs its 100 steps on it
            if (!(fabs(fv) <= fabs(f_last))) return -1;
            f_last = fv;
            const double slope = fma(w1, inv, 2 * asph_dpoly(f, r2));
            dt = -fv / fma(fma(g.u.x, tx, g.u.y * ty), slope, -g.u.z);
            if (i == 100) break;
            t += dt;
            if (dt * dt < tl) { converged = true; break; }
        }
        if (!converged) return -1;
        if (is_base && !shape_inside(S, f.shape, fma(g.u.x, t, a.x), fma(g.u.y, t, a.y))) return -1;
        return in_segment(g, t, tol) ? t : -1;
    }
    default:
        return -1;
    }
}

// Local-frame normal of a face (compute_normal_c of each class).
template <uint32_t F>
RPX_DEV V3 plain_normal(const SceneView &S, const rpx_face_t &f, V3 p) {
    switch (f.type) {
    case RPX_FACE_CIRCULAR:  // cfaces.pyx:180-191
        return v3(0, 0, f.invert_normals ? 1 : -1);
    case RPX_FACE_SHAPED_PLANAR:  // cfaces.pyx:228-236
        return v3(0, 0, 1);
    case RPX_FACE_RECTANGULAR:
    case RPX_FACE_POLYGON:  // cfaces.pyx:399-407, 1110-1118
        return v3(0, 0, -1);
    case RPX_FACE_SPHERICAL:
    case RPX_FACE_SHAPED_SPHERICAL: {
        if constexpr ((F & F_SPHERE) == 0) return p;  // cfaces.pyx:488-498
        const bool shaped = f.type == RPX_FACE_SHAPED_SPHERICAL;
        const double curvature = shaped ? f.p[0] : f.p[1];
        const double z_height = shaped ? f.p[1] : f.p[2];
        p.z -= (z_height - curvature);
        if (curvature < 0) {
            p.z = -p.z;
            p.y = -p.y;
            p.x = -p.x;
        }
        return unit(p);
    }
    case RPX_FACE_EXTRUDED_PLANAR:  // cfaces.pyx:701-702
        return v3(f.p[6], f.p[7], f.p[8]);
    case RPX_FACE_CONIC: {
        if constexpr ((F & F_CONIC) == 0) return p;  // cfaces.pyx:1800-1823
        double R = -f.p[0];
        double beta = 1 + f.p[2];
        int sign = f.invert_normals ? -1 : 1;
        p.z -= f.p[1];
        V3 g;
        g.z = 2 * beta * (R - beta * p.z);
        g.x = -p.x * 2 * beta;
        g.y = -p.y * 2 * beta;
        if ((R * beta) < 0) sign *= -1;
        g.z *= sign;
        g.y *= sign;
        g.x *= sign;
        return unit(g);
    }
    case RPX_FACE_ASPHERIC: {
        if constexpr ((F & F_ASPHERE) == 0) return p;  // cfaces.pyx:1978-2007
        const double R = -f.p[0];
        const int sign = f.invert_normals ? -1 : 1;
        const double r2 = fma(p.x, p.x, p.y * p.y);
        const double w = sqrt(fma(-(1 + f.p[2]) / (R * R), r2, 1.0));
        const double df = 1.0 / (R * w) + 2 * asph_dpoly(f, r2);
        return unit(v3(-df * p.x * sign, -df * p.y * sign, sign));
    }
    default:
        return p;
    }
}

// DistortionFace.intersect_c (cfaces.pyx:2339-2416)
template <uint32_t F>
RPX_DEV double distortion_intersect(const SceneView &S, const rpx_face_t &f, const Seg &g) {
    const rpx_face_t &face = S.faces[f.aux0];
    const int zi = f.aux1;
    double a1, a2;
    const double tolerance = f.p[0];
    a2 = plain_intersect<F>(S, face, g, 0);
    if (a2 > g.slen || a2 < f.tolerance) return -1;
    V3 pt1 = seg_at(g, a2);
    // distance to the tangent plane of base + distortion at pt1
    auto tangent_plane = [&](V3 &pt, double &dz) {
        const V3 grad = zernike_grad(S, zi, pt.x, pt.y);
        V3 n = plain_normal<F>(S, face, pt);
        const double inv = 1.0 / n.z;
        pt.z += grad.z;
        dz = grad.z;
        n.x = fma(n.x, inv, -grad.x);
        n.y = fma(n.y, inv, -grad.y);
        return -dot(sub(g.p1, pt), n) / dot(g.u, n);
    };
    double dz;
    a1 = tangent_plane(pt1, dz);
    if (a1 < fabs(dz)) return -1;
    for (int i = 0; i < 20; ++i) {
        pt1 = seg_at(g, a1);
        if (fabs(a1 - a2) < tolerance) break;
        Seg q = g;
        q.p1.z -= zernike_sag(S, zi, pt1.x, pt1.y);
        a2 = plain_intersect<F>(S, face, q, 0);
        pt1 = seg_at(q, a2);
        const double t = tangent_plane(pt1, dz);
        a2 = a1;
        a1 = t;
    }
    if (!shape_inside(S, f.shape, pt1.x, pt1.y)) return -1;
    return a1;
}

template <uint32_t F>
RPX_DEV double face_intersect(const SceneView &S, const rpx_face_t &f, const Seg &g, int is_base) {
    if constexpr ((F & F_DISTORT) != 0) {
        if (f.type == RPX_FACE_DISTORTION) return distortion_intersect<F>(S, f, g);
    }
    return plain_intersect<F>(S, f, g, is_base);
}

// DistortionFace.compute_normal_c (cfaces.pyx:2418-2431)
template <uint32_t F>
RPX_DEV V3 face_normal(const SceneView &S, const rpx_face_t &f, V3 p) {
    if constexpr ((F & F_DISTORT) == 0) {
        return plain_normal<F>(S, f, p);
    }
    if (f.type != RPX_FACE_DISTORTION) return plain_normal<F>(S, f, p);
    V3 dxdyz = zernike_grad(S, f.aux1, p.x, p.y);
    V3 p1 = p;
    p1.z -= dxdyz.z;
    V3 n = plain_normal<F>(S, S.faces[f.aux0], p1);
    n.x /= n.z;
    n.y /= n.z;
    n.z = 1.0;
    n.x -= dxdyz.x;
    n.y -= dxdyz.y;
    return unit(n);
}

// compute_tangent_c: (1,0,0) by default, (0,0,1) for ExtrudedPlanarFace
// (ctracer.pyx:1786-1791, cfaces.pyx:704-709).
RPX_DEV V3 face_tangent(const rpx_face_t &f) {
    if (f.type == RPX_FACE_EXTRUDED_PLANAR) return v3(0.0, 0.0, 1.0);
    return v3(1.0, 0.0, 0.0);
}

struct Orientation {
    V3 normal, tangent;
};

// FaceList.compute_orientation_c (ctracer.pyx:1939-1953)
template <uint32_t F>
RPX_DEV Orientation compute_orientation(const SceneView &S, const rpx_face_list_t &fl,
                                        const rpx_face_t &f, V3 point) {
    point = to_local(fl, point);
    Orientation o;
    o.normal = face_normal<F>(S, f, point);
    o.tangent = face_tangent(f);
    if (f.invert_normal) {
        o.normal = neg(o.normal);
        o.tangent = neg(o.tangent);
    }
    o.normal = to_global_dir(fl, o.normal);
    o.tangent = to_global_dir(fl, o.tangent);
    return o;
}

// ---------------------------------------------------------- nearest face
struct NearHit {
    double length;
    uint32_t end_face;
    int rec, list;          // face record and face list, -1 without a hit
};

// trace_segment_c / FaceList.intersect_c (ctracer.pyx:2093-2104, 1882-1904), or
// with one_list >= 0 FaceList.intersect_one_face_c (:1861-1879): the first of
// the nearest faces closer than `length`.  Face lists whose frame is the
// global one share one segment.  Face and list indices are the same in every
// lane; with SCALAR the face records are read from `faces` in global memory by
// scalar loads (into SGPRs), otherwise from the LDS copy S holds.
template <uint32_t F, bool SCALAR>
RPX_DEV NearHit nearest_face(const SceneView &S, const rpx_face_t *faces, V3 origin, V3 dir, double max_length,
                             double length, int one_list, int one_face) {
    NearHit h{length, RPX_NO_FACE, -1, -1};
    const V3 point = add(origin, mul(dir, max_length));
    const int l0 = one_list < 0 ? 0 : one_list, l1 = one_list < 0 ? S.n_face_lists : one_list + 1;
    Seg g;
    bool global_frame = false;   // g is in the global frame
    for (int l = l0; l < l1; ++l) {
        const rpx_face_list_t &fl = S.face_lists[l];
        const int flags = __builtin_amdgcn_readfirstlane(fl.pad[0]);
        if (flags & FL_INV_IDENTITY) {
            if (!global_frame) g = make_seg(origin, point);
            global_frame = true;
        } else {
            g = make_seg(transform(fl.inv_trans, origin), transform(fl.inv_trans, point));
            global_frame = false;
        }
        const int k0 = __builtin_amdgcn_readfirstlane(one_list < 0 ? fl.first_face : fl.first_face + one_face);
        const int k1 = __builtin_amdgcn_readfirstlane(one_list < 0 ? fl.first_face + fl.n_faces : k0 + 1);
        for (int k = k0; k < k1; ++k) {
            auto test = [&](const rpx_face_t &fc) {
                if (face_out_of_reach(fc, g.p1.z, g.u.z * h.length, g.slen)) return;
                const double dist = face_intersect<F>(S, fc, g, 1);
                if (fc.tolerance < dist && dist < h.length) {
                    h.length = dist;
                    h.end_face = (uint32_t)fc.global_idx;
                    h.rec = k;
                    h.list = l;
                }
            };
            if constexpr (SCALAR) test(face_uniform(faces, k));
            else test(S.faces[k]);
        }
    }
    return h;
}

}  // namespace rpx
