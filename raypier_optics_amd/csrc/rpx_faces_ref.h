// Face intersections with the reference's own roundings: the segment p1..p2 is
// parametrised by the fraction h, and every expression keeps the operation
// order of cfaces.pyx (the sources that include this are compiled without
// contraction).  Capture selection and the Face.intersect query use them: a
// capture surface may be the face that the ray already ended on, and then the
// last bit of h decides whether h <= 1.  The traces use rpx_faces.h, whose
// nearest hits lie inside their segments.
#pragma once
#include "rpx_faces.h"

namespace rpx {
namespace ref {

// intersect_conic (cfaces.pyx:1695-1747)
RPX_DEV double intersect_conic(V3 a, V3 d, double curvature, double conic_const) {
    double beta = 1 + conic_const;
    double R = -curvature;
    double b2 = beta * beta;
    double A = b2 * (d.z * d.z) + beta * (d.x * d.x) + beta * (d.y * d.y);
    double B = -2 * R * beta * d.z + 2 * a.x * beta * d.x + 2 * a.y * beta * d.y + 2 * a.z * b2 * d.z;
    double C = -2 * R * a.z * beta + (a.x * a.x) * beta + (a.y * a.y) * beta + (a.z * a.z) * b2;
    double D = B * B - 4 * A * C;
    if (D < 0) return -1;
    D = sqrt(D);
    if (R * beta * d.z <= 0) return (-B + D) / (2 * A);
    return (-B - D) / (2 * A);
}

// x^2 .. x^nmax into pw[2..nmax].  x^2 is the rounded product (the
// reference's x**2); higher powers come from a double-double product chain
// rounded once, i.e. correctly rounded like the C library's pow for these
// integer exponents, at a fraction of pow's cost.
RPX_DEV void pow_chain(double x, double *pw, int nmax) {
    double hi = x * x;
    double lo = fma(x, x, -hi);
    pw[2] = hi;
    for (int k = 3; k <= nmax; ++k) {
        double p = hi * x;
        double e = fma(hi, x, -p);
        lo = fma(lo, x, e);
        double s = p + lo;
        lo = lo - (s - p);
        hi = s;
        pw[k] = hi + lo;
    }
}

struct Asph {
    double R, beta, A4, A6, A8, A10, A12, A14, A16, R3;
    V3 a, d;
};

// eval_aspheric_impf (cfaces.pyx:1854-1863)
RPX_DEV double asph_impf(const Asph &A, double alpha) {
    double tx = A.a.x + alpha * A.d.x, ty = A.a.y + alpha * A.d.y;
    double r2 = (tx * tx + ty * ty);
    double pw[9];
    pow_chain(r2, pw, 8);
    double out = r2;
    out /= A.R * (1 + sqrt(1 - A.beta * r2 / (A.R * A.R)));
    out -= A.a.z + alpha * A.d.z;
    out += A.A4 * pw[2] + A.A6 * pw[3] + A.A8 * pw[4] + A.A10 * pw[5] + A.A12 * pw[6] + A.A14 * pw[7] +
           A.A16 * pw[8];
    return out;
}

// eval_aspheric_grad (cfaces.pyx:1866-1882)
RPX_DEV double asph_grad(const Asph &A, double alpha) {
    double tx = A.a.x + alpha * A.d.x, ty = A.a.y + alpha * A.d.y;
    double r2 = (tx * tx + ty * ty);
    double dx = A.d.x * tx;
    double dy = A.d.y * ty;
    double pw[8];
    pow_chain(r2, pw, 7);
    double out = A.A10 * (10 * dx + 10 * dy) * pw[4];
    out += A.A12 * (12 * dx + 12 * dy) * pw[5];
    out += A.A14 * (14 * dx + 14 * dy) * pw[6];
    out += A.A16 * (16 * dx + 16 * dy) * pw[7];
    out += A.A4 * (4 * dx + 4 * dy) * (r2);
    out += A.A6 * (6 * dx + 6 * dy) * pw[2];
    out += A.A8 * (8 * dx + 8 * dy) * pw[3] - A.d.z;
    out += (2 * dx + 2 * dy) / (A.R * (sqrt(1 - A.beta * (r2) / (A.R * A.R)) + 1));
    double s = sqrt(1 - A.beta * r2 / (A.R * A.R));
    double s1 = s + 1;
    out += A.beta * (2 * dx + 2 * dy) * (r2) / (2 * A.R3 * s * (s1 * s1));
    return out;
}

// As rpx::asph_outside_band.
RPX_DEV bool asph_outside_band(const rpx_face_t &f, V3 p1, V3 p2, int is_base) {
    if (!is_base || f.p[12] < 0.0) return false;
    double len = sep(p1, p2);
    double m = f.p[12] + 1e-9 * (1.0 + fabs(f.p[1]) + f.p[12]) + 10.0 * f.p[10] * len * (1.0 + f.p[13]);
    double zlo = fmin(p1.z, p2.z), zhi = fmax(p1.z, p2.z);
    return zhi < f.p[1] - m || zlo > f.p[1] + m;
}

// Base-face intersection, also used by DistortionFace (no recursion into a second
// distortion level: the host refuses nested distortions).
template <uint32_t F>
RPX_DEV double plain_intersect(const SceneView &S, const rpx_face_t &f, V3 p1, V3 p2, int is_base) {
    const double tol = f.tolerance;
    switch (f.type) {
    case RPX_FACE_CIRCULAR: {
        if constexpr ((F & F_PLANE) == 0) return -1;  // cfaces.pyx:151-178
        double max_length = sep(p1, p2);
        double h = (f.p[2] - p1.z) / (p2.z - p1.z);
        double d = f.p[0];
        if ((h < tol) || (h > 1.0)) return -1;
        double X = p1.x + h * (p2.x - p1.x) - f.p[1];
        double Y = p1.y + h * (p2.y - p1.y);
        if (is_base && (X * X + Y * Y) > (d * d / 4)) return -1;
        return h * max_length;
    }
    case RPX_FACE_SHAPED_PLANAR: {
        if constexpr ((F & F_PLANE) == 0) return -1;  // cfaces.pyx:201-226
        double max_length = sep(p1, p2);
        double h = (f.p[0] - p1.z) / (p2.z - p1.z);
        if ((h < tol) || (h > 1.0)) return -1;
        double X = p1.x + h * (p2.x - p1.x);
        double Y = p1.y + h * (p2.y - p1.y);
        if (is_base && !shape_inside(S, f.shape, X, Y)) return -1;
        return h * max_length;
    }
    case RPX_FACE_RECTANGULAR: {
        if constexpr ((F & F_PLANE) == 0) return -1;  // cfaces.pyx:365-397
        double max_length = sep(p1, p2);
        double h = (f.p[3] - p1.z) / (p2.z - p1.z);
        double lngth = f.p[0], wdth = f.p[1];
        if ((h < tol) || (h > 1.0)) return -1;
        if (is_base) {
            double X = p1.x + h * (p2.x - p1.x) - f.p[2];
            double Y = p1.y + h * (p2.y - p1.y);
            if (X * X > lngth * lngth / 4) return -1;
            if (Y * Y > wdth * wdth / 4) return -1;
        }
        return h * max_length;
    }
    case RPX_FACE_POLYGON: {
        if constexpr ((F & F_PLANE) == 0) return -1;  // cfaces.pyx:1093-1108
        double max_length = sep(p1, p2);
        double h = (f.p[0] - p1.z) / (p2.z - p1.z);
        if ((h < tol) || (h > 1.0)) return -1;
        double X = p1.x + h * (p2.x - p1.x);
        double Y = p1.y + h * (p2.y - p1.y);
        if (is_base && polygon_face_inside(S.vertices + 2 * f.aux0, f.aux1, X, Y)) return h * max_length;
        return -1;
    }
    case RPX_FACE_SPHERICAL:
    case RPX_FACE_SHAPED_SPHERICAL: {
        if constexpr ((F & F_SPHERE) == 0) return -1;  // cfaces.pyx:421-486 / 513-576
        const bool shaped = f.type == RPX_FACE_SHAPED_SPHERICAL;
        const double curvature = shaped ? f.p[0] : f.p[1];
        const double z_height = shaped ? f.p[1] : f.p[2];
        V3 s = sub(p2, p1);
        double cz = z_height - curvature;
        V3 d = p1;
        d.z -= cz;
        double A = mag_sq(s);
        double B = 2 * dot(s, d);
        double C = mag_sq(d) - curvature * curvature;
        double D = B * B - 4 * A * C;
        if (D < 0) return -1;
        D = sqrt(D);
        double a1 = (-B + D) / (2 * A);
        V3 pt1 = add(p1, mul(s, a1));
        double a2 = (-B - D) / (2 * A);
        V3 pt2 = add(p1, mul(s, a2));
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
                double DD = f.p[0] * f.p[0] / 4.;
                if ((pt1.x * pt1.x + pt1.y * pt1.y) > DD) a1 = RPX_INF;
                if ((pt2.x * pt2.x + pt2.y * pt2.y) > DD) a2 = RPX_INF;
            }
        }
        if (a2 < a1) a1 = a2;
        if (a1 > 1.0 || a1 < tol) return -1;
        return a1 * sep(p1, p2);
    }
    case RPX_FACE_EXTRUDED_PLANAR: {
        if constexpr ((F & F_PLANE) == 0) return -1;  // cfaces.pyx:665-699
        double ux = f.p[0], uy = f.p[1];
        double vx = f.p[2] - ux, vy = f.p[3] - uy;
        V3 s = sub(p2, p1);
        double a;
        if (is_base) {
            a = (s.y * (ux - p1.x) - s.x * (uy - p1.y)) / (s.x * vy - s.y * vx);
            if (a < 0) return -1;
            if (a > 1) return -1;
        }
        a = (vx * (p1.y - uy) - vy * (p1.x - ux)) / (s.x * vy - s.y * vx);
        if (is_base) {
            double dz = a * (p2.z - p1.z);
            double zz = p1.z + dz;
            if (f.p[4] < zz && zz < f.p[5]) return a * mag(s);
            return -1;
        }
        return a * mag(s);
    }
    case RPX_FACE_CONIC: {
        if constexpr ((F & F_CONIC) == 0) return -1;  // cfaces.pyx:1767-1798
        V3 d = sub(p2, p1);
        V3 a = p1;
        a.z -= f.p[1];
        double a1 = ref::intersect_conic(a, d, f.p[0], f.p[2]);
        V3 pt1 = add(a, mul(d, a1));
        if (is_base && !shape_inside(S, f.shape, pt1.x, pt1.y)) return -1;
        if (a1 > 1.0 || a1 < tol) return -1;
        return a1 * sep(p1, p2);
    }
    case RPX_FACE_ASPHERIC: {
        if constexpr ((F & F_ASPHERE) == 0) return -1;  // cfaces.pyx:1909-1976
        double atol = f.p[10];
        double tl = atol * atol;
        if (asph_outside_band(f, p1, p2, is_base)) return -1;
        V3 d = sub(p2, p1);
        V3 a = p1;
        a.z -= f.p[1];
        double a1 = ref::intersect_conic(a, d, f.p[0], f.p[2]);
        Asph A;
        A.R = -f.p[0];
        A.beta = 1 + f.p[2];
        A.A4 = f.p[3]; A.A6 = f.p[4]; A.A8 = f.p[5]; A.A10 = f.p[6];
        A.A12 = f.p[7]; A.A14 = f.p[8]; A.A16 = f.p[9];
        A.R3 = f.p[11];
        A.a = a;
        A.d = d;
        double fv = asph_impf(A, a1), f_last = fv;
        double dz = -fv / asph_grad(A, a1);
        bool converged = false;
        for (int i = 0; i < 100; ++i) {
            a1 += dz;
            if (dz * dz < tl) { converged = true; break; }
            fv = asph_impf(A, a1);
            if (fabs(fv) > fabs(f_last)) return -1;
            f_last = fv;
            dz = -fv / asph_grad(A, a1);
        }
        if (!converged) return -1;
        V3 pt1 = add(a, mul(d, a1));
        if (is_base && !shape_inside(S, f.shape, pt1.x, pt1.y)) return -1;
        if (a1 > 1.0 || a1 < tol) return -1;
        return a1 * sep(p1, p2);
    }
    default:
        return -1;
    }
}

// DistortionFace.intersect_c (cfaces.pyx:2339-2416)
template <uint32_t F>
RPX_DEV double distortion_intersect(const SceneView &S, const rpx_face_t &f, V3 p1, V3 p2) {
    const rpx_face_t &face = S.faces[f.aux0];
    const int zi = f.aux1;
    double a1, a2, h = sep(p2, p1);
    double tolerance = f.p[0];
    a2 = plain_intersect<F>(S, face, p1, p2, 0);
    if (a2 > h || a2 < f.tolerance) return -1;
    V3 d = sub(p2, p1);
    V3 pt1 = add(p1, mul(d, a2 / h));
    V3 dxdyz = zernike_grad(S, zi, pt1.x, pt1.y);
    V3 n = plain_normal<F>(S, face, pt1);
    pt1.z += dxdyz.z;
    n.x /= n.z;
    n.y /= n.z;
    n.x -= dxdyz.x;
    n.y -= dxdyz.y;
    V3 o = sub(p1, pt1);
    a1 = -h * dot(o, n) / dot(d, n);
    if (a1 < fabs(dxdyz.z)) return -1;
    for (int i = 0; i < 20; ++i) {
        pt1 = add(p1, mul(d, a1 / h));
        if (fabs(a1 - a2) < tolerance) break;
        double z_shift = zernike_sag(S, zi, pt1.x, pt1.y);
        V3 q1 = p1, q2 = p2;
        q1.z -= z_shift;
        q2.z -= z_shift;
        a2 = plain_intersect<F>(S, face, q1, q2, 0);
        pt1 = add(q1, mul(d, a2 / h));
        n = plain_normal<F>(S, face, pt1);
        dxdyz = zernike_grad(S, zi, pt1.x, pt1.y);
        pt1.z += dxdyz.z;
        n.x /= n.z;
        n.y /= n.z;
        n.x -= dxdyz.x;
        n.y -= dxdyz.y;
        o = sub(p1, pt1);
        a2 = a1;
        a1 = -h * dot(o, n) / dot(d, n);
    }
    if (!shape_inside(S, f.shape, pt1.x, pt1.y)) return -1;
    return a1;
}

template <uint32_t F>
RPX_DEV double face_intersect(const SceneView &S, const rpx_face_t &f, V3 p1, V3 p2, int is_base) {
    if constexpr ((F & F_DISTORT) != 0) {
        if (f.type == RPX_FACE_DISTORTION) return distortion_intersect<F>(S, f, p1, p2);
    }
    return plain_intersect<F>(S, f, p1, p2, is_base);
}

}  // namespace ref
}  // namespace rpx
