// Device-side types and arithmetic helpers for the gfx950 tracer.
//
// The float64 sources are compiled with -ffp-contract=off: a product and a sum
// are fused only where the code says fma.  The vector and complex helpers that
// cite the reference (raypier/core/ctracer.pyx:83-262, cmaterials.pyx) keep its
// operation order and round as its x86-64 build does; the face tests of
// rpx_faces_ref.h rest on them.  The traces' own code (rpx_faces.h,
// rpx_materials.h) and the helpers below without a citation reach the same
// values to a few ulp in fewer operations.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include "../../include/rpx.h"

#define RPX_DEV __device__ __forceinline__
#define RPX_INF (__builtin_inf())

namespace rpx {

// ------------------------------------------------------------------ vectors
struct V3 {
    double x, y, z;
};

RPX_DEV V3 v3(double x, double y, double z) { V3 r; r.x = x; r.y = y; r.z = z; return r; }

// transform_c / rotate_c (ctracer.pyx:83-95)
RPX_DEV V3 transform(const rpx_transform_t &t, V3 p) {
    V3 o;
    o.x = p.x * t.m[0] + p.y * t.m[1] + p.z * t.m[2] + t.t[0];
    o.y = p.x * t.m[3] + p.y * t.m[4] + p.z * t.m[5] + t.t[1];
    o.z = p.x * t.m[6] + p.y * t.m[7] + p.z * t.m[8] + t.t[2];
    return o;
}
RPX_DEV V3 rotate(const rpx_transform_t &t, V3 p) {
    V3 o;
    o.x = p.x * t.m[0] + p.y * t.m[1] + p.z * t.m[2];
    o.y = p.x * t.m[3] + p.y * t.m[4] + p.z * t.m[5];
    o.z = p.x * t.m[6] + p.y * t.m[7] + p.z * t.m[8];
    return o;
}
RPX_DEV V3 add(V3 a, V3 b) { return v3(a.x + b.x, a.y + b.y, a.z + b.z); }
RPX_DEV V3 sub(V3 a, V3 b) { return v3(a.x - b.x, a.y - b.y, a.z - b.z); }
RPX_DEV V3 mul(V3 a, double s) { return v3(a.x * s, a.y * s, a.z * s); }
RPX_DEV double dot(V3 a, V3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
RPX_DEV double mag_sq(V3 a) { return a.x * a.x + a.y * a.y + a.z * a.z; }
RPX_DEV double mag(V3 a) { return sqrt(a.x * a.x + a.y * a.y + a.z * a.z); }
RPX_DEV V3 cross(V3 a, V3 b) {
    return v3(a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x);
}
// norm_ divides each component by the magnitude (ctracer.pyx:251-256)
RPX_DEV V3 norm(V3 a) {
    double m = sqrt(a.x * a.x + a.y * a.y + a.z * a.z);
    return v3(a.x / m, a.y / m, a.z / m);
}
// 1/sqrt(a): the hardware estimate (2^-24) and one third-order step
// y (1 + e/2 + 3 e^2 / 8), e = 1 - a y^2, for normal, finite, positive a
// (within an ulp of the rounded value).
RPX_DEV double rsq_third(double a) {
    const double y = __builtin_amdgcn_rsq(a);
    const double e = fma(-(a * y), y, 1.0);
    return fma(y * e, fma(e, 0.375, 0.5), y);
}

// a / |a| by a reciprocal square root: 15 instructions where norm's square
// root and three divisions take about 60.  The sum of squares rounds twice
// (fused) instead of three times, so the result is as close to the unit vector
// as norm's.
RPX_DEV V3 unit(V3 a) {
    const double r = rsq_third(fma(a.x, a.x, fma(a.y, a.y, a.z * a.z)));
    return v3(a.x * r, a.y * r, a.z * r);
}
RPX_DEV V3 neg(V3 a) { return v3(-a.x, -a.y, -a.z); }
// sep_ (ctracer.pyx:109-114)
RPX_DEV double sep(V3 p1, V3 p2) {
    double a = p2.x - p1.x, b = p2.y - p1.y, c = p2.z - p1.z;
    return sqrt((a * a) + (b * b) + (c * c));
}

// ------------------------------------------------------------ complex FP64
// Mixed real/complex expressions of the reference are evaluated with the real
// operand promoted to (x, 0), as the Cython-generated C does.
struct Cx {
    double re, im;
};
RPX_DEV Cx cx(double r, double i) { Cx c; c.re = r; c.im = i; return c; }
RPX_DEV Cx cadd(Cx a, Cx b) { return cx(a.re + b.re, a.im + b.im); }
RPX_DEV Cx csub(Cx a, Cx b) { return cx(a.re - b.re, a.im - b.im); }
RPX_DEV Cx cmul(Cx a, Cx b) {
    return cx(a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re);
}
// Smith's method (R. L. Smith, CACM 5(8) 1962, Algorithm 116), the scheme C
// runtimes use for double-complex division in the normal range.
RPX_DEV Cx cdiv(Cx n, Cx d) {
    double a = n.re, b = n.im, c = d.re, e = d.im;
    double ratio, denom, x, y;
    if (fabs(c) < fabs(e)) {
        ratio = c / e;
        denom = (c * ratio) + e;
        x = ((a * ratio) + b) / denom;
        y = ((b * ratio) - a) / denom;
    } else {
        ratio = e / c;
        denom = (e * ratio) + c;
        x = ((b * ratio) + a) / denom;
        y = (b - (a * ratio)) / denom;
    }
    return cx(x, y);
}
// Principal square root (Kahan's formulation).
RPX_DEV Cx csqrt_(Cx z) {
    double x = z.re, y = z.im;
    if (x == 0.0 && y == 0.0) return cx(0.0, y);
    if (__builtin_isinf(y)) return cx(RPX_INF, y);
    double t = sqrt((fabs(x) + hypot(x, y)) * 0.5);
    if (x >= 0.0) return cx(t, y / (2.0 * t));
    return cx(fabs(y) / (2.0 * t), copysign(t, y));
}
RPX_DEV Cx cexp_(Cx z) {
    double e = exp(z.re);
    double s, c;
    sincos(z.im, &s, &c);
    return cx(e * c, e * s);
}

// ---------------------------------------------------------- feature masks
// Face and material families; generation kernels are instantiated for a few
// masks and a scene runs the smallest one that covers what it uses.
enum : uint32_t {
    F_PLANE = 1u << 0,      // circular, shaped planar, rectangular, polygon, extruded
    F_SPHERE = 1u << 1,     // spherical, shaped spherical
    F_CONIC = 1u << 2,
    F_ASPHERE = 1u << 3,
    F_DISTORT = 1u << 4,
    M_SIMPLE = 1u << 5,     // none, opaque, transparent, PEC, partial, dielectric
    M_FRESNEL = 1u << 6,    // full dielectric, full dispersive
    M_COATED = 1u << 7,     // single layer, coated dispersive
    M_GRATING = 1u << 8,
    V_ALL = 0x1ffu,
    V_LENS = F_PLANE | F_SPHERE | F_CONIC | F_ASPHERE | M_SIMPLE | M_FRESNEL | M_COATED,
    V_SPHERES = F_PLANE | F_SPHERE | M_SIMPLE | M_FRESNEL | M_COATED,
    // flat optics (cubes, plane and distorted mirrors, gratings); the
    // FP32-split generation kernel only, other kernels run V_ALL for it
    V_FLAT = F_PLANE | F_DISTORT | M_SIMPLE | M_FRESNEL | M_GRATING
};

// ------------------------------------------------------------------- scene
// A Zernike distortion as the kernels evaluate it: `n` groups from `first`,
// of at most `terms` coefficients per polynomial.
struct ZTable {
    double inv_radius;
    int32_t first, n, terms, pad;
};

// The coefficients of one |m| whose sag polynomials have one parity, summed:
// polynomials in r^2.  R and the sag carry one more factor r when `odd`, R'
// and R/r when not.  _C: coefficients with m >= 0, _S: with m < 0.
enum : int { ZG_SAG_C, ZG_SAG_S, ZG_R_C, ZG_R_S, ZG_RP_C, ZG_RP_S, ZG_ROR_C, ZG_ROR_S, ZG_POLYS };
#define ZG_TERMS (RPX_ZPOLY / 2)
struct ZGroup {
    int32_t m, odd;
    double p[ZG_POLYS][ZG_TERMS];
};

// Device view of an uploaded scene (pointers into one device allocation).
struct SceneView {
    const rpx_face_list_t *face_lists;
    const rpx_face_t *faces;
    const rpx_material_t *materials;
    const rpx_shape_op_t *shape_ops;
    const double *vertices;
    const ZTable *ztables;
    const ZGroup *zgroups;
    int32_t n_face_lists, n_faces, n_materials, n_shape_ops, n_vertices;
    int32_t n_zernikes;
    int32_t n_list_faces;   // faces that belong to face lists (chain order)
    // the tables a workgroup stages in LDS: the first stage_units 16-byte units
    // of the block that starts with the face lists, then the faces; shape_ops
    // and materials are at these byte offsets in it, or not staged (-1)
    int32_t stage_units, stage_ops, stage_materials;
    int32_t max_children;
};

// Intersection result (ctracer.pxd:77-81, piece/uv unused by these faces)
struct Hit {
    double dist;
    int32_t face;     // face record index, -1 = none
};

}  // namespace rpx
