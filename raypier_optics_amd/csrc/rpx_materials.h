// Interface materials: child-ray emission and parabasal directions (FP64).
//
// Children are produced through an emitter functor in the reference's order
// (reflected before transmitted, cmaterials.pyx:826-872), so one routine serves
// both the counting pass and the writing pass of a generation.
#pragma once
#include "rpx_faces.h"

namespace rpx {

struct Ray {
    V3 origin, direction, normal, E_vector;
    Cx n, E1, E2;
    double length, phase, accum;
    uint32_t wl_idx, parent_idx, end_face_idx, ray_ident, ray_type_id;
};

// Emitters take children in order through operator(); kCap is how many a
// material should build and hand over, skip() counts one more child the
// emitter does not take (a multi-order grating's third order, built again
// after the children's positions are known).
//
// PairEmit collects the (at most two) children of one ray: what a material
// gives both of them alike once (hit point, normal, polarisation basis,
// lengths, wavelength, identity), and direction, index, amplitudes, phase and
// type per child in a two-slot shift register (s0 is the latest child, s1 the
// one before).  Conditional or indexed slot writes make the compiler keep the
// pair in scratch memory; the unconditional shift keeps both in registers,
// 66 of them where two whole records took 94.
struct PairEmit {
    static constexpr int kCap = 2;
    struct Slot {
        V3 direction;
        Cx n, E1, E2;
        double phase;
        uint32_t type;
    };
    V3 origin, normal, E_vector;
    double length, accum;
    uint32_t wl_idx, parent_idx, end_face_idx, ray_ident;
    Slot s0, s1;
    int n = 0;
    RPX_DEV void operator()(const Ray &x) {
        origin = x.origin;
        normal = x.normal;
        E_vector = x.E_vector;
        length = x.length;
        accum = x.accum;
        wl_idx = x.wl_idx;
        parent_idx = x.parent_idx;
        end_face_idx = x.end_face_idx;
        ray_ident = x.ray_ident;
        s1 = s0;
        s0 = Slot{x.direction, x.n, x.E1, x.E2, x.phase, x.ray_type_id};
        ++n;
    }
    RPX_DEV void skip() { ++n; }
    RPX_DEV Ray child(const Slot &s) const {
        Ray r;
        r.origin = origin;
        r.direction = s.direction;
        r.normal = normal;
        r.E_vector = E_vector;
        r.n = s.n;
        r.E1 = s.E1;
        r.E2 = s.E2;
        r.length = length;
        r.phase = s.phase;
        r.accum = accum;
        r.wl_idx = wl_idx;
        r.parent_idx = parent_idx;
        r.end_face_idx = end_face_idx;
        r.ray_ident = ray_ident;
        r.ray_type_id = s.type;
        return r;
    }
    RPX_DEV Ray first() const { return child(n > 1 ? s1 : s0); }
    RPX_DEV Ray second() const { return child(s0); }
};

// Order k (0-based) of a grating: `order`, then the signed bytes of
// more_orders (multi-order gratings, n_orders 2 or 3).
RPX_DEV int grating_order(const rpx_material_t &m, int k) {
    return k == 0 ? m.order : (int)(int8_t)((uint32_t)m.more_orders >> (8 * (k - 1)));
}
RPX_DEV int grating_orders(const rpx_material_t &m) { return m.n_orders > 1 ? m.n_orders : 1; }

RPX_DEV Ray load_ray(const rpx_rays_t &r, uint64_t i) {
    const double *f = r.f64;
    const uint64_t c = r.capacity;
    Ray o;
    o.origin = v3(f[RPX_OX * c + i], f[RPX_OY * c + i], f[RPX_OZ * c + i]);
    o.direction = v3(f[RPX_DX * c + i], f[RPX_DY * c + i], f[RPX_DZ * c + i]);
    o.normal = v3(f[RPX_NX * c + i], f[RPX_NY * c + i], f[RPX_NZ * c + i]);
    o.E_vector = v3(f[RPX_EX * c + i], f[RPX_EY * c + i], f[RPX_EZ * c + i]);
    o.n = cx(f[RPX_N_RE * c + i], f[RPX_N_IM * c + i]);
    o.E1 = cx(f[RPX_E1_RE * c + i], f[RPX_E1_IM * c + i]);
    o.E2 = cx(f[RPX_E2_RE * c + i], f[RPX_E2_IM * c + i]);
    o.length = f[RPX_LENGTH * c + i];
    o.phase = f[RPX_PHASE * c + i];
    o.accum = f[RPX_ACCUM * c + i];
    const uint32_t *u = r.u32;
    o.wl_idx = u[RPX_WL_IDX * c + i];
    o.parent_idx = u[RPX_PARENT_IDX * c + i];
    o.end_face_idx = u[RPX_END_FACE_IDX * c + i];
    o.ray_ident = u[RPX_RAY_IDENT * c + i];
    o.ray_type_id = u[RPX_RAY_TYPE_ID * c + i];
    return o;
}

// The fields of ray i that its children depend on besides its geometry and
// wavelength index; the others are left unset.
RPX_DEV Ray load_ray_rest(const rpx_rays_t &r, uint64_t i) {
    const double *f = r.f64;
    const uint64_t c = r.capacity;
    Ray o;
    o.normal = v3(0, 0, 0);
    o.E_vector = v3(f[RPX_EX * c + i], f[RPX_EY * c + i], f[RPX_EZ * c + i]);
    o.n = cx(f[RPX_N_RE * c + i], f[RPX_N_IM * c + i]);
    o.E1 = cx(f[RPX_E1_RE * c + i], f[RPX_E1_IM * c + i]);
    o.E2 = cx(f[RPX_E2_RE * c + i], f[RPX_E2_IM * c + i]);
    o.phase = f[RPX_PHASE * c + i];
    o.accum = f[RPX_ACCUM * c + i];
    o.parent_idx = 0;
    o.ray_ident = r.u32[RPX_RAY_IDENT * c + i];
    o.ray_type_id = r.u32[RPX_RAY_TYPE_ID * c + i];
    return o;
}

RPX_DEV void store_ray(const rpx_rays_t &r, uint64_t i, const Ray &o) {
    double *f = r.f64;
    const uint64_t c = r.capacity;
    f[RPX_OX * c + i] = o.origin.x;  f[RPX_OY * c + i] = o.origin.y;  f[RPX_OZ * c + i] = o.origin.z;
    f[RPX_DX * c + i] = o.direction.x; f[RPX_DY * c + i] = o.direction.y; f[RPX_DZ * c + i] = o.direction.z;
    f[RPX_NX * c + i] = o.normal.x;  f[RPX_NY * c + i] = o.normal.y;  f[RPX_NZ * c + i] = o.normal.z;
    f[RPX_EX * c + i] = o.E_vector.x; f[RPX_EY * c + i] = o.E_vector.y; f[RPX_EZ * c + i] = o.E_vector.z;
    f[RPX_N_RE * c + i] = o.n.re;    f[RPX_N_IM * c + i] = o.n.im;
    f[RPX_E1_RE * c + i] = o.E1.re;  f[RPX_E1_IM * c + i] = o.E1.im;
    f[RPX_E2_RE * c + i] = o.E2.re;  f[RPX_E2_IM * c + i] = o.E2.im;
    f[RPX_LENGTH * c + i] = o.length;
    f[RPX_PHASE * c + i] = o.phase;
    f[RPX_ACCUM * c + i] = o.accum;
    uint32_t *u = r.u32;
    u[RPX_WL_IDX * c + i] = o.wl_idx;
    u[RPX_PARENT_IDX * c + i] = o.parent_idx;
    u[RPX_END_FACE_IDX * c + i] = o.end_face_idx;
    u[RPX_RAY_IDENT * c + i] = o.ray_ident;
    u[RPX_RAY_TYPE_ID * c + i] = o.ray_type_id;
}

// Parabasal ray (ctracer.pxd:54-58)
struct Para {
    V3 origin, direction, normal;
    double length;
};

// ------------------------------------------------------------- dispersion
// BaseDispersionCurve.c_evaluate_n (cmaterials.pyx:206-228) for one
// wavelength; the host rejects out-of-range wavelengths beforehand.
RPX_DEV Cx eval_dispersion(const rpx_dispersion_t &d, double wvl) {
    double nre;
    const double *c = d.coefs;
    switch (d.formula_id) {
    case 0:  // nondispersive_0 (cmaterials.pyx:107)
        nre = c[0];
        break;
    case 1: {  // sellmeier_1 (cmaterials.pyx:110-119)
        double n2 = 1.0, wl2 = wvl * wvl;
        n2 += c[0];
        for (int i = 0; i < (d.n_coefs - 1) / 2; ++i)
            n2 += c[2 * i + 1] * wl2 / (wl2 - c[2 * i + 2] * c[2 * i + 2]);
        nre = sqrt(n2);
    } break;
    case 2: {  // sellmeier_2 (cmaterials.pyx:121-130)
        double n2 = 1.0, wl2 = wvl * wvl;
        n2 += c[0];
        for (int i = 0; i < (d.n_coefs - 1) / 2; ++i)
            n2 += c[2 * i + 1] * wl2 / (wl2 - c[2 * i + 2]);
        nre = sqrt(n2);
    } break;
    case 3: {  // sellmeier_3 polynomial (cmaterials.pyx:133-140)
        double n2 = c[0];
        for (int i = 1; i < d.n_coefs - 1; i += 2) n2 += c[i] * pow(wvl, c[i + 1]);
        nre = sqrt(n2);
    } break;
    default:  // sellmeier_5 returns nothing (cmaterials.pyx:143-149): 0.0
        nre = 0.0;
        break;
    }
    double n_imag = 0.0001 * d.absorption / (4 * M_PI);
    return cx(nre, n_imag * wvl);
}

// ------------------------------------------------------------- S/P basis
// convert_to_sp (cmaterials.pyx:49-91) for a unit normal (which the
// reference normalises once more).
RPX_DEV Ray convert_to_sp(Ray ray, V3 normal) {
    const V3 S0 = cross(ray.direction, normal);
    if (fabs(S0.x) < 1.0e-10 && fabs(S0.y) < 1.0e-10 && fabs(S0.z) < 1.0e-10) return ray;
    const Cx E1 = ray.E1, E2 = ray.E2;
    const V3 E2v = unit(cross(ray.direction, ray.E_vector));
    const V3 E1v = unit(cross(E2v, ray.direction));
    const V3 S = unit(S0), P = unit(cross(ray.direction, S));
    double A = dot(E1v, S), B = dot(E2v, S);
    ray.E1 = cx(E1.re * A + E2.re * B, E1.im * A + E2.im * B);
    B = dot(E1v, P);
    A = dot(E2v, P);
    ray.E2 = cx(E1.re * B + E2.re * A, E1.im * B + E2.im * A);
    ray.E_vector = S;
    return ray;
}

RPX_DEV Cx R(double x) { return cx(x, 0.0); }

// Indices on the incident (n1), coating (n2) and far (n3) sides.
struct Sides {
    Cx n_in, n_out, n_coat;
};

RPX_DEV Sides material_indices(const rpx_material_t &m, double wvl) {
    Sides s;
    if (m.type == RPX_MAT_FULL_DISPERSIVE || m.type == RPX_MAT_COATED_DISPERSIVE) {
        s.n_in = eval_dispersion(m.disp_inside, wvl);
        s.n_out = eval_dispersion(m.disp_outside, wvl);
        s.n_coat = (m.type == RPX_MAT_COATED_DISPERSIVE) ? eval_dispersion(m.disp_coating, wvl) : cx(0, 0);
    } else {
        s.n_in = cx(m.n_inside[0], m.n_inside[1]);
        s.n_out = cx(m.n_outside[0], m.n_outside[1]);
        s.n_coat = cx(m.n_coating[0], m.n_coating[1]);
    }
    return s;
}

// Wavelength table lookup; an index outside the table yields NaN (the ray's
// children then fail every threshold test) instead of a fault.
struct WlTable {
    const double *wl;
    uint64_t n;
    RPX_DEV double operator[](uint32_t i) const { return (i < n) ? wl[i] : __builtin_nan(""); }
};

// The wavelength of one ray, looked up beforehand.
struct WlOne {
    double v;
    RPX_DEV double operator[](uint32_t) const { return v; }
};

// Whether a material can have children: OpaqueMaterial and the base
// InterfaceMaterial never do, so a ray ending on them needs no material
// evaluation and none of its record beyond the geometry.
RPX_DEV bool material_emits(const rpx_material_t &m) {
    return m.type != RPX_MAT_NONE && m.type != RPX_MAT_OPAQUE;
}

// power / P_in > threshold as a product: no reciprocal, which overflows for
// the subnormal P_in of very faint rays.
template <class T>
RPX_DEV bool passes(T power, T P_in, T threshold) {
    return P_in > 0 ? power > threshold * P_in : power < threshold * P_in;
}

// |a|^2
RPX_DEV double cnorm2(Cx a) { return fma(a.re, a.re, a.im * a.im); }

// Amplitude coefficients of an interface: reflected and transmitted, s and p;
// the transmitted ones carry sqrt(cos3 / cos1).
struct Coefs {
    Cx rs, rp, ts, tp;
};

// Bare interface n1 -> n2 (cmaterials.pyx:790-850).  Two real indices below
// total reflection (`real`): cos2 is the transmitted ray's own cosine, and each
// polarisation's pair shares one reciprocal.
RPX_DEV Coefs fresnel_coefs(Cx n1, Cx n2, double cos1, double sin1, bool real, double cos2r) {
    Coefs c;
    if (real) {
        const double n2c1 = n2.re * cos1, n1c2 = n1.re * cos2r, n2c2 = n2.re * cos2r, n1c1 = n1.re * cos1;
        const double ip = 1.0 / (n2c1 + n1c2), is = 1.0 / (n2c2 + n1c1);
        const double t = 2.0 * n1.re * sqrt(cos1 * cos2r);
        c.rp = cx((n1c2 - n2c1) * ip, 0.0);
        c.rs = cx((n1c1 - n2c2) * is, 0.0);
        c.tp = cx(t * ip, 0.0);
        c.ts = cx(t * is, 0.0);
        return c;
    }
    const Cx sin2 = cdiv(cmul(n1, cx(sin1, 0.0)), n2);
    const Cx cos2 = csqrt_(csub(cx(1, 0), cmul(sin2, sin2)));
    const Cx n2c1 = cmul(n2, cx(cos1, 0)), n1c2 = cmul(n1, cos2);
    const Cx n2c2 = cmul(n2, cos2), n1c1 = cmul(n1, cx(cos1, 0));
    c.rp = cdiv(csub(n1c2, n2c1), cadd(n2c1, n1c2));
    c.rs = cdiv(csub(n1c1, n2c2), cadd(n2c2, n1c1));
    const double aspect = sqrt(cos2.re / cos1);
    const Cx num = cmul(cx(aspect, 0), cmul(cx(2.0 * cos1, 0), n1));
    c.tp = cdiv(num, cadd(n2c1, n1c2));
    c.ts = cdiv(num, cadd(n2c2, n1c1));
    return c;
}

// Interface n1 -> n3 under a film of index n2 (cmaterials.pyx:1026-1182,
// 1228-1391).  With the reference's phi = -i dwc (n2 - sin2^2) / cos2 and, for
// s, a, b = n1 cos1 -+ n2 cos2, c, d = n2 cos2 +- n3 cos3 (for p with the
// cosines of the other side), its matrix elements M00 .. M11 give
//   r = (a c + b d e^-2phi) / (a d e^-2phi + b c),
//   t = M10 + M11 r = -(a^2 - b^2)(c^2 - d^2) e^-phi / (4 n2 cos2 n3 cos3 (..)),
// and a^2 - b^2 is a product again: 4 n1 cos1 n2 cos2 e^-phi over the same
// denominator for s, 4 n1 cos2 n2 cos1 e^-phi for p.  Three real indices below
// total reflection (`real`): e^phi has modulus 1 and the rest is real.
// `n2c2sq`, (n2 cos2)^2 = n2^2 - n1^2 sin1^2, is then above zero as computed, so
// that no rounding of sin2^2 takes cos2 to zero or past it.
RPX_DEV Coefs film_coefs(Cx n1, Cx n2, Cx n3, double cos1, double sin1, double dwc, bool real, double sin1sq,
                         double n2c2sq, double cos3r) {
    Coefs o;
    if (real) {
        const double inv2 = 1.0 / n2.re, q = n1.re * inv2, sin2sq = sin1sq * q * q;
        const double n2c2 = sqrt(n2c2sq), cos2 = n2c2 * inv2;
        double sp, cp;   // e^-phi = cp + i sp
        sincos(dwc * (n2.re - sin2sq) / cos2, &sp, &cp);
        const double er = fma(cp, cp, -(sp * sp)), ei = 2.0 * sp * cp;   // e^-2phi
        const double n1c1 = n1.re * cos1, n3c3 = n3.re * cos3r;
        const double n1c2 = n1.re * cos2, n2c1 = n2.re * cos1, n2c3 = n2.re * cos3r, n3c2 = n3.re * cos2;
        const double aspect = 4.0 * sqrt(cos3r / cos1);
        auto pol = [&](double a, double b, double c, double d, double t, Cx &r_out, Cx &t_out) {
            const double ac = a * c, bd = b * d, ad = a * d, bc = b * c;
            const double dr = fma(ad, er, bc), di = ad * ei;
            const double nr = fma(bd, er, ac), ni = bd * ei;
            const double inv = 1.0 / fma(dr, dr, di * di);
            r_out = cx(fma(nr, dr, ni * di) * inv, fma(ni, dr, -(nr * di)) * inv);
            t *= aspect * inv;
            t_out = cx(fma(cp, dr, sp * di) * t, fma(sp, dr, -(cp * di)) * t);
        };
        pol(n1c1 - n2c2, n1c1 + n2c2, n2c2 + n3c3, n2c2 - n3c3, n1c1 * n2c2, o.rs, o.ts);
        pol(n1c2 - n2c1, n1c2 + n2c1, n2c3 + n3c2, n2c3 - n3c2, n1c2 * n2c1, o.rp, o.tp);
        return o;
    }
    const Cx n1s1 = cmul(n1, cx(sin1, 0));
    const Cx sin2 = cdiv(n1s1, n2), sin3 = cdiv(n1s1, n3);
    const Cx s2 = cmul(sin2, sin2);
    const Cx cos2 = csqrt_(csub(cx(1, 0), s2)), cos3 = csqrt_(csub(cx(1, 0), cmul(sin3, sin3)));
    const Cx mphi = cdiv(cmul(cx(0.0, dwc), csub(n2, s2)), cos2);    // -phi
    const Cx e1 = cexp_(mphi), e2 = cexp_(cmul(cx(2, 0), mphi));
    const Cx n1c1 = cmul(n1, cx(cos1, 0)), n2c2 = cmul(n2, cos2), n3c3 = cmul(n3, cos3);
    const Cx n1c2 = cmul(n1, cos2), n2c1 = cmul(n2, cx(cos1, 0)), n2c3 = cmul(n2, cos3), n3c2 = cmul(n3, cos2);
    const double aspect = 4.0 * sqrt(cos3.re / cos1);
    auto pol = [&](Cx a, Cx b, Cx c, Cx d, Cx t, Cx &r_out, Cx &t_out) {
        const Cx den = cadd(cmul(cmul(a, d), e2), cmul(b, c));
        r_out = cdiv(cadd(cmul(a, c), cmul(cmul(b, d), e2)), den);
        t_out = cdiv(cmul(cmul(t, cx(aspect, 0)), e1), den);
    };
    pol(csub(n1c1, n2c2), cadd(n1c1, n2c2), cadd(n2c2, n3c3), csub(n2c2, n3c3), cmul(n1c1, n2c2), o.rs, o.ts);
    pol(csub(n1c2, n2c1), cadd(n1c2, n2c1), cadd(n2c3, n3c2), csub(n2c3, n3c2), cmul(n1c2, n2c1), o.rp, o.tp);
    return o;
}

// ------------------------------------------------------------- children
// InterfaceMaterial.eval_child_ray_c of every supported material.
// DiffractionGratingMaterial.eval_child_ray_c (cmaterials.pyx:1472-1542):
// one child per propagating order, orders in list order (one order in the
// reference); children past the emitter's kCap are counted, not built.
template <class W, class Emit>
RPX_DEV void grating_children(const rpx_material_t &m, const Ray &in, uint32_t idx, V3 point,
                              const Orientation &orient, const W &wavelengths, Emit &emit) {
    V3 normal = unit(orient.normal);
    V3 tangent = unit(orient.tangent);
    V3 tangent2 = cross(normal, tangent);
    double wavelen = wavelengths[in.wl_idx];
    double line_spacing = 1000.0 / m.lines_per_mm;
    const V3 dir = unit(in.direction);
    const double k_z0 = dot(normal, dir);
    const double k_y = dot(tangent2, dir);
    const double k_x0 = dot(tangent, dir);
    int sign = (k_z0 < 0.0) ? 1 : -1;
    double n_re = in.n.re;
    const int n_orders = grating_orders(m);
    int built = 0;
    for (int o = 0; o < n_orders; ++o) {
        const int order = grating_order(m, o);
        double k_x = k_x0 - order * wavelen / (line_spacing * n_re);
        double k_z = 1 - (k_x * k_x) - (k_y * k_y);
        if (k_z < 0) continue;
        if (built >= Emit::kCap) {
            emit.skip();
            continue;
        }
        ++built;
        k_z = sign * sqrt(k_z);
        V3 reflected = mul(tangent, k_x);
        reflected = add(reflected, mul(tangent2, k_y));
        reflected = add(reflected, mul(normal, k_z));
        Ray sp = convert_to_sp(in, normal);
        sp.accum += sp.length * sp.n.re;
        sp.origin = point;
        sp.normal = normal;
        sp.direction = reflected;
        sp.E1.re = -sp.E1.re * m.efficiency;
        sp.E1.im = -sp.E1.im * m.efficiency;
        sp.E2.re = sp.E2.re * m.efficiency;
        sp.E2.im = sp.E2.im * m.efficiency;
        sp.parent_idx = idx;
        sp.ray_type_id |= RPX_REFL_RAY;
        V3 og = v3(m.origin[0], m.origin[1], m.origin[2]);
        sp.phase += 1000.0 * dot(sub(og, point), tangent) * order * 2 * M_PI / line_spacing;
        emit(sp);
    }
}

template <uint32_t F, class W, class Emit>
RPX_DEV void eval_children(const rpx_material_t &m, const Ray &in, uint32_t idx, V3 point,
                           const Orientation &orient, const W &wavelengths, Emit &emit) {
    switch (m.type) {
    case RPX_MAT_TRANSPARENT: {
        if constexpr ((F & M_SIMPLE) == 0) return;  // cmaterials.pyx:260-278
        V3 normal = unit(orient.normal);
        Ray sp = convert_to_sp(in, normal);
        sp.accum += sp.length * sp.n.re;
        sp.origin = point;
        sp.normal = normal;
        sp.length = RPX_INF;
        sp.parent_idx = idx;
        sp.ray_type_id &= ~RPX_REFL_RAY;
        emit(sp);
    } break;
    case RPX_MAT_PEC: {
        if constexpr ((F & M_SIMPLE) == 0) return;  // cmaterials.pyx:285-319
        V3 normal = unit(orient.normal);
        Ray sp = convert_to_sp(in, normal);
        double cosTheta = dot(normal, in.direction);
        V3 ctn = mul(normal, cosTheta);
        V3 reflected = sub(in.direction, mul(ctn, 2));
        sp.accum += sp.length * sp.n.re;
        sp.origin = point;
        sp.normal = normal;
        sp.direction = reflected;
        sp.length = RPX_INF;
        sp.E1.re = -sp.E1.re;
        sp.E1.im = -sp.E1.im;
        sp.parent_idx = idx;
        sp.ray_type_id |= RPX_REFL_RAY;
        emit(sp);
    } break;
    case RPX_MAT_PARTIAL: {
        if constexpr ((F & M_SIMPLE) == 0) return;  // cmaterials.pyx:345-397
        V3 normal = unit(orient.normal);
        V3 in_dir = unit(in.direction);
        Ray sp = convert_to_sp(in, normal);
        double cosTheta = dot(normal, in_dir);
        V3 ctn = mul(normal, cosTheta);
        sp.accum += sp.length * sp.n.re;
        Ray sp2 = sp;
        double Rr = sqrt(m.reflectivity);
        double T = sqrt(1 - m.reflectivity);
        V3 reflected = sub(in_dir, mul(ctn, 2));
        sp.origin = point;
        sp.normal = normal;
        sp.direction = reflected;
        sp.length = RPX_INF;
        sp.E1 = cmul(sp.E1, R(Rr));
        sp.E2 = cmul(sp.E2, R(Rr));
        sp.parent_idx = idx;
        sp.ray_type_id |= RPX_REFL_RAY;
        emit(sp);
        sp2.origin = point;
        sp2.normal = normal;
        sp2.direction = in_dir;
        sp2.length = RPX_INF;
        sp2.E1 = cmul(sp2.E1, R(T));
        sp2.E2 = cmul(sp2.E2, R(T));
        sp2.parent_idx = idx;
        sp2.ray_type_id &= ~RPX_REFL_RAY;
        emit(sp2);
    } break;
    case RPX_MAT_DIELECTRIC: {
        if constexpr ((F & M_SIMPLE) == 0) return;  // cmaterials.pyx:587-680
        V3 normal = unit(orient.normal);
        V3 in_dir = unit(in.direction);
        Ray sp = convert_to_sp(in, normal);
        sp.accum += sp.length * sp.n.re;
        double cosTheta = dot(normal, in_dir);
        double cos1 = fabs(cosTheta);
        double n1, n2;
        int flip;
        if (cosTheta < 0.0) {
            n1 = m.n_outside[0];
            n2 = m.n_inside[0];
            sp.n = cx(m.n_inside[0], m.n_inside[1]);
            flip = 1;
        } else {
            n1 = m.n_inside[0];
            n2 = m.n_outside[0];
            sp.n = cx(m.n_outside[0], m.n_outside[1]);
            flip = -1;
        }
        double q = n2 / n1;
        double N2 = q * q;
        double N2_sin2 = (cosTheta * cosTheta) + (N2 - 1);
        V3 ctn = mul(normal, cosTheta);
        if (N2_sin2 < 0.0) {
            V3 reflected = sub(in_dir, mul(ctn, 2));
            sp.origin = point;
            sp.normal = normal;
            sp.direction = reflected;
            sp.length = RPX_INF;
            sp.E1.re *= -1; sp.E1.im *= -1;
            sp.E2.re *= -1; sp.E2.im *= -1;
            sp.parent_idx = idx;
            sp.ray_type_id |= RPX_REFL_RAY;
        } else {
            V3 tangent = sub(in_dir, ctn);
            V3 tg2 = mul(tangent, n1 / n2);
            double tan_mag_sq = mag_sq(tg2);
            double c2 = sqrt(1 - tan_mag_sq);
            V3 transmitted = sub(tg2, mul(normal, c2 * flip));
            double cos2 = fabs(dot(transmitted, normal));
            double Two_n1_cos1 = (2 * n1) * cos1;
            double aspect = sqrt(cos2 / cos1) * Two_n1_cos1;
            double T_p = aspect / (n2 * cos1 + n1 * cos2);
            double T_s = aspect / (n2 * cos2 + n1 * cos1);
            sp.origin = point;
            sp.normal = normal;
            sp.direction = transmitted;
            sp.length = RPX_INF;
            sp.E1.re *= T_s; sp.E1.im *= T_s;
            sp.E2.re *= T_p; sp.E2.im *= T_p;
            sp.parent_idx = idx;
            sp.ray_type_id &= ~RPX_REFL_RAY;
        }
        emit(sp);
    } break;
    case RPX_MAT_FULL_DIELECTRIC:
    case RPX_MAT_FULL_DISPERSIVE:
    case RPX_MAT_SINGLE_LAYER:
    case RPX_MAT_COATED_DISPERSIVE: {
        // FullDielectricMaterial and its dispersive form (cmaterials.pyx:755-872,
        // 896-1013), SingleLayerCoated and CoatedDispersive (:1026-1182, 1228-1391)
        if constexpr ((F & (M_FRESNEL | M_COATED)) == 0) return;
        const bool film = m.type == RPX_MAT_SINGLE_LAYER || m.type == RPX_MAT_COATED_DISPERSIVE;
        const double wavelength = m.type == RPX_MAT_FULL_DIELECTRIC ? 0.0 : wavelengths[in.wl_idx];
        const Sides sd = material_indices(m, wavelength);
        V3 normal = unit(orient.normal);
        V3 in_dir = unit(in.direction);
        Ray sp = convert_to_sp(in, normal);
        sp.accum += sp.length * sp.n.re;
        sp.origin = point;
        sp.normal = normal;
        sp.length = RPX_INF;
        sp.parent_idx = idx;
        const Cx E1 = sp.E1, E2 = sp.E2;
        const double cosTheta = dot(normal, in_dir);
        const double cos1 = fabs(cosTheta);
        const bool inward = cosTheta < 0.0;
        const Cx n1 = inward ? sd.n_out : sd.n_in, n3 = inward ? sd.n_in : sd.n_out;
        const double P_in = n1.re * (cnorm2(E1) + cnorm2(E2));
        if (P_in == 0.0) return;
        // the tangential part of the direction, before and after refraction
        const V3 tangent = sub(in_dir, mul(normal, cosTheta));
        const V3 tg2 = mul(tangent, n1.re / n3.re);
        const double tan_mag_sq = mag_sq(tg2);
        const double c2 = sqrt(1 - tan_mag_sq);
        bool real = n1.im == 0.0 && n3.im == 0.0 && n1.re > 0.0 && n3.re > 0.0 && tan_mag_sq < 1.0;
        Coefs k;
        if (film) {
            if constexpr ((F & M_COATED) != 0) {
                const double sin1sq = mag_sq(tangent);
                const double n2c2sq = sd.n_coat.re * sd.n_coat.re - n1.re * n1.re * sin1sq;
                real = real && sd.n_coat.im == 0.0 && sd.n_coat.re > 0.0 && n2c2sq > 0.0;
                k = film_coefs(n1, sd.n_coat, n3, cos1, sqrt(fabs(1 - cos1 * cos1)),
                               2 * M_PI * m.thickness / wavelength, real, sin1sq, n2c2sq, c2);
            } else {
                return;
            }
        } else {
            if constexpr ((F & M_FRESNEL) != 0)
                k = fresnel_coefs(n1, n3, cos1, sqrt(fabs(1 - cos1 * cos1)), real, c2);
            else
                return;
        }
        const Cx R_s = cmul(k.rs, E1), R_p = cmul(k.rp, E2);
        if (passes(n1.re * (cnorm2(R_s) + cnorm2(R_p)), P_in, m.reflection_threshold)) {
            sp.direction = sub(in_dir, mul(mul(normal, cosTheta), 2));
            sp.E1 = R_s;
            sp.E2 = cx(-R_p.re, -R_p.im);
            sp.n = n1;
            sp.ray_type_id |= RPX_REFL_RAY;
            emit(sp);
        }
        const Cx T_s = cmul(k.ts, E1), T_p = cmul(k.tp, E2);
        if (passes(n3.re * (cnorm2(T_s) + cnorm2(T_p)), P_in, m.transmission_threshold)) {
            sp.direction = sub(tg2, mul(normal, inward ? c2 : -c2));
            sp.E1 = T_s;
            sp.E2 = T_p;
            sp.n = n3;
            sp.ray_type_id &= ~RPX_REFL_RAY;
            emit(sp);
        }
    } break;
    case RPX_MAT_GRATING: {
        if constexpr ((F & M_GRATING) == 0) return;
        grating_children(m, in, idx, point, orient, wavelengths, emit);
    } break;
    default:  // RPX_MAT_NONE, RPX_MAT_OPAQUE: no children
        break;
    }
}

// Real indices inside and outside of a refracting material, for its parabasal
// rays (once per gausslet: a dispersive material takes them from its curves).
struct ParaIndex {
    double inside, outside;
};

template <uint32_t F>
RPX_DEV ParaIndex parabasal_index(const rpx_material_t &m, double wavelength) {
    if constexpr ((F & M_COATED) != 0) {
        if (m.type == RPX_MAT_COATED_DISPERSIVE)
            return ParaIndex{eval_dispersion(m.disp_inside, wavelength).re, eval_dispersion(m.disp_outside, wavelength).re};
    }
    return ParaIndex{m.n_inside[0], m.n_outside[0]};
}

// eval_parabasal_ray_c: InterfaceMaterial default (ctracer.pyx:1588-1610),
// DielectricMaterial (cmaterials.pyx:683-724, inherited by FullDielectric and
// SingleLayerCoated), CoatedDispersiveMaterial (:1393-1434), grating (:1544-1599).
// n_re: the base child's index, ray_type_id: its type.
template <uint32_t F>
RPX_DEV Para eval_parabasal(const rpx_material_t &m, const ParaIndex &index, double wavelength, double n_re,
                            V3 direction, V3 point, const Orientation &orient, uint32_t ray_type_id) {
    Para out;
    V3 normal = unit(orient.normal);
    switch (m.type) {
    case RPX_MAT_DIELECTRIC:
    case RPX_MAT_FULL_DIELECTRIC:
    case RPX_MAT_SINGLE_LAYER:
    case RPX_MAT_COATED_DISPERSIVE: {
        if constexpr ((F & (M_SIMPLE | M_FRESNEL | M_COATED)) == 0) break;
        direction = unit(direction);
        double cosTheta = dot(normal, direction);
        V3 ctn = mul(normal, cosTheta);
        if (ray_type_id & RPX_REFL_RAY) {
            out.direction = sub(direction, mul(ctn, 2));
        } else {
            const bool inward = cosTheta < 0.0;
            const double n1 = inward ? index.outside : index.inside, n2 = inward ? index.inside : index.outside;
            V3 tg2 = mul(sub(direction, ctn), n1 / n2);
            double c2 = sqrt(1 - mag_sq(tg2));
            out.direction = sub(tg2, mul(normal, inward ? c2 : -c2));
        }
    } break;
    case RPX_MAT_GRATING: {
        if constexpr ((F & M_GRATING) == 0) break;
        V3 tangent = unit(orient.tangent);
        V3 tangent2 = cross(normal, tangent);
        double line_spacing = 1000.0 / m.lines_per_mm;
        V3 reflected = unit(direction);
        double k_z = dot(normal, reflected);
        double k_y = dot(tangent2, reflected);
        double k_x = dot(tangent, reflected);
        int sign = (k_z < 0.0) ? 1 : -1;
        k_x = k_x - m.order * wavelength / (line_spacing * n_re);
        k_z = 1 - (k_x * k_x) - (k_y * k_y);
        k_z = sign * sqrt(k_z);
        reflected = mul(tangent, k_x);
        reflected = add(reflected, mul(tangent2, k_y));
        reflected = add(reflected, mul(normal, k_z));
        out.direction = reflected;
    } break;
    default:
        if (ray_type_id & RPX_REFL_RAY) {
            double cosTheta = dot(normal, direction);
            V3 ctn = mul(normal, cosTheta);
            out.direction = sub(direction, mul(ctn, 2));
        } else {
            out.direction = direction;
        }
        break;
    }
    out.origin = point;
    out.normal = normal;
    out.length = RPX_INF;
    return out;
}

}  // namespace rpx
