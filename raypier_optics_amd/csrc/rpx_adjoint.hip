// Spot RMS or wavefront RMS of a coaxial sequential lens and its gradient
// with respect to every surface's curvature, conic constant, A4..A10 terms
// and Zernike distortion coefficients.
//
// Forward (k_lens_forward): one thread per ray traces surfaces 0..n-1 and the
// detector plane and writes per-workgroup moment partials.  Adjoint
// (k_lens_adjoint): each thread traces its ray again, keeping the direction
// entering every surface, the distance to it and x and y there, then runs the
// chain rule backwards from the detector, recomputing each surface's normal
// and refraction at the very point; surface parameters receive the
// contributions of the implicit intersection equation and of the normal.
// Per-workgroup parameter partials are summed by a fixed-order reduction.
//
// Both are bound by float64 instruction issue (the rays are 56 bytes each).  A
// surface's w and 1/w come from one reciprocal root, 1/(1+w) and every other
// quotient from reciprocals, and products are fused with the sums that take
// them.  The adjoint also moves the kept states through private memory: 48
// bytes per surface.  (32, with the points stepped back to from the last one,
// take 261 us at the size below, not 281; but a point is then a rounding of the
// segment away from the forward's, which near total reflection is all there is
// of the refracted cosine.)  MI355X, 2,097,152 rays through 6 surfaces:
// forward 315 -> 128 us, adjoint 774 -> 281 us (3 waves per SIMD instead of 5
// cost another 32 us), column sums 15 -> 11 us, against square roots and
// divisions per term, two Newton steps more, and every intersection solved
// twice.
//
// Surface:  G(q) = S(rho) + D(q.x, q.y) - (q.z - z_s) = 0,
//   rho     = q.x^2 + q.y^2,
//   S(rho)  = c rho / (1 + w) + A4 rho^2 + A6 rho^3 + A8 rho^4 + A10 rho^5,
//   w       = sqrt(1 - (1 + k) c^2 rho),
//   S'(rho) = c / (2 w) + 2 A4 rho + 3 A6 rho^2 + 4 A8 rho^3 + 5 A10 rho^4,
//   D       = sum_k C_k (x/Ru)^a_k (y/Ru)^b_k   (0 without a distortion),
//   normal  = m / |m|,  m = (-(2 q.x S' + D_x), -(2 q.y S' + D_y), 1).
// Wavefront: W = accumulated_path + sum_s n_s t_s + n_L (P - q_L) . d_L.
// Refraction (unit d, unit normal N oriented along d, mu = n1 / n2):
//   cos = d.N,  t = mu d + (sqrt(1 - mu^2 (1 - cos^2)) - mu cos) N.
#include <hip/hip_runtime.h>
#include <algorithm>
#include <string>
// the objective and its gradient follow no reference rounding
#pragma clang fp contract(fast)
#include "rpx_internal.h"
#include "rpx_host.h"

using namespace rpx;

namespace {

constexpr int LB = 256;   // workgroup size

// 1/a for normal, finite a: the hardware estimate and one third-order step.
__device__ __forceinline__ double rcp_third(double a) {
    const double y = __builtin_amdgcn_rcp(a);
    const double e = fma(-a, y, 1.0);
    return fma(y, fma(e, e, e), y);
}

// What S and its derivatives at one rho share: y = 1/w.
struct Conic {
    double w, y, w1;    // w1 = 1 + w
};

// With TRACED (the backward pass, at a point where the forward pass had a root)
// it has one always: the two passes may evaluate the same point to a rounding
// of the argument's terms apart, and a ray of a surface's rim then keeps the
// least argument that such a rounding leaves, instead of none.
#define LEAST_ARG 0x1p-53
template <bool TRACED>
__device__ __forceinline__ bool conic(const double *P, double rho, Conic &k) {
    double arg = 1 - (1 + P[1]) * P[0] * P[0] * rho;
    if constexpr (TRACED) arg = fmax(arg, LEAST_ARG);
    else if (!(arg > 0)) return false;
    k.y = rsq_third(arg);
    k.w = arg * k.y;
    k.w1 = 1 + k.w;
    return true;
}

// A4 rho^2 + ... + A10 rho^5
__device__ __forceinline__ double poly(const double *P, double rho) {
    return rho * rho * (P[2] + rho * (P[3] + rho * (P[4] + rho * P[5])));
}

__device__ __forceinline__ double slope(const double *P, double rho, double y) {
    return 0.5 * P[0] * y + rho * (2 * P[2] + rho * (3 * P[3] + rho * (4 * P[4] + rho * (5 * P[5]))));
}

// Monomial k = d(d+1)/2 + (d - a) is x^a y^b with b = d - a, d = 0..6.
constexpr int ZDEG = 6;

// D and its first and second derivatives in x, y (physical units) from the
// monomial coefficients C (normalised coordinates x/Ru, y/Ru).
struct ZEval {
    double D, Dx, Dy, Dxx, Dxy, Dyy;
};

__device__ __forceinline__ void zpowers(double x, double *p) {
    p[0] = 1.0;
#pragma unroll
    for (int i = 1; i <= ZDEG; ++i) p[i] = p[i - 1] * x;
}

__device__ __forceinline__ ZEval zernike_eval(const double *C, double Ru, double x, double y, bool second) {
    ZEval z = {0, 0, 0, 0, 0, 0};
    if (!C) return z;
    const double inv = 1.0 / Ru;
    double xp[ZDEG + 1], yp[ZDEG + 1];
    zpowers(x * inv, xp);
    zpowers(y * inv, yp);
    int k = 0;
#pragma unroll
    for (int d = 0; d <= ZDEG; ++d) {
#pragma unroll
        for (int a = d; a >= 0; --a, ++k) {
            const int b = d - a;
            const double c = C[k];
            z.D += c * xp[a] * yp[b];
            if (a >= 1) z.Dx += c * a * xp[a - 1] * yp[b];
            if (b >= 1) z.Dy += c * b * xp[a] * yp[b - 1];
            if (second) {
                if (a >= 2) z.Dxx += c * a * (a - 1) * xp[a - 2] * yp[b];
                if (a >= 1 && b >= 1) z.Dxy += c * a * b * xp[a - 1] * yp[b - 1];
                if (b >= 2) z.Dyy += c * b * (b - 1) * xp[a] * yp[b - 2];
            }
        }
    }
    z.Dx *= inv;
    z.Dy *= inv;
    z.Dxx *= inv * inv;
    z.Dxy *= inv * inv;
    z.Dyy *= inv * inv;
    return z;
}

// Row of surface s of the monomial table, or null without a distortion.
__device__ __forceinline__ const double *zrow(const rpx_lens_t &L, const double *zc, int s) {
    return (zc && L.zernike_radius[s] > 0) ? zc + (uint64_t)s * RPX_LENS_ZTERMS : nullptr;
}

// Newton on G(t) = S(rho(t)) + D(t) - (p.z + t d.z - z_s), started at the
// vertex plane.  Converged once a step is below 1e-9 (1 + |t|): the point it
// reaches is then within float64 rounding of the root (Newton's error squares
// each step), and one further step there gives the root and, with it, S' and
// the distortion at the intersection.  Each step multiplies G / G' through by
// 1 + w and takes one reciprocal.
__device__ __forceinline__ bool newton_step(const double *P, const double *C, double Ru, double hz, V3 p, V3 d,
                                            double &t, double &dt, double &Sp, ZEval &z) {
    const double qx = p.x + t * d.x, qy = p.y + t * d.y;
    const double rho = qx * qx + qy * qy;
    Conic k;
    if (!conic<false>(P, rho, k)) return false;
    z = zernike_eval(C, Ru, qx, qy, false);
    Sp = slope(P, rho, k.y);
    const double G = P[0] * rho + k.w1 * (poly(P, rho) + z.D - (hz + t * d.z));     // (1 + w) G
    const double Gt = 2 * Sp * (qx * d.x + qy * d.y) + z.Dx * d.x + z.Dy * d.y - d.z;
    dt = -G * rcp_third(k.w1 * Gt);
    t += dt;
    return true;
}

__device__ __forceinline__ bool intersect(const double *P, const double *C, double Ru, double zs, double ap2, V3 p,
                                          V3 d, V3 &q, double &t, double &Sp, ZEval &z) {
    const double hz = p.z - zs;
    double dt = 0;
    t = -hz * rcp_third(d.z);
    bool conv = false;
    for (int it = 0; it < 60 && !conv; ++it) {
        if (!newton_step(P, C, Ru, hz, p, d, t, dt, Sp, z)) return false;
        conv = fabs(dt) <= 1e-9 * (1 + fabs(t));
    }
    if (!conv) return false;
    if (!newton_step(P, C, Ru, hz, p, d, t, dt, Sp, z)) return false;
    if (!(t > 0)) return false;
    q = v3(p.x + t * d.x, p.y + t * d.y, p.z + t * d.z);
    return !(q.x * q.x + q.y * q.y > ap2);
}

struct Refr {
    V3 N;                     // unit normal oriented along d
    double imlen, sgn;        // 1 / |m|, orientation of N
    double cosv, isr, kappa;  // isr = 1 / sqrt(1 - mu^2 (1 - cos^2))
    V3 t;
};

// TRACED as in conic: such a ray is not totally reflected.
template <bool TRACED>
__device__ __forceinline__ bool refract(double x, double y, double Sp, const ZEval &z, V3 d, double mu,
                                        Refr &r) {
    const V3 m = v3(-(2 * x * Sp + z.Dx), -(2 * y * Sp + z.Dy), 1.0);
    r.imlen = rsq_third(m.x * m.x + m.y * m.y + 1.0);
    const double c = (m.x * d.x + m.y * d.y + d.z) * r.imlen;
    r.sgn = c >= 0 ? 1.0 : -1.0;
    r.N = mul(m, r.imlen * r.sgn);
    r.cosv = c * r.sgn;
    double rr = 1 - mu * mu * (1 - r.cosv * r.cosv);
    if constexpr (TRACED) rr = fmax(rr, LEAST_ARG);
    else if (rr < 0) return false;
    r.isr = rr > 0 ? rsq_third(rr) : RPX_INF;
    r.kappa = (rr > 0 ? rr * r.isr : rr) - mu * r.cosv;
    r.t = v3(mu * d.x + r.N.x * r.kappa, mu * d.y + r.N.y * r.kappa, mu * d.z + r.N.z * r.kappa);
    return true;
}

struct LensArgs {
    rpx_lens_t L;
    rpx_rays_t rays;
    uint64_t n;
    const double *n_table;
    uint64_t n_wl;
    const double *zc;    // monomial table (n_surfaces x RPX_LENS_ZTERMS) or null
    int objective;
};

// Where a ray met a surface, and how far it came.
struct Kept {
    double x, y, t;
};

// Traces one ray: detector point (px, py), its wavefront path W and
// wavelength index; when `keep`, the direction entering every surface and its
// Kept, and the point on the last one.
template <bool ZK, bool WF>
__device__ __forceinline__ bool trace_ray(const LensArgs &A, uint64_t i, double &px, double &py, double &W,
                                          uint32_t &wl, V3 &last, V3 *sd, Kept *sq, bool keep) {
    const double *f = A.rays.f64;
    const uint64_t cap = A.rays.capacity;
    V3 p = v3(f[RPX_OX * cap + i], f[RPX_OY * cap + i], f[RPX_OZ * cap + i]);
    V3 d = unit(v3(f[RPX_DX * cap + i], f[RPX_DY * cap + i], f[RPX_DZ * cap + i]));
    wl = A.rays.u32[RPX_WL_IDX * cap + i];
    if (wl >= A.n_wl) return false;
    const double *nt = A.n_table + (uint64_t)wl * A.L.n_media;
    if constexpr (WF) W = f[RPX_ACCUM * cap + i];
    for (int s = 0; s < A.L.n_surfaces; ++s) {
        if (keep) sd[s] = d;
        const double *C = ZK ? zrow(A.L, A.zc, s) : nullptr;
        V3 q;
        double t, Sp;
        ZEval z;
        if (!intersect(A.L.param[s], C, A.L.zernike_radius[s], A.L.z[s], A.L.aperture[s] * A.L.aperture[s], p, d,
                       q, t, Sp, z))
            return false;
        Refr r;
        if (!refract<false>(q.x, q.y, Sp, z, d, nt[A.L.medium_before[s]] / nt[A.L.medium_after[s]], r)) return false;
        if constexpr (WF) W += nt[A.L.medium_before[s]] * t;
        if (keep) sq[s] = Kept{q.x, q.y, t};
        p = q;
        d = r.t;
    }
    if (!(d.z > 0)) return false;
    const double t = (A.L.detector_z - p.z) / d.z;
    px = p.x + t * d.x;
    py = p.y + t * d.y;
    if constexpr (WF) {
        const double nL = nt[A.L.medium_after[A.L.n_surfaces - 1]];
        W += nL * (-p.x * d.x - p.y * d.y + (A.L.detector_z - p.z) * d.z);
    }
    if (keep) {
        last = p;
        sd[A.L.n_surfaces] = d;
    }
    return true;
}

// Sums over the wavefront of four (two) values at once, in a fixed order: rows
// of 16 lanes trade places so that each row ends with one value's sum, in 7
// (6) adds where a butterfly takes 6 per value; lanes (l & 15) == 0 of row k
// (of rows 2k) hold value k's.
template <bool ROWS>
__device__ __forceinline__ double swap_add(double a, double b) {
    const uint64_t x = __double_as_longlong(a), y = __double_as_longlong(b);
    uint32_t lo[2], hi[2];
    if constexpr (ROWS) {
        const auto l = __builtin_amdgcn_permlane16_swap((uint32_t)x, (uint32_t)y, false, false);
        const auto h = __builtin_amdgcn_permlane16_swap((uint32_t)(x >> 32), (uint32_t)(y >> 32), false, false);
        lo[0] = l[0]; lo[1] = l[1]; hi[0] = h[0]; hi[1] = h[1];
    } else {
        const auto l = __builtin_amdgcn_permlane32_swap((uint32_t)x, (uint32_t)y, false, false);
        const auto h = __builtin_amdgcn_permlane32_swap((uint32_t)(x >> 32), (uint32_t)(y >> 32), false, false);
        lo[0] = l[0]; lo[1] = l[1]; hi[0] = h[0]; hi[1] = h[1];
    }
    return __longlong_as_double(((uint64_t)hi[0] << 32) | lo[0]) +
           __longlong_as_double(((uint64_t)hi[1] << 32) | lo[1]);
}

template <int N>
__device__ __forceinline__ double row_rotate(double v) {
    const uint64_t x = __double_as_longlong(v);
    const uint32_t lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)x, 0x120 + N, 0xF, 0xF, true);
    const uint32_t hi = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)(x >> 32), 0x120 + N, 0xF, 0xF, true);
    return __longlong_as_double(((uint64_t)hi << 32) | lo);
}

__device__ __forceinline__ double row_sum(double v) {
    v += row_rotate<8>(v);
    v += row_rotate<4>(v);
    v += row_rotate<2>(v);
    return v + row_rotate<1>(v);
}
__device__ __forceinline__ double wave_sum4(double v0, double v1, double v2, double v3) {
    return row_sum(swap_add<true>(swap_add<false>(v0, v2), swap_add<false>(v1, v3)));
}
__device__ __forceinline__ double wave_sum2(double v0, double v1) {
    const double a = swap_add<false>(v0, v1);
    return row_sum(swap_add<true>(a, a));
}
// Row k's sum (of wave_sum4) goes to out[k]; row 2k's (of wave_sum2) to out[k].
__device__ __forceinline__ void put4(double *out, int lane, double v) {
    if ((lane & 15) == 0) out[lane >> 4] = v;
}
__device__ __forceinline__ void put2(double *out, int lane, double v) {
    if ((lane & 31) == 0) out[lane >> 5] = v;
}

// Per-workgroup partials of the objective's moments (ZK: some surface has a
// distortion).  Spot RMS (width 4):
// kept rays, sum x, sum y, sum x^2 + y^2.  Wavefront RMS, pass 0 (width
// 2 n_wl): per wavelength, kept rays and sum W; pass 1 (width 2): kept rays
// and sum (W - mean_l)^2 with the per-wavelength means of pass 0 (read from
// moments).  Sums within a workgroup run in a fixed order.
template <bool ZK, bool WF>
__global__ __launch_bounds__(LB) void k_lens_forward(LensArgs A, int pass, const double *moments, double *partials) {
    __shared__ double red[LB / 64][2 * RPX_LENS_MAX_WFE_WAVELENGTHS];
    const uint64_t i = (uint64_t)blockIdx.x * LB + threadIdx.x;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    double px = 0, py = 0, W = 0;
    uint32_t wl = 0;
    V3 last;
    const bool ok = i < A.n && trace_ray<ZK, WF>(A, i, px, py, W, wl, last, nullptr, nullptr, false);
    int width;
    if constexpr (!WF) {
        width = 4;
        put4(red[wave], lane, wave_sum4(ok ? 1.0 : 0.0, ok ? px : 0.0, ok ? py : 0.0, ok ? px * px + py * py : 0.0));
    } else if (pass == 0) {
        width = 2 * (int)A.n_wl;
        for (int l = 0; l < (int)A.n_wl; ++l) {
            const bool m = ok && wl == (uint32_t)l;
            put2(&red[wave][2 * l], lane, wave_sum2(m ? 1.0 : 0.0, m ? W : 0.0));
        }
    } else {
        width = 2;
        double dv = 0;
        if (ok) {
            const double mu = moments[3 + 2 * wl] / moments[2 + 2 * wl];
            dv = (W - mu) * (W - mu);
        }
        put2(red[wave], lane, wave_sum2(ok ? 1.0 : 0.0, dv));
    }
    __syncthreads();
    if ((int)threadIdx.x < width) {
        double v = 0;
        for (int w = 0; w < LB / 64; ++w) v += red[w][threadIdx.x];
        partials[(uint64_t)threadIdx.x * gridDim.x + blockIdx.x] = v;
    }
}

// out[q] = sum over blocks b of partials[q * nb + b], fixed order; one
// workgroup per column q.  Columns from `width` on have no partials: zero.
__global__ __launch_bounds__(256) void k_lens_reduce(const double *partials, uint64_t nb, int width, double *out) {
    __shared__ double red[256];
    const int q = blockIdx.x;
    double v = 0;
    if (q < width)
        for (uint64_t b = threadIdx.x; b < nb; b += 256) v += partials[q * nb + b];
    red[threadIdx.x] = v;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (threadIdx.x < (unsigned)w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[q] = red[0];
}

// Objective value from its moments.
__device__ __forceinline__ double objective_value(int objective, const double *m) {
    if (objective == RPX_LENS_SPOT_RMS) {
        const double cx = m[1] / m[0], cy = m[2] / m[0];
        const double var = m[3] / m[0] - (cx * cx + cy * cy);
        return sqrt(var > 0 ? var : 0.0);
    }
    const double var = m[1] / m[0];
    return sqrt(var > 0 ? var : 0.0);
}

// Partials, column by column: the parameter block (6 n_surfaces), then with
// distortions the monomial block (RPX_LENS_ZTERMS n_surfaces).
template <bool ZK, bool WF>
__device__ __forceinline__ void lens_adjoint(const LensArgs &A, const double *moments, double *partials) {
    __shared__ double gsum[LB / 64][RPX_LENS_MAX_SURFACES * (6 + (ZK ? RPX_LENS_ZTERMS : 0))];
    const int S = A.L.n_surfaces, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int zbase = 6 * S;
    const uint64_t i = (uint64_t)blockIdx.x * LB + threadIdx.x;
    const double cnt = moments[0];
    const double obj = cnt > 0 ? objective_value(WF ? RPX_LENS_WAVEFRONT_RMS : RPX_LENS_SPOT_RMS, moments) : 0.0;
    V3 last = v3(0, 0, 0), sd[RPX_LENS_MAX_SURFACES + 1];
    Kept sq[RPX_LENS_MAX_SURFACES];
    double px = 0, py = 0, W = 0;
    uint32_t wl = 0;
    bool ok = (i < A.n) && cnt > 0 && obj > 0 && trace_ray<ZK, WF>(A, i, px, py, W, wl, last, sd, sq, true);
    const double *nt = ok ? A.n_table + (uint64_t)wl * A.L.n_media : A.n_table;
    // seeds: adjoints of (p, d) leaving the last surface, and the weight of
    // each segment's optical path (wavefront objective)
    V3 pb = v3(0, 0, 0), db = v3(0, 0, 0);
    double omega = 0;
    if (ok) {
        const V3 p = last, d = sd[S];
        if constexpr (!WF) {
            // d sigma / d (px, py) = (p - centroid) / (N sigma)
            const double cx = moments[1] / cnt, cy = moments[2] / cnt;
            const double gx = (px - cx) / (cnt * obj), gy = (py - cy) / (cnt * obj);
            const double t = (A.L.detector_z - p.z) / d.z;
            pb = v3(gx, gy, 0);
            db = v3(t * gx, t * gy, 0);
            const double tb = gx * d.x + gy * d.y;
            pb.z += -tb / d.z;
            db.z += -tb * t / d.z;
        } else {
            // d wfe / d W = (W - mean_l) / (N wfe); W's last term
            // n_L (P - p) . d with P = (0, 0, detector_z)
            const double mu = moments[3 + 2 * wl] / moments[2 + 2 * wl];
            omega = (W - mu) / (cnt * obj);
            const double nL = nt[A.L.medium_after[S - 1]];
            pb = mul(d, -nL * omega);
            db = mul(v3(-p.x, -p.y, A.L.detector_z - p.z), nL * omega);
        }
    }
    for (int s = S - 1; s >= 0; --s) {
        double th[6] = {0, 0, 0, 0, 0, 0};
        double zth[ZK ? RPX_LENS_ZTERMS : 1];
        const double *C = ZK ? zrow(A.L, A.zc, s) : nullptr;
        const double Ru = A.L.zernike_radius[s];
#pragma unroll
        for (int k = 0; k < (ZK ? RPX_LENS_ZTERMS : 1); ++k) zth[k] = 0;
        if (ok) {
            const double *P = A.L.param[s];
            const V3 d = sd[s];
            const Kept q = sq[s];
            const double t = q.t, rho = q.x * q.x + q.y * q.y;
            Conic k;
            conic<true>(P, rho, k);
            const double Sp = slope(P, rho, k.y);
            const ZEval z = zernike_eval(C, Ru, q.x, q.y, true);
            const double mu = nt[A.L.medium_before[s]] / nt[A.L.medium_after[s]];
            Refr r;
            refract<true>(q.x, q.y, Sp, z, d, mu, r);
            // outputs of the step: q (adjoint pb), r.t (adjoint db)
            const V3 tb = db;
            V3 qb = pb;
            V3 dbar = mul(tb, mu);
            V3 Nb = mul(tb, r.kappa);
            const double kb = dot(tb, r.N);
            const double srb = kb;
            const double cb = mu * (srb * r.isr * mu * r.cosv - kb);
            dbar = add(dbar, mul(r.N, cb));
            Nb = add(Nb, mul(d, cb));
            // oriented unit normal -> unnormalised m = (-(2 x S' + Dx), -(2 y S' + Dy), 1)
            const V3 Nu = mul(r.N, r.sgn), Nub = mul(Nb, r.sgn);
            const V3 mb = mul(sub(Nub, mul(Nu, dot(Nub, Nu))), r.imlen);
            const double Spb = -2 * (q.x * mb.x + q.y * mb.y);
            const double Dxb = -mb.x, Dyb = -mb.y;
            qb.x += -2 * Sp * mb.x + Dxb * z.Dxx + Dyb * z.Dxy;
            qb.y += -2 * Sp * mb.y + Dxb * z.Dxy + Dyb * z.Dyy;
            // with y = 1/w and v = 1/(1+w), u = (1 + k) c^2:
            //   S'' = c u y^3 / 4 + 2 A4 + 6 A6 rho + 12 A8 rho^2 + 20 A10 rho^3
            //   dS/dc = rho v + u rho^2 y v^2,    dS'/dc = y / 2 + u rho y^3 / 2
            //   dS/dk = c^3 rho^2 y v^2 / 2,      dS'/dk = c^3 rho y^3 / 4
            const double c = P[0], u = (1 + P[1]) * c * c, y3 = k.y * k.y * k.y, v = rcp_third(k.w1);
            const double yv2 = k.y * v * v, r2 = rho * rho, r3 = r2 * rho, c3 = c * c * c;
            const double rhob =
                Spb * (0.25 * c * u * y3 + 2 * P[2] + rho * (6 * P[3] + rho * (12 * P[4] + rho * (20 * P[5]))));
            qb.x += 2 * q.x * rhob;
            qb.y += 2 * q.y * rhob;
            // intersection q = p + t d with G(t; p, d, param) = 0; the
            // segment's optical path n_before t adds to t's adjoint
            V3 pbar = qb;
            dbar = add(dbar, mul(qb, t));
            const double tbar = WF ? dot(qb, d) + omega * nt[A.L.medium_before[s]] : dot(qb, d);
            const V3 Gp = v3(2 * q.x * Sp + z.Dx, 2 * q.y * Sp + z.Dy, -1.0);
            const double Gt = dot(Gp, d);
            const double lam = -tbar * rcp_third(Gt);
            pbar = add(pbar, mul(Gp, lam));
            dbar = add(dbar, mul(Gp, lam * t));
            th[0] = lam * (rho * v + u * r2 * yv2) + Spb * (0.5 * k.y + 0.5 * u * rho * y3);
            th[1] = lam * (0.5 * c3 * r2 * yv2) + Spb * (0.25 * c3 * rho * y3);
            th[2] = lam * r2 + Spb * (2 * rho);
            th[3] = lam * r3 + Spb * (3 * r2);
            th[4] = lam * (r2 * r2) + Spb * (4 * r3);
            th[5] = lam * (r2 * r3) + Spb * (5 * (r2 * r2));
            if constexpr (ZK) {
              if (C) {
                // dG/dC_k = M_k(q); dm/dC_k = -(dM_k/dx, dM_k/dy, 0)
                const double inv = 1.0 / Ru;
                double xp[ZDEG + 1], yp[ZDEG + 1];
                zpowers(q.x * inv, xp);
                zpowers(q.y * inv, yp);
                int k = 0;
#pragma unroll
                for (int dg = 0; dg <= ZDEG; ++dg) {
#pragma unroll
                    for (int a = dg; a >= 0; --a, ++k) {
                        const int b = dg - a;
                        double v = lam * xp[a] * yp[b];
                        if (a >= 1) v += Dxb * a * xp[a - 1] * yp[b] * inv;
                        if (b >= 1) v += Dyb * b * xp[a] * yp[b - 1] * inv;
                        zth[k] = v;
                    }
                }
              }
            }
            pb = pbar;
            db = dbar;
        }
        put4(&gsum[wave][s * 6], lane, wave_sum4(th[0], th[1], th[2], th[3]));
        put2(&gsum[wave][s * 6 + 4], lane, wave_sum2(th[4], th[5]));
        if constexpr (ZK) {
            double *g = &gsum[wave][zbase + s * RPX_LENS_ZTERMS];
            if (C) {
#pragma unroll
                for (int k = 0; k < RPX_LENS_ZTERMS; k += 4)
                    put4(g + k, lane, wave_sum4(zth[k], zth[k + 1], zth[k + 2], zth[k + 3]));
            } else if (lane < RPX_LENS_ZTERMS) {
                g[lane] = 0.0;
            }
        }
    }
    __syncthreads();
    const int width = S * (6 + (ZK ? RPX_LENS_ZTERMS : 0));
    for (int k = threadIdx.x; k < width; k += LB) {
        double v = 0;
        for (int w = 0; w < LB / 64; ++w) v += gsum[w][k];
        partials[(uint64_t)k * gridDim.x + blockIdx.x] = v;
    }
}

// Without distortions the adjoint fits 5 waves per SIMD (84 VGPRs).
template <bool WF>
__global__ __launch_bounds__(LB) __attribute__((amdgpu_waves_per_eu(5))) void k_lens_adjoint(
    LensArgs A, const double *moments, double *partials) {
    lens_adjoint<false, WF>(A, moments, partials);
}

template <bool WF>
__global__ __launch_bounds__(LB) void k_lens_adjoint_zernike(LensArgs A, const double *moments, double *partials) {
    lens_adjoint<true, WF>(A, moments, partials);
}

rpx_status_t check_lens(const rpx_lens_t *L, const rpx_rays_t *rays, uint64_t n, const double *n_table,
                        uint64_t n_wl) {
    if (!L || !rays) return rpx_set_error(RPX_E_INVALID, "null lens or rays");
    if (L->n_surfaces < 1 || L->n_surfaces > RPX_LENS_MAX_SURFACES)
        return rpx_set_error(RPX_E_INVALID, "lens must have 1..16 surfaces");
    if (L->n_media < 1) return rpx_set_error(RPX_E_INVALID, "lens has no media");
    for (int s = 0; s < L->n_surfaces; ++s)
        if (L->medium_before[s] < 0 || L->medium_before[s] >= L->n_media || L->medium_after[s] < 0 ||
            L->medium_after[s] >= L->n_media)
            return rpx_set_error(RPX_E_INVALID, "surface medium index out of range");
    if (rays->capacity < n || (n && (!rays->f64 || !rays->u32))) return rpx_set_error(RPX_E_INVALID, "rays");
    if (!n_table || n_wl == 0) return rpx_set_error(RPX_E_INVALID, "index table is empty");
    if (n > 0xFFFFFFFFull) return rpx_set_error(RPX_E_UNSUPPORTED, "more than 2^32-1 rays");
    return RPX_OK;
}

rpx_status_t check_objective(const rpx_lens_t *L, const double *zcart, uint64_t n_wl, int32_t objective) {
    if (objective != RPX_LENS_SPOT_RMS && objective != RPX_LENS_WAVEFRONT_RMS)
        return rpx_set_error(RPX_E_INVALID, "unknown lens objective");
    if (objective == RPX_LENS_WAVEFRONT_RMS && n_wl > RPX_LENS_MAX_WFE_WAVELENGTHS)
        return rpx_set_error(RPX_E_UNSUPPORTED, "the wavefront objective takes at most 16 wavelengths");
    for (int s = 0; s < L->n_surfaces; ++s)
        if (L->zernike_radius[s] > 0 && !zcart)
            return rpx_set_error(RPX_E_INVALID, "a surface has a distortion but the monomial table is null");
    return RPX_OK;
}

bool has_distortion(const rpx_lens_t *L, const double *zcart) {
    if (!zcart) return false;
    for (int s = 0; s < L->n_surfaces; ++s)
        if (L->zernike_radius[s] > 0) return true;
    return false;
}

uint64_t lens_width(int32_t n_surfaces) {
    return (uint64_t)std::max(RPX_LENS_MOMENTS, (6 + RPX_LENS_ZTERMS) * std::max(1, (int)n_surfaces));
}

rpx_status_t lens_eval(const rpx_lens_t *lens, const double *zcart, const rpx_rays_t *rays, uint64_t n_rays,
                       const double *n_table, uint64_t n_wavelengths, int32_t objective, double *moments,
                       void *workspace, uint64_t workspace_bytes, hipStream_t s) {
    if (!moments) return rpx_set_error(RPX_E_INVALID, "moments is null");
    if (!workspace || workspace_bytes < rpx_lens_workspace_bytes(n_rays, lens->n_surfaces))
        return rpx_set_error(RPX_E_INVALID, "workspace too small");
    const uint64_t nb = std::max<uint64_t>((n_rays + LB - 1) / LB, 1);
    LensArgs A{*lens, *rays, n_rays, n_table, n_wavelengths, zcart, objective};
    double *part = (double *)workspace;
    const bool zk = has_distortion(lens, zcart), wf = objective == RPX_LENS_WAVEFRONT_RMS;
    auto forward = zk ? (wf ? k_lens_forward<true, true> : k_lens_forward<true, false>)
                      : (wf ? k_lens_forward<false, true> : k_lens_forward<false, false>);
    if (objective == RPX_LENS_SPOT_RMS) {
        hipLaunchKernelGGL(forward, dim3((unsigned)nb), dim3(LB), 0, s, A, 0, (const double *)moments, part);
        RPX_HIP_TRY(hipGetLastError());
        hipLaunchKernelGGL(k_lens_reduce, dim3(4), dim3(256), 0, s, (const double *)part, nb, 4, moments);
        RPX_HIP_TRY(hipGetLastError());
        return RPX_OK;
    }
    const int w0 = 2 * (int)n_wavelengths;
    hipLaunchKernelGGL(forward, dim3((unsigned)nb), dim3(LB), 0, s, A, 0, (const double *)moments, part);
    RPX_HIP_TRY(hipGetLastError());
    hipLaunchKernelGGL(k_lens_reduce, dim3(w0), dim3(256), 0, s, (const double *)part, nb, w0, moments + 2);
    RPX_HIP_TRY(hipGetLastError());
    hipLaunchKernelGGL(forward, dim3((unsigned)nb), dim3(LB), 0, s, A, 1, (const double *)moments, part);
    RPX_HIP_TRY(hipGetLastError());
    hipLaunchKernelGGL(k_lens_reduce, dim3(2), dim3(256), 0, s, (const double *)part, nb, 2, moments);
    RPX_HIP_TRY(hipGetLastError());
    return RPX_OK;
}

rpx_status_t lens_grad(const rpx_lens_t *lens, const double *zcart, const rpx_rays_t *rays, uint64_t n_rays,
                       const double *n_table, uint64_t n_wavelengths, int32_t objective, const double *moments,
                       double *grad, int columns, void *workspace, uint64_t workspace_bytes, hipStream_t s) {
    if (!moments || !grad) return rpx_set_error(RPX_E_INVALID, "moments or grad is null");
    if (!workspace || workspace_bytes < rpx_lens_workspace_bytes(n_rays, lens->n_surfaces))
        return rpx_set_error(RPX_E_INVALID, "workspace too small");
    const uint64_t nb = std::max<uint64_t>((n_rays + LB - 1) / LB, 1);
    LensArgs A{*lens, *rays, n_rays, n_table, n_wavelengths, zcart, objective};
    const bool zk = has_distortion(lens, zcart), wf = objective == RPX_LENS_WAVEFRONT_RMS;
    const int width = (6 + (zk ? RPX_LENS_ZTERMS : 0)) * lens->n_surfaces;
    auto adjoint = zk ? (wf ? k_lens_adjoint_zernike<true> : k_lens_adjoint_zernike<false>)
                      : (wf ? k_lens_adjoint<true> : k_lens_adjoint<false>);
    hipLaunchKernelGGL(adjoint, dim3((unsigned)nb), dim3(LB), 0, s, A, moments, (double *)workspace);
    RPX_HIP_TRY(hipGetLastError());
    hipLaunchKernelGGL(k_lens_reduce, dim3(columns), dim3(256), 0, s, (const double *)workspace, nb, width, grad);
    RPX_HIP_TRY(hipGetLastError());
    return RPX_OK;
}

}  // namespace

extern "C" uint64_t rpx_lens_workspace_bytes(uint64_t n_rays, int32_t n_surfaces) {
    const uint64_t nb = (n_rays + LB - 1) / LB;
    return std::max<uint64_t>(nb, 1) * lens_width(n_surfaces) * 8;
}

extern "C" rpx_status_t rpx_lens_eval(const rpx_lens_t *lens, const double *zcart, const rpx_rays_t *rays,
                                      uint64_t n_rays, const double *n_table, uint64_t n_wavelengths,
                                      int32_t objective, double *moments, void *workspace, uint64_t workspace_bytes,
                                      void *stream) {
    rpx_status_t st = check_lens(lens, rays, n_rays, n_table, n_wavelengths);
    if (!st) st = check_objective(lens, zcart, n_wavelengths, objective);
    if (st) return st;
    return lens_eval(lens, zcart, rays, n_rays, n_table, n_wavelengths, objective, moments, workspace,
                     workspace_bytes, (hipStream_t)stream);
}

extern "C" rpx_status_t rpx_lens_grad(const rpx_lens_t *lens, const double *zcart, const rpx_rays_t *rays,
                                      uint64_t n_rays, const double *n_table, uint64_t n_wavelengths,
                                      int32_t objective, const double *moments, double *grad, void *workspace,
                                      uint64_t workspace_bytes, void *stream) {
    rpx_status_t st = check_lens(lens, rays, n_rays, n_table, n_wavelengths);
    if (!st) st = check_objective(lens, zcart, n_wavelengths, objective);
    if (st) return st;
    return lens_grad(lens, zcart, rays, n_rays, n_table, n_wavelengths, objective, moments, grad,
                     (6 + RPX_LENS_ZTERMS) * lens->n_surfaces, workspace, workspace_bytes, (hipStream_t)stream);
}

extern "C" rpx_status_t rpx_lens_spot(const rpx_lens_t *lens, const rpx_rays_t *rays, uint64_t n_rays,
                                      const double *n_table, uint64_t n_wavelengths, double *moments, void *workspace,
                                      uint64_t workspace_bytes, void *stream) {
    rpx_status_t st = check_lens(lens, rays, n_rays, n_table, n_wavelengths);
    if (st) return st;
    rpx_lens_t L = *lens;
    for (int s = 0; s < RPX_LENS_MAX_SURFACES; ++s) L.zernike_radius[s] = 0;
    return lens_eval(&L, nullptr, rays, n_rays, n_table, n_wavelengths, RPX_LENS_SPOT_RMS, moments, workspace,
                     workspace_bytes, (hipStream_t)stream);
}

extern "C" rpx_status_t rpx_lens_spot_grad(const rpx_lens_t *lens, const rpx_rays_t *rays, uint64_t n_rays,
                                           const double *n_table, uint64_t n_wavelengths, const double *moments,
                                           double *grad, void *workspace, uint64_t workspace_bytes, void *stream) {
    rpx_status_t st = check_lens(lens, rays, n_rays, n_table, n_wavelengths);
    if (st) return st;
    rpx_lens_t L = *lens;
    for (int s = 0; s < RPX_LENS_MAX_SURFACES; ++s) L.zernike_radius[s] = 0;
    return lens_grad(&L, nullptr, rays, n_rays, n_table, n_wavelengths, RPX_LENS_SPOT_RMS, moments, grad,
                     6 * lens->n_surfaces, workspace, workspace_bytes, (hipStream_t)stream);
}
