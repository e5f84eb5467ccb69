// Gausslet E-field summation on gfx950.
//
//   k_modes_gc    one gausslet per lane: parabasal offsets/slopes
//                 (evaluate_neighbours_gc, core/fields.py:114-136) fused with
//                 the closed-form 3x3 least-squares mode fit
//                 (evaluate_one_mode, cfields.pyx:156-215).
//   k_field_prep  per-gausslet invariants of sum_gaussian_modes
//                 (cfields.pyx:76-99), one 288-byte record per gausslet.
//   k_field_sum   one evaluation point per lane; the gausslet is the same in
//                 every lane, so its record comes by scalar loads into SGPRs.
//                 A lane sums a chunk of gausslets in order; k_field_reduce
//                 adds the chunks' sums in a fixed order.
#include <hip/hip_runtime.h>
#include <mutex>
#include <algorithm>
#include <string>
#include "rpx_materials.h"
#include "rpx_host.h"
#include "rpx_gen.h"

using namespace rpx;

// --------------------------------------------------------------- mode fit
RPX_DEV void fit_one_mode(const double *x, const double *y, const double *dx, const double *dy, int size,
                          double blending, double *o) {
    double a00 = 0, a01 = 0, a02 = 0, a11 = 0, a12 = 0, a22 = 0, b0 = 0, b1 = 0, b2 = 0;
    for (int i = 0; i < size; ++i) {
        double xi2 = x[i] * x[i];
        double yi2 = y[i] * y[i];
        a00 += xi2 * xi2;
        a01 += 2 * xi2 * x[i] * y[i];
        a02 += xi2 * yi2;
        a11 += 4 * xi2 * yi2;
        a12 += 2 * x[i] * y[i] * yi2;
        a22 += yi2 * yi2;
        b0 += xi2;
        b1 += 2 * x[i] * y[i];
        b2 += yi2;
    }
    double den = (-a00 * a11 * a22 + a00 * (a12 * a12) + (a01 * a01) * a22 - 2 * a01 * a02 * a12 + (a02 * a02) * a11);
    o[1] = blending * (-b0 * (a11 * a22 - (a12 * a12)) + b1 * (a01 * a22 - a02 * a12) - b2 * (a01 * a12 - a02 * a11)) / den;
    o[3] = -blending * (b0 * (a01 * a22 - a02 * a12) - b1 * (a00 * a22 - (a02 * a02)) + b2 * (a00 * a12 - a01 * a02)) / den;
    o[5] = blending * (-b0 * (a01 * a12 - a02 * a11) + b1 * (a00 * a12 - a01 * a02) - b2 * (a00 * a11 - (a01 * a01))) / den;
    a00 = a01 = a02 = a11 = a12 = a22 = b0 = b1 = b2 = 0;
    for (int i = 0; i < size; ++i) {
        double xi2 = x[i] * x[i];
        double yi2 = y[i] * y[i];
        a00 += xi2;
        a01 += x[i] * y[i];
        a11 += xi2 + yi2;
        a22 += yi2;
        b0 += dx[i] * x[i];
        b1 += dx[i] * y[i] + dy[i] * x[i];
        b2 += dy[i] * y[i];
    }
    a12 = a01 * a01;
    den = (a00 * a12 - a00 * a11 * a22 + a12 * a22);
    o[0] = (-a12 * b2 + a01 * a22 * b1 + b0 * (a12 - a11 * a22)) / den;
    o[2] = -(a00 * a01 * b2 - a00 * a22 * b1 + a01 * a22 * b0) / den;
    o[4] = (a00 * a01 * b1 - a12 * b0 - b2 * (a00 * a11 - a12)) / den;
}

__global__ void k_modes_gc(rpx_rays_t g, uint64_t n, double blending, double *modes) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint64_t c = g.capacity;
    const double *f = g.f64;
    V3 o = v3(f[RPX_OX * c + i], f[RPX_OY * c + i], f[RPX_OZ * c + i]);
    V3 d = v3(f[RPX_DX * c + i], f[RPX_DY * c + i], f[RPX_DZ * c + i]);
    V3 E = v3(f[RPX_EX * c + i], f[RPX_EY * c + i], f[RPX_EZ * c + i]);
    V3 H = cross(E, d);  // numpy.cross(E, direction)
    double x[6], y[6], dx[6], dy[6];
    for (int j = 0; j < RPX_N_PARA; ++j) {
        const uint64_t b = (uint64_t)j * RPX_PARA_FIELDS;
        V3 po = v3(g.para[(b + 0) * c + i], g.para[(b + 1) * c + i], g.para[(b + 2) * c + i]);
        V3 nd = v3(g.para[(b + 3) * c + i], g.para[(b + 4) * c + i], g.para[(b + 5) * c + i]);
        V3 off = sub(po, o);
        double dz = (nd.x * d.x + nd.y * d.y) + nd.z * d.z;
        x[j] = (off.x * E.x + off.y * E.y) + off.z * E.z;
        y[j] = (off.x * H.x + off.y * H.y) + off.z * H.z;
        dx[j] = ((nd.x * E.x + nd.y * E.y) + nd.z * E.z) / dz;
        dy[j] = ((nd.x * H.x + nd.y * H.y) + nd.z * H.z) / dz;
    }
    fit_one_mode(x, y, dx, dy, RPX_N_PARA, blending, modes + 6 * i);
}

#define RPX_MAX_ROW 32

__global__ void k_modes_xy(const double *X, const double *Y, const double *DX, const double *DY, uint64_t n,
                           int row, double blending, double *modes) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    fit_one_mode(X + i * row, Y + i * row, DX + i * row, DY + i * row, row, blending, modes + 6 * i);
}

extern "C" rpx_status_t rpx_gausslet_modes(const rpx_rays_t *g, uint64_t n, double blending, double *modes,
                                           void *stream) {
    if (n == 0) return RPX_OK;
    if (!g || !g->f64 || !g->para || !modes || g->capacity < n)
        return rpx_set_error(RPX_E_INVALID, "gausslet buffers");
    hipLaunchKernelGGL(k_modes_gc, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream, *g, n,
                       blending, modes);
    RPX_HIP_TRY(hipGetLastError());
    return RPX_OK;
}

extern "C" rpx_status_t rpx_evaluate_modes(const double *x, const double *y, const double *dx, const double *dy,
                                           uint64_t n, int32_t row, double blending, double *modes, void *stream) {
    if (n == 0) return RPX_OK;
    if (!x || !y || !dx || !dy || !modes || row < 1 || row > RPX_MAX_ROW)
        return rpx_set_error(RPX_E_INVALID, "mode-fit buffers or row size");
    hipLaunchKernelGGL(k_modes_xy, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream, x, y, dx,
                       dy, n, row, blending, modes);
    RPX_HIP_TRY(hipGetLastError());
    return RPX_OK;
}

// ------------------------------------------------------ ray-field modes
// The RayField path of eval_Efield_from_rays (core/fields.py:196-218):
//   k_project_sphere    project_to_sphere (core/fields.py:51-80): rays whose
//                       line meets the sphere move back to the nearer
//                       intersection; the others are dropped (compacted in
//                       ray order).
//   k_ray_field_modes   evaluate_neighbours (core/fields.py:83-111) fused with
//                       the mode fit: rays with six neighbours >= 0 project
//                       each neighbour onto their own origin plane, fit the
//                       mode, and are compacted with it in ray order.
// numpy's sum over a length-3 axis accumulates from +0.0: ((0 + a) + b) + c
// (the leading zero only changes the sign of an exactly zero result).
__device__ __forceinline__ double np_sum3(double a, double b, double c) { return ((0.0 + a) + b) + c; }

__global__ __launch_bounds__(RPX_BLOCK) void k_project_sphere(rpx_rays_t in, uint64_t n, V3 centre, double radius_sq,
                                                              rpx_rays_t out, Workspace w) {
    __shared__ uint32_t lds_wave[RPX_BLOCK / 64];
    __shared__ uint32_t lds_tile;
    __shared__ uint64_t lds_excl;
    if (threadIdx.x == 0) lds_tile = atomicAdd(&w.ctl->tile_counter, 1u);
    __syncthreads();
    const uint32_t tile = lds_tile;
    const uint64_t i = (uint64_t)tile * RPX_BLOCK + threadIdx.x;
    bool sel = false;
    double alpha = 0.0;
    if (i < n) {
        const double *f = in.f64;
        const uint64_t c = in.capacity;
        const V3 o = sub(v3(f[RPX_OX * c + i], f[RPX_OY * c + i], f[RPX_OZ * c + i]), centre);
        const V3 d = v3(f[RPX_DX * c + i], f[RPX_DY * c + i], f[RPX_DZ * c + i]);
        const double cc = np_sum3(o.x * o.x, o.y * o.y, o.z * o.z) - radius_sq;
        const double b = 2 * np_sum3(d.x * o.x, d.y * o.y, d.z * o.z);
        const double disc = b * b - 4 * cc;
        sel = disc >= 0.0;
        if (sel) {
            const double sq = sqrt(disc);
            const double root1 = (-b + sq) / 2, root2 = (-b - sq) / 2;
            alpha = root2 < root1 ? root2 : root1;
        }
    }
    uint32_t block_total;
    const uint32_t local = block_scan_small(sel ? 1u : 0u, lds_wave, &block_total);
    if (threadIdx.x < 64) {
        const uint64_t excl = lookback(w.tile_status, tile, 0, block_total, &w.ctl->error);
        if (threadIdx.x == 0) lds_excl = excl;
    }
    __syncthreads();
    const uint64_t pos = lds_excl + local;
    if (sel && pos < out.capacity) {
        Ray r = load_ray(in, i);
        r.origin = add(r.origin, mul(r.direction, alpha));
        r.accum = r.accum + alpha * r.n.re;
        store_ray(out, pos, r);
    }
    if (threadIdx.x == 0 && (uint64_t)tile == (n - 1) / RPX_BLOCK) w.ctl->children = lds_excl + block_total;
}

__global__ __launch_bounds__(RPX_BLOCK) void k_ray_field_modes(rpx_rays_t in, uint64_t n, const int32_t *nb,
                                                               double blending, rpx_rays_t out, double *modes,
                                                               double *xy, Workspace w) {
    __shared__ uint32_t lds_wave[RPX_BLOCK / 64];
    __shared__ uint32_t lds_tile;
    __shared__ uint64_t lds_excl;
    if (threadIdx.x == 0) lds_tile = atomicAdd(&w.ctl->tile_counter, 1u);
    __syncthreads();
    const uint32_t tile = lds_tile;
    const uint64_t i = (uint64_t)tile * RPX_BLOCK + threadIdx.x;
    bool sel = false;
    double m[6], x[6], y[6], dx[6], dy[6];
    if (i < n) {
        int32_t k6[6];
        sel = true;
        for (int j = 0; j < 6; ++j) {
            k6[j] = nb[i * 6 + j];
            if (k6[j] < 0) sel = false;
        }
        if (sel) {
            for (int j = 0; j < 6; ++j)
                if ((uint64_t)k6[j] >= n) {
                    atomicAdd((unsigned long long *)&w.ctl->hits, 1ull);
                    sel = false;
                }
        }
        if (sel) {
            const double *f = in.f64;
            const uint64_t c = in.capacity;
            const V3 o = v3(f[RPX_OX * c + i], f[RPX_OY * c + i], f[RPX_OZ * c + i]);
            const V3 d = v3(f[RPX_DX * c + i], f[RPX_DY * c + i], f[RPX_DZ * c + i]);
            const V3 E = v3(f[RPX_EX * c + i], f[RPX_EY * c + i], f[RPX_EZ * c + i]);
            const V3 H = cross(E, d);  // numpy.cross(E, direction)
            for (int j = 0; j < 6; ++j) {
                const uint64_t q = (uint64_t)k6[j];
                const V3 no = v3(f[RPX_OX * c + q], f[RPX_OY * c + q], f[RPX_OZ * c + q]);
                const V3 nd = v3(f[RPX_DX * c + q], f[RPX_DY * c + q], f[RPX_DZ * c + q]);
                const V3 off = sub(no, o);
                const double dz = np_sum3(nd.x * d.x, nd.y * d.y, nd.z * d.z);
                const double alpha = (-np_sum3(off.x * d.x, off.y * d.y, off.z * d.z)) / dz;
                const V3 pr = add(off, mul(nd, alpha));
                x[j] = np_sum3(pr.x * E.x, pr.y * E.y, pr.z * E.z);
                y[j] = np_sum3(pr.x * H.x, pr.y * H.y, pr.z * H.z);
                dx[j] = np_sum3(nd.x * E.x, nd.y * E.y, nd.z * E.z) / dz;
                dy[j] = np_sum3(nd.x * H.x, nd.y * H.y, nd.z * H.z) / dz;
            }
            fit_one_mode(x, y, dx, dy, 6, blending, m);
        }
    }
    uint32_t block_total;
    const uint32_t local = block_scan_small(sel ? 1u : 0u, lds_wave, &block_total);
    if (threadIdx.x < 64) {
        const uint64_t excl = lookback(w.tile_status, tile, 0, block_total, &w.ctl->error);
        if (threadIdx.x == 0) lds_excl = excl;
    }
    __syncthreads();
    const uint64_t pos = lds_excl + local;
    if (sel && pos < out.capacity) {
        store_ray(out, pos, load_ray(in, i));
        for (int q = 0; q < 6; ++q) modes[6 * pos + q] = m[q];
        if (xy) {
            for (int q = 0; q < 6; ++q) {
                xy[24 * pos + q] = x[q];
                xy[24 * pos + 6 + q] = y[q];
                xy[24 * pos + 12 + q] = dx[q];
                xy[24 * pos + 18 + q] = dy[q];
            }
        }
    }
    if (threadIdx.x == 0 && (uint64_t)tile == (n - 1) / RPX_BLOCK) w.ctl->children = lds_excl + block_total;
}

static rpx_status_t compact_launch_checks(const rpx_rays_t *in, uint64_t n, const rpx_rays_t *out, uint64_t ws_bytes,
                                          void *ws) {
    if (!in || in->capacity < n) return rpx_set_error(RPX_E_INVALID, "input rays");
    if (n > 0 && (!in->f64 || !in->u32)) return rpx_set_error(RPX_E_INVALID, "input rays have null fields");
    if (!out || (out->capacity > 0 && (!out->f64 || !out->u32))) return rpx_set_error(RPX_E_INVALID, "output rays");
    if (n > 0xFFFFFFFFull) return rpx_set_error(RPX_E_UNSUPPORTED, "more than 2^32-1 rays");
    if (n > 0 && (!ws || ws_bytes < rpx_trace_workspace_bytes(n))) return rpx_set_error(RPX_E_INVALID, "workspace too small");
    return RPX_OK;
}

static rpx_status_t finish_compaction(const Workspace &w, uint64_t capacity, uint64_t *n_out, hipStream_t stream,
                                      const char *what) {
    GenControl ctl;
    RPX_HIP_TRY(read_control(ctl, w.ctl, stream));
    if (ctl.error) return rpx_set_error(RPX_E_HIP, std::string(what) + ": a look-back wait exceeded its poll limit");
    *n_out = ctl.children;
    if (ctl.hits)
        return rpx_set_error(RPX_E_INVALID, std::to_string(ctl.hits) + " rays have a neighbour index outside the rays");
    if (ctl.children > capacity)
        return rpx_set_error(RPX_E_CAPACITY, std::string(what) + ": output capacity below " +
                                                 std::to_string(ctl.children));
    return RPX_OK;
}

extern "C" rpx_status_t rpx_project_to_sphere(const rpx_rays_t *in, uint64_t n, const double *centre, double radius,
                                              rpx_rays_t *out, uint64_t *n_out, void *workspace,
                                              uint64_t workspace_bytes, void *stream_) {
    if (!n_out) return rpx_set_error(RPX_E_INVALID, "n_out is null");
    *n_out = 0;
    if (!centre) return rpx_set_error(RPX_E_INVALID, "centre is null");
    if (rpx_status_t st = compact_launch_checks(in, n, out, workspace_bytes, workspace)) return st;
    if (n == 0) return RPX_OK;
    hipStream_t stream = (hipStream_t)stream_;
    Workspace w = carve(workspace, n);
    const uint64_t nb = (n + RPX_BLOCK - 1) / RPX_BLOCK;
    hipLaunchKernelGGL(k_clear, dim3((unsigned)((std::max<uint64_t>(nb, RPX_SHARDS * RPX_LDS_FACES) + 255) / 256)),
                       dim3(256), 0, stream, w.tile_status, nb, w.ctl);
    RPX_HIP_TRY(hipGetLastError());
    V3 c;
    c.x = centre[0];
    c.y = centre[1];
    c.z = centre[2];
    hipLaunchKernelGGL(k_project_sphere, dim3((unsigned)nb), dim3(RPX_BLOCK), 0, stream, *in, n, c, radius * radius,
                       *out, w);
    RPX_HIP_TRY(hipGetLastError());
    return finish_compaction(w, out->capacity, n_out, stream, "project_to_sphere");
}

extern "C" rpx_status_t rpx_ray_field_modes(const rpx_rays_t *rays, uint64_t n, const int32_t *neighbours,
                                            double blending, rpx_rays_t *out, double *modes, double *neighbour_xy,
                                            uint64_t *n_out, void *workspace, uint64_t workspace_bytes,
                                            void *stream_) {
    if (!n_out) return rpx_set_error(RPX_E_INVALID, "n_out is null");
    *n_out = 0;
    if (rpx_status_t st = compact_launch_checks(rays, n, out, workspace_bytes, workspace)) return st;
    if (n == 0) return RPX_OK;
    if (!neighbours) return rpx_set_error(RPX_E_INVALID, "neighbours are null");
    if (out->capacity > 0 && !modes) return rpx_set_error(RPX_E_INVALID, "modes are null");
    hipStream_t stream = (hipStream_t)stream_;
    Workspace w = carve(workspace, n);
    const uint64_t nb = (n + RPX_BLOCK - 1) / RPX_BLOCK;
    hipLaunchKernelGGL(k_clear, dim3((unsigned)((std::max<uint64_t>(nb, RPX_SHARDS * RPX_LDS_FACES) + 255) / 256)),
                       dim3(256), 0, stream, w.tile_status, nb, w.ctl);
    RPX_HIP_TRY(hipGetLastError());
    hipLaunchKernelGGL(k_ray_field_modes, dim3((unsigned)nb), dim3(RPX_BLOCK), 0, stream, *rays, n, neighbours,
                       blending, *out, modes, neighbour_xy, w);
    RPX_HIP_TRY(hipGetLastError());
    return finish_compaction(w, out->capacity, n_out, stream, "ray field modes");
}

// ----------------------------------------------- decomposition mode maths
// calc_mode_curvature (cfields.pyx:231-293): mode basis and curvature
// coefficients from the wavefront's first and second derivatives.
__global__ __launch_bounds__(256) void k_mode_curvature(const double *dx, const double *dy, const double *dx2,
                                                        const double *dy2, const double *dxdy, uint64_t n,
                                                        double *A, double *B, double *C, double *x, double *y,
                                                        double *z) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    V3 c = norm(v3(-dx[i], -dy[i], 1.0));
    V3 b = v3(0.0, 0.0, 1.0);
    const V3 a = norm(cross(b, c));
    b = cross(c, a);
    x[3 * i] = a.x; x[3 * i + 1] = a.y; x[3 * i + 2] = a.z;
    y[3 * i] = b.x; y[3 * i + 1] = b.y; y[3 * i + 2] = b.z;
    z[3 * i] = c.x; z[3 * i + 1] = c.y; z[3 * i + 2] = c.z;
    const double Fz = c.x * dx[i] + c.y * dy[i] + c.z;
    A[i] = -(a.x * a.x * dx2[i] + 2 * a.x * a.y * dxdy[i] + a.y * a.y * dy2[i]) / Fz;
    B[i] = -(a.x * b.x * dx2[i] + (a.x * b.y + b.x * a.y) * dxdy[i] + a.y * b.y * dy2[i]) / Fz;
    C[i] = -(b.x * b.x * dx2[i] + 2 * b.x * b.y * dxdy[i] + b.y * b.y * dy2[i]) / Fz;
}

extern "C" rpx_status_t rpx_calc_mode_curvature(const double *dx, const double *dy, const double *dx2,
                                                const double *dy2, const double *dxdy, uint64_t n, double *A,
                                                double *B, double *C, double *x, double *y, double *z,
                                                void *stream) {
    if (n == 0) return RPX_OK;
    if (!dx || !dy || !dx2 || !dy2 || !dxdy || !A || !B || !C || !x || !y || !z)
        return rpx_set_error(RPX_E_INVALID, "mode curvature buffers");
    hipLaunchKernelGGL(k_mode_curvature, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream, dx, dy,
                       dx2, dy2, dxdy, n, A, B, C, x, y, z);
    RPX_HIP_TRY(hipGetLastError());
    return RPX_OK;
}

// apply_mode_curvature (cfields.pyx:397-424): tilts each parabasal direction
// by the curvature coefficients in the base ray's (E, E x d) frame.
__global__ __launch_bounds__(256) void k_apply_mode_curvature(rpx_rays_t g, uint64_t n, const double *A,
                                                              const double *B, const double *C) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double *f = g.f64;
    const uint64_t c = g.capacity;
    const V3 o = v3(f[RPX_OX * c + i], f[RPX_OY * c + i], f[RPX_OZ * c + i]);
    const V3 zz = v3(f[RPX_DX * c + i], f[RPX_DY * c + i], f[RPX_DZ * c + i]);
    const V3 xx = v3(f[RPX_EX * c + i], f[RPX_EY * c + i], f[RPX_EZ * c + i]);
    const V3 yy = cross(xx, zz);
    const double a = A[i], b = B[i], cc = C[i];
    for (int j = 0; j < RPX_N_PARA; ++j) {
        const uint64_t q = (uint64_t)j * RPX_PARA_FIELDS;
        const V3 po = v3(g.para[(q + 0) * c + i], g.para[(q + 1) * c + i], g.para[(q + 2) * c + i]);
        const V3 pd = v3(g.para[(q + 3) * c + i], g.para[(q + 4) * c + i], g.para[(q + 5) * c + i]);
        const V3 r = sub(po, o);
        const double px = dot(r, xx), py = dot(r, yy);
        V3 shift = mul(xx, (-a * px - b * py));
        shift = add(shift, mul(yy, (-cc * py - b * px)));
        const V3 nd = norm(add(shift, pd));
        g.para[(q + 3) * c + i] = nd.x;
        g.para[(q + 4) * c + i] = nd.y;
        g.para[(q + 5) * c + i] = nd.z;
    }
}

extern "C" rpx_status_t rpx_apply_mode_curvature(rpx_rays_t *gausslets, uint64_t n, const double *A, const double *B,
                                                 const double *C, void *stream) {
    if (n == 0) return RPX_OK;
    if (!gausslets || gausslets->capacity < n || !gausslets->f64 || !gausslets->para || !A || !B || !C)
        return rpx_set_error(RPX_E_INVALID, "mode curvature buffers");
    hipLaunchKernelGGL(k_apply_mode_curvature, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                       *gausslets, n, A, B, C);
    RPX_HIP_TRY(hipGetLastError());
    return RPX_OK;
}

// calc_mode_U (cfields.pyx:118-151), statement by statement.
RPX_DEV Cx calc_mode_u(Cx A, Cx B, Cx C, Cx detG0, V3 pt, V3 E, V3 H, V3 dir, Cx k, double phase,
                       double inv_root_area) {
    const Cx I = cx(0.0, 1.0);
    const Cx rootI = cx(sqrt(0.5), sqrt(0.5));
    const double x = dot(pt, E), y = dot(pt, H), z = dot(pt, dir);
    const Cx denom = cmul(cadd(cadd(cx(1, 0), cmul(cx(z, 0), cadd(A, C))), cmul(cx(z * z, 0), detG0)), cx(2, 0));
    const Cx zd = cmul(cx(z, 0), detG0);
    const Cx AA = cdiv(cadd(A, zd), denom);
    const Cx CC = cdiv(cadd(C, zd), denom);
    Cx inner = cadd(cx(z, 0), cmul(AA, cx(x * x, 0)));
    inner = cadd(inner, cdiv(cmul(B, cx(2 * x * y, 0)), denom));
    inner = cadd(inner, cmul(CC, cx(y * y, 0)));
    Cx U = cexp_(cmul(I, cadd(cx(phase, 0), cmul(k, inner))));
    const Cx q1 = cadd(cx(1, 0), cmul(cx(z, 0), A));
    const Cx q2 = cadd(cx(1, 0), cmul(cx(z, 0), C));
    const Cx zb = cmul(cx(z, 0), B);
    U = cdiv(U, csqrt_(cmul(csub(cmul(q1, q2), cmul(zb, zb)), I)));
    return cmul(U, cmul(cx(inv_root_area, 0), rootI));
}

// build_interaction_matrix (cfields.pyx:295-395): the COO entries (i, j,
// E_ij) for every mode i and test point j within max_spacing, in (i, j)
// order -- one lane per pair of the flattened index i * L + j, placed by the
// look-back.
struct InteractionArgs {
    const double *rx, *ry, *tx, *ty, *A, *B, *C, *x, *y, *z;
    uint64_t n, l;
    double k, impart, max2;
    double *data;
    uint64_t *ij;
    uint64_t capacity;
    Workspace ws;
};

__global__ __launch_bounds__(RPX_BLOCK) void k_interaction(InteractionArgs P) {
    __shared__ uint32_t lds_wave[RPX_BLOCK / 64];
    __shared__ uint32_t lds_tile;
    __shared__ uint64_t lds_excl;
    if (threadIdx.x == 0) lds_tile = atomicAdd(&P.ws.ctl->tile_counter, 1u);
    __syncthreads();
    const uint32_t tile = lds_tile;
    const uint64_t total = P.n * P.l;
    const uint64_t t = (uint64_t)tile * RPX_BLOCK + threadIdx.x;
    bool sel = false;
    uint64_t i = 0, j = 0;
    V3 pt = v3(0, 0, 0);
    if (t < total) {
        i = t / P.l;
        j = t - i * P.l;
        pt = sub(v3(P.tx[j], P.ty[j], 0.0), v3(P.rx[i], P.ry[i], 0.0));
        sel = ((pt.x * pt.x) + (pt.y * pt.y)) <= P.max2;
    }
    Cx U = cx(0, 0);
    if (sel) {
        const Cx A = cx(P.A[i], P.impart), B = cx(P.B[i], 0.0), C = cx(P.C[i], P.impart);
        const Cx detG0 = cmul(A, C);
        const V3 a = v3(P.x[3 * i], P.x[3 * i + 1], P.x[3 * i + 2]);
        const V3 b = v3(P.y[3 * i], P.y[3 * i + 1], P.y[3 * i + 2]);
        const V3 c = v3(P.z[3 * i], P.z[3 * i + 1], P.z[3 * i + 2]);
        U = calc_mode_u(A, B, C, detG0, pt, a, b, c, cx(P.k, 0.0), 0.0, 1.0);
    }
    uint32_t block_total;
    const uint32_t local = block_scan_small(sel ? 1u : 0u, lds_wave, &block_total);
    if (threadIdx.x < 64) {
        const uint64_t excl = lookback(P.ws.tile_status, tile, 0, block_total, &P.ws.ctl->error);
        if (threadIdx.x == 0) lds_excl = excl;
    }
    __syncthreads();
    const uint64_t pos = lds_excl + local;
    if (sel && pos < P.capacity) {
        P.data[2 * pos] = U.re;
        P.data[2 * pos + 1] = U.im;
        P.ij[pos] = i;
        P.ij[P.capacity + pos] = j;
    }
    if (threadIdx.x == 0 && (uint64_t)tile == (total - 1) / RPX_BLOCK) P.ws.ctl->children = lds_excl + block_total;
}

extern "C" rpx_status_t rpx_build_interaction_matrix(const double *rx, const double *ry, uint64_t n,
                                                     const double *tx, const double *ty, uint64_t l,
                                                     const double *A, const double *B, const double *C,
                                                     const double *x, const double *y, const double *z,
                                                     double wavelength, double spacing, double max_spacing,
                                                     double blending, double *data, uint64_t *ij,
                                                     uint64_t capacity, uint64_t *n_out, void *workspace,
                                                     uint64_t workspace_bytes, void *stream_) {
    if (!n_out) return rpx_set_error(RPX_E_INVALID, "n_out is null");
    *n_out = 0;
    const uint64_t total = n * l;
    if (total == 0) return RPX_OK;
    if (l != 0 && total / l != n) return rpx_set_error(RPX_E_UNSUPPORTED, "n * l overflows");
    if (total > 0xFFFFFF00ull) return rpx_set_error(RPX_E_UNSUPPORTED, "more than 2^32-256 mode / point pairs");
    if (!rx || !ry || !tx || !ty || !A || !B || !C || !x || !y || !z)
        return rpx_set_error(RPX_E_INVALID, "interaction matrix inputs");
    if (capacity > 0 && (!data || !ij)) return rpx_set_error(RPX_E_INVALID, "interaction matrix outputs");
    if (!workspace || workspace_bytes < rpx_trace_workspace_bytes(total))
        return rpx_set_error(RPX_E_INVALID, "workspace too small");
    hipStream_t stream = (hipStream_t)stream_;
    InteractionArgs P;
    P.rx = rx; P.ry = ry; P.tx = tx; P.ty = ty; P.A = A; P.B = B; P.C = C; P.x = x; P.y = y; P.z = z;
    P.n = n;
    P.l = l;
    P.k = 2000.0 * M_PI / wavelength;
    P.impart = 2 * (blending * blending) / (P.k * spacing * spacing);
    P.max2 = max_spacing * max_spacing;
    P.data = data;
    P.ij = ij;
    P.capacity = capacity;
    P.ws = carve(workspace, total);
    const uint64_t nb = (total + RPX_BLOCK - 1) / RPX_BLOCK;
    hipLaunchKernelGGL(k_clear, dim3((unsigned)((std::max<uint64_t>(nb, RPX_SHARDS * RPX_LDS_FACES) + 255) / 256)),
                       dim3(256), 0, stream, P.ws.tile_status, nb, P.ws.ctl);
    RPX_HIP_TRY(hipGetLastError());
    hipLaunchKernelGGL(k_interaction, dim3((unsigned)nb), dim3(RPX_BLOCK), 0, stream, P);
    RPX_HIP_TRY(hipGetLastError());
    return finish_compaction(P.ws, capacity, n_out, stream, "interaction matrix");
}

// ------------------------------------------------------------ field sum
// calc_mode_U (cfields.pyx:118-151) of one gausslet at one point, in its frame
// (x, y, z) = ((p - O).E, (p - O).H, (p - O).d):
//   w   = (1 + z A)(1 + z C) - (z B)^2        (= 1 + z (A + C) + z^2 detG0),
//   arg = phase + kz (z + N / (2 w)),  N = (A + z detG0) x^2 + 2 B x y + (C + z detG0) y^2,
//   U   = exp(i arg) / sqrt(i w) * inv_root_area sqrt(i),  field += U (E1 E + E2 H).
// The reference's `denom` is 2 w, so one w (in the product form, which does
// not cancel near a focus) and one 1/|w| serve both the quadratic phase and
// the root.  With h = |w|, i w = a + i b, M = |a| + h:
//   sqrt(i w) = (t, q) or, for a < 0, (|q|, copysign(t, b)),
//   t = M g, q = b g, g = 1 / sqrt(2 M), and 1 / sqrt(i w) = conj(sqrt) / h.
//
// Per-gausslet invariants: one record of RPX_GP doubles (288 B).  The pair
// kernels read records through the constant address space: the gausslet is
// the same in every lane, so a record arrives by scalar loads in SGPRs, which
// the vector instructions read directly -- no LDS staging, no barriers, and
// no vector register or issue slot per invariant.  kz / 2 is folded into
// the coefficients of N, sqrt(1/2) and inv_root_area sqrt(i) into
// V = (E1 E + E2 H), and the constant phase is reduced modulo 2 pi.
#define RPX_GP 36
// float64 record (35 of RPX_GP): the shared part, then A C B^2 | kz/2 times A 2B C detG0 | V
enum : int { GP_O = 0, GP_E = 3, GP_H = 6, GP_D = 9, GP_KZ = 12, GP_PHASE = 13, GP_V = 14, GP_KZI = 20, GP_A = 21,
             GP_C = 23, GP_B2 = 25, GP_KA = 27, GP_KB = 29, GP_KC = 31, GP_KD = 33 };
// FP32-split record: the shared part and V in float64 (0..19), then as floats
// from double GP_KZI on: Im kz, A, C, B^2, kz/2 times A 2B C detG0 (15 floats)
enum : int { GF_KZI = 0, GF_A = 1, GF_C = 3, GF_B2 = 5, GF_KA = 7, GF_KB = 9, GF_KC = 11, GF_KD = 13, GF_N = 15 };

template <bool SPLIT>
__global__ __launch_bounds__(256) void k_field_prep(rpx_rays_t r, uint64_t n, const double *modes, WlTable wl,
                                                    double ct, double *gp) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    Ray ray = load_ray(r, i);
    V3 E = norm(ray.E_vector);
    V3 H = norm(cross(ray.direction, E));
    double k = 2000.0 * M_PI / wl[ray.wl_idx];
    double phase = ray.phase + (ray.accum * k) - (ct * k / ray.n.re);
    Cx kz = cmul(ray.n, cx(k, 0.0));
    double invk = 2. / kz.re;
    Cx A = cx(modes[6 * i], modes[6 * i + 1]);
    Cx B = cx(modes[6 * i + 2], modes[6 * i + 3]);
    Cx C = cx(modes[6 * i + 4], modes[6 * i + 5]);
    double ira = sqrt(sqrt(A.im * C.im - (B.im * B.im)) * (2.0 / M_PI));
    A.im *= invk;
    B.im *= invk;
    C.im *= invk;
    const Cx B2 = cmul(B, B);
    const Cx detG0 = csub(cmul(A, C), B2);
    // sqrt(1/2) sqrt(i) = (1 + i) / 2
    const Cx w = cx(0.5 * ira, 0.5 * ira);
    const Cx Vx = cmul(cadd(cmul(ray.E1, cx(E.x, 0)), cmul(ray.E2, cx(H.x, 0))), w);
    const Cx Vy = cmul(cadd(cmul(ray.E1, cx(E.y, 0)), cmul(ray.E2, cx(H.y, 0))), w);
    const Cx Vz = cmul(cadd(cmul(ray.E1, cx(E.z, 0)), cmul(ray.E2, cx(H.z, 0))), w);
    // phase mod 2 pi: 2 pi as a double and its remainder, each step one
    // rounding of a result below 2 pi (phases beyond 2^40 turns, whose own
    // spacing is above 1e-3 rad, stay as they are)
    const double turns = rint(phase * 0.15915494309189535);
    if (fabs(turns) < 1099511627776.0)
        phase = fma(-turns, 2.4492935982947064e-16, fma(-turns, 6.283185307179586, phase));
    const Cx h = cx(0.5 * kz.re, 0.5 * kz.im);
    const Cx KA = cmul(h, A), KB = cmul(kz, B), KC = cmul(h, C), KD = cmul(h, detG0);
    double *o = gp + i * RPX_GP;
    const double v[20] = {ray.origin.x, ray.origin.y, ray.origin.z, E.x, E.y, E.z, H.x, H.y, H.z,
                          ray.direction.x, ray.direction.y, ray.direction.z, kz.re, phase,
                          Vx.re, Vx.im, Vy.re, Vy.im, Vz.re, Vz.im};
    for (int q = 0; q < 20; ++q) o[q] = v[q];
    const double m[15] = {kz.im, A.re, A.im, C.re, C.im, B2.re, B2.im, KA.re, KA.im, KB.re, KB.im, KC.re, KC.im,
                          KD.re, KD.im};
    if constexpr (SPLIT) {
        float *of = (float *)(o + GP_KZI);
        for (int q = 0; q < GF_N; ++q) of[q] = (float)m[q];
    } else {
        for (int q = 0; q < 15; ++q) o[GP_KZI + q] = m[q];
    }
}

#define FS_BLOCK 256
// smallest chunk of gausslets on grid y, and the unit chunks are rounded to
#define FS_TILE 32

typedef __attribute__((address_space(4))) const double GpK;
typedef __attribute__((address_space(4))) const float GpKf;

// sin(j pi / 128), j = 0..64, rounded to float64
static __device__ const double QUARTER_SINE[65] = {
    0.0, 0.024541228522912288, 0.049067674327418015, 0.07356456359966743,
    0.0980171403295606, 0.1224106751992162, 0.14673047445536175, 0.17096188876030122,
    0.19509032201612828, 0.2191012401568698, 0.2429801799032639, 0.26671275747489837,
    0.2902846772544624, 0.31368174039889146, 0.33688985339222005, 0.35989503653498817,
    0.3826834323650898, 0.40524131400498986, 0.4275550934302821, 0.4496113296546066,
    0.47139673682599764, 0.49289819222978404, 0.5141027441932218, 0.5349976198870973,
    0.5555702330196022, 0.5758081914178453, 0.5956993044924334, 0.6152315905806268,
    0.6343932841636455, 0.6531728429537768, 0.6715589548470184, 0.6895405447370669,
    0.7071067811865476, 0.7242470829514669, 0.7409511253549591, 0.7572088465064846,
    0.773010453362737, 0.7883464276266062, 0.8032075314806449, 0.8175848131515837,
    0.8314696123025452, 0.8448535652497071, 0.8577286100002721, 0.8700869911087115,
    0.881921264348355, 0.8932243011955153, 0.9039892931234433, 0.9142097557035307,
    0.9238795325112867, 0.9329927988347388, 0.9415440651830208, 0.9495281805930367,
    0.9569403357322088, 0.9637760657954398, 0.970031253194544, 0.9757021300385286,
    0.9807852804032304, 0.9852776423889412, 0.989176509964781, 0.99247953459871,
    0.9951847266721969, 0.9972904566786902, 0.9987954562051724, 0.9996988186962042,
    1.0};

// Fills one entry per lane of a 256-entry table of (cos, sin)(j pi / 128).
template <class T>
__device__ __forceinline__ void fill_turn_table(T (*tab)[2]) {
    static_assert(FS_BLOCK == 256, "one entry per lane");
    const int j = threadIdx.x & 63, quadrant = (threadIdx.x >> 6) & 3;
    const double s = QUARTER_SINE[j], c = QUARTER_SINE[64 - j];
    const double cq = quadrant == 0 ? c : quadrant == 1 ? -s : quadrant == 2 ? -c : s;
    const double sq = quadrant == 0 ? s : quadrant == 1 ? c : quadrant == 2 ? -s : -c;
    tab[threadIdx.x][0] = (T)cq;
    tab[threadIdx.x][1] = (T)sq;
}

// x = n pi / 128 + r, |r| <= pi / 256: n from the low bits of x (128 / pi) +
// 1.5 2^52 (valid for |x| < 2^45), pi / 128 as a double and its remainder;
// fma forms each n C exactly, so r is good to 2^-59.  Returns r; *n is n mod 2^32.
#define TURN_MAX 35184372088832.0   // 2^45
__device__ __forceinline__ double turn_reduce(double x, uint32_t *n) {
    const double t = fma(x, 40.74366543152521, 6755399441055744.0);
    *n = (uint32_t)__double2loint(t);
    const double nd = t - 6755399441055744.0;
    return fma(-nd, 9.567553118338697e-19, fma(-nd, 0.02454369260617026, x));
}

// A literal held in scalar registers: a Horner step then reads it as the
// addend of v_fma_f64, where a literal held in vector registers costs a copy
// per step (the compiler turns the step into v_fmac_f64, which overwrites it).
__device__ __forceinline__ double in_sgpr(double v) {
    asm("" : "+s"(v));
    return v;
}

// exp(x): x = n ln2 + r, |r| <= ln2 / 2, a degree-11 polynomial (interpolation
// of exp at the Chebyshev nodes of that interval, error below 4e-18) and
// ldexp.  Below -1000 the result is 0; above ldexp's range inf.
struct ExpCheb {
    double c[10];
    __device__ __forceinline__ ExpCheb() {
        c[0] = in_sgpr(0.5000000000000019);
        c[1] = in_sgpr(0.1666666666666668);
        c[2] = in_sgpr(0.04166666666648795);
        c[3] = in_sgpr(0.008333333333319589);
        c[4] = in_sgpr(0.0013888888952352863);
        c[5] = in_sgpr(0.00019841269890076403);
        c[6] = in_sgpr(2.4801485441561313e-05);
        c[7] = in_sgpr(2.755724088722987e-06);
        c[8] = in_sgpr(2.763265472252779e-07);
        c[9] = 2.5110049204818658e-08;
    }
    __device__ __forceinline__ double operator()(double x) const {
        x = fmin(fmax(x, -1000.0), 1000.0);
        const double t = fma(x, 1.4426950408889634, 6755399441055744.0);
        const double nd = t - 6755399441055744.0;
        const double r = fma(-nd, 2.3190468138462996e-17, fma(-nd, 0.6931471805599453, x));
        double p = fma(c[9], r, c[8]);
#pragma unroll
        for (int i = 7; i >= 0; --i) p = fma(p, r, c[i]);
        p = fma(p, r, 1.0);
        p = fma(p, r, 1.0);
        return ldexp(p, __double2loint(t));
    }
};

struct FieldAcc {
    double r0 = 0, i0 = 0, r1 = 0, i1 = 0, r2 = 0, i2 = 0;
    // += (ur + i ui) V, V the record's last factor
    __device__ __forceinline__ void add(double ur, double ui, const GpK *V) {
        r0 = fma(ur, V[0], fma(-ui, V[1], r0));
        i0 = fma(ur, V[1], fma(ui, V[0], i0));
        r1 = fma(ur, V[2], fma(-ui, V[3], r1));
        i1 = fma(ur, V[3], fma(ui, V[2], i1));
        r2 = fma(ur, V[4], fma(-ui, V[5], r2));
        i2 = fma(ur, V[5], fma(ui, V[4], i2));
    }
};

// Sums records g, g + RPX_GP, .. (`n` of them) at p0 in order.  Phases of
// 2^45 rad and above are beyond turn_reduce: the sum without LIBRARY sets
// *large for the lane that met one, and is then taken again with LIBRARY.
template <bool LIBRARY>
__device__ __forceinline__ FieldAcc pair_sum(const GpK *g, uint64_t n, V3 p0, const double (*turn)[2], bool *large) {
    FieldAcc acc;
    const ExpCheb exp_cheb;
    const double s5 = 8.333333333333333e-03, s3 = in_sgpr(-1.6666666666666666e-01);
    const double c6 = -1.388888888888889e-03, c4 = in_sgpr(4.1666666666666664e-02);
    bool big = false;
    for (; n > 0; --n, g += RPX_GP) {
        const double dx = p0.x - g[GP_O], dy = p0.y - g[GP_O + 1], dz = p0.z - g[GP_O + 2];
        const double x = fma(dx, g[GP_E], fma(dy, g[GP_E + 1], dz * g[GP_E + 2]));
        const double y = fma(dx, g[GP_H], fma(dy, g[GP_H + 1], dz * g[GP_H + 2]));
        const double z = fma(dx, g[GP_D], fma(dy, g[GP_D + 1], dz * g[GP_D + 2]));
        const double x2 = x * x, y2 = y * y, xy = x * y, z2 = z * z, zr2 = z * (x2 + y2);
        const double q1r = fma(z, g[GP_A], 1.0), q1i = z * g[GP_A + 1];
        const double q2r = fma(z, g[GP_C], 1.0), q2i = z * g[GP_C + 1];
        const double wr = fma(-z2, g[GP_B2], fma(q1r, q2r, -(q1i * q2i)));
        const double wi = fma(-z2, g[GP_B2 + 1], fma(q1r, q2i, q1i * q2r));
        const double hh = fma(wr, wr, wi * wi);
        const double rh = rsq_third(hh);      // 1 / |w|
        // kz N / 2, then times conj(w) / |w|^2
        const double nr = fma(zr2, g[GP_KD], fma(x2, g[GP_KA], fma(xy, g[GP_KB], y2 * g[GP_KC])));
        const double ni = fma(zr2, g[GP_KD + 1], fma(x2, g[GP_KA + 1], fma(xy, g[GP_KB + 1], y2 * g[GP_KC + 1])));
        const double s = rh * rh;
        const double ar = fma(s, fma(nr, wr, ni * wi), fma(z, g[GP_KZ], g[GP_PHASE]));
        const double ai = fma(s, fma(ni, wr, -(nr * wi)), z * g[GP_KZI]);
        double sn, cs;
        if constexpr (LIBRARY) {
            sincos(ar, &sn, &cs);
        } else {
            big = big || fabs(ar) >= TURN_MAX;
            uint32_t k;
            const double r = turn_reduce(ar, &k);
            const double ct = turn[k & 255][0], st = turn[k & 255][1];
            // sin r and cos r - 1 to r^5 and r^6 (truncation below 1e-17)
            const double u = r * r;
            const double sr = fma(r * u, fma(u, s5, s3), r);
            const double cm = u * fma(u, fma(u, c6, c4), -0.5);
            cs = fma(-st, sr, fma(ct, cm, ct));
            sn = fma(ct, sr, fma(st, cm, st));
        }
        const double mag = exp_cheb(-ai) * rh;
        // i w = (-wi, wr)
        const double m = fma(hh, rh, fabs(wi));
        const double gg = rsq_third(m) * mag;
        const double t = m * gg, q = wr * gg;
        const double sqr = wi <= 0.0 ? t : fabs(q), sqi = wi <= 0.0 ? q : copysign(t, wr);
        acc.add(fma(cs, sqr, sn * sqi), fma(sn, sqr, -(cs * sqi)), g + GP_V);
    }
    *large = big;
    return acc;
}

__device__ __forceinline__ void store_field(double *out, const FieldAcc &a) {
    out[0] = a.r0; out[1] = a.i0;
    out[2] = a.r1; out[3] = a.i1;
    out[4] = a.r2; out[5] = a.i2;
}

// The float64 pair sum.  Block (x, y): points x*FS_BLOCK.., gausslets
// [y*chunk, min(G, (y+1)*chunk)), summed in gausslet order into out + y*6*M;
// one point per lane.  Bound by VALU issue: 124 vector instructions per pair
// (220 before, when the quotients by `denom` and the root had a complex |.|^2
// and a reciprocal each, sin and cos were degree-15/16 series on pi/4, and 31
// invariants were read from LDS).  262,144 gausslets x 65,536 points on
// MI355X: 113.4 -> 66.2 ms per call; 30,000 x 300 points: 339 -> 191 us.
// Six waves per SIMD: the loop fits 80 registers; the rare library loop
// spills.
__global__ __launch_bounds__(FS_BLOCK) __attribute__((amdgpu_waves_per_eu(6)))
void k_field_sum(const double *gp, uint64_t G, uint64_t chunk, const double *points, uint64_t M, double *out) {
    __shared__ double turn[256][2];
    fill_turn_table(turn);
    __syncthreads();
    const uint64_t ip = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const uint64_t g0 = (uint64_t)blockIdx.y * chunk, g1 = min(G, g0 + chunk);
    if (ip >= M) return;
    const V3 p0 = v3(points[3 * ip], points[3 * ip + 1], points[3 * ip + 2]);
    const GpK *g = (const GpK *)(gp + g0 * RPX_GP);
    bool large = false;
    FieldAcc acc = pair_sum<false>(g, g1 - g0, p0, turn, &large);
    if (large) acc = pair_sum<true>(g, g1 - g0, p0, turn, &large);
    store_field(out + (uint64_t)blockIdx.y * 6 * M + 6 * ip, acc);
}

// The FP32-split pair: the same term with float32 amplitude arithmetic.
// In float64: the local coordinates (x, y, z) (|p - O| is tens of mm), the
// phase phi + Re(kz) z + the quadratic phase and its reduction to |r| <= pi /
// 256, and the accumulation U V.  In float32: w, N (whose phase is tens of
// rad), the sine and cosine of r, the exponential and 1/sqrt(i w).  U goes to
// float64 before the product with V (14 instructions, where six float32
// products converted and added one by one took 24).  111 vector instructions
// per pair (167 before); 262,144 gausslets x 16,384 points on MI355X: 14.3 ->
// 10.4 ms per call.
template <bool LIBRARY>
__device__ __forceinline__ FieldAcc pair_sum_split(const GpK *g, uint64_t n, V3 p0, const float (*turn)[2],
                                                   bool *large) {
    FieldAcc acc;
    bool big = false;
    for (; n > 0; --n, g += RPX_GP) {
        const GpKf *f = (const GpKf *)(g + GP_KZI);
        const double dx = p0.x - g[GP_O], dy = p0.y - g[GP_O + 1], dz = p0.z - g[GP_O + 2];
        const double xd = fma(dx, g[GP_E], fma(dy, g[GP_E + 1], dz * g[GP_E + 2]));
        const double yd = fma(dx, g[GP_H], fma(dy, g[GP_H + 1], dz * g[GP_H + 2]));
        const double zd = fma(dx, g[GP_D], fma(dy, g[GP_D + 1], dz * g[GP_D + 2]));
        const float x = (float)xd, y = (float)yd, z = (float)zd;
        const float x2 = x * x, y2 = y * y, xy = x * y, z2 = z * z, zr2 = z * (x2 + y2);
        const float q1r = fmaf(z, f[GF_A], 1.0f), q1i = z * f[GF_A + 1];
        const float q2r = fmaf(z, f[GF_C], 1.0f), q2i = z * f[GF_C + 1];
        const float wr = fmaf(-z2, f[GF_B2], fmaf(q1r, q2r, -(q1i * q2i)));
        const float wi = fmaf(-z2, f[GF_B2 + 1], fmaf(q1r, q2i, q1i * q2r));
        const float hh = fmaf(wr, wr, wi * wi);
        const float rh = __builtin_amdgcn_rsqf(hh);
        const float nr = fmaf(zr2, f[GF_KD], fmaf(x2, f[GF_KA], fmaf(xy, f[GF_KB], y2 * f[GF_KC])));
        const float ni = fmaf(zr2, f[GF_KD + 1], fmaf(x2, f[GF_KA + 1], fmaf(xy, f[GF_KB + 1], y2 * f[GF_KC + 1])));
        const float s = rh * rh;
        const double ar = fma(zd, g[GP_KZ], g[GP_PHASE]) + (double)(s * fmaf(nr, wr, ni * wi));
        const float ai = fmaf(s, fmaf(ni, wr, -(nr * wi)), z * f[GF_KZI]);
        float sn, cs;
        if constexpr (LIBRARY) {
            double sd, cd;
            sincos(ar, &sd, &cd);
            sn = (float)sd;
            cs = (float)cd;
        } else {
            big = big || fabs(ar) >= TURN_MAX;
            uint32_t k;
            const float r = (float)turn_reduce(ar, &k);
            const float ct = turn[k & 255][0], st = turn[k & 255][1];
            // sin r to r^3, cos r - 1 to r^2 (truncation below 1e-9)
            const float u = r * r;
            const float sr = fmaf(r * u, -1.6666667163372040e-01f, r);
            const float cm = -0.5f * u;
            cs = fmaf(-st, sr, fmaf(ct, cm, ct));
            sn = fmaf(ct, sr, fmaf(st, cm, st));
        }
        const float mag = expf(-ai) * rh;
        const float m = fmaf(hh, rh, fabsf(wi));
        const float gg = __builtin_amdgcn_rsqf(m) * mag;
        const float t = m * gg, q = wr * gg;
        const float sqr = wi <= 0.0f ? t : fabsf(q), sqi = wi <= 0.0f ? q : copysignf(t, wr);
        acc.add((double)fmaf(cs, sqr, sn * sqi), (double)fmaf(sn, sqr, -(cs * sqi)), g + GP_V);
    }
    *large = big;
    return acc;
}

__global__ __launch_bounds__(FS_BLOCK) __attribute__((amdgpu_waves_per_eu(8)))
void k_field_sum_split(const double *gp, uint64_t G, uint64_t chunk, const double *points, uint64_t M, double *out) {
    __shared__ float turn[256][2];
    fill_turn_table(turn);
    __syncthreads();
    const uint64_t ip = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const uint64_t g0 = (uint64_t)blockIdx.y * chunk, g1 = min(G, g0 + chunk);
    if (ip >= M) return;
    const V3 p0 = v3(points[3 * ip], points[3 * ip + 1], points[3 * ip + 2]);
    const GpK *g = (const GpK *)(gp + g0 * RPX_GP);
    bool large = false;
    FieldAcc acc = pair_sum_split<false>(g, g1 - g0, p0, turn, &large);
    if (large) acc = pair_sum_split<true>(g, g1 - g0, p0, turn, &large);
    store_field(out + (uint64_t)blockIdx.y * 6 * M + 6 * ip, acc);
}

// out[e] = sum over chunks c of part[c*n + e]: FR_GROUPS lanes per element sum
// every FR_GROUPS-th chunk, then the groups are added in order.  (One lane per
// element is a serial chain of loads: 469 chunks of 1,800 elements took 117 us
// on eight workgroups.)
#define FR_GROUPS 16
__global__ __launch_bounds__(256) void k_field_reduce(const double *part, uint32_t n_chunks, uint64_t n,
                                                      double *out) {
    __shared__ double red[FR_GROUPS][256 / FR_GROUPS];
    constexpr int W = 256 / FR_GROUPS;
    const int col = threadIdx.x % W, group = threadIdx.x / W;
    const uint64_t e = (uint64_t)blockIdx.x * W + col;
    double s = 0;
    if (e < n) {
#pragma unroll 4
        for (uint32_t c = group; c < n_chunks; c += FR_GROUPS) s += part[(uint64_t)c * n + e];
    }
    red[group][col] = s;
    __syncthreads();
    if (group == 0 && e < n) {
        for (int k = 1; k < FR_GROUPS; ++k) s += red[k][col];
        out[e] = s;
    }
}

// Workgroups of FS_BLOCK threads of `kernel` resident at once on the current
// device (occupancy per CU times CUs), cached per kernel and device.
static uint64_t field_resident(const void *kernel) {
    static std::mutex mu;
    static struct { const void *k; int dev; uint64_t n; } cache[8];
    static int n_cache = 0;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) dev = 0;
    {
        std::lock_guard<std::mutex> g(mu);
        for (int i = 0; i < n_cache; ++i)
            if (cache[i].k == kernel && cache[i].dev == dev) return cache[i].n;
    }
    int per_cu = 0, cus = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, FS_BLOCK, 0) != hipSuccess || per_cu < 1) {
        (void)hipGetLastError();
        per_cu = 1;
    }
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1) {
        (void)hipGetLastError();
        cus = 1;
    }
    const uint64_t n = (uint64_t)per_cu * (uint64_t)cus;
    std::lock_guard<std::mutex> g(mu);
    if (n_cache < 8) {
        cache[n_cache].k = kernel;
        cache[n_cache].dev = dev;
        cache[n_cache].n = n;
        ++n_cache;
    }
    return n;
}

// Gausslets per chunk for the 2-D field-sum grid: enough chunks that the grid
// is about four rounds of resident workgroups (fewer point blocks than that
// leave CUs idle, and a grid of 1.3 rounds idles most of them in its second
// round), a whole number of tiles per chunk, and a partial-sum buffer of at
// most 512 MB.
static uint64_t field_chunk(const void *kernel, uint64_t G, uint64_t M, uint64_t tile) {
    const uint64_t pb = (M + FS_BLOCK - 1) / FS_BLOCK;
    const uint64_t tiles = (G + tile - 1) / tile;
    uint64_t c = (4 * field_resident(kernel) + pb - 1) / pb;
    const uint64_t cap = (512ull << 20) / (48 * M);
    c = std::max<uint64_t>(1, std::min(c, std::min<uint64_t>(tiles, std::max<uint64_t>(cap, 1))));
    c = std::min<uint64_t>(c, 65535);
    return ((tiles + c - 1) / c) * tile;
}

static rpx_status_t field_sum_checks(const rpx_rays_t *rays, uint64_t n_rays, const double *modes,
                                     const double *points, uint64_t n_pts, double *out, int32_t precision) {
    if (precision != 0 && precision != 1) return rpx_set_error(RPX_E_INVALID, "precision must be 0 or 1");
    if (n_pts == 0) return RPX_OK;
    if (!points || !out) return rpx_set_error(RPX_E_INVALID, "null point/output buffer");
    if (n_rays == 0) return RPX_OK;
    if (!rays || !rays->f64 || !rays->u32 || rays->capacity < n_rays || !modes)
        return rpx_set_error(RPX_E_INVALID, "ray/mode buffers");
    return RPX_OK;
}

// Gausslet chunks on grid y for this precision (see field_chunk).
static uint64_t field_sum_chunk(uint64_t n_rays, uint64_t n_pts, int32_t precision) {
    const void *kern = precision == 0 ? (const void *)k_field_sum : (const void *)k_field_sum_split;
    return field_chunk(kern, n_rays, n_pts, FS_TILE);
}

// The field-sum launches: invariants into gp (RPX_GP * n_rays doubles), the
// pair kernel over gausslet chunks of `chunk` (partial sums into `part`,
// 6 * n_pts doubles per chunk, when there is more than one chunk), then the
// chunk-ordered reduction into out.  n_rays > 0 and n_pts > 0.
// With `timed`, the pair kernel is bracketed by events whose elapsed time is
// added to its timing slot once the stream has completed.
static hipError_t field_sum_launch(const rpx_rays_t *rays, uint64_t n_rays, const double *modes, WlTable wl,
                                   const double *points, uint64_t n_pts, double time_ps, double *out,
                                   int32_t precision, uint64_t chunk, double *gp, double *part,
                                   hipStream_t stream, bool timed = false) {
    const double ct = 0.299792458 * time_ps;
    hipLaunchKernelGGL((precision == 0 ? k_field_prep<false> : k_field_prep<true>),
                       dim3((unsigned)((n_rays + 255) / 256)), dim3(256), 0, stream, *rays, n_rays, modes, wl, ct, gp);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const uint64_t n_chunks = (n_rays + chunk - 1) / chunk;
    double *dst = n_chunks > 1 ? part : out;
    const dim3 grid((unsigned)((n_pts + FS_BLOCK - 1) / FS_BLOCK), (unsigned)n_chunks);
    hipEvent_t ev[2] = {nullptr, nullptr};
    if (timed && (hipEventCreate(&ev[0]) != hipSuccess || hipEventCreate(&ev[1]) != hipSuccess)) timed = false;
    if (timed) (void)hipEventRecord(ev[0], stream);
    if (precision == 0)
        hipLaunchKernelGGL(k_field_sum, grid, dim3(FS_BLOCK), 0, stream, gp, n_rays, chunk, points, n_pts, dst);
    else
        hipLaunchKernelGGL(k_field_sum_split, grid, dim3(FS_BLOCK), 0, stream, gp, n_rays, chunk, points, n_pts,
                           dst);
    e = hipGetLastError();
    if (timed) {
        float ms = 0;
        if (e == hipSuccess && hipEventRecord(ev[1], stream) == hipSuccess &&
            hipEventSynchronize(ev[1]) == hipSuccess && hipEventElapsedTime(&ms, ev[0], ev[1]) == hipSuccess)
            rpx_timing_add(precision == 0 ? RPX_TIMING_FIELD_SUM : RPX_TIMING_FIELD_SUM_SPLIT, ms,
                           (double)n_rays * (double)n_pts);
        (void)hipEventDestroy(ev[0]);
        (void)hipEventDestroy(ev[1]);
    }
    if (e != hipSuccess || n_chunks == 1) return e;
    const uint64_t per_block = 256 / FR_GROUPS;
    hipLaunchKernelGGL(k_field_reduce, dim3((unsigned)((6 * n_pts + per_block - 1) / per_block)), dim3(256), 0, stream,
                       (const double *)part, (uint32_t)n_chunks, 6 * n_pts, out);
    return hipGetLastError();
}

extern "C" rpx_status_t rpx_sum_gaussian_modes(const rpx_rays_t *rays, uint64_t n_rays, const double *modes,
                                               const double *wavelengths, uint64_t n_wavelengths,
                                               const double *points, uint64_t n_pts, double time_ps, double *out,
                                               int32_t precision, void *stream_) {
    hipStream_t stream = (hipStream_t)stream_;
    if (rpx_status_t st = field_sum_checks(rays, n_rays, modes, points, n_pts, out, precision)) return st;
    if (n_pts == 0) return RPX_OK;
    if (n_rays == 0) {
        RPX_HIP_TRY(hipMemsetAsync(out, 0, sizeof(double) * 6 * n_pts, stream));
        return RPX_OK;
    }
    WlTable wl;
    wl.wl = wavelengths;
    wl.n = wavelengths ? n_wavelengths : 0;
    const uint64_t chunk = field_sum_chunk(n_rays, n_pts, precision);
    const uint64_t n_chunks = (n_rays + chunk - 1) / chunk;
    double *gp = nullptr, *part = nullptr;
    RPX_HIP_TRY(hipMallocAsync((void **)&gp, sizeof(double) * RPX_GP * n_rays, stream));
    hipError_t e = hipSuccess;
    if (n_chunks > 1) e = hipMallocAsync((void **)&part, sizeof(double) * 6 * n_pts * n_chunks, stream);
    if (e == hipSuccess)
        e = field_sum_launch(rays, n_rays, modes, wl, points, n_pts, time_ps, out, precision, chunk, gp, part, stream,
                             rpx_timing_is_on());
    hipError_t e2 = hipFreeAsync(gp, stream);
    if (part) {
        hipError_t e3 = hipFreeAsync(part, stream);
        if (e2 == hipSuccess) e2 = e3;
    }
    if (e != hipSuccess) return rpx_set_error(RPX_E_HIP, std::string("field sum launch: ") + hipGetErrorString(e));
    if (e2 != hipSuccess) return rpx_set_error(RPX_E_HIP, std::string("field sum free: ") + hipGetErrorString(e2));
    return RPX_OK;
}

// --------------------------------------------- field sum without allocation
// rpx_sum_gaussian_modes_noalloc keeps the invariants table and the chunk
// partial sums in this file-scope device array instead of stream-ordered
// allocations.  Each device holds its own copy until the process ends; host
// code uses the per-device address from hipGetSymbolAddress, never the
// array's name (which is a host-side stand-in).
static __device__ __align__(256) double scratch[RPX_FIELD_SCRATCH_BYTES / sizeof(double)];

#define RPX_MAX_DEVICES 64

// Device address of `scratch` on the current device, looked up once per
// device; nullptr (with the error recorded) if the lookup fails.
static double *field_scratch(rpx_status_t *st) {
    static std::mutex mu;
    static double *ptrs[RPX_MAX_DEVICES] = {};
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) {
        *st = rpx_set_error(RPX_E_HIP, std::string("hipGetDevice: ") + hipGetErrorString(e));
        return nullptr;
    }
    if (dev < 0 || dev >= RPX_MAX_DEVICES) {
        *st = rpx_set_error(RPX_E_INVALID, "device ordinal beyond the no-alloc scratch table");
        return nullptr;
    }
    std::lock_guard<std::mutex> g(mu);
    if (!ptrs[dev]) {
        void *p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            *st = rpx_set_error(RPX_E_HIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
            return nullptr;
        }
        ptrs[dev] = (double *)p;
    }
    return ptrs[dev];
}

// out[i] = 0 for i < n (a kernel rather than a memset node, so that the call
// can be captured into a graph).
__global__ void k_fill_zero(double *out, uint64_t n) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = 0.0;
}

extern "C" uint64_t rpx_field_noalloc_max_rays(void) {
    return RPX_FIELD_SCRATCH_BYTES / (sizeof(double) * RPX_GP);
}

extern "C" rpx_status_t rpx_sum_gaussian_modes_noalloc(const rpx_rays_t *rays, uint64_t n_rays, const double *modes,
                                                       const double *wavelengths, uint64_t n_wavelengths,
                                                       const double *points, uint64_t n_pts, double time_ps,
                                                       double *out, int32_t precision, void *stream_) {
    hipStream_t stream = (hipStream_t)stream_;
    if (rpx_status_t st = field_sum_checks(rays, n_rays, modes, points, n_pts, out, precision)) return st;
    if (n_pts == 0) return RPX_OK;
    if (n_rays > rpx_field_noalloc_max_rays())
        return rpx_set_error(RPX_E_CAPACITY, "rpx_sum_gaussian_modes_noalloc: " + std::to_string(n_rays) +
                                                 " gausslets exceed the scratch limit of " +
                                                 std::to_string(rpx_field_noalloc_max_rays()));
    rpx_status_t st = RPX_OK;
    double *base = field_scratch(&st);
    if (!base) return st;
    if (n_rays == 0) {
        hipLaunchKernelGGL(k_fill_zero, dim3((unsigned)((6 * n_pts + 255) / 256)), dim3(256), 0, stream, out,
                           6 * n_pts);
        RPX_HIP_TRY(hipGetLastError());
        return RPX_OK;
    }
    WlTable wl;
    wl.wl = wavelengths;
    wl.n = wavelengths ? n_wavelengths : 0;
    // the invariants table first, the partial sums after it; the chunk count
    // of the allocating entry point when its partial sums fit (then the two
    // entry points sum in the same order), else as many chunks as fit, else
    // one chunk summed straight into out
    const uint64_t gp_doubles = ((RPX_GP * n_rays + 31) / 32) * 32;
    const uint64_t left = RPX_FIELD_SCRATCH_BYTES / sizeof(double) - gp_doubles;
    const uint64_t tile = FS_TILE;
    uint64_t chunk = field_sum_chunk(n_rays, n_pts, precision);
    uint64_t n_chunks = (n_rays + chunk - 1) / chunk;
    if (n_chunks > 1 && 6 * n_pts * n_chunks > left) {
        const uint64_t fit = left / (6 * n_pts);
        const uint64_t tiles = (n_rays + tile - 1) / tile;
        chunk = fit < 2 ? n_rays : ((tiles + fit - 1) / fit) * tile;
        n_chunks = (n_rays + chunk - 1) / chunk;
    }
    double *part = n_chunks > 1 ? base + gp_doubles : nullptr;
    hipError_t e =
        field_sum_launch(rays, n_rays, modes, wl, points, n_pts, time_ps, out, precision, chunk, base, part, stream);
    if (e != hipSuccess) return rpx_set_error(RPX_E_HIP, std::string("field sum launch: ") + hipGetErrorString(e));
    return RPX_OK;
}
