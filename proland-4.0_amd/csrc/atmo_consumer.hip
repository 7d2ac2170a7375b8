// atmo_consumer.hip — the table consumer on gfx950: skyRadiance, inScattering,
// sunRadiance and skyIrradiance of src/atmo/examples/atmo/atmosphereShader.glsl
// evaluated on the .raw-layout tables (RGB T and E, RGBA S) with GL LINEAR +
// CLAMP_TO_EDGE filtering.  One thread per ray / point / (r, muS) pair.
//
// Precision follows the preprocess kernels: ray geometry (camera radius, r mu,
// the top-sphere and ground discriminants, the texture4D coordinates) in FP64,
// filtering, phase functions and the radiance combination in FP32.
//
// Every shader constant comes from atmo_params instead of the shader's
// hard-coded Earth (atmosphereShader.glsl:72-125); lengths are in the
// parameters' unit, and the 600 m near-ground offset of inScattering (:472)
// is 600 / meters_per_unit.  Where the shader (built with OPTIMIZE) takes
// sqrt of a negative number for a ray that misses the atmosphere from
// outside, max(NaN, 0) evaluates to 0 on GPUs, so din = 0 here.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdio>

#include "../../include/atmo_consumer.h"
#include "atmo_device.h"

namespace atmo {
atmo_status set_error(atmo_status st, const char *msg);
}

namespace atmo {
namespace {

struct CDesc {
    double Rg, Rt, H, near;       // H = sqrt(Rt^2 - Rg^2); near = Rg + 600 m
    double cam[3], sun[3], shaft;
    float bR[3];
    float kR, kM, g2p1, m2g;      // phase-function constants
    float f_tMu;                  // tan(1.5) / 1.15
    float f_inv_dRt;              // 1 / (Rt - Rg)
    int TW, TH, SW, SH, RR, RMU, RMUS, RNU, W4;
    const float *T, *S, *E;
    // What every ray of a camera inside the atmosphere without light shafts shares
    // (host): the camera's radius and sun, their column, layer and T row
    double cm[3], r, invr, rho, rho2, invrH, H2, muS, lim;
    int i0, k0, k1, tj0, tj1;
    float ia, kg, tb;
    double near_f;   // the radius that :472 gives a camera below `near`, over its own
    int inside;
};

constexpr float kSunIntensity = 100.0f;  // atmosphereShader.glsl:66

typedef __attribute__((address_space(1))) const float gfloat;

// bilinear RGB fetch from a [H][W][3] table at texel coordinates (x, y)
__device__ __forceinline__ float3 rgb_bilinear(const float *tab, int W, int H, float x, float y) {
    int i0, i1, j0, j1;
    float a, b;
    gl_axis(x, W, i0, i1, a);
    gl_axis(y, H, j0, j1, b);
    const gfloat *t = (const gfloat *)tab;
    auto at = [&](int j, int i) {
        const gfloat *q = t + ((size_t)j * W + i) * 3;
        return make_float3(q[0], q[1], q[2]);
    };
    return lerp3(lerp3(at(j0, i0), at(j0, i1), a), lerp3(at(j1, i0), at(j1, i1), a), b);
}

// getTransmittanceUV + transmittance(r, mu) (atmosphereShader.glsl:141-151, 232-235)
__device__ __forceinline__ float3 T_at(const CDesc &d, double r, double mu) {
    const float uR = sqrtf((float)fmax(r - d.Rg, 0.0) * d.f_inv_dRt);
    const float uMu = atanf(((float)mu + 0.15f) * d.f_tMu) * (1.0f / 1.5f);
    return rgb_bilinear(d.T, d.TW, d.TH, uMu * d.TW - 0.5f, uR * d.TH - 0.5f);
}

// 1/x in FP64 from the hardware estimate (4.5e-8) and Newton steps: 1.11e-16 relative over
// 1e-6 .. 3e7, as a division.  NaN at 0 and infinity: a point without a direction, which
// is NaN in any case (0 / 0), or at the planet's centre, likewise.
__device__ __forceinline__ double rcp64(double x) {
    double y = __builtin_amdgcn_rcp(x);
    y = fma(y, fma(-x, y, 1.0), y);
    return fma(y, fma(-x, y, 1.0), y);
}

// texture4D's mu axis (atmosphereShader.glsl:175-199, INSCATTER_NON_LINEAR) as a texel
// coordinate; the ground branch in the cancellation-free form -rho / (sqrt(delta) - r mu).
// (A root's argument is cut at 1e-280, whose root is 0 to a coordinate.)
__device__ __forceinline__ double mu_coord(const CDesc &d, double rmu, double rho, double rho2, double invrH) {
    const double delta = rmu * rmu - rho2, hr = 0.5 * d.RMU - 1.0;
    if (rmu < 0.0 && delta > 0.0) return hr - hr * (rho * rcp64(sqrt64_pos(delta) - rmu));
    return fma((sqrt64_pos(fmax(delta + d.H2, 1e-280)) - rmu) * invrH, hr, 0.5 * d.RMU);
}
// Its mu_s axis as a texel coordinate inside a slice: the FP64 arctangent in every lane, so
// that a ray's value does not depend on the rays beside it (an FP32 polynomial from the
// camera's sun, in waves whose lanes were all near it, took 37.9 us for 1280 x 720 points, this 35.4)
__device__ __forceinline__ double mus_coord(const CDesc &d, double muS) {
    const double x = fmax(muS, -0.1975) * tan(1.26 * 1.1);
    return fma(atan(x), 1.0 / 1.1, 1.0 - 0.26) * (0.5 * (d.RMUS - 1.0));
}
// The nu slices: slice and fraction of the shader's lerp.  Beyond -1 and RNU both slices
// clamp to the table's edge.
__device__ __forceinline__ int nu_coord(const CDesc &d, double nu, float &w) {
    const double t = fmin(fmax((nu + 1.0) * 0.5 * (d.RNU - 1.0), -1.0), (double)d.RNU), f = floor(t);
    w = (float)(t - f);
    return (int)f;
}
__device__ __forceinline__ float4 lerp4(float4 u, float4 v, float w) {
    return make_float4(fmaf(w, v.x - u.x, u.x), fmaf(w, v.y - u.y, u.y), fmaf(w, v.z - u.z, u.z), fmaf(w, v.w - u.w, u.w));
}

// texture4D: the two trilinear fetches share all but the slice
__device__ __forceinline__ float4 texture4D(const CDesc &d, double r, double mu, double muS, double nu) {
    const double rho2 = r * r - d.Rg * d.Rg, rho = sqrt64_pos(fmax(rho2, 1e-280));
    int j0, j1, k0, k1;
    float b, g, w;
    gl_axis_d(mu_coord(d, r * mu, rho, rho2, rcp64(rho + d.H)), d.RMU, j0, j1, b);
    gl_axis_d(rho * ((d.RR - 1.0) / d.H), d.RR, k0, k1, g);
    const double xs = mus_coord(d, muS), fx = floor(xs);
    const float a = (float)(xs - fx);
    const int i0 = nu_coord(d, nu, w) * d.RMUS + (int)fx, last = d.W4 - 1;
    const int x0 = min(max(i0, 0), last), x1 = min(max(i0 + 1, 0), last), x2 = min(max(i0 + d.RMUS, 0), last),
              x3 = min(max(i0 + d.RMUS + 1, 0), last);
    const gfloat *t = (const gfloat *)d.S;
    auto row = [&](int k, int j) {   // both slices of one row
        const gfloat *q = t + ((size_t)k * d.RMU + j) * d.W4 * 4;
        auto at = [&](int x) { return make_float4(q[4 * x], q[4 * x + 1], q[4 * x + 2], q[4 * x + 3]); };
        return lerp4(lerp4(at(x0), at(x1), a), lerp4(at(x2), at(x3), a), w);
    };
    return lerp4(lerp4(row(k0, j0), row(k0, j1), b), lerp4(row(k1, j0), row(k1, j1), b), g);
}

// The tables as a camera inside the atmosphere sees them: r and mu_s are the same for
// every ray, so S blends to [RMU][RNU + 3] (slices -1 to RNU + 1, each column clamped as the
// fetch clamps it) and T to one row of columns.  STAGED: once per workgroup in LDS, where a
// lookup reads 4 and 2 entries instead of 16 texels and 4; otherwise a lookup blends the
// entries it needs itself, with the same bits.
template <bool STAGED>
struct ViewTables {
    const float4 *S, *T;
    int stride;   // RNU + 3
};
__host__ __device__ __forceinline__ size_t view_entries(const CDesc &d) {
    return (size_t)(d.RMU + 1) * (d.RNU + 3) + d.TW + 1;
}
typedef __attribute__((address_space(1))) const char gchar;
// (a layer of S, at most 2^27 texels of 16 bytes, and the rows of T: scalar bases and 32-bit
// byte offsets)
__device__ __forceinline__ float4 view_entry_S(const CDesc &d, int j, int slice) {   // mu row j
    const size_t layer = (size_t)d.RMU * d.W4 * 16;
    const gchar *t0 = (const gchar *)d.S + d.k0 * layer, *t1 = (const gchar *)d.S + d.k1 * layer;
    const int i = slice * d.RMUS + d.i0, last = d.W4 - 1;
    const unsigned x0 = (unsigned)(j * d.W4 + min(max(i, 0), last)) * 16u, x1 = (unsigned)(j * d.W4 + min(max(i + 1, 0), last)) * 16u;
    auto at = [](const gchar *t, unsigned x) {
        const gfloat *q = (const gfloat *)(t + x);
        return make_float4(q[0], q[1], q[2], q[3]);
    };
    return lerp4(lerp4(at(t0, x0), at(t0, x1), d.ia), lerp4(at(t1, x0), at(t1, x1), d.ia), d.kg);
}
__device__ __forceinline__ float3 view_entry_T(const CDesc &d, int x) {
    const gchar *t = (const gchar *)d.T;
    const unsigned o = (unsigned)min(x, d.TW - 1) * 12u;
    const gfloat *p = (const gfloat *)(t + (size_t)d.tj0 * d.TW * 12 + o), *q = (const gfloat *)(t + (size_t)d.tj1 * d.TW * 12 + o);
    return lerp3(make_float3(p[0], p[1], p[2]), make_float3(q[0], q[1], q[2]), d.tb);
}
template <bool STAGED>
__device__ __forceinline__ ViewTables<STAGED> stage_view(const CDesc &d, float4 *lds) {
    if (!STAGED) return {nullptr, nullptr, 0};
    const int stride = d.RNU + 3, nS = d.RMU * stride;
    float4 *T = lds + (d.RMU + 1) * stride;
    for (int e = threadIdx.x; e < nS + stride; e += blockDim.x)
        // below the last row, where the fraction is 0: nothing
        lds[e] = e < nS ? view_entry_S(d, e / stride, e % stride - 1) : make_float4(0.f, 0.f, 0.f, 0.f);
    for (int x = threadIdx.x; x <= d.TW; x += blockDim.x) {
        const float3 v = view_entry_T(d, x);
        T[x] = make_float4(v.x, v.y, v.z, 0.f);
    }
    __syncthreads();
    return {lds, T, stride};
}
// texture4D at the camera's r and sun
template <bool STAGED>
__device__ __forceinline__ float4 view_S(const CDesc &d, const ViewTables<STAGED> &v, double rmu, int e, float w) {
    const double y = fmin(fmax(mu_coord(d, rmu, d.rho, d.rho2, d.invrH), 0.0), d.RMU - 1.0), fy = floor(y);
    const float b = (float)(y - fy);
    if constexpr (STAGED) {
        const float4 *p = v.S + (int)fy * v.stride + e + 1, *q = p + v.stride;
        return lerp4(lerp4(p[0], p[1], w), lerp4(q[0], q[1], w), b);
    } else {
        const int j0 = (int)fy, j1 = min(j0 + 1, d.RMU - 1);
        return lerp4(lerp4(view_entry_S(d, j0, e), view_entry_S(d, j0, e + 1), w),
                     lerp4(view_entry_S(d, j1, e), view_entry_S(d, j1, e + 1), w), b);
    }
}
// T at the camera's r
template <bool STAGED>
__device__ __forceinline__ float3 view_T(const CDesc &d, const ViewTables<STAGED> &v, double mu) {
    const float uMu = atanf(((float)mu + 0.15f) * d.f_tMu) * (1.0f / 1.5f);
    const float x = __builtin_amdgcn_fmed3f(uMu * d.TW - 0.5f, 0.0f, (float)(d.TW - 1)), f = floorf(x);
    if constexpr (STAGED) {
        const float4 *p = v.T + (int)f;
        return lerp3(f3(p[0]), f3(p[1]), x - f);
    } else {
        return lerp3(view_entry_T(d, (int)f), view_entry_T(d, (int)f + 1), x - f);
    }
}

__host__ __device__ __forceinline__ double dot3(const double *a, const double *b) {
    return a[0] * b[0] + a[1] * b[1] + a[2] * b[2];
}

// rgb of inScatter * phaseR(nu) + getMie(inScatter) * phaseM(nu), times SUN_INTENSITY
// (:300-302 getMie, :290-297 phases)
__device__ __forceinline__ float4 combine(const CDesc &d, float4 is, double nu) {
    const float n = (float)nu;
    const float pr = d.kR * fmaf(n, n, 1.0f);
    const float y = rsqrtf(fmaf(d.m2g, n, d.g2p1));
    const float pm = d.kM * fmaf(n, n, 1.0f) * (y * y * y);
    const float k = is.w / fmaxf(is.x, 1e-4f);
    const float m0 = is.x * k, m1 = is.y * k * (d.bR[0] / d.bR[1]), m2 = is.z * k * (d.bR[0] / d.bR[2]);
    return make_float4(fmaf(is.x, pr, m0 * pm) * kSunIntensity, fmaf(is.y, pr, m1 * pm) * kSunIntensity,
                       fmaf(is.z, pr, m2 * pm) * kSunIntensity, 0.f);
}

// transmittance between points A and B of a ray, as the shaders write it:
// up ? T(A)/T(B) : T(B reversed)/T(A reversed), clamped to 1
__device__ __forceinline__ float3 T_ratio(const CDesc &d, double ra, double mua, double rb, double mub,
                                         bool up) {
    float3 a, b;
    if (up) {
        a = T_at(d, ra, mua);
        b = T_at(d, rb, mub);
    } else {
        a = T_at(d, rb, -mub);
        b = T_at(d, ra, -mua);
    }
    return make_float3(fminf(a.x / b.x, 1.f), fminf(a.y / b.y, 1.f), fminf(a.z / b.z, 1.f));
}

// skyRadiance, atmosphereShader.glsl:371-418
__global__ __launch_bounds__(256) void k_sky_radiance(CDesc d, const float4 *__restrict__ dirs, int n,
                                                      float4 *__restrict__ rad, float4 *__restrict__ ext) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float4 v4 = dirs[i];
    const double v[3] = {v4.x, v4.y, v4.z};
    double cam[3];
    for (int c = 0; c < 3; ++c) cam[c] = d.cam[c] + v[c] * fmax(d.shaft, 0.0);
    double r = sqrt(dot3(cam, cam));
    double rMu = dot3(cam, v);
    double mu = rMu / r;
    const double r0 = r, mu0 = mu;
    const double q = rMu * rMu - r * r + d.Rt * d.Rt;
    const double din = q >= 0.0 ? fmax(-rMu - sqrt(q), 0.0) : 0.0;
    if (din > 0.0) {
        for (int c = 0; c < 3; ++c) cam[c] += din * v[c];
        rMu += din;
        mu = rMu / d.Rt;
        r = d.Rt;
    }
    float4 out = make_float4(0.f, 0.f, 0.f, 0.f), ex = make_float4(1.f, 1.f, 1.f, 0.f);
    if (r <= d.Rt) {
        const double nu = dot3(v, d.sun);
        const double muS = dot3(cam, d.sun) / r;
        float4 is = texture4D(d, r, rMu / r, muS, nu);
        if (d.shaft > 0.0) {
            const float3 f = T_ratio(d, r0, mu0, r, mu, mu > 0.0);
            is = make_float4(is.x * f.x, is.y * f.y, is.z * f.z, is.w * f.x);
        }
        const float3 e = T_at(d, r, mu);
        ex = make_float4(e.x, e.y, e.z, 0.f);
        out = combine(d, is, nu);
    }
    rad[i] = out;
    if (ext) ext[i] = ex;
}

// skyRadiance from inside the atmosphere without light shafts: no ray enters from
// outside (din = 0).  STAGED: workgroups stage the view's tables once and walk the rays.
// 1920 x 1080 rays on the 32x128x32x8 tables: 45 -> 22 us.
template <bool STAGED>
__global__ __launch_bounds__(STAGED ? 512 : 256) void k_sky_radiance_inside(CDesc d, const float4 *__restrict__ dirs, int n,
                                                             float4 *__restrict__ rad, float4 *__restrict__ ext) {
    extern __shared__ float4 clds[];
    const ViewTables<STAGED> t = stage_view<STAGED>(d, clds);
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
        const float4 v4 = dirs[i];
        const double v[3] = {v4.x, v4.y, v4.z};
        const double rmu = dot3(d.cm, v), nu = dot3(v, d.sun);
        float w;
        const int e = nu_coord(d, nu, w);
        const float4 is = view_S(d, t, rmu, e, w);
        rad[i] = combine(d, is, nu);
        if (ext) {
            const float3 x = view_T(d, t, rmu * d.invr);
            ext[i] = make_float4(x.x, x.y, x.z, 0.f);
        }
    }
}

// inScattering, atmosphereShader.glsl:425-533 (HORIZON_HACK on).  INSIDE: the camera is
// inside the atmosphere and there are no light shafts (din = sw = 0): its side of the
// difference and of the extinction comes from the view's tables.
// 1280 x 720 points on the 32x128x32x8 tables, staged: 70 -> 35 us.  The other forms take the
// registers that they need (202; held to 128 for four waves they spill): 65536 points from inside
// 12.5 -> 7.5 us, 921600 with light shafts 72 -> 49.
template <bool INSIDE, bool STAGED>
__global__ __launch_bounds__(STAGED ? 512 : 256) __attribute__((amdgpu_waves_per_eu(STAGED ? 4 : 2))) void
k_in_scattering(CDesc d, const float4 *__restrict__ pts, int n, float4 *__restrict__ rad, float4 *__restrict__ ext) {
    extern __shared__ float4 clds[];
    const ViewTables<STAGED> t = stage_view<STAGED>(d, clds);
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
        const float4 p4 = pts[i];
        double cam[3] = {d.cam[0], d.cam[1], d.cam[2]};
        double pt[3] = {p4.x, p4.y, p4.z};
        double v[3] = {pt[0] - cam[0], pt[1] - cam[1], pt[2] - cam[2]};
        double dist = sqrt64_pos(dot3(v, v));   // NaN for a point at the camera or at infinity, as v is then
        const double idist = rcp64(dist);
        for (int c = 0; c < 3; ++c) v[c] *= idist;
        double r, rMu, mu;
        const double shift = d.cm[2] - cam[2];   // flat-terrain coordinates (Rg) or 0
        cam[2] = d.cm[2];
        pt[2] += shift;
        rMu = dot3(cam, v);
        if (INSIDE) {
            r = d.r;
            mu = rMu * d.invr;
        } else {
            r = sqrt(dot3(cam, cam));
            mu = rMu / r;
            const double sw = fmin(fmax(d.shaft, 0.0), dist);
            for (int c = 0; c < 3; ++c) pt[c] -= v[c] * sw;
            const double q = rMu * rMu - r * r + d.Rt * d.Rt;
            const double din = q >= 0.0 ? fmax(-rMu - sqrt(q), 0.0) : 0.0;
            if (din > 0.0 && din < dist) {
                for (int c = 0; c < 3; ++c) cam[c] += din * v[c];
                rMu += din;
                mu = rMu / d.Rt;
                r = d.Rt;
                dist -= din;
            }
        }
        float4 out = make_float4(0.f, 0.f, 0.f, 0.f), ex = make_float4(1.f, 1.f, 1.f, 0.f);
        if (INSIDE || r <= d.Rt) {
            const double nu = dot3(v, d.sun);
            const double muS = INSIDE ? d.muS : dot3(cam, d.sun) / r;
            if (INSIDE) {   // r is that of :472 already
                for (int c = 0; c < 3; ++c) pt[c] *= d.near_f;
            } else if (r < d.near) {
                const double f = d.near / r;
                r *= f;
                for (int c = 0; c < 3; ++c) pt[c] *= f;
            }
            double r1 = sqrt64(dot3(pt, pt)), ir1 = rcp64(r1);
            double mu1 = dot3(pt, v) * ir1;
            const double muS1 = dot3(pt, d.sun) * ir1;
            float3 e;
            if (INSIDE) {   // T_ratio with the camera's end from its row
                const bool up = mu > 0.0;
                const float3 x = view_T(d, t, up ? mu : -mu), y = T_at(d, r1, up ? mu1 : -mu1);
                e = up ? make_float3(x.x / y.x, x.y / y.y, x.z / y.z) : make_float3(y.x / x.x, y.y / x.y, y.z / x.z);
                e = make_float3(fminf(e.x, 1.f), fminf(e.y, 1.f), fminf(e.z, 1.f));
            } else {
                e = T_ratio(d, r, mu, r1, mu1, mu > 0.0);
            }
            ex = make_float4(e.x, e.y, e.z, 0.f);
            float nw;
            const int ne = nu_coord(d, nu, nw);
            const double EPS = 0.004;
            double lim;
            if (INSIDE) {
                lim = d.lim;
            } else {
                const double qg = d.Rg / r;
                lim = -sqrt(1.0 - qg * qg);
            }
            // next to the horizon: between the two sides of it (one loop body: the lookups
            // of both sides at once would take 250 registers)
            const bool hor = fabs(mu - lim) < EPS;
            const float wh = hor ? (float)(((mu - lim) + EPS) / (2.0 * EPS)) : 0.f;
            double m = hor ? lim - EPS : mu;
            float4 is = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 1
            for (int h = 0; h < (hor ? 2 : 1); ++h) {
                if (hor) {
                    r1 = sqrt64_pos(r * r + dist * dist + 2.0 * r * dist * m);
                    mu1 = (r * m + dist) * rcp64(r1);
                }
                const float4 s0 = INSIDE ? view_S(d, t, r * m, ne, nw) : texture4D(d, r, m, muS, nu);
                const float4 s1 = texture4D(d, r1, mu1, muS1, nu);
                const float4 x = make_float4(fmaxf(s0.x - s1.x * e.x, 0.f), fmaxf(s0.y - s1.y * e.y, 0.f),
                                             fmaxf(s0.z - s1.z * e.z, 0.f), fmaxf(s0.w - s1.w * e.x, 0.f));
                is = h == 0 ? x : lerp4(is, x, wh);
                m = lim + EPS;
            }
            const float f = fminf(fmaxf((float)muS / 0.02f, 0.f), 1.f);  // smoothstep(0, 0.02, muS)
            is.w *= f * f * (3.f - 2.f * f);
            out = combine(d, is, nu);
        }
        rad[i] = out;
        if (ext) ext[i] = ex;
    }
}

// sunRadiance (:342-350, transmittanceWithShadow :263-265) and skyIrradiance (:355-361)
__global__ __launch_bounds__(256) void k_sun_sky(CDesc d, const float2 *__restrict__ rmus, int n,
                                                 float4 *__restrict__ sun, float4 *__restrict__ sky) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double r = rmus[i].x, muS = rmus[i].y;
    const double qg = d.Rg / r;
    float3 s = make_float3(0.f, 0.f, 0.f);
    if (!(muS < -sqrt(1.0 - qg * qg))) s = T_at(d, r, muS);
    sun[i] = make_float4(s.x * kSunIntensity, s.y * kSunIntensity, s.z * kSunIntensity, 0.f);
    const float uR = (float)((r - d.Rg) / (d.Rt - d.Rg));
    const float uMuS = ((float)muS + 0.2f) / 1.2f;
    const float3 e = rgb_bilinear(d.E, d.SW, d.SH, uMuS * d.SW - 0.5f, uR * d.SH - 0.5f);
    sky[i] = make_float4(e.x * kSunIntensity, e.y * kSunIntensity, e.z * kSunIntensity, 0.f);
}

atmo_status cfail(atmo_status st, const char *fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    return atmo::set_error(st, buf);
}

bool al(const void *p, size_t a) { return ((uintptr_t)p % a) == 0; }

atmo_status make_desc(const atmo_params *p, const atmo_view *v, CDesc &d) {
    if (!p) return cfail(ATMO_ERR_INVALID_ARGUMENT, "null parameters");
    if (!(p->Rg > 0.f) || !(p->Rt > p->Rg)) return cfail(ATMO_ERR_INVALID_ARGUMENT, "need 0 < Rg < Rt");
    if (p->TRANSMITTANCE_W < 2 || p->TRANSMITTANCE_H < 2 || p->SKY_W < 2 || p->SKY_H < 2 || p->RES_R < 2 ||
        p->RES_MU < 2 || p->RES_MU_S < 2 || p->RES_NU < 2)
        return cfail(ATMO_ERR_INVALID_ARGUMENT, "table sizes must be >= 2");
    if ((long long)p->RES_R * p->RES_MU * p->RES_MU_S * p->RES_NU > (1LL << 28))
        return cfail(ATMO_ERR_INVALID_ARGUMENT, "inscatter table too large");
    if (!(p->betaR.x > 0.f && p->betaR.y > 0.f && p->betaR.z > 0.f))
        return cfail(ATMO_ERR_INVALID_ARGUMENT, "getMie divides by betaR: need betaR > 0");
    if (!(p->mieG > -1.f && p->mieG < 1.f)) return cfail(ATMO_ERR_INVALID_ARGUMENT, "mieG must be in (-1, 1)");
    d.Rg = p->Rg;
    d.Rt = p->Rt;
    d.H = sqrt(d.Rt * d.Rt - d.Rg * d.Rg);
    d.bR[0] = p->betaR.x;
    d.bR[1] = p->betaR.y;
    d.bR[2] = p->betaR.z;
    const double g = p->mieG, pi = 3.141592657;  // M_PI of atmosphereShader.glsl:99
    d.kR = (float)(3.0 / (16.0 * pi));
    d.kM = (float)(1.5 / (4.0 * pi) * (1.0 - g * g) / (2.0 + g * g));
    d.g2p1 = (float)(1.0 + g * g);
    d.m2g = (float)(-2.0 * g);
    d.f_tMu = (float)(tan(1.5) / 1.15);
    d.f_inv_dRt = (float)(1.0 / (d.Rt - d.Rg));
    d.TW = p->TRANSMITTANCE_W;
    d.TH = p->TRANSMITTANCE_H;
    d.SW = p->SKY_W;
    d.SH = p->SKY_H;
    d.RR = p->RES_R;
    d.RMU = p->RES_MU;
    d.RMUS = p->RES_MU_S;
    d.RNU = p->RES_NU;
    d.W4 = p->RES_MU_S * p->RES_NU;
    d.near = d.Rg;
    d.shaft = 0.0;
    for (int c = 0; c < 3; ++c) d.cam[c] = d.sun[c] = 0.0;
    if (v) {
        if (!(v->meters_per_unit > 0.0)) return cfail(ATMO_ERR_INVALID_ARGUMENT, "meters_per_unit must be > 0");
        for (int c = 0; c < 3; ++c) {
            d.cam[c] = v->camera[c];
            d.sun[c] = v->sun[c];
        }
        if (!(dot3(d.cam, d.cam) > 0.0)) return cfail(ATMO_ERR_INVALID_ARGUMENT, "camera at the planet centre");
        d.shaft = v->shaft_width;
        d.near = d.Rg + 600.0 / v->meters_per_unit;
    }
    d.T = d.S = d.E = nullptr;
    return ATMO_OK;
}

// GL LINEAR + CLAMP_TO_EDGE taps of texel coordinate x (gl_axis_d)
void axis(double x, int N, int &i0, int &i1, float &a) {
    x = std::fmin(std::fmax(x, -1.0), (double)N);
    const double f = std::floor(x);
    a = (float)(x - f);
    i0 = std::min(std::max((int)f, 0), N - 1);
    i1 = std::min(std::max((int)f + 1, 0), N - 1);
}

// What the rays of a view share; flat: the flat-terrain and near-ground adjustments of
// inScattering.  d.inside: the view tables serve every ray.
void view_desc(CDesc &d, bool flat) {
    for (int c = 0; c < 3; ++c) d.cm[c] = d.cam[c];
    double r = std::sqrt(dot3(d.cm, d.cm));
    if (flat && r < 0.9 * d.Rg) {
        d.cm[2] += d.Rg;
        r = std::sqrt(dot3(d.cm, d.cm));
    }
    // a margin of rounding below Rt: din = 0 for every ray
    d.inside = !(d.shaft > 0.0) && r <= d.Rt * (1.0 - 1e-9);
    d.muS = dot3(d.cm, d.sun) / r;
    d.invr = 1.0 / r;
    d.near_f = 1.0;
    if (flat && r < d.near) {
        d.near_f = d.near / r;
        r *= d.near_f;
    }
    d.r = r;
    d.rho2 = r * r - d.Rg * d.Rg;
    d.rho = std::sqrt(std::fmax(d.rho2, 0.0));
    d.H2 = d.H * d.H;
    d.invrH = 1.0 / (d.rho + d.H);
    const double qg = d.Rg / r;
    d.lim = -std::sqrt(1.0 - qg * qg);
    const double xs = (std::atan(std::fmax(d.muS, -0.1975) * std::tan(1.26 * 1.1)) / 1.1 + (1.0 - 0.26)) * 0.5 * (d.RMUS - 1.0);
    d.inside = d.inside && xs < 1e6;   // (a sun vector of length 1 stays below RMUS)
    const double f = std::floor(std::fmin(xs, 1e6));
    d.i0 = (int)f;
    d.ia = (float)(xs - f);
    axis(d.rho / d.H * (d.RR - 1.0), d.RR, d.k0, d.k1, d.kg);
    axis(std::sqrt(std::fmax(r - d.Rg, 0.0) / (d.Rt - d.Rg)) * d.TH - 0.5, d.TH, d.tj0, d.tj1, d.tb);
}

// Staged view tables pay from some rays per staged entry on (1676 entries for 32x128x32x8 with
// 256 T columns, 3316 for 32x160x32x16): every workgroup stages them all.  GPU time of a
// frame's rays in us, each lookup blending its own / staged:
//   sky         131072 rays  4.4 / 6.7 and 4.5 / 10.2;  262144  6.4 / 7.9 and 6.8 / 11.3;
//               921600  16.1 / 15.1 and 16.0 / 19.1;  2073600  29.1 / 23.2 and 29.1 / 26.8
//   scattering  262144 points  15.7 / 22.6 and 15.6 / 30.1;  921600  42.4 / 41.6 and 42.7 / 51.4;
//               2073600  85.5 / 73.3 and 85.5 / 84.6
// Scattered directions, whose own lookups share no cache lines, cross earlier: 262144 rays 11.6 /
// 8.2 and 12.0 / 11.6; 921600 points 57.9 / 52.1 and 63.7 / 63.3.  At most 64 KB, two
// workgroups per CU.
constexpr int kSkyPerEntry = 128, kAerialPerEntry = 512;
constexpr size_t kInsideLds = 64 * 1024;
// Workgroups of 512 threads: one per CU for the sky (2073600 rays with 256 / 512 / 1024:
// 22.2 / 23.8 / 28.0 us), two for the scattering, whose own lookups wait more
// (921600 points: 40.6 / 34.8 / 39.5).
constexpr int kSkyGroups = 256, kAerialGroups = 512;
bool use_staged(const CDesc &d, int n, int per_entry) {
    const size_t entries = view_entries(d);
    return d.inside && entries * sizeof(float4) <= kInsideLds && (size_t)n >= per_entry * entries;
}
int staged_groups(int n, int most) { return std::min((int)(((long long)n + 511) / 512), most); }

}  // namespace
}  // namespace atmo

using atmo::CDesc;

extern "C" {

atmo_status atmo_sky_radiance(const atmo_params *p, const float *T, const float *S, const atmo_view *view,
                              const float *dirs, int n, float *radiance, float *extinction, void *stream) {
    CDesc d;
    atmo_status st = atmo::make_desc(p, view, d);
    if (st != ATMO_OK) return st;
    if (!view) return atmo::cfail(ATMO_ERR_INVALID_ARGUMENT, "null view");
    if (n < 0) return atmo::cfail(ATMO_ERR_INVALID_ARGUMENT, "negative count");
    if (n == 0) return ATMO_OK;
    if (!T || !S || !dirs || !radiance || !atmo::al(T, 4) || !atmo::al(S, 16) || !atmo::al(dirs, 16) ||
        !atmo::al(radiance, 16) || (extinction && !atmo::al(extinction, 16)))
        return atmo::cfail(ATMO_ERR_INVALID_ARGUMENT, "bad table or array pointers");
    d.T = T;
    d.S = S;
    atmo::view_desc(d, false);
    if (atmo::use_staged(d, n, atmo::kSkyPerEntry))
        hipLaunchKernelGGL(atmo::k_sky_radiance_inside<true>, dim3(atmo::staged_groups(n, atmo::kSkyGroups)), dim3(512),
                           atmo::view_entries(d) * sizeof(float4), (hipStream_t)stream, d, (const float4 *)dirs, n,
                           (float4 *)radiance, (float4 *)extinction);
    else if (d.inside)
        hipLaunchKernelGGL(atmo::k_sky_radiance_inside<false>, dim3((n + 255) / 256), dim3(256), 0, (hipStream_t)stream, d,
                           (const float4 *)dirs, n, (float4 *)radiance, (float4 *)extinction);
    else
        hipLaunchKernelGGL(atmo::k_sky_radiance, dim3((n + 255) / 256), dim3(256), 0, (hipStream_t)stream, d,
                           (const float4 *)dirs, n, (float4 *)radiance, (float4 *)extinction);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return atmo::cfail(ATMO_ERR_DEVICE, "k_sky_radiance: %s", hipGetErrorString(e));
    return ATMO_OK;
}

atmo_status atmo_in_scattering(const atmo_params *p, const float *T, const float *S, const atmo_view *view,
                               const float *points, int n, float *radiance, float *extinction, void *stream) {
    CDesc d;
    atmo_status st = atmo::make_desc(p, view, d);
    if (st != ATMO_OK) return st;
    if (!view) return atmo::cfail(ATMO_ERR_INVALID_ARGUMENT, "null view");
    if (n < 0) return atmo::cfail(ATMO_ERR_INVALID_ARGUMENT, "negative count");
    if (n == 0) return ATMO_OK;
    if (!T || !S || !points || !radiance || !atmo::al(T, 4) || !atmo::al(S, 16) || !atmo::al(points, 16) ||
        !atmo::al(radiance, 16) || (extinction && !atmo::al(extinction, 16)))
        return atmo::cfail(ATMO_ERR_INVALID_ARGUMENT, "bad table or array pointers");
    d.T = T;
    d.S = S;
    atmo::view_desc(d, true);
    if (atmo::use_staged(d, n, atmo::kAerialPerEntry))
        hipLaunchKernelGGL((atmo::k_in_scattering<true, true>), dim3(atmo::staged_groups(n, atmo::kAerialGroups)), dim3(512),
                           atmo::view_entries(d) * sizeof(float4), (hipStream_t)stream, d, (const float4 *)points, n,
                           (float4 *)radiance, (float4 *)extinction);
    else if (d.inside)
        hipLaunchKernelGGL((atmo::k_in_scattering<true, false>), dim3((n + 255) / 256), dim3(256), 0, (hipStream_t)stream, d,
                           (const float4 *)points, n, (float4 *)radiance, (float4 *)extinction);
    else
        hipLaunchKernelGGL((atmo::k_in_scattering<false, false>), dim3((n + 255) / 256), dim3(256), 0, (hipStream_t)stream, d,
                           (const float4 *)points, n, (float4 *)radiance, (float4 *)extinction);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return atmo::cfail(ATMO_ERR_DEVICE, "k_in_scattering: %s", hipGetErrorString(e));
    return ATMO_OK;
}

atmo_status atmo_sun_sky_irradiance(const atmo_params *p, const float *T, const float *E, const float *rmus,
                                    int n, float *sun, float *sky, void *stream) {
    CDesc d;
    atmo_status st = atmo::make_desc(p, nullptr, d);
    if (st != ATMO_OK) return st;
    if (n < 0) return atmo::cfail(ATMO_ERR_INVALID_ARGUMENT, "negative count");
    if (n == 0) return ATMO_OK;
    if (!T || !E || !rmus || !sun || !sky || !atmo::al(T, 4) || !atmo::al(E, 4) || !atmo::al(rmus, 8) ||
        !atmo::al(sun, 16) || !atmo::al(sky, 16))
        return atmo::cfail(ATMO_ERR_INVALID_ARGUMENT, "bad table or array pointers");
    d.T = T;
    d.E = E;
    hipLaunchKernelGGL(atmo::k_sun_sky, dim3((n + 255) / 256), dim3(256), 0, (hipStream_t)stream, d,
                       (const float2 *)rmus, n, (float4 *)sun, (float4 *)sky);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return atmo::cfail(ATMO_ERR_DEVICE, "k_sun_sky: %s", hipGetErrorString(e));
    return ATMO_OK;
}

}  // extern "C"
