// atmo_kernels.hip — gfx950 kernels of the atmo precompute, one per reference pass.
//
// Every kernel is launched once per pass for a whole batch of parameter sets:
// blockIdx.x indexes a tile table of (set, tile) pairs built by the host plan,
// so sets of different resolutions share one launch.
#include "atmo_kernels.h"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace atmo {

// 2^y for y <= 1000, at least 2^-1000 (also for NaN), 1.4e-16 relative: a polynomial in the
// fraction (degree 11, interpolated in Chebyshev points of |f| <= 1/2), the integer part
// added to the exponent.
constexpr double kLog2e = 1.4426950408889634;
__device__ __forceinline__ double exp2_64(double y) {
    constexpr double kRound64 = 6755399441055744.0;   // 1.5 2^52
    y = fmax(y, -1000.0);
    const double t = y + kRound64, f = y - (t - kRound64);
    double p = fma(f, 4.4554725442721574e-10, 7.0742005955524935e-09);
    p = fma(f, p, 1.0178059245425577e-07);
    p = fma(f, p, 1.3215432498125634e-06);
    p = fma(f, p, 1.5252733836823374e-05);
    p = fma(f, p, 0.00015403530463804289);
    p = fma(f, p, 0.0013333558146410734);
    p = fma(f, p, 0.009618129107587189);
    p = fma(f, p, 0.05550410866482161);
    p = fma(f, p, 0.2402265069591016);
    p = fma(f, p, 0.6931471805599453);
    p = fma(f, p, 1.0);
    return __hiloint2double(__double2hiint(p) + (__double2loint(t) << 20), __double2loint(p));
}

// tan x for x in [0, 1.5], 5.5e-16 relative (x = 1.5 m itself is rounded, which moves tan x by
// up to 2.3e-15): from the Taylor series of sine and cosine at half of x, or of pi/2 - x
// from 0.8 on (terms below 1e-17 left out).  A tenth of the library's code, which reduces
// any argument.
__device__ __forceinline__ double tan_col(double x) {
    const bool co = x > 0.8;
    const double y = 0.5 * (co ? (1.5707963267948966 - x) + 6.123233995736766e-17 : x), z = y * y;
    double s = fma(z, 1.6059043836821613e-10, -2.505210838544172e-08);
    s = fma(z, s, 2.7557319223985893e-06);
    s = fma(z, s, -0.0001984126984126984);
    s = fma(z, s, 0.008333333333333333);
    s = fma(z, s, -0.16666666666666666);
    s = fma(y * z, s, y);
    double c = fma(z, 2.08767569878681e-09, -2.755731922398589e-07);
    c = fma(z, c, 2.48015873015873e-05);
    c = fma(z, c, -0.001388888888888889);
    c = fma(z, c, 0.041666666666666664);
    c = fma(z, c, -0.5);
    c = fma(z, c, 1.0);
    const double n = 2.0 * s * c, d = fma(-s, s, c * c);
    return co ? d / n : n / d;
}

// ---------------------------------------------------------------------------
// Pass T — transmittance.glsl:78-98.  FP64 trapezoid of exp(-h/H) for both
// scale heights at once; 16 lanes share one texel's samples.
// tile = 16 consecutive texels.  Bound by FP64 issue: the library's exp and square
// root take about 95 instructions a sample, exp2_64 and sqrt64_pos 54, and the tables are
// FP32 (256x64 texels, 500 samples: 28 -> 21 us); nearly half of the texels of the
// tangent parameterisation look at the ground and need no samples, and straight code
// without the library's argument reductions is fetched in time (-> 20; 24 sets 515 ->
// 310 us).  A single set is left with its latency: 4 waves per SIMD, half of them idle.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_transmittance(const SetDesc *__restrict__ sets,
                                                       const uint2 *__restrict__ tiles,
                                                       int nsamp) {
    const uint2 tl = tiles[blockIdx.x];
    const SetDesc &s = sets[tl.x];
    const int lane = threadIdx.x & 15;
    const int t = ((int)tl.y * kTileY + (int)blockIdx.y) * 16 + (threadIdx.x >> 4);
    const bool valid = t < s.TW * s.TH;
    const int tt = valid ? t : 0;
    const int i = tt % s.TW, j = tt / s.TW;
    // getTransmittanceRMu (common.glsl:126-136), gl_FragCoord = (i + .5, j + .5)
    double rr = (j + 0.5) / s.TH;
    double m = (i + 0.5) / s.TW;
    double r, mu;
    const double tm = tan_col(1.5 * m);
    if (s.linT) {
        r = s.Rg + rr * (s.Rt - s.Rg);
        mu = -0.15 + m * (1.0 + 0.15);
    } else {
        r = s.Rg + rr * rr * (s.Rt - s.Rg);
        mu = -0.15 + tm * (1.15 / 14.101419947171719);   // tan(1.5)
    }
    double dx = limit_d(s, r, mu) / nsamp;
    double sR = 0.0, sM = 0.0;
    const double eR = -kLog2e / s.HR, eM = -kLog2e / s.HM;
    const double r2 = r * r, rmu2 = 2.0 * r * mu;
    const double q = s.Rg / r;
    const bool below = mu < -sqrt(1.0 - q * q);   // the ground is in the way: no integral
    for (int k = below ? nsamp + 1 : lane; k <= nsamp; k += 16) {
        const double x = k * dx;
        const double h = sqrt64_pos(fma(x, x + rmu2, r2)) - s.Rg;   // >= 0: the ray ends at the ground
        const double w = (k == 0 || k == nsamp) ? 0.5 : 1.0;
        sR = fma(w, exp2_64(h * eR), sR);
        sM = fma(w, exp2_64(h * eM), sM);
    }
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) {
        sR += __shfl_xor(sR, off, 16);
        sM += __shfl_xor(sM, off, 16);
    }
    if (lane == 0 && valid) {
        // sun_centres: the bits of tan(1.5 m), the upper half in row 0 and the lower in row 1
        const float ck = __int_as_float(j == 0 ? __double2hiint(tm) : j == 1 ? __double2loint(tm) : 0);
        // no number where the ray's length is none (the sums above are finite in any case)
        double dR = below ? 1e9 : fma(sR, dx, dx - dx);
        double dM = below ? 1e9 : fma(sM, dx, dx - dx);
        double tau[3], T[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            tau[k] = (double)s.bR[k] * dR + (double)s.bME[k] * dM;
            T[k] = tau[k] == tau[k] ? exp2_64(tau[k] * -kLog2e) : tau[k];
        }
        float4 o = make_float4((float)T[0], (float)T[1], (float)T[2], 0.0f);
        o = q16(o, s.hs);
        s.T4[t] = o;
        if (s.tau4)
            s.tau4[t] = make_float4((float)tau[0], (float)tau[1], (float)tau[2], ck);
        if (s.outT) {
            s.outT[3 * t + 0] = o.x;
            s.outT[3 * t + 1] = o.y;
            s.outT[3 * t + 2] = o.z;
        }
    }
}

// ---------------------------------------------------------------------------
// Pass dE1 — irradiance1.glsl:78-82, fused with copyIrradiance k = 0
// (PreprocessAtmo.cpp:298-303: E = 0).  tile = 256 texels.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_irradiance1(const SetDesc *__restrict__ sets,
                                                     const uint2 *__restrict__ tiles) {
    const uint2 tl = tiles[blockIdx.x];
    const SetDesc &s = sets[tl.x];
    const int t = (int)tl.y * 256 + threadIdx.x;
    if (t >= s.SW * s.SH) return;
    const int i = t % s.SW, j = t / s.SW;
    // getIrradianceRMuS (common.glsl:144-147): r - Rg = j/(SH-1) (Rt - Rg)
    double h = (double)j / (s.SH - 1.0) * (s.Rt - s.Rg);
    double muS = -0.2 + (double)i / (s.SW - 1.0) * (1.0 + 0.2);
    float3 T = T_lookup(s, (float)h, (float)muS);
    float c = (float)fmax(muS, 0.0);
    if (s.dE4) s.dE4[t] = q16(make_float4(T.x * c, T.y * c, T.z * c, 0.0f), s.hs);
    if (s.E4) s.E4[t] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (s.outE) {
        s.outE[3 * t + 0] = 0.0f;
        s.outE[3 * t + 1] = 0.0f;
        s.outE[3 * t + 2] = 0.0f;
    }
}

constexpr int kNChunk = 64;   // k_inscatterN form 2: samples staged per chunk
// LDS byte address of an entry in two FMA-class instructions (about 2 cycles per
// wave on gfx950, where a conversion and a shift-add take 4 each).  u + kRound,
// kRound = 1.5 2^23, is kRound + k with k = u rounded to the nearest integer;
// times STRIDE 2^-149, plus (base - STRIDE kRound) 2^-149, it is the denormal
// whose bit pattern is base + STRIDE k.  Exact: the addend is a multiple of
// STRIDE below 2^24 STRIDE (base is a multiple of STRIDE), the result is an
// integer below 2^23.  At a tie either neighbour may come out: the two lines meet
// there.
constexpr float kRound = 12582912.0f;
template <int STRIDE>
__device__ __forceinline__ float lds_addend(unsigned base) {   // (base - STRIDE kRound) 2^-149
    return ((float)base - (float)STRIDE * kRound) * 1.40129846e-45f;
}
template <int STRIDE>
__device__ __forceinline__ unsigned lds_entry(float u, float addend) {
    return __float_as_uint(fmaf(u + kRound, (float)STRIDE * 1.40129846e-45f, addend));
}
__device__ __forceinline__ float4 lds4(unsigned a, int off = 0) {
    typedef float v4 __attribute__((ext_vector_type(4)));
    const v4 v = *(__attribute__((address_space(3))) const v4 *)(size_t)(a + off);
    return make_float4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ float2 lds2(unsigned a, int off = 0) {
    typedef float v2 __attribute__((ext_vector_type(2)));
    const v2 v = *(__attribute__((address_space(3))) const v2 *)(size_t)(a + off);
    return make_float2(v.x, v.y);
}

// ---------------------------------------------------------------------------
// Pass dS1 — inscatter1.glsl:104-150 fused with copyInscatter1.glsl:104-109.
// A texel's view ray depends only on its r layer and mu row, so everything of
// an integration sample that does not involve the sun — its distance and
// radius, the view-ray transmittance T(r, mu, t), the scale-height factors and
// the r-row of the T(r_i, mu_s_i) lookup — is shared by the RNU x RMU_S texels
// of the row.  A workgroup computes those terms (FP64 geometry) for its row in LDS,
// and a texel then needs only the sun's visibility, mu_s_i and the mu axis of the
// T lookup per sample.
//
// Two forms.  k_inscatter1_rows: the two T rows of the sample, weighted by the
// r fraction and by T(r, mu, t), are blended once into an LDS row that the row's
// texels look up; the rows are loaded coalesced, one sample ahead, into registers by
// the parity of the row number, so a step to the next row loads one.
// k_inscatter1: every texel gathers its four T texels.  Gathers of 64 lanes cost
// the texture path about 27 cycles each, a staged row costs 64 per CU for all its
// texels: 32x128x32x8 (256 texels, 256 columns) 159 -> 105 us; 48 sets of the mixed
// batch 14.9 -> 7.8 ms; 64x256x64x16 2.34 -> 1.14 ms.
// ---------------------------------------------------------------------------
struct __attribute__((aligned(16))) S1Entry {
    double ti;       // sample distance
    double thr;      // the sun is visible where r_i mu_s_i >= thr
    double iri;      // 1 / r_i, times the factor of the mu axis' argument
    float eR, eM;    // exp(-h_i/HR), exp(-h_i/HM)
    float p0[3];     // weights of the T row of even and of odd number: r fraction x T(r, mu, t_i) x
    unsigned j0;     // trapezoid weight; rows of r_i (k_inscatter1: p0 without the r fraction, p1[0] the fraction)
    float p1[3];
    unsigned j1;
};

constexpr int kS1Chunk = 64;
constexpr int kXkMin = 64;     // columns from which a few terms of the arctangent's series do

// The mu axis of the sun's T lookup next to the horizon, where T is steep: an FP32
// texel coordinate is good to ~3e-5 of a texel at TW = 512, which moves a grazing
// sun's T by ~1e-4.  So the filter fraction is taken from a column centre x_k =
// tan(1.5 (k + 0.5) / TW), staged once per workgroup:  u - u_k = (atan x - atan x_k)
// / 1.5 = atan((x - x_k) / (1 + x x_k)) / 1.5, x = (mu_s_i + 0.15) tan(1.5) / 1.15 and
// the difference in FP64; the centre is any within about a column of x (its column
// comes from a fit of atan in x / (1 + |x|), good to 7.1e-4), the integer part of the
// offset moves to the column, and the arctangent of the small offset is its series (three
// terms, 6e-9 relative from kXkMin columns on; below, atanf).
enum { kSunTab, kSunLin, kSunWide, kSunFew };   // centres; linear parameterisation; more than kXkMax columns
                                                // (FP32); centres, fewer than kXkMin columns
struct SunAxis {
    double c;      // argument at mu_s_i = 0
    double scale;  // argument per mu_s_i
    float last, sc;   // TW - 1, TW / 1.5
    float xk;      // LDS address of the centres (lds_addend form, base only)
};
template <int AX>
__device__ __forceinline__ SunAxis sun_axis(const SetDesc &s, const double *xk) {
    SunAxis x;
    x.c = AX == kSunLin ? 0.15 / 1.15 * s.TW - 0.5 : 0.15 * s.tMu;
    x.scale = AX == kSunLin ? s.TW / 1.15 : s.tMu;
    x.last = (float)(s.TW - 1);
    x.sc = (float)s.TW / 1.5f;
    x.xk = (float)(unsigned)(size_t)(__attribute__((address_space(3))) const char *)xk * 1.40129846e-45f;
    return x;
}
// The column (a whole number in [0, TW - 1]) and the fraction of r_i mu_s_i = num, in two
// steps: the argument and a centre near it (an LDS read), then the offset from it.
struct SunCell {
    double x, xk;   // argument, centre
    float xf, k;    // argument, column of the centre
};
template <int AX>
__device__ __forceinline__ SunCell sun_cell(const SunAxis &x, double num, double iri) {
    SunCell c;
    c.x = fma(num, iri, x.c);
    if constexpr (AX == kSunTab || AX == kSunFew) {
        c.xf = (float)c.x;
        const float t = c.xf * __builtin_amdgcn_rcpf(1.0f + fabsf(c.xf));
        const float ta = __uint_as_float(__float_as_uint(t) & 0x7fffffffu);
        float q = fmaf(ta, 2.434126615524292f, -6.0853166580200195f);
        q = fmaf(ta, q, 3.8018410205841064f);
        q = fmaf(ta, q, 0.38255468010902405f);
        q = fmaf(ta, q, 1.0375903844833374f);
        c.k = __builtin_amdgcn_fmed3f((fmaf(t * x.sc, q, -0.5f) + kRound) - kRound, 0.0f, x.last);
        const unsigned xa = __float_as_uint(fmaf(c.k, 8.0f * 1.40129846e-45f, x.xk));
        c.xk = *(__attribute__((address_space(3))) const double *)(size_t)xa;
    }
    return c;
}
template <int AX>
__device__ __forceinline__ void sun_column(const SunAxis &x, const SunCell &c, float &col, float &a) {
    if constexpr (AX == kSunLin) {
        const double p = fmin(fmax(c.x, 0.0), (double)x.last), f = floor(p);
        col = (float)f;
        a = (float)(p - f);
    } else if constexpr (AX == kSunWide) {
        const float p = __builtin_amdgcn_fmed3f(fmaf(atanf((float)c.x), x.sc, -0.5f), 0.0f, x.last);
        col = floorf(p);
        a = p - col;
    } else {
        const float d = (float)(c.x - c.xk);
        const float g = d * __builtin_amdgcn_rcpf(fmaf(c.xf, c.xf - d, 1.0f));
        float o;   // offset from the centre, in columns
        if constexpr (AX == kSunTab) {
            const float z = g * g, e = g * x.sc;
            o = fmaf(e, z * fmaf(z, 0.2f, -1.0f / 3.0f), e);
        } else {
            o = atanf(g) * x.sc;
        }
        o = __builtin_amdgcn_fmed3f(o, -c.k, x.last - c.k);   // CLAMP_TO_EDGE
        const float f = floorf(o);
        a = o - f;
        col = c.k + f;
    }
}
// Centres of the T table's columns: from the spare component of the first two rows of
// optical depths (k_transmittance), upper and lower half of their bits, where there are any.
__device__ __forceinline__ void sun_centres(const SetDesc &s, double *xk) {
    for (int k = threadIdx.x; k < s.TW; k += blockDim.x)
        xk[k] = s.tau4 ? __hiloint2double(__float_as_int(s.tau4[k].w), __float_as_int(s.tau4[s.TW + k].w)) : tan(1.5 * (k + 0.5) / s.TW);
}
// nu and r mu_s of the texel in column x
__device__ __forceinline__ void s1_texel(const SetDesc &s, int x, double r, double &nu, double &muSr) {
    const ColGeom c = s.cols[x % s.RMUS];
    nu = -1.0 + (double)(x / s.RMUS) / (s.RNU - 1.0) * 2.0;
    muSr = c.mus64 * r;
}
// The terms of sample i of the row (l, y); BY_PARITY: row weights for k_inscatter1_rows.
// Stores the row's sample distance in dx.
template <bool BY_PARITY>
__device__ __forceinline__ S1Entry s1_entry(const SetDesc &s, int l, int y, int i, int nsamp, const SunAxis &ax, float &sdx) {
    const double r = s.layers[l].r;
    double mu, muS_u, nu_u;
    mu_mus_nu(s, s.layers[l], 0, y, mu, muS_u, nu_u);
    const double dx = limit_d(s, r, mu) / nsamp;
    if (i == 0) sdx = (float)dx;
    const double rho2 = r * r - s.Rg2;
    const double rmu = r * mu;
    const bool up = mu > 0.0;
    S1Entry en;
    en.ti = i * dx;
    const double q = rho2 + en.ti * (en.ti + 2.0 * rmu);       // ri^2 - Rg^2
    // muSi >= -sqrt(1 - Rg^2 / max(Rg, ri)^2)  <=>  ri muSi >= -sqrt(ri^2 - Rg^2)
    en.thr = q > 0.0 ? -sqrt(q) : 0.0;
    const float ri = sqrtf((float)(q + s.Rg2));
    const float h1 = (float)q / (ri + s.f_Rg);                 // ri - Rg (< 0 at a ground hit)
    const float mu1 = (float)(rmu + en.ti) / ri;
    // transmittance(r, mu, t_i) (common.glsl:272-282)
    const float3 Tseg = s.tview ? ld3(gptr(s.tview) + ((size_t)l * s.RMU + y) * (nsamp + 1) + i)
                      : up      ? T_ratio_lin(s, (float)(r - s.Rg), (float)mu, h1, mu1)
                                : T_ratio_lin(s, h1, -mu1, (float)(r - s.Rg), (float)-mu);
    const float w = !s.tview && (i == 0 || i == nsamp) ? 0.5f : 1.0f;
    const float T[3] = {Tseg.x * w, Tseg.y * w, Tseg.z * w};
    const double rid = sqrt(q + s.Rg2);
    en.iri = ax.scale / rid;
    const float hc = fmaxf(h1, 0.0f);                          // ri = max(Rg, ri)
    en.eR = __expf(-hc * (float)(1.0 / s.HR));
    en.eM = __expf(-hc * (float)(1.0 / s.HM));
    // r axis of T(max(Rg, ri), muSi): common.glsl:114-124 (FP64 coordinate)
    int j0, j1;
    double bd;
    gl_axis_dd(T_ur_d(s, q / (rid + s.Rg)) * s.TH - 0.5, s.TH, j0, j1, bd);
    const float b = (float)bd;
    if (BY_PARITY) {   // rows j0 and j0 + 1, or the one row of an edge
        const float w0 = j1 == j0 ? 1.0f : 1.0f - b, w1 = j1 == j0 ? 0.0f : b;
        const float we = j0 & 1 ? w1 : w0, wo = j0 & 1 ? w0 : w1;
#pragma unroll
        for (int c = 0; c < 3; ++c) { en.p0[c] = we * T[c]; en.p1[c] = wo * T[c]; }
        en.j0 = (unsigned)(j0 & 1 ? j1 : j0);   // even (an edge's: either parity, weight 0)
        en.j1 = (unsigned)(j0 & 1 ? j0 : j1);
    } else {
#pragma unroll
        for (int c = 0; c < 3; ++c) en.p0[c] = T[c];
        en.p1[0] = b; en.p1[1] = en.p1[2] = 0.f;
        en.j0 = (unsigned)(j0 * s.TW) * 16u;
        en.j1 = (unsigned)(j1 * s.TW) * 16u;
    }
    return en;
}
__device__ __forceinline__ void s1_store(const SetDesc &s, size_t t, float fdx, const float r[3], const float m[3]) {
    const float4 oR = q16(make_float4(r[0] * fdx * s.bR[0], r[1] * fdx * s.bR[1], r[2] * fdx * s.bR[2], 0.f), s.hs);
    const float4 oM = q16(make_float4(m[0] * fdx * s.bMS[0], m[1] * fdx * s.bMS[1], m[2] * fdx * s.bMS[2], 0.f), s.hs);
    s.dSR4[t] = oR;
    s.dSM4[t] = oM;
    if (s.S4) s.S4[t] = make_float4(oR.x, oR.y, oR.z, oM.x);
}

// One mu row per workgroup, NM texels and NC T columns per thread.  Dynamic LDS:
// [2][NC threads + 1] row entries (the last one zero: the second tap of the last
// column, whose fraction is 0), [TW] centres.
template <int AX, int NM, int NC>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(NM >= 3 ? 4 : 5))) void
k_inscatter1_rows(const SetDesc *__restrict__ sets, const uint2 *__restrict__ tiles, int nsamp) {
    extern __shared__ __attribute__((aligned(32))) float4 lds[];
    __shared__ __attribute__((aligned(16))) S1Entry ent[kS1Chunk];
    __shared__ float s_dx;
    const uint2 tl = tiles[blockIdx.x];
    const SetDesc &s = sets[tl.x];
    const int TW = s.TW, W4 = s.W4, nthr = (int)blockDim.x;
    const int RS = NC * nthr + 1;
    double *xk = (double *)(lds + 2 * RS);
    if (AX == kSunTab) sun_centres(s, xk);
    if (threadIdx.x < 2) lds[threadIdx.x * RS + RS - 1] = make_float4(0.f, 0.f, 0.f, 0.f);
    const SunAxis ax = sun_axis<AX>(s, xk);
    const int line = (int)tl.y * kTileRows + (int)blockIdx.y;
    if (line >= s.RR * s.RMU) return;
    const int l = line / s.RMU, y = line % s.RMU;
    const double r = s.layers[l].r;
    double nud[NM], muSr[NM];
    float aR[NM][3], aM[NM][3];
#pragma unroll
    for (int j = 0; j < NM; ++j) {
        s1_texel(s, min((int)threadIdx.x + j * nthr, W4 - 1), r, nud[j], muSr[j]);
#pragma unroll
        for (int c = 0; c < 3; ++c) aR[j][c] = aM[j][c] = 0.f;
    }
    const __amdgpu_buffer_rsrc_t Tr = table_rsrc(s.T4, (unsigned)((size_t)TW * s.TH * sizeof(float4)));
    unsigned xo[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) xo[c] = (unsigned)min((int)threadIdx.x + c * nthr, TW - 1) * 16u;
    float3 t0[NC], t1[NC];   // the held rows of even and of odd number
#pragma unroll
    for (int c = 0; c < NC; ++c) t0[c] = t1[c] = make_float3(0.f, 0.f, 0.f);
    int held0 = -1, held1 = -1;
    struct Stage {   // S1Entry's part for the staging
        float4 p0, p1;
    } st;
    auto get_stage = [&](int js) {
        const float4 *q = (const float4 *)&ent[js];
        st.p0 = q[2];
        st.p1 = q[3];
    };
    auto load_rows = [&]() {   // those that the registers do not hold yet
        const int j0 = __builtin_amdgcn_readfirstlane(__float_as_int(st.p0.w)), j1 = __builtin_amdgcn_readfirstlane(__float_as_int(st.p1.w));
        auto load = [&](int j, float3 t[NC]) {
#pragma unroll
            for (int c = 0; c < NC; ++c) t[c] = ld3b(Tr, xo[c], (unsigned)(j * TW) * 16u);
        };
        if (j0 != held0) load(held0 = j0, t0);
        if (j1 != held1) load(held1 = j1, t1);
    };
    for (int c0 = 0; c0 <= nsamp; c0 += kS1Chunk) {
        const int nc = min(kS1Chunk, nsamp + 1 - c0);
        if (c0 > 0) __syncthreads();
        for (int js = threadIdx.x; js < nc; js += nthr) ent[js] = s1_entry<true>(s, l, y, c0 + js, nsamp, ax, s_dx);
        __syncthreads();
        get_stage(0);
        load_rows();
        for (int js = 0; js < nc; ++js) {
            float4 *row = lds + (js & 1) * RS;
#pragma unroll
            for (int c = 0; c < NC; ++c)
                row[(int)threadIdx.x + c * nthr] =
                    make_float4(fmaf(t0[c].x, st.p0.x, t1[c].x * st.p1.x), fmaf(t0[c].y, st.p0.y, t1[c].y * st.p1.y),
                                fmaf(t0[c].z, st.p0.z, t1[c].z * st.p1.z), 0.f);
            // this sample's terms and the next one's rows, read before the barrier
            const double ti = ent[js].ti, thr = ent[js].thr, iri = ent[js].iri;
            const float eR = ent[js].eR, eM = ent[js].eM;
            get_stage(min(js + 1, nc - 1));
            __syncthreads();
            if (js + 1 < nc) load_rows();
            const float rb = (float)(unsigned)(size_t)(__attribute__((address_space(3))) const char *)row * 1.40129846e-45f;
            // the texels step by step together: a step's LDS reads are in flight at once
            SunCell cell[NM];
            float vis[NM], col[NM], a[NM];
            float4 v0[NM], v1[NM];
#pragma unroll
            for (int j = 0; j < NM; ++j) {
                const double num = fma(nud[j], ti, muSr[j]);        // ri * muSi
                vis[j] = num >= thr ? 1.0f : 0.0f;
                cell[j] = sun_cell<AX>(ax, num, iri);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < NM; ++j) {
                sun_column<AX>(ax, cell[j], col[j], a[j]);
                const unsigned p = __float_as_uint(fmaf(col[j], 16.0f * 1.40129846e-45f, rb));
                v0[j] = lds4(p);
                v1[j] = lds4(p, 16);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < NM; ++j) {
                const float wR = vis[j] * eR, wM = vis[j] * eM;
                const float3 v = lerp3(f3(v0[j]), f3(v1[j]), a[j]);
                aR[j][0] = fmaf(v.x, wR, aR[j][0]); aR[j][1] = fmaf(v.y, wR, aR[j][1]); aR[j][2] = fmaf(v.z, wR, aR[j][2]);
                aM[j][0] = fmaf(v.x, wM, aM[j][0]); aM[j][1] = fmaf(v.y, wM, aM[j][1]); aM[j][2] = fmaf(v.z, wM, aM[j][2]);
            }
        }
    }
#pragma unroll
    for (int j = 0; j < NM; ++j) {
        const int x = (int)threadIdx.x + j * nthr;
        if (x < W4) s1_store(s, ((size_t)l * s.RMU + y) * W4 + x, s_dx, aR[j], aM[j]);
    }
}

// One mu row per workgroup.  Rows of at most 128 texels deal their samples to 4
// (at most 64 texels) or 2 slots of threads, whose sums are added through LDS in slot
// order: 16x64x16x4, whose 1024 rows would give a SIMD one wave, takes 19 us instead of 36.
// Samples that do not see the sun load nothing: over wide T tables, whose rows no cache
// holds, the loads are most of the time (rows of 512 texels, 32 x 64 of them: 1536 columns 387
// us with all loads, 228 so; 4096 columns 547 and 304).
// Dynamic LDS: [TW] centres.
template <int AX>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void
k_inscatter1(const SetDesc *__restrict__ sets, const uint2 *__restrict__ tiles, int nsamp) {
    extern __shared__ __attribute__((aligned(32))) float4 lds[];
    __shared__ __attribute__((aligned(16))) S1Entry ent[kS1Chunk];
    __shared__ float s_dx;
    __shared__ float part[6][192];
    const uint2 tl = tiles[blockIdx.x];
    const SetDesc &s = sets[tl.x];
    const int TW = s.TW, W4 = s.W4;
    double *xk = (double *)lds;
    if (AX == kSunTab || AX == kSunFew) sun_centres(s, xk);
    const SunAxis ax = sun_axis<AX>(s, xk);
    const int line = (int)tl.y * kTileRows + (int)blockIdx.y;
    if (line >= s.RR * s.RMU) return;
    const int l = line / s.RMU, y = line % s.RMU;
    const double r = s.layers[l].r;
    const int slots = W4 <= 64 ? 4 : W4 <= 128 ? 2 : 1, nthr = 256 / slots;
    const int slot = __builtin_amdgcn_readfirstlane((int)threadIdx.x / nthr), lane = (int)threadIdx.x - slot * nthr;
    constexpr int MAXT = 4;   // W4 <= 1024 (validated on the host)
    double nud[MAXT], muSr[MAXT];
    float aR[MAXT][3], aM[MAXT][3];
#pragma unroll
    for (int j = 0; j < MAXT; ++j) {
#pragma unroll
        for (int c = 0; c < 3; ++c) aR[j][c] = aM[j][c] = 0.f;
        nud[j] = muSr[j] = 0.0;
        if (j * nthr < W4) s1_texel(s, min(lane + j * nthr, W4 - 1), r, nud[j], muSr[j]);
    }
    const __amdgpu_buffer_rsrc_t Tr = table_rsrc(s.T4, (unsigned)((size_t)TW * s.TH * sizeof(float4)));
    const unsigned lastb = (unsigned)(TW - 1) * 16u;
    for (int c0 = 0; c0 <= nsamp; c0 += kS1Chunk) {   // a multiple of the slots
        const int nc = min(kS1Chunk, nsamp + 1 - c0);
        __syncthreads();
        for (int js = threadIdx.x; js < nc; js += blockDim.x) ent[js] = s1_entry<false>(s, l, y, c0 + js, nsamp, ax, s_dx);
        __syncthreads();
#pragma unroll
        for (int j = 0; j < MAXT; ++j) {
            if (j * nthr >= W4) break;
#pragma unroll 2
            for (int js = slot; js < nc; js += slots) {
                const S1Entry &en = ent[js];
                const double num = fma(nud[j], en.ti, muSr[j]);        // ri * muSi
                if (!(num >= en.thr)) continue;                        // the sun has set: no loads
                float col, a;
                sun_column<AX>(ax, sun_cell<AX>(ax, num, en.iri), col, a);
                const unsigned o0 = __float2uint_rz(col) * 16u, o1 = min(o0 + 16u, lastb);
                const float3 t00 = ld3b(Tr, en.j0 + o0, 0u), t01 = ld3b(Tr, en.j0 + o1, 0u);
                const float3 t10 = ld3b(Tr, en.j1 + o0, 0u), t11 = ld3b(Tr, en.j1 + o1, 0u);
                const float3 Ts = lerp3(lerp3(t00, t01, a), lerp3(t10, t11, a), en.p1[0]);
                const float tx = en.p0[0] * Ts.x, ty = en.p0[1] * Ts.y, tz = en.p0[2] * Ts.z;
                aR[j][0] = fmaf(tx, en.eR, aR[j][0]); aR[j][1] = fmaf(ty, en.eR, aR[j][1]); aR[j][2] = fmaf(tz, en.eR, aR[j][2]);
                aM[j][0] = fmaf(tx, en.eM, aM[j][0]); aM[j][1] = fmaf(ty, en.eM, aM[j][1]); aM[j][2] = fmaf(tz, en.eM, aM[j][2]);
            }
        }
    }
    if (slots > 1) {
        if (slot > 0) {
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                part[c][threadIdx.x - nthr] = aR[0][c];
                part[3 + c][threadIdx.x - nthr] = aM[0][c];
            }
        }
        __syncthreads();
        if (slot > 0) return;
        for (int q = 0; q + 1 < slots; ++q)
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                aR[0][c] += part[c][q * nthr + lane];
                aM[0][c] += part[3 + c][q * nthr + lane];
            }
    }
#pragma unroll
    for (int j = 0; j < MAXT; ++j) {
        const int x = lane + j * nthr;
        if (x < W4 && j * nthr < W4) s1_store(s, ((size_t)l * s.RMU + y) * W4 + x, s_dx, aR[j], aM[j]);
    }
}

// The table rows of theta row `it` of N at radius r (squared height over the ground's: rho2).
__device__ __forceinline__ void theta_taps(const SetDesc &s, double r, double rho2, double ct, ThetaRow &row) {
    const double rmu = r * ct;
    double tz, ty;
    tex4d_rmu(s, rho2, rmu, rmu * rmu - rho2, ct, tz, ty);
    int z0, z1, y0, y1;
    gl_axis_d(tz, s.RR, z0, z1, row.az);
    gl_axis_d(ty, s.RMU, y0, y1, row.ay);
    row.base = (z0 * s.RMU + y0) * s.W4;
    row.dy = (y1 - y0) * s.W4;
    row.dz = (z1 - z0) * s.RMU * s.W4;
}

// ---------------------------------------------------------------------------
// Shared staging of the spherical integrals (inscatterS, irradianceN).
//
// For a fixed r and mu_s, texture4D(table, r, cos(theta), mu_s, nu) is a
// linear interpolation in nu between RNU + 2 "slice values" (slices -1 and
// RNU are the CLAMP_TO_EDGE columns), each slice value being the trilinear
// filter of the 8 texels around (r, cos theta, mu_s).  Trilinear filtering is
// separable, so the 4D lookup of every direction (theta, phi) reduces to a
// 2-entry lerp of LDS data once those slice values are staged.
//
// Staged pairs per theta row, kk = 0..RNU, with pos = (nu+1)/2 (RNU-1) + 1,
// kk = floor(pos), f = pos - kk, A = V[kk-1], D = V[kk] - V[kk-1]:
// irradianceN stores {A, D} and looks up A + f D; inscatterS stores
// {A - kk D, D} (rounded once from FP64) and looks up fma(pos, D, A - kk D),
// the same line without the fraction.
// ---------------------------------------------------------------------------
template <int NT>
__device__ __forceinline__ void stage_slice(const SetDesc &s, const float4 *const *tabs,
                                            const ThetaRow &row, double txs, int k,
                                            float4 *out) {
    int x0, x1;
    float ax;
    const float ay = row.ay, az = row.az;
    gl_axis_d((double)k * s.RMUS + txs, s.W4, x0, x1, ax);
#pragma unroll
    for (int n = 0; n < NT; ++n) {
        const gfloat4 *tb = gptr(tabs[n]);
        const gfloat4 *t0 = tb + row.base, *t1 = t0 + row.dz;
        float3 c000 = ld3(t0 + x0), c001 = ld3(t0 + x1), c010 = ld3(t0 + row.dy + x0), c011 = ld3(t0 + row.dy + x1);
        float3 c100 = ld3(t1 + x0), c101 = ld3(t1 + x1), c110 = ld3(t1 + row.dy + x0), c111 = ld3(t1 + row.dy + x1);
        float3 v = lerp3(lerp3(lerp3(c000, c001, ax), lerp3(c010, c011, ax), ay),
                         lerp3(lerp3(c100, c101, ax), lerp3(c110, c111, ax), ay), az);
        out[n] = make_float4(v.x, v.y, v.z, 0.f);
    }
}

// ---------------------------------------------------------------------------
// Pass dJn — inscatterS.glsl:111-189.  One workgroup per (set, r layer,
// mu_s column); its RMU x RNU texels share r and mu_s, hence the staged
// slice values.  FIRST = order 2 (Rayleigh and Mie stored separately).
//
// Each thread integrates G texels of one mu row (G nu slices): they share
// the view vector v, so the phase factors of nu2 = v.w are evaluated once per
// direction for all G, and since v has no y component the directions phi and
// 2 pi - phi share them too; the thread walks the grid in such mirrored pairs
// and folds both phases and the scattering coefficients into one rgb weight
// per pair, as the reference's sum does per direction.  Per direction and
// texel the lookup position is pos = (nu1 + 1)/2 (RNU - 1) + 1 =
// posA s'.w + posB, with s' = posA s folded in per texel and the mu_s term
// folded in per theta.
//
// Bound by vector instruction issue, then by LDS reads: at 64x256x64x16 and
// 32 x 64 directions an order >= 3 takes 7.8 ms, 7.2 with the lookups' LDS reads
// left out.  On gfx950 an add, multiply or FMA of registers and literals issues
// in about 2 cycles per wave; with a scalar-register operand, and a conversion,
// floor, shift or integer multiply-add, in 4.  So the loop keeps its operands in
// vector registers and forms LDS addresses with FMAs (lds_entry): 8.6 -> 7.8 ms;
// 16x64x16x4 is bound by the latency of one wave per SIMD instead: order 2
// 130 -> 116 us, order 3 73 -> 60, and 42 and 26 us with the theta rows split.
// ---------------------------------------------------------------------------
// Entries of padding in front of the staged ground-irradiance row: texel
// coordinates down to -(0.8/1.2) SW - 0.5 (mu_s = -1) plus rounding.
__host__ __device__ __forceinline__ int e_pad(int SW) { return (2 * SW) / 3 + 3; }
// The lookup positions pos = (nu1 + 1)/2 (RNU - 1) + 1 of a direction lie in
// [1, RNU] up to FP32 rounding (|nu1| <= 1 + a few ulp); the merged ground rows
// cover [kPosLo, RNU + kPosHi].
constexpr float kPosLo = 1.0f - 1.0f / 256.0f, kPosHi = 1.0f / 256.0f;

// The staged rows are functions of a coordinate u = pos - 1/2 (ground row of
// order 2: xg - 1/2), whose rounding to an integer is the entry k = floor(pos).
// An entry holds its line's value at u = 0: with slope d through (pos = k, a),
// a - (k - 1/2) d, from FP64 and rounded once; a lookup is then fma(u, d, .).
__device__ __forceinline__ float at_zero(float a, float d, int k) {
    return (float)((double)a - ((double)k - 0.5) * (double)d);
}

struct DirJ {      // per-theta constants of the NS x 2NS grid
    float ct, st, dw, pad;
};

// CHUNK: the theta rows are staged CH at a time (when the staging of all NS
// rows exceeds the LDS budget); between chunks a thread keeps its running sums
// in the dJ table itself and resumes them, so the sum over theta runs in the
// same order, and gives the same bits, as with all rows staged at once
// (!CHUNK, CH = NS: one round, compiled without the chunk bookkeeping).
// At most 128 VGPRs (four waves per SIMD, as the LDS of a typical staging
// allows): G = 8 then keeps its direction loops free of spills (its per-group
// set-up spills a few registers) and runs 2 % faster than G = 4 at 32 x 64
// directions; at 166 VGPRs (three waves) it ran 14 % slower.
//
// SPLIT: sets with too few columns to fill the chip (16x64x16x4 has 256
// workgroups of 64 groups, one wave on a quarter of the SIMDs): the workgroup has
// DS slots of threads for its groups, each takes every DS-th theta row, and the
// slots' sums are added through LDS in slot order.
template <bool FIRST, int G, int MODE>
__global__ __launch_bounds__(MODE == kJSplit ? kJSplitThreads : 256) __attribute__((amdgpu_waves_per_eu(4))) void
k_inscatterS(const SetDesc *__restrict__ sets, const uint2 *__restrict__ tiles, int NS, int CH, int JX, int DS,
             const DirJ *__restrict__ dirT, const float2 *__restrict__ dirW) {
    constexpr bool CHUNK = MODE == kJChunk, SPLIT = MODE == kJSplit;
    constexpr int NT = FIRST ? 2 : 1;
    constexpr int PW = FIRST ? 3 : 2;      // float4 per staged pair entry
    extern __shared__ __attribute__((aligned(32))) float4 lds[];   // lds_entry: 32-byte strides
    const uint2 tl = tiles[blockIdx.x];
    const SetDesc &s = sets[tl.x];
    const int l = (int)tl.y / s.RMUS;
    const int m = (int)tl.y % s.RMUS;
    const int NU = s.RNU;
    const int NP = NU + 1;                 // pairs per theta
    const int NV = NU + 2;                 // slice values per theta
    const int EPAD = e_pad(s.SW);
    // orders >= 3: a ground row holds NP + (its E cells - 1) merged entries
    // (sky + ground terms); JX bounds the extra entries of a chunk's rows
    const int JXr = FIRST ? 0 : JX;
    const size_t npairs = (size_t)CH * NP + (size_t)JXr;
    __shared__ int s_jxmax;
    __shared__ double s_u[4];   // mu_s, 1 - mu_s^2, sqrt(1 - mu_s^2), posA
    // order 2, unchunked: the entries' three float4 as planes kJ1Plane apart
    // (16-byte stride in each: a lookup's reads spread over the LDS banks, and
    // one address serves all three with immediate offsets); otherwise whole
    constexpr bool PLANES = FIRST && !CHUNK;
    constexpr int ES = PLANES ? 1 : PW;                    // entry stride (float4)
    constexpr int CS = PLANES ? kJ1Plane : 1;              // component stride (float4)
    if (PLANES && npairs > (size_t)kJ1Plane) return;       // the host never launches this
    float4 *pairs = lds;                                   // rows of NP (+ JX) entries
    // [CH][NV][NT] slice values (the planes compute each entry's two directly)
    float4 *vtmp = pairs + (PLANES ? 2 * kJ1Plane + npairs : npairs * PW);
    // [EPAD + SW + 1][2] (order 2), 32-byte aligned
    float4 *epair = lds + (((vtmp - lds) + (PLANES ? 0 : (size_t)CH * NV * NT) + 1) & ~(size_t)1);
    float4 *gdat = epair + (FIRST ? (size_t)(EPAD + s.SW + 1) * 2 : 0);   // [CH][3]
    float *part = (float *)(gdat + 3 * CH);   // SPLIT: [DS - 1][3][threads / DS] partial sums

    const LayerGeom L = s.layers[l];
    const double r = fmin(fmax(L.r, s.Rg), s.Rt);          // inscatterS.glsl:112
    const double rho2 = r * r - s.Rg2;
    // rows and the sun's column from the tables, where there are any (k_geometry): their FP64
    // terms, 2,500 instructions of straight code, were half of a workgroup's set-up
    const ThetaRow *rowJ = s.rowJ ? s.rowJ + (size_t)l * NS : nullptr;
    double muS, txs;
    if (rowJ) {
        muS = s.sunJ[m].mus;
        txs = s.sunJ[m].txs;
    } else {
        muS = fmin(fmax(texel_mus(s, m), -1.0), 1.0);   // :114
        txs = tex4d_umus(s, muS) * s.RMUS - 0.5;
    }
    const float4 *tabs[2] = {s.dSR4, s.dSM4};
    const double posAd = 0.5 * (NU - 1), posBd = posAd + 1.0;

    // (2) order 2: row 0 of dE (irradiance at r = Rg reads only row 0 under
    // CLAMP_TO_EDGE), with EPAD copies of texel 0 in front and one of texel
    // SW-1 behind (zero differences): every texel coordinate the ground term can
    // produce, (mu_s + 0.2)/1.2 SW - 0.5 for |mu_s| <= 1, then lands on an entry
    // that reproduces the clamp, and the lookup needs no clamp instruction
    for (int k = threadIdx.x; FIRST && k < EPAD + s.SW + 1; k += blockDim.x) {
        const int k0 = min(max(k - EPAD, 0), s.SW - 1), k1 = min(max(k - EPAD + 1, 0), s.SW - 1);
        const float4 a = s.dE4[k0];
        const float4 b = s.dE4[k1];
        // the lookup at texel coordinate xg is fma(xg - 1/2, d, .) (at_zero)
        const float dx = b.x - a.x, dy = b.y - a.y, dz = b.z - a.z;
        epair[2 * k] = make_float4(at_zero(a.x, dx, k), at_zero(a.y, dy, k), at_zero(a.z, dz, k), dx);
        epair[2 * k + 1] = make_float4(dy, dz, 0.f, 0.f);
    }

    // per-layer scattering coefficients (phase constants folded in)
    const double hr = r - s.Rg;
    const float eR = rowJ ? rowJ[0].eR : (float)exp(-hr / s.HR), eM = rowJ ? rowJ[0].eM : (float)exp(-hr / s.HM);
    const float A0 = s.bR[0] * eR * s.kR, A1 = s.bR[1] * eR * s.kR, A2 = s.bR[2] * eR * s.kR;
    const float B0 = s.bMS[0] * eM * s.kM, B1 = s.bMS[1] * eM * s.kM, B2 = s.bMS[2] * eM * s.kM;
    const float iposA = (float)(1.0 / posAd), nposBi = (float)((0.5 - posBd) / posAd);   // nu1 from u
    const float g2p1 = s.g2p1, m2g = s.m2g;
    if (threadIdx.x == 0) {
        s_u[0] = muS;
        s_u[1] = fma(-muS, muS, 1.0);
        s_u[2] = sqrt(s_u[1]);
        s_u[3] = posAd;
    }
    const int ngk = (NU + G - 1) / G;
    const int ngroups = s.RMU * ngk;
    // LDS byte addresses of the staged rows
    const unsigned pairs_b = (unsigned)(size_t)(__attribute__((address_space(3))) char *)pairs;
    const float epb = lds_addend<32>((unsigned)(size_t)(__attribute__((address_space(3))) char *)epair);

    for (int c0 = 0; c0 < NS; c0 += CH) {
        const int nth = CHUNK ? min(CH, NS - c0) : NS;
        const bool last = !CHUNK || c0 + nth == NS;
        if (CHUNK && c0 > 0) __syncthreads();   // every thread is done with the previous chunk's rows
        // (1) slice values V[it][kk], kk = slice + 1
        auto slice_value = [&](int it, int kk, float4 v[NT]) {
            ThetaRow row;
            if (rowJ) row = rowJ[it];
            else theta_taps(s, r, rho2, cos((it + 0.5) * (kPI / NS)), row);
            stage_slice<NT>(s, tabs, row, txs, kk - 1, v);
            if (FIRST) {  // fold the phase-function constants in
                v[0].x *= s.kR; v[0].y *= s.kR; v[0].z *= s.kR;
                v[NT - 1].x *= s.kM; v[NT - 1].y *= s.kM; v[NT - 1].z *= s.kM;
            }
        };
        for (int e = threadIdx.x; !PLANES && e < nth * NV; e += blockDim.x) {
            float4 v[NT];
            slice_value(c0 + e / NV, e % NV, v);
    #pragma unroll
            for (int n = 0; n < NT; ++n) vtmp[(size_t)e * NT + n] = v[n];
        }
        // (3) per theta: ground visibility, ground-to-x transmittance (:129-138), and
        // the theta-uniform parts of the lookup positions
        for (int itl = threadIdx.x; itl < nth; itl += blockDim.x) {
            const int it = c0 + itl;
            const double sc = s.SW / 1.2;
            double ct, e1 = 0.0;   // e1: E texels per unit of nu1
            float dwt;
            bool ground;
            float3 tr = make_float3(0.f, 0.f, 0.f);
            if (rowJ) {
                const float4 t = s.tground[(size_t)l * NS + it];
                ct = rowJ[it].ct;
                e1 = rowJ[it].e1;
                dwt = rowJ[it].dw;
                ground = t.w != 0.0f;
                tr = f3(t);
            } else {
                ct = cos((it + 0.5) * (kPI / NS));
                dwt = (float)((kPI / NS) * (kPI / NS) * sin((it + 0.5) * (kPI / NS)));
                const double q = s.Rg / r;
                ground = ct < -sqrt(1.0 - q * q);
                if (ground) {
                    const double dg = -r * ct - sqrt(r * r * (ct * ct - 1.0) + s.Rg2);
                    const double mug = -(r * ct + dg) / s.Rg;
                    // transmittance(Rg, mug, dg) (common.glsl:272-282); its end point is x itself
                    const double r1sq = s.Rg2 + dg * dg + 2.0 * s.Rg * mug * dg;
                    const double r1 = sqrt(r1sq);
                    const double mu1 = (s.Rg * mug + dg) / r1;
                    const float h1 = (float)((r1sq - s.Rg2) / (r1 + s.Rg));
                    tr = s.tground ? ld3(gptr(s.tground) + (size_t)l * NS + it)
                       : mug > 0.0 ? T_ratio_lin(s, 0.0f, (float)mug, h1, (float)mu1)
                                   : T_ratio_lin(s, h1, (float)-mu1, 0.0f, (float)-mug);
                    e1 = dg / s.Rg * sc;
                }
            }
            float4 g0 = make_float4(0.f, 0.f, 0.f, 0.f);
            double c1 = 0.0, ce0 = 0.0;
            int jlo = 0, jhi = 0;
            if (ground) {
                const float gr = (float)(s.alpha / kPI);
                g0 = make_float4(gr * tr.x, gr * tr.y, gr * tr.z, 1.0f);
                // E texel coordinate ((r muS + dg nu1)/Rg + 0.2)/1.2 SW - 0.5 as c1 u + ce0
                const double e0 = (r * muS / s.Rg + 0.2) * sc - 0.5 + EPAD;
                c1 = e1 / posAd;
                ce0 = e0 + e1 * (0.5 - posBd) / posAd;   // xg = c1 u + ce0
                // E cells the lookups of this row can reach: positions [1, NU] up to rounding
                const float fc1 = (float)c1, fce0 = (float)ce0;
                jlo = (int)__float2uint_rz(fmaf(kPosLo - 0.5f, fc1, fce0));
                jhi = (int)__float2uint_rz(fmaf((float)NU + kPosHi - 0.5f, fc1, fce0));
                // the lookups move xg by at most c1 (RNU - 1 + 2/256) <= 2.0158 e1
                // (RNU >= 2): at most that many + 1 cells; the host sizes the rows
                // with ceil(2.05 e1) + 2 per ground row (merged_extra)
                jhi = min(jhi, jlo + (int)ceil(2.05 * e1) + 1);
            }
            gdat[3 * itl] = g0;
            // order 2's ground lookup takes xg - 1/2 (its entries' coordinate)
            gdat[3 * itl + 1] = make_float4((float)c1, (float)(FIRST ? ce0 - 0.5 : ce0), (float)(posAd * muS * ct + posBd - 0.5), dwt);
            gdat[3 * itl + 2] = make_float4(__int_as_float(jlo), __int_as_float(jhi),
                                            __int_as_float(FIRST ? NP : NP + (jhi - jlo)), 0.f);
        }
        __syncthreads();
        // first entry of every row: the sum of the entries of the rows before it
        // (a ground row needs NP + jhi - jlo), and the widest ground row
        if (threadIdx.x == 0) s_jxmax = 0;
        for (int itl = threadIdx.x; itl < nth; itl += blockDim.x) {
            int off = 0;
            for (int i = 0; i < itl; ++i) off += __float_as_int(gdat[3 * i + 2].z);
            gdat[3 * itl + 2].w = __int_as_float(off);
        }
        __syncthreads();
        if (!FIRST)
            for (int itl = threadIdx.x; itl < nth; itl += blockDim.x)
                atomicMax(&s_jxmax, __float_as_int(gdat[3 * itl + 2].z) - NP);
        // ground rows are a suffix of the chunk (ct decreases with theta): the
        // first one, found by bisection on the flags
        int ig0 = nth;
        if (!FIRST) {
            int lo = 0, hi = nth;
            while (lo < hi) {
                const int mid = (lo + hi) >> 1;
                if (gdat[3 * mid].w != 0.0f) hi = mid; else lo = mid + 1;
            }
            ig0 = lo;
        }
        auto rowoff = [&](int itl) { return __float_as_int(gdat[3 * itl + 2].w); };
        __syncthreads();   // s_jxmax
        // (4) pairs {V[kk-1], V[kk] - V[kk-1]}
        for (int e = threadIdx.x; e < nth * NP; e += blockDim.x) {
            const int it = e / NP, kk = e % NP;
            if (!FIRST && it >= ig0) continue;   // merged ground row (4b)
            float4 va[NT], vb[NT];   // V[kk-1], V[kk]
            if (PLANES) {            // computed here: no slice-value staging (LDS)
                slice_value(c0 + it, kk, va);
                slice_value(c0 + it, kk + 1, vb);
            } else {
    #pragma unroll
                for (int n = 0; n < NT; ++n) {
                    va[n] = vtmp[((size_t)it * NV + kk) * NT + n];
                    vb[n] = vtmp[((size_t)it * NV + kk + 1) * NT + n];
                }
            }
            const float4 a = va[0], b = vb[0];
            float4 *q = pairs + ((size_t)rowoff(it) + kk) * ES;
            const float dx = b.x - a.x, dy = b.y - a.y, dz = b.z - a.z;
            const float px = at_zero(a.x, dx, kk), py = at_zero(a.y, dy, kk), pz = at_zero(a.z, dz, kk);
            if (!FIRST) {
                // (P.rgb, D.r), (D.g, D.b): one 16-byte and one 8-byte LDS read
                q[0] = make_float4(px, py, pz, dx);
                q[1] = make_float4(dy, dz, 0.f, 0.f);
            } else {
                // Rayleigh and Mie pairs in 48 bytes: three 16-byte LDS reads
                const float4 am = va[NT - 1], bm = vb[NT - 1];
                const float ex = bm.x - am.x, ey = bm.y - am.y, ez = bm.z - am.z;
                q[0] = make_float4(px, py, pz, dx);
                q[CS] = make_float4(dy, dz, at_zero(am.x, ex, kk), at_zero(am.y, ey, kk));
                q[2 * CS] = make_float4(at_zero(am.z, ez, kk), ex, ey, ez);
            }
        }
        // (4b) orders >= 3, ground rows: the lookup of a ground direction is
        // S(pos) + g0 E(xg(pos)) with xg = c1 u + ce0, u = pos - 1/2, two piecewise-linear
        // functions of the same position, with knots at the integers (slices) and
        // where xg crosses an integer (E texels).  The merged row holds one entry
        // per segment between consecutive knots of either kind: the slope Q and
        // the value at u = 0 of the line through (p0, P), the segment's start, so
        // that a lookup is fma(u, Q, .).  The segment of (kk, jg) = (floor(pos), floor(xg)) is
        // entry kk + jg - jlo (each knot raises one of the two by one); segments
        // are found by intersecting every slice cell with every E cell of the row
        // (FP64), so entries of zero-length segments at coinciding knots exist too.
        if (!FIRST && ig0 < nth) {
            const int nj = s_jxmax + 1, per_row = NP * nj;
            for (int e = threadIdx.x; e < (nth - ig0) * per_row; e += blockDim.x) {
                const int itl = ig0 + e / per_row, kk = (e % per_row) / nj, jj = e % nj;
                // the whole merged row must lie inside the staging (guaranteed by
                // the host's bound; a row that would not fit is left unwritten)
                if (rowoff(itl) + __float_as_int(gdat[3 * itl + 2].z) > (int)npairs) continue;
                const float4 g0 = gdat[3 * itl], g1 = gdat[3 * itl + 1], g2 = gdat[3 * itl + 2];
                const int jlo = __float_as_int(g2.x), jhi = __float_as_int(g2.y), jg = jlo + jj;
                if (jg > jhi) continue;
                const double c1 = g1.x, ce0 = g1.y;
                double lo = kk == 0 ? (double)kPosLo : (double)kk;
                double hi = kk == NU ? (double)NU + kPosHi : kk + 1.0;
                if (c1 > 0.0) {
                    lo = fmax(lo, (jg - ce0) / c1 + 0.5);
                    hi = fmin(hi, (jg + 1 - ce0) / c1 + 0.5);
                }
                if (lo > hi) continue;
                const float4 a = vtmp[((size_t)itl * NV + kk) * NT];
                const float4 b = vtmp[((size_t)itl * NV + kk + 1) * NT];
                const float4 ea = s.dE4[min(max(jg - EPAD, 0), s.SW - 1)];
                const float4 eb = s.dE4[min(max(jg + 1 - EPAD, 0), s.SW - 1)];
                const double u = lo - kk, v = (lo - 0.5) * c1 + ce0 - jg;   // fractions at p0
                const double dx = (double)b.x - a.x, dy = (double)b.y - a.y, dz = (double)b.z - a.z;
                const double fx = (double)eb.x - ea.x, fy = (double)eb.y - ea.y, fz = (double)eb.z - ea.z;
                const double Px = a.x + u * dx + g0.x * (ea.x + v * fx);
                const double Py = a.y + u * dy + g0.y * (ea.y + v * fy);
                const double Pz = a.z + u * dz + g0.z * (ea.z + v * fz);
                const float Qx = (float)(dx + g0.x * c1 * fx), Qy = (float)(dy + g0.y * c1 * fy),
                            Qz = (float)(dz + g0.z * c1 * fz);
                // the FP32 slope's line through (p0, P), at u = 0
                float4 *q = pairs + ((size_t)rowoff(itl) + kk + jj) * PW;
                const double l0 = lo - 0.5;
                q[0] = make_float4((float)(Px - l0 * Qx), (float)(Py - l0 * Qy), (float)(Pz - l0 * Qz), Qx);
                q[1] = make_float4(Qy, Qz, 0.f, 0.f);
            }
        }
        __syncthreads();

        // SPLIT: the threads are DS slots of gpi threads (whole waves); slot ds takes
        // the theta rows ds, ds + DS, ... of the groups of all slots
        const int gpi = SPLIT ? (int)blockDim.x / DS : (int)blockDim.x;
        const int ds = SPLIT ? __builtin_amdgcn_readfirstlane((int)threadIdx.x / gpi) : 0;
        const int gt = (int)threadIdx.x - ds * gpi;
        for (int base = 0; base < ngroups; base += gpi) {
            if (!SPLIT && base + gt >= ngroups) break;
            const int grp = SPLIT ? min(base + gt, ngroups - 1) : base + gt;
            const int y = grp % s.RMU, kb = (grp / s.RMU) * G;
            // the G texels' set-up (inscatterS.glsl:113-122, FP64); products rounded
            // on their own and explicit fma: every G gives the same bits.  Its uniform
            // terms are read from LDS by each group, so that no FP64 value takes a
            // register over the direction loop.
            float vx, vz, sxp[G], syp[G];
            {
                asm volatile("" ::: "memory");
                const volatile double *us = s_u;
                const double uS = us[0], uq = us[1], ur = us[2], up = us[3];
                double mu, muS_t, nu0;
                mu_mus_nu(s, s.layers[l], kb * s.RMUS + m, y, mu, muS_t, nu0);
                mu = fmin(fmax(mu, -1.0), 1.0);
                const double vxd = sqrt(fma(-mu, mu, 1.0)), var = __dmul_rn(vxd, ur), mm = __dmul_rn(uS, mu);
                vx = (float)vxd;
                vz = (float)mu;
    #pragma unroll
                for (int g = 0; g < G; ++g) {
                    const int k = min(kb + g, NU - 1);
                    double nu = -1.0 + (double)k / (s.RNU - 1.0) * 2.0;
                    nu = fmin(fmax(nu, mm - var), mm + var);
                    const double sxd = vxd == 0.0 ? 0.0 : (nu - mm) / vxd;
                    const double syd = sqrt(fmax(0.0, fma(-sxd, sxd, uq)));
                    sxp[g] = (float)(up * sxd);
                    syp[g] = (float)(up * syd);
                }
            }
            const float cx1 = m2g * vx;
            int vzero;
            asm("v_mov_b32 %0, 0" : "=v"(vzero));
            float acc[G][3];
    #pragma unroll
            for (int g = 0; g < G; ++g)
    #pragma unroll
                for (int c = 0; c < 3; ++c) acc[g][c] = 0.f;
            if (CHUNK && c0 > 0) {   // resume the sums of the previous chunks (written by this thread)
    #pragma unroll
                for (int g = 0; g < G; ++g) {
                    const int k = kb + g;
                    if (k < NU) {
                        const size_t o = ((size_t)l * s.RMU + y) * s.W4 + (size_t)k * s.RMUS + m;
                        if (s.dJb == 12) {
                            const float *q = (const float *)s.dJ4 + 3 * o;
                            acc[g][0] = q[0]; acc[g][1] = q[1]; acc[g][2] = q[2];
                        } else {
                            const float4 q = s.dJ4[o];
                            acc[g][0] = q.x; acc[g][1] = q.y; acc[g][2] = q.z;
                        }
                    }
                }
            }

            // 4D lookup of one direction from the staged pairs: the clamp of the
            // nu slice is implicit, |s.w| <= 1 keeps pos in [1, RNU] (+ rounding)
            // and the entry in [0, RNU] = the staged pair range.
            // (order 2: the Rayleigh and Mie values weighted by the phase functions of
            // nu1 = s.w, as q1 (R + z1 M) with q1 = 1 + nu1^2, z1 = (1+g^2-2g nu1)^-3/2;
            // the caller applies q1, whose per-set constants are folded into the staging)
            // Orders >= 3, ground direction: the merged sky + ground entry of the
            // segment holding pos (4b).  floor(xg) is exact (v_floor): the row's cells
            // are those of its floor, so a tie has to go up.
            struct Tap {
                float u;
                float4 a, b, c;   // orders >= 3: a, b.xy
            };
            auto fetch = [&](auto gr, float pt, unsigned pi, float gb, float cg1, float cg0, float u) {
                Tap t;
                t.u = u;
                unsigned pp;
                if constexpr (!FIRST && decltype(gr)::value) {
                    const float fg = floorf(fmaf(u, cg1, cg0));   // >= 0: EPAD is folded into cg0
                    pp = __float_as_uint(fmaf(fg, 32.0f * 1.40129846e-45f, fmaf(u + kRound, 32.0f * 1.40129846e-45f, gb)));
                } else if constexpr (ES == 3) {   // 48-byte entries: the addend has no exact FP32 form
                    pp = pi + __umul24(__float2uint_rz(u + 0.5f), 48u);
                } else {
                    pp = lds_entry<16 * ES>(u, pt);
                }
                t.a = lds4(pp);
                if (FIRST) {
                    t.b = lds4(pp, 16 * CS);
                    t.c = lds4(pp, 32 * CS);
                } else {
                    const float2 d = lds2(pp, 16);
                    t.b.x = d.x;
                    t.b.y = d.y;
                }
                return t;
            };
            auto value = [&](const Tap &t, float out[3], float &q1) {
                const float u = t.u;
                if (!FIRST) {
                    out[0] = fmaf(u, t.a.w, t.a.x);
                    out[1] = fmaf(u, t.b.x, t.a.y);
                    out[2] = fmaf(u, t.b.y, t.a.z);
                    q1 = 1.0f;
                } else {
                    const float nu1 = fmaf(u, iposA, nposBi);
                    q1 = fmaf(nu1, nu1, 1.0f);
                    const float y1 = __builtin_amdgcn_rsqf(fmaf(m2g, nu1, g2p1));
                    const float z1 = y1 * y1 * y1;
                    const float m0 = fmaf(u, t.c.y, t.b.z), m1 = fmaf(u, t.c.z, t.b.w), m2 = fmaf(u, t.c.w, t.c.x);
                    out[0] = fmaf(m0, z1, fmaf(u, t.a.w, t.a.x));
                    out[1] = fmaf(m1, z1, fmaf(u, t.b.x, t.a.y));
                    out[2] = fmaf(m2, z1, fmaf(u, t.b.y, t.a.z));
                }
            };
            // irradiance at the ground point seen in direction w, row 0 of dE
            auto ground_e = [&](float u, float cg1, float cg0, float out[3]) {
                const float xg = fmaf(u, cg1, cg0);   // texel coordinate - 1/2
                const unsigned pe = lds_entry<32>(xg, epb);
                const float4 ea = lds4(pe);
                const float2 ed = lds2(pe, 16);
                out[0] = fmaf(xg, ea.w, ea.x);
                out[1] = fmaf(xg, ed.x, ea.y);
                out[2] = fmaf(xg, ed.y, ea.z);
            };

            for (int itl = SPLIT ? ds : 0; itl < nth; itl += SPLIT ? DS : 1) {
                const int it = c0 + itl;
                const float ct = dirT[it].ct;
                const float4 g0 = gdat[3 * itl], g1 = gdat[3 * itl + 1];
                const bool ground = g0.w != 0.0f;
                const float vzwz = vz * ct;
                const float cx0 = fmaf(m2g, vzwz, g2p1);
                const float dw = g1.w, cp = g1.z;
                const unsigned pi = pairs_b + (unsigned)rowoff(itl) * 16 * ES;
                const float pt = lds_addend<16 * ES>(pi);
                // merged ground row: entry (floor(pos) + floor(xg)) - jlo (the exact
                // sum of the two products is base + 32 (k + floor(xg) - jlo))
                const float gbase = ((float)(int)(pairs_b + 32 * (rowoff(itl) - __float_as_int(gdat[3 * itl + 2].x))) -
                                     32.0f * kRound) * 1.40129846e-45f;
                // through a vector address: in a scalar register, w would halve the
                // rate of every FMA that takes it
                const float2 *wrow = dirW + (size_t)it * 2 * NS + vzero;
                // the directions of one theta row; GR: a merged ground row of orders
                // >= 3 (a compile-time branch, so the lookups of all G texels stay
                // one straight sequence)
                auto phi_row = [&](auto gr) {
                    float2 wn = wrow[0];
                    // Orders >= 3: the lookups of texel g + 1 are read while texel g's are
                    // used; without the second set in flight four waves per SIMD do not
                    // cover the LDS (8.6 against 7.9 ms per order, G = 8, 64x256x64x16).
                    constexpr int AHEAD = FIRST ? 0 : 1;   // (order 2 has no registers for it)
                    Tap ta[2], tb[2];
                    auto fetch_pair = [&](int g, float2 w) {
                        const float base = fmaf(sxp[g], w.x, cp);
                        ta[g & 1] = fetch(gr, pt, pi, gbase, g1.x, g1.y, fmaf(syp[g], w.y, base));
                        tb[g & 1] = fetch(gr, pt, pi, gbase, g1.x, g1.y, fmaf(-syp[g], w.y, base));
                    };
                    // directions phi and 2 pi - phi together: same w.x, opposite w.y,
                    // hence the same nu2 = v.w (v has no y component) and weights
                    for (int ip = 0; ip < NS; ++ip) {
                        const float2 w = wn;
                        if (ip + 1 < NS) wn = wrow[ip + 1];  // prefetch of the next direction
                        if (AHEAD) fetch_pair(0, w);
                        const float nu2 = fmaf(vx, w.x, vzwz);
                        const float q2 = fmaf(nu2 * dw, nu2, dw);
                        const float y2 = __builtin_amdgcn_rsqf(fmaf(cx1, w.x, cx0));
                        const float t2 = q2 * (y2 * y2 * y2);
                        // betaR e^(-h/HR) pR(nu2) dw + betaMSca e^(-h/HM) pM(nu2) dw (:182-185)
                        const float W0 = fmaf(A0, q2, B0 * t2), W1 = fmaf(A1, q2, B1 * t2),
                                    W2 = fmaf(A2, q2, B2 * t2);
    #pragma unroll
                        for (int g = 0; g < G; ++g) {
                            if (g + AHEAD < G) fetch_pair(g + AHEAD, w);
                            if (AHEAD) __builtin_amdgcn_sched_barrier(0);
                            const Tap &a = ta[g & 1], &b = tb[g & 1];
                            float la[3], lb[3], lv[3], qa, qb;
                            value(a, la, qa);
                            value(b, lb, qb);
                            if (FIRST) {
    #pragma unroll
                                for (int c = 0; c < 3; ++c) lv[c] = fmaf(qa, la[c], qb * lb[c]);
                            } else {
    #pragma unroll
                                for (int c = 0; c < 3; ++c) lv[c] = la[c] + lb[c];
                            }
                            if (FIRST && ground) {   // order 2: the separate ground term (uniform branch)
                                float ea[3], eb[3];
                                ground_e(a.u, g1.x, g1.y, ea);
                                ground_e(b.u, g1.x, g1.y, eb);
                                lv[0] = fmaf(g0.x, ea[0] + eb[0], lv[0]);
                                lv[1] = fmaf(g0.y, ea[1] + eb[1], lv[1]);
                                lv[2] = fmaf(g0.z, ea[2] + eb[2], lv[2]);
                            }
                            acc[g][0] = fmaf(lv[0], W0, acc[g][0]);
                            acc[g][1] = fmaf(lv[1], W1, acc[g][1]);
                            acc[g][2] = fmaf(lv[2], W2, acc[g][2]);
                        }
                    }
                };
                if (!FIRST && ground) phi_row(std::true_type{});
                else phi_row(std::false_type{});
            }
            if (SPLIT) {   // the slots' sums, added in slot order
    #pragma unroll
                for (int g = 0; g < G; ++g) {
                    float *q = part + ((ds - 1) * 3) * gpi + gt;
                    if (ds > 0) {
                        q[0] = acc[g][0]; q[gpi] = acc[g][1]; q[2 * gpi] = acc[g][2];
                    }
                    __syncthreads();
                    for (int j = 0; ds == 0 && j < 3 * (DS - 1); j += 3) {
                        acc[g][0] += part[j * gpi + gt];
                        acc[g][1] += part[(j + 1) * gpi + gt];
                        acc[g][2] += part[(j + 2) * gpi + gt];
                    }
                    __syncthreads();
                }
                if (ds > 0 || base + gt >= ngroups) continue;
            }
    #pragma unroll
            for (int g = 0; g < G; ++g) {
                const int k = kb + g;
                if (k < NU) {
                    const size_t o = ((size_t)l * s.RMU + y) * s.W4 + (size_t)k * s.RMUS + m;
                    if (!FIRST && last) {
                        // dJ is a sum of non-negative terms; a merged ground entry
                        // (FP32 P and Q) can undershoot a zero value by rounding
                        acc[g][0] = fmaxf(acc[g][0], 0.f); acc[g][1] = fmaxf(acc[g][1], 0.f);
                        acc[g][2] = fmaxf(acc[g][2], 0.f);
                    }
                    if (s.hs && last) {
                        acc[g][0] = q16(acc[g][0]); acc[g][1] = q16(acc[g][1]); acc[g][2] = q16(acc[g][2]);
                    }
                    if (s.dJb == 12) {
                        float *q = (float *)s.dJ4 + 3 * o;
                        q[0] = acc[g][0]; q[1] = acc[g][1]; q[2] = acc[g][2];
                    } else {
                        s.dJ4[o] = make_float4(acc[g][0], acc[g][1], acc[g][2], 0.f);
                    }
                }
            }
        }
        if (!CHUNK) break;
    }
}

// ---------------------------------------------------------------------------
// Pass dEn — irradianceN.glsl:85-114, fused with copyIrradiance k = 1 and its
// ADD blend (PreprocessAtmo.cpp:335-341).  One workgroup per E texel.
// ---------------------------------------------------------------------------
struct DirE {      // per-direction constants of the hemisphere grid
    float wx, wz, wzdw, pad;
};

// The NI/2 theta rows are staged CH at a time (CH = NI/2 unless they exceed
// the LDS budget).
template <bool FIRST>
__global__ __launch_bounds__(256) void k_irradianceN(const SetDesc *__restrict__ sets,
                                                     const uint2 *__restrict__ tiles, int NI, int CH,
                                                     const DirE *__restrict__ dirs) {
    constexpr int NT = FIRST ? 2 : 1;
    extern __shared__ float4 lds[];
    const uint2 tl = tiles[blockIdx.x];
    const SetDesc &s = sets[tl.x];
    const int t = (int)tl.y;
    const int i = t % s.SW, j = t / s.SW;
    const int NU = s.RNU, NP = NU + 1, NV = NU + 2;
    const int NTH = NI / 2;
    float4 *pairs = lds;                                   // [CH][NP][NT][2]
    float4 *vtmp = pairs + (size_t)CH * NP * NT * 2;       // [CH][NV][NT]
    float *red = (float *)(vtmp + (size_t)CH * NV * NT);   // [3][blockDim/64]

    const double h = (double)j / (s.SH - 1.0) * (s.Rt - s.Rg);
    const double r = s.Rg + h;
    const double muS = -0.2 + (double)i / (s.SW - 1.0) * (1.0 + 0.2);
    const double rho2 = h * (2.0 * s.Rg + h);
    const ThetaRow *rowE = s.rowE ? s.rowE + (size_t)j * NTH : nullptr;
    const double txs = rowE ? s.sunE[i].txs : tex4d_umus(s, muS) * s.RMUS - 0.5;
    const float4 *tabs[2] = {s.dSR4, s.dSM4};
    const float sx = (float)sqrt(fmax(1.0 - muS * muS, 0.0)), sz = (float)muS;
    const float posA = 0.5f * (NU - 1), posB = 0.5f * (NU - 1) + 1.0f;
    float a0 = 0.f, a1 = 0.f, a2 = 0.f;
    for (int c0 = 0; c0 < NTH; c0 += CH) {
        const int nth = min(CH, NTH - c0);
        if (c0 > 0) __syncthreads();   // every thread is done with the previous chunk's rows
        for (int e = threadIdx.x; e < nth * NV; e += blockDim.x) {
            const int it = c0 + e / NV, kk = e % NV;
            ThetaRow row;
            if (rowE) row = rowE[it];
            else theta_taps(s, r, rho2, cos((it + 0.5) * (kPI / NI)), row);
            float4 v[NT];
            stage_slice<NT>(s, tabs, row, txs, kk - 1, v);
            if (FIRST) {
                v[0].x *= s.kR; v[0].y *= s.kR; v[0].z *= s.kR;
                v[NT - 1].x *= s.kM; v[NT - 1].y *= s.kM; v[NT - 1].z *= s.kM;
            }
    #pragma unroll
            for (int n = 0; n < NT; ++n) vtmp[(size_t)e * NT + n] = v[n];
        }
        __syncthreads();
        for (int e = threadIdx.x; e < nth * NP * NT; e += blockDim.x) {
            const int n = e % NT, ek = e / NT;
            const int it = ek / NP, kk = ek % NP;
            float4 a = vtmp[((size_t)it * NV + kk) * NT + n];
            float4 b = vtmp[((size_t)it * NV + kk + 1) * NT + n];
            pairs[((size_t)(it * NP + kk) * NT + n) * 2] = a;
            pairs[((size_t)(it * NP + kk) * NT + n) * 2 + 1] =
                make_float4(b.x - a.x, b.y - a.y, b.z - a.z, 0.f);
        }
        __syncthreads();

        // directions d = phi * NTH + theta of this chunk's theta rows
        const int ndir = 2 * NI * nth;
        for (int dl = threadIdx.x; dl < ndir; dl += blockDim.x) {
            const int it = dl % nth;   // staged row
            const DirE w = dirs[(dl / nth) * NTH + c0 + it];
            const float nu = fmaf(sx, w.wx, sz * w.wz);
            float pos = fmaf(nu, posA, posB);
            float fl = floorf(pos);
            float f = pos - fl;
            int kk = min(max((int)fl, 0), NU);
            const float4 *pp = pairs + ((size_t)it * NP + kk) * NT * 2;
            float4 a = pp[0], dd = pp[1];
            float l0 = fmaf(f, dd.x, a.x), l1 = fmaf(f, dd.y, a.y), l2 = fmaf(f, dd.z, a.z);
            if (FIRST) {
                float4 am = pp[2], dm = pp[3];
                float m0 = fmaf(f, dm.x, am.x), m1 = fmaf(f, dm.y, am.y), m2 = fmaf(f, dm.z, am.z);
                const float q1 = fmaf(nu, nu, 1.0f);
                const float y1 = rsqrtf(fmaf(s.m2g, nu, s.g2p1));
                const float t1 = q1 * (y1 * y1 * y1);
                l0 = fmaf(l0, q1, m0 * t1);
                l1 = fmaf(l1, q1, m1 * t1);
                l2 = fmaf(l2, q1, m2 * t1);
            }
            a0 = fmaf(l0, w.wzdw, a0);
            a1 = fmaf(l1, w.wzdw, a1);
            a2 = fmaf(l2, w.wzdw, a2);
        }
    }
    // block reduction
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        a0 += __shfl_xor(a0, off, 64);
        a1 += __shfl_xor(a1, off, 64);
        a2 += __shfl_xor(a2, off, 64);
    }
    const int nw = blockDim.x >> 6, wv = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        red[wv] = a0;
        red[nw + wv] = a1;
        red[2 * nw + wv] = a2;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        float s0 = 0.f, s1 = 0.f, s2 = 0.f;
        for (int w = 0; w < nw; ++w) {
            s0 += red[w];
            s1 += red[nw + w];
            s2 += red[2 * nw + w];
        }
        if (s.hs) {   // dE stored as FP16, then the FP16 ADD blend E = FP16(E + dE)
            s0 = q16(s0); s1 = q16(s1); s2 = q16(s2);
        }
        s.dE4[t] = make_float4(s0, s1, s2, 1.0f);
        if (s.E4) {
            float4 e = s.E4[t];
            e.x += s0; e.y += s1; e.z += s2;
            e = q16(e, s.hs);
            s.E4[t] = e;
            if (s.outE) {
                s.outE[3 * t + 0] = e.x;
                s.outE[3 * t + 1] = e.y;
                s.outE[3 * t + 2] = e.z;
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Pass dSn — inscatterN.glsl:105-131 fused with copyInscatterN.glsl:105-110 +
// ADD blend (S.rgb += dS / phaseR(nu)).
//
// The view ray (r, mu) of a texel depends only on its layer and mu row, so
// every quantity of an integration sample that does not involve the sun
// (sample radius and zenith cosine, the texture4D r and mu coordinates and
// filter weights, the transmittance T(r, mu, t)) is shared by the
// RNU x RMU_S texels of the row, which one workgroup covers: k_snview computes
// those per-sample terms once per precompute (FP64 geometry), and each thread
// integrates its texels with only the mu_s-dependent work.
// ---------------------------------------------------------------------------
// Sample i of the view ray of mu row y, layer l (FP64 geometry).
__device__ __forceinline__ SnView sn_view(const SetDesc &s, const LayerGeom &L, int y, int i, int nsamp,
                                          double &mu, double &h1, double &mu1, float &tr) {
    const double r = L.r, rho2 = r * r - s.Rg2;
    double muS_u, nu_u;
    mu_mus_nu(s, L, 0, y, mu, muS_u, nu_u);
    const double rmu = r * mu;
    const double delta = rmu * rmu - rho2;            // constant along the ray
    const double dx = limit_d(s, r, mu) / nsamp;
    const double ti = i * dx;
    const double q = rho2 + ti * (ti + 2.0 * rmu);    // ri^2 - Rg^2
    const double rmui = rmu + ti;                     // ri * mui
    const double ri = sqrt(q + s.Rg2);
    const double rho = sqrt(fmax(q, 0.0));
    double f, c;
    if (rmui < 0.0 && delta > 0.0) {
        f = -rho / (sqrt(delta) - rmui);
        c = 0.5 - 0.5 / s.RMU;
    } else {
        f = (sqrt(fmax(delta + s.H * s.H, 0.0)) - rmui) / (rho + s.H);
        c = 0.5 + 0.5 / s.RMU;
    }
    const double ty = s.lin4 ? (0.5 / s.RMU + (rmui / ri + 1.0) / 2.0 * (1.0 - 1.0 / s.RMU)) * s.RMU - 0.5
                             : (c + f * (0.5 - 1.0 / s.RMU)) * s.RMU - 0.5;
    const double tz = rho / s.H * (s.RR - 1.0);
    int z0, z1, y0, y1;
    float az, ay;
    gl_axis_d(tz, s.RR, z0, z1, az);
    gl_axis_d(ty, s.RMU, y0, y1, ay);
    h1 = q / (ri + s.Rg);
    mu1 = rmui / ri;
    tr = (float)(ti / ri);
    SnView v;
    const bool dy = y1 != y0, dz = z1 != z0, oy = y0 & 1, oz = z0 & 1;
    // weights of the odd ones; at an edge both taps are the same row, whose name takes it all
    v.ay = dy ? (oy ? 1.f - ay : ay) : (oy ? 1.f : 0.f);
    v.az = dz ? (oz ? 1.f - az : az) : (oz ? 1.f : 0.f);
    v.row = 8 * (z0 * s.RMU + y0) + (dy ? 1 : 0) + (dz ? 2 : 0) + (oz ? 4 : 0);
    v.dr = i == 0 ? (float)dx : (float)((ri - r) / ri);
    return v;
}
// Row indices (layer RMU + mu row) of a sample: x even layer, even mu row; y even,
// odd; z odd, even; w odd, odd.  (RMU is even, so an index has its mu row's parity.)
__device__ __forceinline__ int4 sn_rows4(int RMU, int row) {
    const int p = row >> 3, oy = p & 1, dy = row & 1, dz = (row & 2) ? RMU : 0;
    const int ye = oy ? dy : 0, yo = oy ? 0 : dy;                     // from p to the even / odd mu row
    const int ze = (row & 4) ? dz : 0, zo = (row & 4) ? 0 : dz;       // from p to the even / odd layer
    return make_int4(p + ze + ye, p + ze + yo, p + zo + ye, p + zo + yo);
}
// Blend weights of the 4 rows in the order of sn_rows4.
__device__ __forceinline__ float4 sn_weights(float az, float ay) {
    return make_float4((1.f - az) * (1.f - ay), (1.f - az) * ay, az * (1.f - ay), az * ay);
}

// The (r, mu) blend of one table column x: sum_q w_q dJ[row_q][x], in one fixed
// FP32 order.  Both forms of k_inscatterN (direct gathers, LDS-staged rows)
// blend with this, then lerp two columns in x as fma(ax, b1 - b0, b0), so
// they give the same bits.
__device__ __forceinline__ float3 sn_blend(const float4 &w, float3 t0, float3 t1, float3 t2, float3 t3) {
    return make_float3(fmaf(w.w, t3.x, fmaf(w.z, t2.x, fmaf(w.y, t1.x, w.x * t0.x))),
                       fmaf(w.w, t3.y, fmaf(w.z, t2.y, fmaf(w.y, t1.y, w.x * t0.y))),
                       fmaf(w.w, t3.z, fmaf(w.z, t2.z, fmaf(w.y, t1.z, w.x * t0.z))));
}
__device__ __forceinline__ float3 sn_lerp(float ax, float3 b0, float3 b1) {
    return make_float3(fmaf(ax, b1.x - b0.x, b0.x), fmaf(ax, b1.y - b0.y, b0.y), fmaf(ax, b1.z - b0.z, b0.z));
}

// Texel offset of the sample's mu_s_i = (nu t + mu_s r) / r_i inside a nu
// slice (texture4D's uMuS * RMUS - 0.5), evaluated relative to the texel's own
// mu_s.  Near the start of a long, nearly horizontal ray mu_s_i moves away from
// mu_s by 1e-5 and less per sample, and where a thin layer's dJ rises steeply
// out of the shadow between two mu_s columns the lookup is proportional to
// that move: an FP32 mu_s_i (~2e-8 absolute) put through the coordinate
// formula (whose + 0.74, resp. + 0.2, cancels at the low end) would give it
// only to a few 1e-3.  So:
//   linear (:165): offset proportional to mu_s_i + 0.2 =
//     nu t / r_i - mu_s (r_i - r) / r_i + (mu_s + 0.2);
//   non-linear (:161), txb = the texel's own offset (FP64): with
//     d = max(mu_s_i, -0.1975) - mu_b, mu_b = max(mu_s, -0.1975), and
//     mu_s_i - mu_s = (nu t - mu_s (r_i - r)) / r_i,
//     offset = txb + C atan(k d / (1 + k mu_b k (mu_b + d))), k = tan(1.386),
//     C = 0.5 (RMUS - 1) / 1.1 (atan a - atan b = atan((a - b) / (1 + a b)),
//     used while |k d| < 0.5, where the argument is below 0.5334); larger moves
//     take the reference's form, which has no cancellation there.
// The per-column terms, k folded in (ColGeom), leave two FMAs for k d; the near
// arctangent is its own odd polynomial (weighted least-squares fit of
// (atan(x)/x - 1)/x^2 on |x| <= 0.534, 7.2e-8 relative in FP32 arithmetic) and
// the far form is entered only by waves in which a lane needs it: 19 VALU
// slots instead of 36 for a wave of near moves.  A lane's value does not depend
// on its wave's vote.
struct SnTexel {
    float nu;    // k nu (linear: nu)
    ColGeom c;
};
template <bool LIN4>
__device__ __forceinline__ float sn_txs(const SetDesc &s, const SnTexel &x, float tr, float dr) {
    const float half = 0.5f * (float)(s.RMUS - 1);
    // every sum of products is an explicit fmaf, so that the inlined copies of
    // the kernel's forms agree bit for bit
    if (LIN4) return fmaxf(fmaf(x.nu, tr, fmaf(-x.c.mus, dr, x.c.txb)), 0.0f) * (1.0f / 1.2f) * (2.0f * half);
    const float c = half * (1.0f / 1.1f);
    const float kd = fmaxf(fmaf(x.nu, tr, fmaf(-x.c.mus, dr, x.c.ck)), x.c.lo);
    const bool near = fabsf(kd) < 0.5f;
    const float a = kd * __builtin_amdgcn_rcpf(fmaf(x.c.kb, kd, x.c.kb2));
    const float z = a * a;
    float p = fmaf(z, -0.04780794680118561f, 0.09955135732889175f);
    p = fmaf(z, p, -0.14134405553340912f);
    p = fmaf(z, p, 0.19991108775138855f);
    p = fmaf(z, p, -0.3333316147327423f);
    float o = fmaf(c, fmaf(a, z * p, a), x.c.txb);
    if (!__all(near)) {
        const float far = fmaf(c, atanf(x.c.kb + kd), 0.74f * half);
        o = near ? o : far;
    }
    return o;
}

// Waves per SIMD the register budget of a k_inscatterN instantiation is cut to:
// the most that need no spill (40, 70 and 108 VGPRs).  A spill in the sample loop
// costs more than any number of waves gives: 3 texels per thread with 9 registers
// spilled at five waves took 13.1 ms per order for the 48-set mixed batch,
// without them at four 8.9 ms.
// Form 2, whose FP64 terms need about 100 VGPRs, runs at four.
constexpr int sn_waves(int form, int NM) { return form == 2 ? 4 : NM == 1 ? 8 : NM == 2 ? 6 : 4; }

// One mu row of RNU*RMU_S texels per workgroup, NM texels per thread.  FORM:
//   0  each texel gathers its 8 taps per sample from dJ directly (global loads);
//   1  per sample the workgroup first blends the 4 (r, mu) table rows around it
//      into one row B[x] = sum_q w_q dJ[row_q][x] in LDS (coalesced loads), then
//      each texel reads two neighbours of B and lerps in x;
//   2  as 1, without SetDesc::view: the workgroup computes the samples' terms
//      into LDS itself, 64 at a time.
// The direct form blends the two columns it needs in the same order (sn_blend,
// sn_lerp), so all forms give the same bits.  The staged row is double-buffered:
// a sample's rows are loaded during the lookups of the one before it, and there
// is one barrier per sample.  A row that the sample before it had too (the same
// layer and mu row, kept in registers under the parities of both) is not loaded
// again: 1.6 of 4 rows per sample are loaded at 32x128x32x8, 2.6 at
// 64x256x64x16.  The samples' terms are workgroup-uniform, in scalar registers.
//
// What it measured per order, before (several rows per workgroup, samples' terms
// computed by each workgroup in every order, 4 row loads and two barriers per
// sample, 77 VALU slots per texel-sample) and now (about 50): 32x128x32x8 170 ->
// 99 us, 64x256x64x16 2.21 -> 1.51 ms, the 48-set mixed batch 16.2 -> 8.5 ms.  It
// is held by its VALU (about 70 %) and the row loads between them.
template <int FORM, bool LIN4, int NM>   // LIN4: linear inscatter parameterisation (per-sample mu_s)
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(sn_waves(FORM, NM))))
void k_inscatterN(const SetDesc *__restrict__ sets, const uint2 *__restrict__ tiles, int nsamp) {
    struct Entry {
        SnView v;
        float4 tw;   // T(r, mu, t) * trapezoid weight (rgb), t / r_i
    };
    __shared__ Entry ent[FORM == 2 ? kNChunk : 1];
    extern __shared__ float4 blend[];   // [2][W4 + 1]
    const uint2 tl = tiles[blockIdx.x];
    const SetDesc &s = sets[tl.x];
    const int l = (int)tl.y / s.RMU, y = (int)tl.y % s.RMU;
    const int nthr = blockDim.x, W4 = s.W4;
    float acc[NM][3];
    SnTexel tx[NM];
    unsigned kbase[NM];   // first column of the texel's nu slice
    // nu = -1 + 2 k / (RNU - 1) is on slice k of the table, so the nu lerp of
    // texture4D has weight 0 and a lookup reads slice k only
    auto texel_nu = [&](int x) { return -1.0 + (double)(x / s.RMUS) / (s.RNU - 1.0) * 2.0; };
#pragma unroll
    for (int j = 0; j < NM; ++j) {
        acc[j][0] = acc[j][1] = acc[j][2] = 0.f;
        const int x = min((int)threadIdx.x + j * nthr, W4 - 1);   // past the row's end: nothing is stored
        kbase[j] = (unsigned)(x / s.RMUS * s.RMUS);
        tx[j].nu = (float)(LIN4 ? texel_nu(x) : (double)s.f_tMuS * texel_nu(x));
        tx[j].c = s.cols[x % s.RMUS];
    }
    // the dJ table as a buffer (< 2^31 bytes: at most 2^27 texels of 16 bytes)
    const __amdgpu_buffer_rsrc_t Jr = table_rsrc(s.dJ4, (unsigned)((size_t)s.n4 * s.dJb));
    const unsigned jb = (unsigned)s.dJb, rowb = (unsigned)W4 * jb;   // bytes per dJ texel and row

    // sample i, as uniform values
    typedef __attribute__((address_space(4))) const SnView cview;
    typedef __attribute__((address_space(4))) const F4 cf4;
    const size_t v0 = ((size_t)l * s.RMU + y) * (nsamp + 1);
    const cview *gv = (const cview *)(s.view + v0);
    const cf4 *gt = (const cf4 *)(s.tview + v0);
    int c0 = 0;
    float dx = 0.f;   // the row's trapezoid step
    auto get = [&](int i) {
        Entry e;
        if constexpr (FORM == 2) {
            const Entry &q = ent[i - c0];
            auto u = [](float f) { return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(f))); };
            e.v.az = u(q.v.az); e.v.ay = u(q.v.ay); e.v.dr = u(q.v.dr);
            e.v.row = __builtin_amdgcn_readfirstlane(q.v.row);
            e.tw = make_float4(u(q.tw.x), u(q.tw.y), u(q.tw.z), u(q.tw.w));
        } else {
            e.v.az = gv[i].az; e.v.ay = gv[i].ay; e.v.row = gv[i].row; e.v.dr = gv[i].dr;
            e.tw = make_float4(gt[i].x, gt[i].y, gt[i].z, gt[i].w);
        }
        if (i == 0) {
            dx = e.v.dr;
            e.v.dr = 0.f;
        }
        return e;
    };
    auto stage = [&](int c) {   // FORM 2: the terms of samples c .. c + 63
        c0 = c;
        __syncthreads();
        for (int js = threadIdx.x; js < min(kNChunk, nsamp + 1 - c); js += nthr) {
            const int i = c + js;
            const LayerGeom &L = s.layers[l];
            double mu, h1, mu1;
            float tr;
            Entry en;
            en.v = sn_view(s, L, y, i, nsamp, mu, h1, mu1, tr);
            if (s.tview) {
                en.tw = s.tview[v0 + i];
            } else {   // transmittance(r, mu, ti) (common.glsl:272-282)
                const float hl = (float)(L.r - s.Rg), wt = (i == 0 || i == nsamp) ? 0.5f : 1.0f;
                const float3 T = mu > 0.0 ? T_ratio_lin(s, hl, (float)mu, (float)h1, (float)mu1)
                                          : T_ratio_lin(s, (float)h1, (float)-mu1, hl, (float)-mu);
                en.tw = make_float4(T.x * wt, T.y * wt, T.z * wt, tr);
            }
            ent[js] = en;
        }
        __syncthreads();
    };
    // A lookup's texel column is kbase + txs, txs the offset inside the slice,
    // kept apart so that the fraction ax has full FP32 precision.  txs runs past
    // RMU_S - 1 into the next slice when mu_s_i > 1 (as GL's coordinate does);
    // only the row's last column clamps (CLAMP_TO_EDGE): at txs = W4 - 1 - kbase
    // the fraction is 0 and the second tap is the padding column W4, a copy of
    // the last.
    if constexpr (FORM == 0) {
#pragma unroll
        for (int j = 0; j < NM; ++j) {
            const unsigned last = (unsigned)W4 - 1 - kbase[j];
            for (int i = 0; i <= nsamp; ++i) {
                const Entry en = get(i);
                const float4 w = sn_weights(en.v.az, en.v.ay);
                const int4 rows = sn_rows4(s.RMU, en.v.row);
                const float txs = __builtin_amdgcn_fmed3f(sn_txs<LIN4>(s, tx[j], en.tw.w, en.v.dr), 0.0f, (float)last);
                const unsigned is = __float2uint_rz(txs);
                // the blended columns is and is + 1 (as the staged form's rows hold them)
                auto column = [&](unsigned x) {
                    const unsigned o = (kbase[j] + x) * jb;
                    return sn_blend(w, ld3b(Jr, o, (unsigned)rows.x * rowb), ld3b(Jr, o, (unsigned)rows.y * rowb),
                                    ld3b(Jr, o, (unsigned)rows.z * rowb), ld3b(Jr, o, (unsigned)rows.w * rowb));
                };
                const float3 v = sn_lerp(__builtin_amdgcn_fractf(txs), column(is), column(min(is + 1, last)));
                acc[j][0] = fmaf(v.x, en.tw.x, acc[j][0]);
                acc[j][1] = fmaf(v.y, en.tw.y, acc[j][1]);
                acc[j][2] = fmaf(v.z, en.tw.z, acc[j][2]);
            }
        }
    } else {
        unsigned xo[NM];   // byte offset of each texel's column in a table row
#pragma unroll
        for (int j = 0; j < NM; ++j) xo[j] = (unsigned)min((int)threadIdx.x + j * nthr, W4 - 1) * jb;
        float3 t[4][NM];
        int held[4] = {-1, -1, -1, -1};
        auto load_rows = [&](int row) {   // the rows that the registers do not hold yet
            const int4 r4 = sn_rows4(s.RMU, row);
            const int want[4] = {r4.x, r4.y, r4.z, r4.w};
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (want[q] != held[q]) {
                    held[q] = want[q];
#pragma unroll
                    for (int j = 0; j < NM; ++j) t[q][j] = ld3b(Jr, xo[j], (unsigned)want[q] * rowb);
                }
        };
        if (FORM == 2) stage(0);
        Entry cur = get(0);
        load_rows(cur.v.row);
        float4 *B = blend;
        for (int i = 0; i <= nsamp; ++i) {
            const float4 w = sn_weights(cur.v.az, cur.v.ay);
#pragma unroll
            for (int j = 0; j < NM; ++j) {
                const int x = threadIdx.x + j * nthr;
                const float3 b = sn_blend(w, t[0][j], t[1][j], t[2][j], t[3][j]);
                if (x < W4) B[x] = make_float4(b.x, b.y, b.z, 0.f);
                if (x == W4 - 1) B[W4] = make_float4(b.x, b.y, b.z, 0.f);
            }
            if (FORM == 2 && (i & (kNChunk - 1)) == kNChunk - 1 && i < nsamp) stage(i + 1);
            const Entry nxt = get(min(i + 1, nsamp));
            __syncthreads();
            load_rows(nxt.v.row);   // in flight during the lookups
#pragma unroll
            for (int j = 0; j < NM; ++j) {
                const float txs = __builtin_amdgcn_fmed3f(sn_txs<LIN4>(s, tx[j], cur.tw.w, cur.v.dr), 0.0f,
                                                          (float)(W4 - 1 - (int)kbase[j]));
                const float4 *p = B + kbase[j] + __float2uint_rz(txs);
                const float3 v = sn_lerp(__builtin_amdgcn_fractf(txs), f3(p[0]), f3(p[1]));
                acc[j][0] = fmaf(v.x, cur.tw.x, acc[j][0]);
                acc[j][1] = fmaf(v.y, cur.tw.y, acc[j][1]);
                acc[j][2] = fmaf(v.z, cur.tw.z, acc[j][2]);
            }
            cur = nxt;
            B = B == blend ? blend + W4 + 1 : blend;
        }
    }
#pragma unroll
    for (int j = 0; j < NM; ++j) {
        const int x = threadIdx.x + j * nthr;
        if (x >= W4) break;
        const size_t t = ((size_t)l * s.RMU + y) * W4 + x;
        const float4 o = q16(make_float4(acc[j][0] * dx, acc[j][1] * dx, acc[j][2] * dx, 0.f), s.hs);
        s.dSR4[t] = o;
        if (s.S4) {
            const double nu = (float)texel_nu(x);
            const float pr = (float)((3.0 / (16.0 * kPI)) * (1.0 + nu * nu));
            float4 S = s.S4[t];
            S.x += o.x / pr;
            S.y += o.y / pr;
            S.z += o.z / pr;
            s.S4[t] = q16(S, s.hs);   // FP16 ADD blend: S = FP16(S + dS / pR)
        }
    }
}

// The view-ray samples' terms of the dSn passes (SetDesc::view), once per
// precompute: they depend on the geometry only.  Inside k_inscatterN their FP64
// chain runs on one wave of each workgroup while the others wait, in every order.
__global__ __launch_bounds__(256) void k_snview(const SetDesc *__restrict__ sets, const uint2 *__restrict__ tiles,
                                                int nsamp) {
    const uint2 tl = tiles[blockIdx.x];
    const SetDesc &s = sets[tl.x];
    const size_t e = ((size_t)tl.y * kTileY + blockIdx.y) * 256 + threadIdx.x;
    const int row = (int)(e / (nsamp + 1));
    if (row >= s.RR * s.RMU) return;
    double mu, h1, mu1;
    float tr;
    s.view[e] = sn_view(s, s.layers[row / s.RMU], row % s.RMU, (int)(e % (nsamp + 1)), nsamp, mu, h1, mu1, tr);
}

// ---------------------------------------------------------------------------
// Geometry and transmittance tables of one precompute (after the T pass, before the
// passes that use them): every ratio T(x)/T(y) of common.glsl:272-282 the later passes
// take, and the table rows of their integrals, depend only on the T table and the
// geometry, not on the order.  One launch, the theta rows' workgroups first:
//  theta_items: T from the ground point seen in direction theta to the layer
//             radius (inscatterS.glsl:129-138) per (layer, theta row), and the rows
//             and columns of the dJ and dE integrals (ThetaRow, SunColumn);
//  view_item: T(r, mu, t_i), times the trapezoid weight of sample i, along the view ray
//             of each (layer, mu row) at the inscatter samples t_i = i limit(r, mu) / nsamp
//             (inscatter1.glsl, inscatterN.glsl).
// Both use T_ratio_d (FP64 coordinates; underflow-free with the optical-depth
// table).
// ---------------------------------------------------------------------------
__device__ __forceinline__ void view_item(const SetDesc &s, size_t e, int nsamp) {
    const int line = (int)(e / (nsamp + 1)), i = (int)(e % (nsamp + 1));
    if (line >= s.RR * s.RMU) return;
    const LayerGeom L = s.layers[line / s.RMU];
    const double r = L.r;
    const double rho2 = r * r - s.Rg2;
    double mu, muS_u, nu_u;
    mu_mus_nu(s, L, 0, line % s.RMU, mu, muS_u, nu_u);
    const double rmu = r * mu;
    const double ti = i * (limit_d(s, r, mu) / nsamp);
    const double q = rho2 + ti * (ti + 2.0 * rmu);   // ri^2 - Rg^2
    const double ri = sqrt(q + s.Rg2);
    const double h1 = q / (ri + s.Rg);
    const double mu1 = (rmu + ti) / ri;
    const float3 t = mu > 0.0 ? T_ratio_d(s, r - s.Rg, mu, h1, mu1)
                              : T_ratio_d(s, h1, -mu1, r - s.Rg, -mu);
    const float wt = (i == 0 || i == nsamp) ? 0.5f : 1.0f;   // trapezoid weight
    s.tview[e] = make_float4(t.x * wt, t.y * wt, t.z * wt, (float)(ti / ri));
}

// Item e of a set's theta tables: ground transmittances of the dJ rows, the dJ rows, the
// dE rows, the columns, each kind from a multiple of 64 on (a wave has one kind).  A kind has
// at most 2^30 items (2^23 layers or irradiance rows of 128), all of them less than 2^32.
__host__ __device__ __forceinline__ unsigned theta_pad(unsigned n) { return (n + 63u) & ~63u; }
__device__ __forceinline__ void theta_items(const SetDesc &s, unsigned e, int NS, int NI) {
    const unsigned nJ = s.RR * NS, NTH = NI / 2, nE = s.SH * NTH;
    auto layer_r = [&](int l) { return fmin(fmax(s.layers[l].r, s.Rg), s.Rt); };   // inscatterS.glsl:112
    if (e < theta_pad(nJ)) {
        if (e >= nJ) return;
        const double r = layer_r(e / NS), ct = cos((e % NS + 0.5) * (kPI / NS)), q = s.Rg / r;
        float3 tr = make_float3(0.f, 0.f, 0.f);
        double e1 = 0.0;
        const bool ground = ct < -sqrt(1.0 - q * q);
        if (ground) {
            const double dg = -r * ct - sqrt(r * r * (ct * ct - 1.0) + s.Rg2);
            const double mug = -(r * ct + dg) / s.Rg;
            const double r1sq = s.Rg2 + dg * dg + 2.0 * s.Rg * mug * dg;
            const double r1 = sqrt(r1sq);
            const double mu1 = (s.Rg * mug + dg) / r1;
            const double h1 = (r1sq - s.Rg2) / (r1 + s.Rg);
            tr = mug > 0.0 ? T_ratio_d(s, 0.0, mug, h1, mu1) : T_ratio_d(s, h1, -mu1, 0.0, -mug);
            e1 = dg / s.Rg * (s.SW / 1.2);
        }
        s.tground[e] = make_float4(tr.x, tr.y, tr.z, ground ? 1.f : 0.f);
        if (s.rowJ) s.rowJ[e].e1 = e1;
        return;
    }
    e -= theta_pad(nJ);
    if (!s.rowJ) return;
    if (e < theta_pad(nJ)) {
        if (e >= nJ) return;
        const double r = layer_r(e / NS), th = (e % NS + 0.5) * (kPI / NS), hr = r - s.Rg;
        ThetaRow row;
        row.ct = cos(th);
        theta_taps(s, r, r * r - s.Rg2, row.ct, row);
        ThetaRow &o = s.rowJ[e];   // all but e1
        o.ct = row.ct;
        o.base = row.base; o.dy = row.dy; o.dz = row.dz;
        o.ay = row.ay; o.az = row.az;
        o.dw = (float)((kPI / NS) * (kPI / NS) * sin(th));
        o.eR = (float)exp(-hr / s.HR);
        o.eM = (float)exp(-hr / s.HM);
        return;
    }
    e -= theta_pad(nJ);
    if (e < theta_pad(nE)) {
        if (e >= nE) return;
        const double h = (double)(e / NTH) / (s.SH - 1.0) * (s.Rt - s.Rg);
        ThetaRow row = {};
        row.ct = cos((e % NTH + 0.5) * (kPI / NI));
        theta_taps(s, s.Rg + h, h * (2.0 * s.Rg + h), row.ct, row);
        s.rowE[e] = row;
        return;
    }
    e -= theta_pad(nE);
    const unsigned SW = s.SW;
    if (e >= SW + s.RMUS) return;
    SunColumn c;
    c.mus = e < SW ? -0.2 + (double)e / (s.SW - 1.0) * (1.0 + 0.2) : fmin(fmax(texel_mus(s, (int)(e - SW)), -1.0), 1.0);
    c.txs = tex4d_umus(s, c.mus) * s.RMUS - 0.5;
    (e < SW ? s.sunE[e] : s.sunJ[e - SW]) = c;
}

// ntheta workgroups of theta items, wpt of them per set from set0 on, then nview tiles of
// view items
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void
k_geometry(const SetDesc *__restrict__ sets, int set0, const uint2 *__restrict__ tiles, int ntheta, int wpt, int nview, int nsamp,
           int NS, int NI) {
    const int b = (int)blockIdx.x;
    if (b < ntheta) {
        theta_items(sets[set0 + b / wpt], (unsigned)(b % wpt) * 256u + threadIdx.x, NS, NI);
    } else {
        const int v = b - ntheta;
        const uint2 tl = tiles[v % nview];
        view_item(sets[tl.x], ((size_t)tl.y * kTileY + v / nview) * 256 + threadIdx.x, nsamp);
    }
}

// ---------------------------------------------------------------------------
// Numeric validation of finished tables: counts non-finite values, T outside
// [0, 1] and negative E / S entries into flags[set].
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_check(const SetDesc *__restrict__ sets,
                                               const uint2 *__restrict__ tiles,
                                               unsigned int *__restrict__ flags) {
    const uint2 tl = tiles[blockIdx.x];
    const SetDesc &s = sets[tl.x];
    const int t = ((int)tl.y * kTileY + (int)blockIdx.y) * 256 + (int)threadIdx.x;
    bool bad = false;
    if (t < s.n4) {
        float4 v = s.S4[t];
        bad |= !(isfinite(v.x) && isfinite(v.y) && isfinite(v.z) && isfinite(v.w));
        bad |= v.x < 0.f || v.y < 0.f || v.z < 0.f || v.w < 0.f;
    }
    if (t < s.TW * s.TH) {
        float4 v = s.T4[t];
        bad |= !(v.x >= 0.f && v.x <= 1.f && v.y >= 0.f && v.y <= 1.f && v.z >= 0.f && v.z <= 1.f);
    }
    if (t < s.SW * s.SH && s.E4) {
        float4 v = s.E4[t];
        bad |= !(isfinite(v.x) && isfinite(v.y) && isfinite(v.z));
        bad |= v.x < 0.f || v.y < 0.f || v.z < 0.f;
    }
    if (bad) atomicAdd(&flags[tl.x], 1u);
}

// ---------------------------------------------------------------------------
// Host launchers
// ---------------------------------------------------------------------------
bool inscatterS_chunked(int NS, int CH, int RNU, bool first) {
    return CH < NS || (first && (size_t)CH * (RNU + 1) > (size_t)kJ1Plane);
}
size_t lds_inscatterS(int NS, int CH, int RNU, int SW, int JX, bool first) {
    const int NT = first ? 2 : 1, PW = first ? 3 : 2;
    const size_t npairs = (size_t)CH * (RNU + 1) + (first ? 0 : (size_t)JX);
    const bool planes = first && !inscatterS_chunked(NS, CH, RNU, first);
    return sizeof(float4) * ((planes ? 2 * (size_t)kJ1Plane + npairs : npairs * PW) +
                             (planes ? 0 : (size_t)CH * (RNU + 2) * NT) + 1 +
                             (first ? (size_t)(e_pad(SW) + SW + 1) * 2 : 0) + (size_t)CH * 3);
}
int merged_row_extra(double r, double Rg, double Rt, int SW, int NS, int it) {
    // the kernel's r, clamped as inscatterS.glsl:112 does, and its ground test
    r = std::min(std::max(r, Rg), Rt);
    const double ct = std::cos((it + 0.5) * (kPI / NS));
    if (ct >= 1e-9) return 0;   // theta < 90 deg: never a ground row
    const double q = Rg / r, cthetamin = -std::sqrt(1.0 - q * q);
    // ground distance, or (where the device's ground test could round either
    // way) the tangent distance, which bounds the ground distance of every ray
    // that hits the ground
    const double dg = ct < cthetamin - 1e-9 ? -r * ct - std::sqrt(r * r * (ct * ct - 1.0) + Rg * Rg)
                                            : std::sqrt(std::max(r * r - Rg * Rg, 0.0));
    const double e1 = dg / Rg * (SW / 1.2);
    // the kernel keeps at most ceil(2.05 e1) + 1 extra entries in a row
    return (int)std::ceil(2.05 * e1) + 2;
}
size_t lds_irradianceN(int CH, int RNU, bool first) {
    const int NT = first ? 2 : 1;
    return sizeof(float4) * ((size_t)CH * (RNU + 1) * NT * 2 + (size_t)CH * (RNU + 2) * NT) +
           sizeof(float) * 3 * 16;
}
int chunk_inscatterS(int NS, int RNU, int SW, const std::function<int(int)> &jx_of_ch, bool first) {
    for (int ch = NS; ch >= 1; --ch)
        if (lds_inscatterS(NS, ch, RNU, SW, first ? 0 : jx_of_ch(ch), first) <= kSphLdsBudget) return ch;
    return 0;
}
int chunk_irradianceN(int NI, int RNU, bool first) {
    for (int ch = NI / 2; ch >= 1; --ch)
        if (lds_irradianceN(ch, RNU, first) <= kSphLdsBudget) return ch;
    return 0;
}

hipError_t launch_transmittance(const SetDesc *sets, const uint2 *tiles, int ntiles, int nsamp,
                                hipStream_t st) {
    if (ntiles <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_transmittance, dim3(ntiles, kTileY), dim3(256), 0, st, sets, tiles, nsamp);
    return hipGetLastError();
}
int theta_workgroups(int RR, int RMUS, int SW, int SH, int NS, int NI) {
    const long long items = 2LL * theta_pad((unsigned)RR * NS) + theta_pad((unsigned)SH * (NI / 2)) + SW + RMUS;
    return (int)((items + 255) / 256);
}
hipError_t launch_geometry(const SetDesc *sets, int nsets, int wpt, const uint2 *tiles, int nview, int nsamp, int NS, int NI,
                           hipStream_t st) {
    if (nview <= 0) return hipSuccess;
    // a launch has less than 2^32 threads: what is beyond takes further ones
    constexpr int kMost = (1 << 24) - 1;
    const int each = wpt > 0 ? std::max(1, kMost / wpt) : nsets;   // sets of a launch
    for (int s0 = 0, v0 = 0; s0 < nsets || v0 < nview;) {
        const int ns = std::min(nsets - s0, each), ntheta = ns * wpt;
        const int nv = std::min(nview - v0, (kMost - ntheta) / kTileY);
        hipLaunchKernelGGL(k_geometry, dim3(ntheta + nv * kTileY), dim3(256), 0, st, sets, s0, tiles + v0, ntheta, std::max(wpt, 1),
                           nv, nsamp, NS, NI);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        s0 += ns;
        v0 += nv;
    }
    return hipSuccess;
}
hipError_t launch_irradiance1(const SetDesc *sets, const uint2 *tiles, int ntiles,
                              hipStream_t st) {
    if (ntiles <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_irradiance1, dim3(ntiles), dim3(256), 0, st, sets, tiles);
    return hipGetLastError();
}
// The texels per thread of k_inscatter1_rows with the least waves x (5 texels + 4 + T
// columns per thread): a texel costs a wave about 150 issue cycles per sample, the
// sample's own terms and the barrier 120, a staged column 30.  us at 51 samples, with 1 /
// 2 / 3 / 4 texels: 32x128x32x8 (rows of 256) 119 / 103 / 125 / 190 (spills),
// 21x90x27x5 (135) 58 / 54 / 48 / 85 (spills), 64x256x64x16 (1024, 512 columns)
// - / 1434 / 1932 / 1143.  So: four columns per thread only where no spill
// comes with them (three texels).  More columns than that cost more than the gathers
// they save, and rows of at most 64 texels gather (k_inscatter1's slots).  The most LDS is
// that of 3 texels and 4 columns with 384 threads, for 961 to 1024 texels and T of 1536
// columns: 60 KB dynamic and 4 KB static, of the 160 KB a workgroup can have.
S1Shape s1_shape(int W4, int TW, bool linT) {
    const int ax = linT ? kSunLin : TW > kXkMax ? kSunWide : TW < kXkMin ? kSunFew : kSunTab;
    S1Shape best = {ax, 0, 0, 256};
    if (W4 <= 64 || ax == kSunFew) return best;
    int least = 1 << 30;
    for (int n = 1; n <= 4; ++n) {
        const int waves = (W4 + 64 * n - 1) / (64 * n), nc = (TW + 64 * waves - 1) / (64 * waves);
        if (waves > 8 || nc > (n == 3 ? 4 : 2)) continue;
        const int columns = nc > 2 ? 4 : nc, cost = waves * (5 * n + 4 + columns);
        if (cost < least) {
            least = cost;
            best = {ax, n, columns, 64 * waves};
        }
    }
    return best;
}
hipError_t launch_inscatter1(const SetDesc *sets, const uint2 *tiles, int ntiles, int nsamp, S1Shape sh, int TWmax,
                             hipStream_t st) {
    if (ntiles <= 0) return hipSuccess;
    if (sh.texels > 0 && (sh.threads > 512 || sh.columns * sh.threads < TWmax)) return hipErrorInvalidValue;
    const size_t tab = sh.axis == kSunLin || sh.axis == kSunWide ? 0 : sizeof(double) * TWmax;
    const size_t lds = tab + (sh.texels ? 2 * sizeof(float4) * (sh.columns * sh.threads + 1) : 0);
#define ATMO_L1(...) hipLaunchKernelGGL((__VA_ARGS__), dim3(ntiles, kTileRows), dim3(sh.threads), lds, st, sets, tiles, nsamp)
#define ATMO_L1C(NM, NC)                                                                   \
    if (sh.axis == kSunLin) ATMO_L1(k_inscatter1_rows<kSunLin, NM, NC>);                   \
    else ATMO_L1(k_inscatter1_rows<kSunTab, NM, NC>)
#define ATMO_L1R(NM) \
    if (sh.columns == 1) { ATMO_L1C(NM, 1); } else { ATMO_L1C(NM, 2); }
    if (sh.texels == 0) {
        if (sh.axis == kSunLin) ATMO_L1(k_inscatter1<kSunLin>);
        else if (sh.axis == kSunWide) ATMO_L1(k_inscatter1<kSunWide>);
        else if (sh.axis == kSunFew) ATMO_L1(k_inscatter1<kSunFew>);
        else ATMO_L1(k_inscatter1<kSunTab>);
    } else if (sh.texels == 1) {
        ATMO_L1R(1)
    } else if (sh.texels == 2) {
        ATMO_L1R(2)
    } else if (sh.texels == 3) {
        if (sh.columns == 4) { ATMO_L1C(3, 4); } else { ATMO_L1R(3) }
    } else {
        ATMO_L1R(4)
    }
#undef ATMO_L1C
#undef ATMO_L1R
#undef ATMO_L1
    return hipGetLastError();
}
hipError_t launch_inscatterS(const SetDesc *sets, const uint2 *tiles, int ntiles, int NS, int CH, int RNU,
                             int JX, const void *dirT, const void *dirW, bool first, size_t lds, int G,
                             int DS, int threads, hipStream_t st) {
    if (ntiles <= 0) return hipSuccess;
    if (CH < 1 || CH > NS || JX < 0) return hipErrorInvalidValue;
    if (G != 2 && G != 3 && G != 4 && G != 8) return hipErrorInvalidValue;
    const bool chunked = inscatterS_chunked(NS, CH, RNU, first);
    if (DS < 1 || threads < 64 || threads % (64 * DS) || threads > (DS > 1 ? kJSplitThreads : 256) || (DS > 1 && chunked))
        return hipErrorInvalidValue;
    if (DS > 1) lds += sizeof(float) * 3 * (size_t)(threads - threads / DS);
#define ATMO_LJ(F, GG, M)                                                                              \
    hipLaunchKernelGGL((k_inscatterS<F, GG, M>), dim3(ntiles), dim3(threads), lds, st, sets, tiles, NS, \
                       CH, JX, DS, (const DirJ *)dirT, (const float2 *)dirW)
#define ATMO_LJG(F, M)                \
    switch (G) {                      \
    case 2: ATMO_LJ(F, 2, M); break;  \
    case 3: ATMO_LJ(F, 3, M); break;  \
    case 4: ATMO_LJ(F, 4, M); break;  \
    default: ATMO_LJ(F, 8, M); break; \
    }
    if (chunked) {   // chunked staging: one variant (all G give the same bits)
        if (first) ATMO_LJ(true, 4, kJChunk); else ATMO_LJ(false, 4, kJChunk);
    } else if (DS > 1) {
        if (first) ATMO_LJG(true, kJSplit) else ATMO_LJG(false, kJSplit)
    } else {
        if (first) ATMO_LJG(true, kJPlain) else ATMO_LJG(false, kJPlain)
    }
#undef ATMO_LJG
#undef ATMO_LJ
    return hipGetLastError();
}
hipError_t launch_irradianceN(const SetDesc *sets, const uint2 *tiles, int ntiles, int NI, int CH,
                              const void *dirs, bool first, size_t lds, hipStream_t st) {
    if (ntiles <= 0) return hipSuccess;
    if (CH < 1 || CH > NI / 2) return hipErrorInvalidValue;
    if (first)
        hipLaunchKernelGGL(k_irradianceN<true>, dim3(ntiles), dim3(256), lds, st, sets, tiles, NI,
                           CH, (const DirE *)dirs);
    else
        hipLaunchKernelGGL(k_irradianceN<false>, dim3(ntiles), dim3(256), lds, st, sets, tiles, NI,
                           CH, (const DirE *)dirs);
    return hipGetLastError();
}
// Two texels per thread share a sample's uniform work and give a wave two
// independent lookups: 32x128x32x8 (rows of 256 texels) 116 us per order with one
// texel per thread, 99 with two, 145 with four (one wave per row); 1024 texels
// 1.51 ms with two (512 threads), 1.60 with four; 135 texels 48 us with one, 47
// with two.  Three where two leave 8 % or more of the threads' slots idle beyond
// what three do: 576 texels (640 slots against 576) 9.5 ms with two, 8.5 with
// three for the 48-set mixed batch.  Rows of at most a wave have one.
SnShape sn_shape(int W4) {
    const int t2 = 64 * ((W4 + 127) / 128), t3 = 64 * ((W4 + 191) / 192);
    if (W4 <= 64) return {1, 64};
    return W4 > 256 && 3 * t3 * 100 <= 2 * t2 * 92 ? SnShape{3, t3} : SnShape{2, t2};
}
template <int NM>
static void launch_sn(const SetDesc *sets, const uint2 *tiles, int ntiles, int nsamp, int form, int threads, int W4max,
                      bool lin4, hipStream_t st) {
    const size_t lds = form == 0 ? 0 : sizeof(float4) * 2 * ((size_t)W4max + 1);
#define ATMO_LN(F, L) \
    hipLaunchKernelGGL((k_inscatterN<F, L, NM>), dim3(ntiles), dim3(threads), lds, st, sets, tiles, nsamp)
    if (form == 0) {
        if (lin4) ATMO_LN(0, true); else ATMO_LN(0, false);
    } else if (form == 1) {
        if (lin4) ATMO_LN(1, true); else ATMO_LN(1, false);
    } else {
        if (lin4) ATMO_LN(2, true); else ATMO_LN(2, false);
    }
#undef ATMO_LN
}
hipError_t launch_inscatterN(const SetDesc *sets, const uint2 *tiles, int ntiles, int nsamp, int form, SnShape sh,
                             int W4max, bool lin4, hipStream_t st) {
    if (ntiles <= 0) return hipSuccess;
    if (form < 0 || form > 2 || sh.threads < 64 || sh.threads > 512 || sh.threads % 64 ||
        W4max > sh.texels * sh.threads)
        return hipErrorInvalidValue;
    switch (sh.texels) {
    case 1: launch_sn<1>(sets, tiles, ntiles, nsamp, form, sh.threads, W4max, lin4, st); break;
    case 2: launch_sn<2>(sets, tiles, ntiles, nsamp, form, sh.threads, W4max, lin4, st); break;
    case 3: launch_sn<3>(sets, tiles, ntiles, nsamp, form, sh.threads, W4max, lin4, st); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}
hipError_t launch_snview(const SetDesc *sets, const uint2 *tiles, int ntiles, int nsamp, hipStream_t st) {
    if (ntiles <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_snview, dim3(ntiles, kTileY), dim3(256), 0, st, sets, tiles, nsamp);
    return hipGetLastError();
}
hipError_t launch_check(const SetDesc *sets, const uint2 *tiles, int ntiles, unsigned int *flags,
                        hipStream_t st) {
    if (ntiles <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_check, dim3(ntiles, kTileY), dim3(256), 0, st, sets, tiles, flags);
    return hipGetLastError();
}

}  // namespace atmo
