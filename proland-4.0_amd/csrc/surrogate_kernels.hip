// surrogate_kernels.hip — kernels of the learned multiple-scattering surrogate.
//
// MLP 14 -> 256 -> 256 -> 256 -> 4 (kNL = 3 hidden layers), act() on the hidden
// layers.  Layers are numbered as for four hidden layers: the output layer is
// "layer 5" and the last hidden layer's activations "H4" whatever kNL is.  The
// kNG = kNL - 1 256x256 layers hold 96 % of the FLOPs.
//   inference (k_mlp_infer): all layers of a set's texels in one kernel, FP16 on the
//     matrix cores with FP32 accumulation;
//   training (k_train_rows, k_train_dw, k_train_reduce): forward and backward of a
//     batch, bf16 hidden products, everything else FP32;
//   predict: a kernel per layer (k_layer1_fwd, k_gemm_act, k_layer5), bf16 hidden
//     products.
#include "surrogate_kernels.h"

#include <algorithm>
#include <mutex>

namespace atmo {
namespace sg {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(8 * sizeof(_Float16)))) _Float16 f16x8;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16;

// Hidden activation: z gated by a smoothstep, act(z) = z s(t), t = clamp(z / 6
// + 1/2, 0, 1), s = t^2 (3 - 2 t).  Like SiLU (z sigmoid(z)) it is C1 with
// gate 1/2 and gate slope 1/4 at 0, but it is linear (z or 0) beyond |z| = 3 and
// takes 6 full-rate instructions where SiLU needs two quarter-rate
// transcendentals (exp, rcp) and three more: the activations of the fused
// inference kernel are a bound of its speed.  act'(z) = s + z t (1 - t).
__device__ __forceinline__ float gate_t(float z) {
    return __builtin_amdgcn_fmed3f(fmaf(z, 1.0f / 6.0f, 0.5f), 0.0f, 1.0f);
}
__device__ __forceinline__ float act(float z) {
    const float t = gate_t(z);
    return z * (t * t * fmaf(-2.0f, t, 3.0f));
}
__device__ __forceinline__ float dact(float z) {
    const float t = gate_t(z);
    return fmaf(z, t * (1.0f - t), t * t * fmaf(-2.0f, t, 3.0f));
}

// ---------------------------------------------------------------------------
// H_out[M x 256] = act(A[M x 256] . B^T + bias), bf16 in and out, FP32 accumulate; B
// stored [N][K].  Tile 128 x 128 x 32, 4 waves of 64 x 64 (2 x 2 MFMA 32x32 tiles).
// M, N multiples of 128, K a multiple of 32 (checked by the host).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_gemm_act(const __bf16 *__restrict__ A, const __bf16 *__restrict__ Bm, int M,
                                                  int N, int K, const float *__restrict__ bias,
                                                  __bf16 *__restrict__ hout) {
    __shared__ __attribute__((aligned(16))) __bf16 As[128][40];
    __shared__ __attribute__((aligned(16))) __bf16 Bs[128][40];
    const int n0 = blockIdx.x * 128, m0 = blockIdx.y * 128;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, wm = w >> 1, wn = w & 1;
    f32x16 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

    for (int k0 = 0; k0 < K; k0 += 32) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int c = tid + i * 256, row = c >> 2, kc = (c & 3) * 8;
            *(uint4 *)&As[row][kc] = *(const uint4 *)(A + (size_t)(m0 + row) * K + k0 + kc);
            *(uint4 *)&Bs[row][kc] = *(const uint4 *)(Bm + (size_t)(n0 + row) * K + k0 + kc);
        }
        __syncthreads();
#pragma unroll
        for (int ks = 0; ks < 32; ks += 16) {
            bf16x8 a[2], b[2];
            const int kk = ks + 8 * (lane >> 5);
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                a[t] = *(const bf16x8 *)&As[wm * 64 + t * 32 + (lane & 31)][kk];
                b[t] = *(const bf16x8 *)&Bs[wn * 64 + t * 32 + (lane & 31)][kk];
            }
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
        }
    }
    // epilogue: lane holds rows 8(r/4) + 4(lane/32) + r%4 of column lane%32 of each 32x32 tile
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int row = m0 + wm * 64 + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                const int col = n0 + wn * 64 + j * 32 + (lane & 31);
                hout[(size_t)row * N + col] = (__bf16)act(acc[i][j][r] + bias[col]);
            }
}

// ---------------------------------------------------------------------------
// Layer 1 (14 -> 256), FP32: H1 = act(X W1 + b1).  X rows are 16
// floats (14 used).  One thread per (row, column).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_layer1_fwd(const float *__restrict__ X,
                                                    const float *__restrict__ W1,
                                                    const float *__restrict__ b1, int rows,
                                                    __bf16 *__restrict__ H1) {
    const size_t t = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= (size_t)rows * kNH) return;
    const int n = (int)(t % kNH);
    const size_t b = t / kNH;
    float z = b1[n];
#pragma unroll
    for (int i = 0; i < kNIN; ++i) z = fmaf(X[b * kXS + i], W1[i * kNH + n], z);
    H1[t] = (__bf16)act(z);
}

// ---------------------------------------------------------------------------
// Layer 5 (256 -> 4), FP32 from bf16 H4: a wave takes a row at a time (16 rows), each
// lane 4 of the 256 inputs, shuffles for the dot products.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_layer5(const __bf16 *__restrict__ H4,
                                                const float *__restrict__ W5,
                                                const float *__restrict__ b5, int rows,
                                                float *__restrict__ Y) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    for (int rr = 0; rr < 16; ++rr) {
        const size_t b = (size_t)blockIdx.x * 64 + wv * 16 + rr;
        if (b >= (size_t)rows) break;
        float acc[kNOUT] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int k = lane * 4 + q;
            const float h = (float)H4[b * kNH + k];
#pragma unroll
            for (int o = 0; o < kNOUT; ++o) acc[o] = fmaf(h, W5[k * kNOUT + o], acc[o]);
        }
#pragma unroll
        for (int o = 0; o < kNOUT; ++o)
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) acc[o] += __shfl_xor(acc[o], off, 64);
        if (lane == 0) {
#pragma unroll
            for (int o = 0; o < kNOUT; ++o) Y[b * kNOUT + o] = acc[o] + b5[o];
        }
    }
}

// Adam (bias-corrected) on the flat FP32 parameter vector.
__global__ __launch_bounds__(256) void k_adam(float *__restrict__ p, const float *__restrict__ g,
                                              float *__restrict__ m, float *__restrict__ v, int n,
                                              float lr, float b1, float b2, float eps, float c1,
                                              float c2) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr * (mi * c1) / (sqrtf(vi * c2) + eps);
}

// bf16 copies of a 256x256 weight: W (row-major [in][out]) and Wt ([out][in]).
__global__ __launch_bounds__(256) void k_to_bf16(const float *__restrict__ W, __bf16 *__restrict__ Wb,
                                                 __bf16 *__restrict__ Wt) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= kNH * kNH) return;
    const int r = i / kNH, c = i % kNH;
    const __bf16 v = (__bf16)W[i];
    Wb[i] = v;
    Wt[c * kNH + r] = v;
}

// ---------------------------------------------------------------------------
// Features of table texels and dataset assembly
// ---------------------------------------------------------------------------
constexpr float kHorizonGap = 0.25f;

// The mu coordinate of row y of layer l.
__device__ __forceinline__ float row_coordinate(const FeatSet &fs, int l, int y) {
    // mu rows: the row's ray length d (getMuMuSNu, common.glsl:175-190, with
    // the layer radius of setLayer, PreprocessAtmo.cpp:255-271) on one log
    // scale for the whole set, from 1 m (the shortest ray of the table: up
    // from the highest layer) to 2 sqrt(Rt^2 - Rg^2) (longer than any ray),
    // the ground-ray half in [-1, -kHorizonGap] and the sky half in
    // [kHorizonGap, 1].  The table rows are linear in d up to a clamp at the
    // shortest ray of a layer (10 m down from the lowest layer), where the
    // inscatter, proportional to d, drops by 10-100x from one row to the
    // next; on a log scale common to all layers that drop is the same slope
    // everywhere, and the gap separates the straight-down and straight-up
    // rows, which are neighbours in the table only.
    const int half = fs.RMU / 2;
    const double Rg = fs.Rg, Rt = fs.Rt, Rg2 = Rg * Rg;
    double rl = (double)l / (fs.RR - 1);
    rl = sqrt(Rg2 + rl * rl * (Rt * Rt - Rg2)) + (l == 0 ? 0.01 : (l == fs.RR - 1 ? -0.001 : 0.0));
    const double rho = sqrt(fmax(rl * rl - Rg2, 0.0)), H = sqrt(Rt * Rt - Rg2);
    double dmin, dmax, d;
    if (y < half) {
        dmin = rl - Rg;
        dmax = 0.999 * rho;
        d = (1.0 - (double)y / (half - 1)) * rho;
    } else {
        dmin = Rt - rl;
        dmax = 0.999 * (rho + H);
        d = (double)(y - half) / (half - 1) * (rho + H);
    }
    d = fmin(fmax(d, dmin), dmax);
    const double dlo = 1e-3, dhi = 2.0 * H;   // in the parameters' length unit (km)
    const float t = (float)fmin(fmax(log(d / dlo) / log(dhi / dlo), 0.0), 1.0);
    return y < half ? fmaf(-(1.f - kHorizonGap), t, -kHorizonGap) : fmaf(1.f - kHorizonGap, t, kHorizonGap);
}

// Resolution-independent texel coordinates in [-1, 1] (the arguments of
// getMuMuSNu, common.glsl:175-201), the 7 normalised atmosphere features, and
// the exactly computed orders' value at the texel (ex: S.rgb of an inscatter
// texel, E of an irradiance texel) on a log scale: 0.25 (log(v + 1e-6) + 5),
// about -2 .. 1 over the tables' range.  The higher orders follow the lower
// ones closely (where the view ray meets the ground, where the sun sets), so
// the network learns them relative to what the exact part already resolves.
// E texels use the irradiance coordinates in slots 0 and 2 and -2 in 1 and 3.
// mu: row_coordinate of every (layer, row), or nullptr.
__device__ __forceinline__ void texel_features(const FeatSet &fs, unsigned code, const float *ex, float *x,
                                               const float *mu = nullptr) {
    if (code & 0x80000000u) {
        const unsigned t = code & 0x7fffffffu;
        const int i = t % fs.SW, j = t / fs.SW;
        x[0] = 2.f * j / (fs.SH - 1) - 1.f;
        x[1] = -2.f;
        x[2] = 2.f * i / (fs.SW - 1) - 1.f;
        x[3] = -2.f;
    } else {
        const int W4 = fs.RMUS * fs.RNU;
        const int xx = code % W4, y = (code / W4) % fs.RMU, l = code / (W4 * fs.RMU);
        x[0] = 2.f * l / (fs.RR - 1) - 1.f;
        x[1] = mu ? mu[code / W4] : row_coordinate(fs, l, y);
        x[2] = 2.f * (xx % fs.RMUS) / (fs.RMUS - 1) - 1.f;
        x[3] = 2.f * (xx / fs.RMUS) / (fs.RNU - 1) - 1.f;
    }
#pragma unroll
    for (int k = 0; k < 7; ++k) x[4 + k] = fs.f[k];
#pragma unroll
    for (int c = 0; c < 3; ++c) x[11 + c] = 0.25f * (__logf(fmaxf(ex[c], 0.f) + 1e-6f) + 5.0f);
}

// The exact part's value at a texel (S.rgb, or E of an irradiance texel).
__device__ __forceinline__ void exact_value(const FeatSet &fs, unsigned code, const float4 *S1, const float *E1,
                                            float *ex) {
    if (code & 0x80000000u) {
        const unsigned e = code & 0x7fffffffu;
        ex[0] = E1[3 * e];
        ex[1] = E1[3 * e + 1];
        ex[2] = E1[3 * e + 2];
    } else {
        const float4 v = S1[code];
        ex[0] = v.x;
        ex[1] = v.y;
        ex[2] = v.z;
    }
}

__device__ __forceinline__ unsigned hash32(unsigned long long z) {
    z += 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return (unsigned)((z ^ (z >> 31)) >> 32);
}

// Training rows of one set: `ns` seeded S texels (a quarter of them near the
// horizon) then all E texels.
// target c = (log(max(v_c, 0) + eps) - mu_c) / sd_c, v = S(orders<=N) - S(orders<=K) for S
// texels (rgb) and E(orders<=N) - E(orders<=K) for E texels, K the exactly computed
// orders (S1, E1); the fourth target is 0 (the orders above 1 add 0 to alpha).
__global__ __launch_bounds__(256) void k_make_rows(FeatSet fs, const float4 *__restrict__ S4,
                                                   const float4 *__restrict__ S1,
                                                   const float *__restrict__ E,
                                                   const float *__restrict__ E1, int ns,
                                                   unsigned long long seed, float *__restrict__ X,
                                                   float *__restrict__ Tg, TargetNorm tn) {
    const int t = blockIdx.x * 256 + threadIdx.x;
    const int nE = fs.SW * fs.SH;
    if (t >= ns + nE) return;
    unsigned code;
    float v[3], ex[3];
    if (t < ns) {
        const unsigned hh = hash32(seed * 0x100000001ull + t);
        if ((t & 3) == 0 && fs.RMU >= 8) {
            // a quarter of the samples from the 8 mu rows around the horizon,
            // where each set's worst texels sit (the last ground rows, the
            // first sky rows); the rest uniform over the table
            const unsigned W4 = (unsigned)(fs.RMUS * fs.RNU);
            const unsigned l = hh % (unsigned)fs.RR, y = (unsigned)(fs.RMU / 2 - 4) + (hh / (unsigned)fs.RR) % 8u;
            code = (l * (unsigned)fs.RMU + y) * W4 + (hh / ((unsigned)fs.RR * 8u)) % W4;
        } else {
            code = hh % (unsigned)fs.n4;
        }
        const float4 a = S4[code], b = S1[code];
        v[0] = a.x - b.x; v[1] = a.y - b.y; v[2] = a.z - b.z;
        ex[0] = b.x; ex[1] = b.y; ex[2] = b.z;
    } else {
        const int e = t - ns;
        code = 0x80000000u | (unsigned)e;
        v[0] = E[3 * e] - E1[3 * e]; v[1] = E[3 * e + 1] - E1[3 * e + 1]; v[2] = E[3 * e + 2] - E1[3 * e + 2];
        ex[0] = E1[3 * e]; ex[1] = E1[3 * e + 1]; ex[2] = E1[3 * e + 2];
    }
    float x[kNIN];
    texel_features(fs, code, ex, x);
#pragma unroll
    for (int i = 0; i < kNIN; ++i) X[(size_t)t * kXS + i] = x[i];
#pragma unroll
    for (int i = kNIN; i < kXS; ++i) X[(size_t)t * kXS + i] = 0.f;
#pragma unroll
    for (int c = 0; c < 3; ++c) Tg[(size_t)t * kNOUT + c] = (logf(fmaxf(v[c], 0.f) + tn.eps) - tn.mu[c]) / tn.sd[c];
    Tg[(size_t)t * kNOUT + 3] = 0.f;
}

// Rows for caller-given texel codes.
__global__ __launch_bounds__(256) void k_code_rows(FeatSet fs, const unsigned *__restrict__ codes,
                                                   int n, const float4 *__restrict__ S1,
                                                   const float *__restrict__ E1, float *__restrict__ X) {
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= n) return;
    float ex[3], x[kNIN];
    exact_value(fs, codes[t], S1, E1, ex);
    texel_features(fs, codes[t], ex, x);
#pragma unroll
    for (int i = 0; i < kNIN; ++i) X[(size_t)t * kXS + i] = x[i];
#pragma unroll
    for (int i = kNIN; i < kXS; ++i) X[(size_t)t * kXS + i] = 0.f;
}

// Sum and sum of squares of the three rgb targets over n rows (FP64, for the
// output standardisation): out[0..2] sums, out[3..5] sums of squares.
__global__ __launch_bounds__(256) void k_target_stats(const float *__restrict__ Tg, size_t n,
                                                      double *__restrict__ out) {
    double a[6] = {0, 0, 0, 0, 0, 0};
    for (size_t t = (size_t)blockIdx.x * 256 + threadIdx.x; t < n; t += (size_t)gridDim.x * 256) {
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const double v = Tg[t * kNOUT + c];
            a[c] += v;
            a[3 + c] += v * v;
        }
    }
    __shared__ double red[6][256];
#pragma unroll
    for (int k = 0; k < 6; ++k) red[k][threadIdx.x] = a[k];
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w)
#pragma unroll
            for (int k = 0; k < 6; ++k) red[k][threadIdx.x] += red[k][threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x < 6) atomicAdd(&out[threadIdx.x], red[threadIdx.x][0]);
}

// In-place standardisation of the three rgb targets.
__global__ __launch_bounds__(256) void k_norm_targets(float *__restrict__ Tg, size_t n, TargetNorm tn) {
    const size_t t = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= n) return;
#pragma unroll
    for (int c = 0; c < 3; ++c) Tg[t * kNOUT + c] = (Tg[t * kNOUT + c] - tn.mu[c]) / tn.sd[c];
}


// Random training batch: rows idx = hash(seed, b) mod n copied from the dataset.
__global__ __launch_bounds__(256) void k_gather(const float *__restrict__ Xa, const float *__restrict__ Ta,
                                                size_t n, int B, unsigned long long seed,
                                                float *__restrict__ X, float *__restrict__ Tg) {
    const int b = blockIdx.x * 256 + threadIdx.x;
    if (b >= B) return;
    const unsigned long long h = ((unsigned long long)hash32(seed * 0x9E3779B1ull + 2 * b) << 32) |
                                 hash32(seed * 0x9E3779B1ull + 2 * b + 1);
    const size_t i = (size_t)(h % n);
#pragma unroll
    for (int k = 0; k < kXS; ++k) X[(size_t)b * kXS + k] = Xa[i * kXS + k];
#pragma unroll
    for (int k = 0; k < kNOUT; ++k) Tg[(size_t)b * kNOUT + k] = Ta[i * kNOUT + k];
}

// Per-set max relative error of a surrogate table against the plain one,
// floored at 1e-4 of the plain table's largest magnitude (scale given).
__global__ __launch_bounds__(256) void k_relerr(const float *__restrict__ a, const float *__restrict__ b,
                                                size_t n, int stride, int ncomp, float floorv,
                                                unsigned int *__restrict__ out) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    float e = 0.f;
    if (i < n) {
        for (int c = 0; c < ncomp; ++c) {
            const float x = a[i * stride + c], y = b[i * stride + c];
            const float den = fmaxf(fabsf(y), floorv);
            float r = fabsf(x - y) / den;
            if (!(r == r)) r = 3.0e38f;  // NaN counts as a failure
            e = fmaxf(e, r);
        }
    }
    for (int off = 32; off > 0; off >>= 1) e = fmaxf(e, __shfl_xor(e, off, 64));
    if ((threadIdx.x & 63) == 0) atomicMax(out, __float_as_uint(e));
}

// max |v| over a table (for the relative-error floor)
__global__ __launch_bounds__(256) void k_absmax(const float *__restrict__ a, size_t n, int stride,
                                                int ncomp, unsigned int *__restrict__ out) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    float e = 0.f;
    if (i < n)
        for (int c = 0; c < ncomp; ++c) e = fmaxf(e, fabsf(a[i * stride + c]));
    for (int off = 32; off > 0; off >>= 1) e = fmaxf(e, __shfl_xor(e, off, 64));
    if ((threadIdx.x & 63) == 0) atomicMax(out, __float_as_uint(e));
}

// ---------------------------------------------------------------------------
// Fused inference: texel features -> layer 1 -> kNG x (256x256 + bias + act)
// -> layer 5 -> orders >= 2 added to S / written to E, all in one kernel with
// the activations in registers.
//
// The products are computed transposed, D = W^T H^T (output features x rows),
// with v_mfma_f32_32x32x16_f16 (FP16 weights and activations, FP32
// accumulation; layer 1 with the _bf16 form): the A operand is a 32-feature x 16-k slice of
// the weight (W^T rows, staged in LDS), the B operand a 16-k x 32-row slice of
// the activations, held by each lane for its own row (lane l: row l%32,
// features 16kb + 8(l/32) .. +7 of every k block kb).  A D tile gives lane l
// the features 8q + 4(l/32) + t (q, t < 4) of row l%32; one swap of 4 values
// with lane l^32 turns it into the B layout of the next layer.  Each wave owns
// 32*RBW rows through all five layers; a workgroup stages one 256x256 weight
// (rows padded to 528 B, conflict-free 16-byte LDS reads) per layer.
// Layers 1 and 5 split their FP32 weights into hi + lo parts, bf16 for layer 1
// (x W ~ xh Wh + xh Wl + xl Wh, its bias riding in input column 14) and FP16
// for layer 5 (its input is FP16 already, so Wh + Wl only): relative error
// ~1e-5 and ~1e-6, inside the FP16 rounding of the activations.
// ---------------------------------------------------------------------------
constexpr int kRowPad = 264;   // 16-bit values per staged weight row (512 B + 16 B pad)

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// act of a (low half) and b (high half) in packed FP16: one v_cvt_pk_f16_f32
// (round to nearest even) and five v_pk_*_f16, the clamp of t riding on the
// first FMA.  FP16 keeps 11 significant bits where the bf16 activations of the
// training path keep 8, and its range covers the pre-activations (|z| < 65504).
__device__ __forceinline__ unsigned act_pk(float a, float b) {
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
    const f16x2 z = __builtin_convertvector((f32x2){a, b}, f16x2);
    const _Float16 k6 = (_Float16)(1.0f / 6.0f);
    const f16x2 c6 = {k6, k6}, c05 = {(_Float16)0.5f, (_Float16)0.5f};
    const f16x2 zero = {(_Float16)0.0f, (_Float16)0.0f}, one = {(_Float16)1.0f, (_Float16)1.0f};
    const f16x2 m2 = {(_Float16)-2.0f, (_Float16)-2.0f}, three = {(_Float16)3.0f, (_Float16)3.0f};
    f16x2 t = __builtin_elementwise_fma(z, c6, c05);
    t = __builtin_elementwise_min(__builtin_elementwise_max(t, zero), one);
    const f16x2 u = __builtin_elementwise_fma(m2, t, three);
    return __builtin_bit_cast(unsigned, z * (t * t * u));
}

// D tile (features x 32 rows) -> act(D) as the FP16 B operands of k blocks 2nt (lo)
// and 2nt + 1 (hi).
__device__ __forceinline__ void tile_to_b(const f32x16 &acc, int h, f16x8 &lo, f16x8 &hi) {
    unsigned P[4][2];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        P[q][0] = act_pk(acc[4 * q], acc[4 * q + 1]);
        P[q][1] = act_pk(acc[4 * q + 2], acc[4 * q + 3]);
    }
    // lane h = 0 keeps features 0-3, 16-19 and needs 4-7, 20-23 from lane l^32;
    // lane h = 1 keeps 12-15, 28-31 and needs 8-11, 24-27.  v_permlane32_swap
    // exchanges the upper 32 lanes of its first operand with the lower 32 lanes
    // of its second: swapping (P[0], P[1]) leaves lanes h = 0 with their own
    // P[0] and their partner's P[0], lanes h = 1 with their partner's P[1] and
    // their own P[1], i.e. features 8h .. 8h + 7 in order in both halves (and
    // (P[2], P[3]) the same for 16 + 8h ..), with no lane-dependent selects.
    unsigned X[2], Y[2], Z[2], W[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const auto a = __builtin_amdgcn_permlane32_swap(P[0][i], P[1][i], false, false);
        const auto b = __builtin_amdgcn_permlane32_swap(P[2][i], P[3][i], false, false);
        X[i] = a[0]; Y[i] = a[1]; Z[i] = b[0]; W[i] = b[1];
    }
    const u32x4 L = u32x4{X[0], X[1], Y[0], Y[1]};
    const u32x4 Hh = u32x4{Z[0], Z[1], W[0], W[1]};
    lo = __builtin_bit_cast(f16x8, L);
    hi = __builtin_bit_cast(f16x8, Hh);
}

typedef __attribute__((address_space(3))) void lds_void;

// Asynchronous copy of 128 rows of 256 FP16 weights into a
// padded LDS image (global_load_lds_dwordx4: each active lane moves 16 B
// straight into LDS; one row = 32 lanes).  Each of the NW waves moves 128/NW rows.
template <int NW>
__device__ __forceinline__ void stage_half_async(const _Float16 *W, _Float16 *wl, int wv, int lane) {
    constexpr int RPWV = 128 / NW;
    if (lane < 32) {
#pragma unroll 8
        for (int r = 0; r < RPWV; ++r) {
            const int row = RPWV * wv + r;
            __builtin_amdgcn_global_load_lds((const void *)(W + row * kNH + lane * 8),
                                             (lds_void *)(wl + row * kRowPad), 16, 0, 0);
        }
    }
}

// Output tiles nt0 .. nt0+3 of one hidden layer from the staged weight rows.  The
// weight operands are read kAhead products ahead and tile nt - 1's activations are
// dealt over tile nt's products (the group barriers: one product, one or two reads, a
// few vector instructions).  The first product's addend is the tile's biases (element
// 4q + t of lane (c, h) is feature 8q + 4h + t).
constexpr int kAhead = 8;

#define ATMO_SG_PRODUCT(READS, VALU)                        \
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);     \
    __builtin_amdgcn_sched_group_barrier(0x100, READS, 0); \
    __builtin_amdgcn_sched_group_barrier(0x002, VALU, 0)

__device__ __forceinline__ void hidden_half(const _Float16 *wl, const float *bias, int nt0, int c, int h,
                                            const f16x8 (&H)[16], f16x8 (&Hn)[16]) {
    f32x16 acc[2], bq[2];
    f16x8 a[kAhead];
    const _Float16 *wrow = wl + c * kRowPad + 8 * h;
    auto bias_tile = [&](int i) {
        const float4 *p = (const float4 *)(bias + 32 * (nt0 + i) + 4 * h);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float4 v = p[2 * q];
            bq[i & 1][4 * q] = v.x; bq[i & 1][4 * q + 1] = v.y; bq[i & 1][4 * q + 2] = v.z; bq[i & 1][4 * q + 3] = v.w;
        }
    };
    auto read = [&](int st) { a[st % kAhead] = *(const f16x8 *)(wrow + 32 * (st / 16) * kRowPad + 16 * (st % 16)); };
    bias_tile(0);
#pragma unroll
    for (int st = 0; st < kAhead; ++st) read(st);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 5; ++i) {
        if (i < 4) {
#pragma unroll
            for (int kb = 0; kb < 16; ++kb) {
                const int st = 16 * i + kb;
                acc[i & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[st % kAhead], H[kb], kb == 0 ? bq[i & 1] : acc[i & 1], 0, 0, 0);
                if (st + kAhead < 64) read(st + kAhead);
            }
            if (i < 3) bias_tile(i + 1);
        }
        if (i > 0) {
            const int nt = nt0 + i - 1;
            tile_to_b(acc[(i - 1) & 1], h, Hn[2 * nt], Hn[2 * nt + 1]);
        }
        ATMO_SG_PRODUCT(1, 0); ATMO_SG_PRODUCT(1, 0); ATMO_SG_PRODUCT(1, 4); ATMO_SG_PRODUCT(1, 4);
        ATMO_SG_PRODUCT(1, 4); ATMO_SG_PRODUCT(1, 4); ATMO_SG_PRODUCT(1, 4); ATMO_SG_PRODUCT(1, 4);
        ATMO_SG_PRODUCT(1, 4); ATMO_SG_PRODUCT(1, 4); ATMO_SG_PRODUCT(1, 4); ATMO_SG_PRODUCT(1, 4);
        ATMO_SG_PRODUCT(2, 4); ATMO_SG_PRODUCT(2, 4); ATMO_SG_PRODUCT(2, 4); ATMO_SG_PRODUCT(2, 4);
        __builtin_amdgcn_sched_barrier(0);
    }
}

__device__ __forceinline__ void wait_all_and_sync() {
    __builtin_amdgcn_s_waitcnt(0);  // the LDS-direct loads of this wave have landed
    __syncthreads();
}

// row_coordinate of every layer and row of every set, into its mu table.
__global__ __launch_bounds__(256) void k_infer_rows(const InferSet *__restrict__ sets) {
    const InferSet &is = sets[blockIdx.y];
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t < is.fs.RR * is.fs.RMU) is.mu[t] = row_coordinate(is.fs, t / is.fs.RMU, t % is.fs.RMU);
}

// A workgroup stays on its CU and walks the tiles of 256 rows (blockIdx.x, + gridDim.x,
// ...): the weights of layers 1 and 5 and the biases are staged once, a tile's exact
// values and the first half of its layer 2 are loaded during the tile before.  LDS:
// rows 0..127 of the current weight in wA, rows 128..255 in wB (528-byte rows), while
// one half is read by the matrix cores the other is refilled for the next step; two
// arrays, not one, so that the compiler does not wait for the one before it reads the
// other.  24 sets of 32x128x32x8 (6.8 TFLOP): a workgroup per tile, with its own
// search, staging, FP64 row coordinates and second read of S, spent 3.0 of 8.2 ms
// outside the hidden layers; the whole call, exact part included, takes 10.15 ms
// against 11.1.  64 rows per wave and 4 waves (half the LDS reads) took 12.4.
template <int NW>
__global__ __launch_bounds__(64 * NW) void k_mlp_infer(const InferSet *__restrict__ sets, int nsets, int ntiles,
                                                       FusedWeights fw, TargetNorm tn) {
    static_assert(kNG == 2, "the layers alternate between two register arrays");
    __shared__ __attribute__((aligned(16))) _Float16 wA[128 * kRowPad], wB[128 * kRowPad];
    __shared__ __attribute__((aligned(16))) __bf16 w1[2 * kNH * 16];           // hi, lo: [256][16]
    __shared__ __attribute__((aligned(16))) _Float16 w5[2 * kNOUT * kRowPad];   // hi rows, lo rows
    __shared__ float bs[kNG][kNH];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, h = lane >> 5, c = lane & 31;
    for (int i = threadIdx.x; i < 1024; i += 64 * NW)
        *(uint4 *)(w1 + i * 8) = *(const uint4 *)((i < 512 ? fw.a1h : fw.a1l) + (i & 511) * 8);
    for (int i = threadIdx.x; i < 256; i += 64 * NW)
        *(uint4 *)(w5 + (i >> 5) * kRowPad + (i & 31) * 8) = *(const uint4 *)((i < 128 ? fw.a5h : fw.a5l) + (i & 127) * 8);
    for (int i = threadIdx.x; i < kNG * kNH; i += 64 * NW) (&bs[0][0])[i] = fw.bh[i];
    __syncthreads();
    stage_half_async<NW>(fw.wt, wA, wv, lane);

    int tile = blockIdx.x, si = 0;   // si: the last set whose first tile is at most `tile`
    for (int hi = nsets - 1; si < hi;) {
        const int mid = (si + hi + 1) >> 1;
        if (sets[mid].tile0 <= tile) si = mid; else hi = mid - 1;
    }
    // this lane's row of a tile, its code and the exact part there, before this kernel adds to it
    auto row_of = [&](const InferSet &is, int tl) { return (tl - is.tile0) * (32 * NW) + wv * 32 + c; };
    auto code_of = [&](const FeatSet &fs, int r) {
        r = min(r, fs.n4 + fs.SW * fs.SH - 1);
        return r < fs.n4 ? (unsigned)r : (0x80000000u | (unsigned)(r - fs.n4));
    };
    auto exact_of = [&](const InferSet &is, int tl) {
        const unsigned code = code_of(is.fs, row_of(is, tl));
        if (!(code & 0x80000000u)) return is.S[code];
        const float *e = is.E + 3 * (size_t)(code & 0x7fffffffu);
        return make_float4(e[0], e[1], e[2], 0.f);
    };
    float4 ex = exact_of(sets[si], tile);
    for (;;) {
        const InferSet &is = sets[si];
        const int next = tile + (int)gridDim.x;
        const bool more = next < ntiles;
        int sn = si;
        while (more && sn + 1 < nsets && sets[sn + 1].tile0 <= next) ++sn;
        f16x8 H[16], Hn[16];
        // (1) features and layer 1
        {
            const FeatSet fs = is.fs;
            const float e3[3] = {ex.x, ex.y, ex.z};
            float x[kNIN];
            texel_features(fs, code_of(fs, row_of(is, tile)), e3, x, is.mu);
            float xe[16];
#pragma unroll
            for (int k = 0; k < 16; ++k) xe[k] = k < kNIN ? x[k] : (k == kNIN ? 1.0f : 0.0f);
            bf16x8 xh, xl;
            const unsigned hm = 0u - (unsigned)h;  // all ones on lanes 32..63
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                // lane half h takes input columns 8h .. 8h+7 (bit select, no indexed array)
                const float v = __uint_as_float((__float_as_uint(xe[i]) & ~hm) | (__float_as_uint(xe[8 + i]) & hm));
                const __bf16 vh = (__bf16)v;
                xh[i] = vh;
                xl[i] = (__bf16)(v - (float)vh);
            }
#pragma unroll
            for (int nt = 0; nt < 8; ++nt) {
                const bf16x8 ah = *(const bf16x8 *)(w1 + (32 * nt + c) * 16 + 8 * h);
                const bf16x8 al = *(const bf16x8 *)(w1 + kNH * 16 + (32 * nt + c) * 16 + 8 * h);
                f32x16 acc;
#pragma unroll
                for (int j = 0; j < 16; ++j) acc[j] = 0.0f;
                acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, xh, acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al, xh, acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, xl, acc, 0, 0, 0);
                tile_to_b(acc, h, H[2 * nt], H[2 * nt + 1]);
            }
        }
        // (2) hidden layers 2 and 3
        float4 exn = ex;
#pragma unroll
        for (int L = 0; L < kNG; ++L) {
            const _Float16 *W = fw.wt + (size_t)L * kNH * kNH;
            wait_all_and_sync();                                        // wA holds rows 0..127; wB is free
            stage_half_async<NW>(W + 128 * kNH, wB, wv, lane);
            hidden_half(wA, bs[L], 0, c, h, L ? Hn : H, L ? H : Hn);
            wait_all_and_sync();                                        // wB holds rows 128..255; wA is free
            if (L < kNG - 1) {
                stage_half_async<NW>(W + (size_t)kNH * kNH, wA, wv, lane);
            } else if (more) {   // for the next tile
                stage_half_async<NW>(fw.wt, wA, wv, lane);
                exn = exact_of(sets[sn], next);
            }
            hidden_half(wB, bs[L], 4, c, h, L ? Hn : H, L ? H : Hn);
        }
        // (3) layer 5, its hi rows in D rows 0..3 and its lo rows in 4..7 (the other rows repeat
        // them and are not used), and the combination with the exact part
        f32x16 acc;
#pragma unroll
        for (int j = 0; j < 16; ++j) acc[j] = 0.0f;
#pragma unroll
        for (int kb = 0; kb < 16; ++kb)
            acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(*(const f16x8 *)(w5 + (c & 7) * kRowPad + 16 * kb + 8 * h), H[kb], acc, 0, 0, 0);
        const int r = row_of(is, tile);
        float v[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) {   // lanes h = 0: hi rows in acc[0..3], lanes h = 1: lo rows
            const float y = acc[k] + __shfl_xor(acc[k], 32, 64);
            v[k] = fmaxf(__expf((y + fw.b5[k]) * tn.sd[k] + tn.mu[k]) - tn.eps, 0.f);
        }
        if (h == 0 && r < is.fs.n4) {
            is.S[r] = make_float4(ex.x + v[0], ex.y + v[1], ex.z + v[2], ex.w);
        } else if (h == 0 && r < is.fs.n4 + is.fs.SW * is.fs.SH) {
            float *e = is.E + 3 * (size_t)(r - is.fs.n4);
            e[0] = ex.x + v[0]; e[1] = ex.y + v[1]; e[2] = ex.z + v[2];
        }
        if (!more) break;
        tile = next;
        si = sn;
        ex = exn;
    }
}

// ---------------------------------------------------------------------------
// Training pass, forward and backward of a batch in one kernel (k_train_rows), the
// hidden layers' weight gradients in a second (k_train_dw) and the sums over
// workgroups in a third (k_train_reduce).
//
// k_train_rows keeps 32 rows per wave in registers as k_mlp_infer does (products
// transposed, D = W^T H^T, bf16 weights of one or two layers staged in LDS) and
// recomputes pre-activations where the backward pass needs them instead of storing
// them: layer 3's when its output gradient is known, layer 2's beside the products
// that make its gradient, layer 1's likewise.  Two more 256x256 products per row cost
// less than 400 MB of FP32 pre-activations and gradients written and read.  Every
// value is rounded where a layer-by-layer pass rounds it (bf16 activations and
// gradients, FP32 pre-activations) and summed in its order: k ascending on the matrix
// cores, layer 1 as an FMA chain from the bias (v_mfma_f32_32x32x2_f32 gives an FMA
// chain's bits), layer 5 over the butterfly's tree.
//
// The activations and gradients that the weight gradients contract over the rows
// leave it transposed, as operand fragments: a product with the identity turns a
// register tile (lane = row) into lane = feature, 16 rows per lane, exactly; each
// store is one contiguous KB per wave and k_train_dw loads fragments straight into
// registers.  The row order inside a block of 16 is the C layout's (8q + 4h + t) for
// both operands of a product, so it cancels.
//
// 65,536 rows: 103 us, k_train_dw 35, k_train_reduce 18; the layer-by-layer kernels took 790
// (GEMMs 420, bias sums 80, layers 1 and 5 250, sums 34).
// ---------------------------------------------------------------------------
typedef float f32x4 __attribute__((ext_vector_type(4)));
constexpr int kTrainWaves = 8;
constexpr int kPart5 = kNH * kNOUT + 8;   // dW5, db5, loss of a wave
struct TrainLds {
    __bf16 w[kNH * kRowPad];              // staged weights; at the end the FP32 transposes and sums
    float w1[kNIN * kNH], b[3 * kNH];     // layer 1's weights; b1, b2, b3
    float4 w5[kNH];
    float4 dy[kTrainWaves][32];
};

// D tile (features x 32 rows, FP32) -> bf16 B operands of k blocks 2nt (lo), 2nt + 1 (hi): tile_to_b's relayout
__device__ __forceinline__ void tile_to_bf16(const float (&v)[16], bf16x8 &lo, bf16x8 &hi) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    unsigned P[4][2];
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const bf16x2 p = {(__bf16)v[4 * q + 2 * i], (__bf16)v[4 * q + 2 * i + 1]};
            P[q][i] = __builtin_bit_cast(unsigned, p);
        }
    u32x4 L, H;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const auto a = __builtin_amdgcn_permlane32_swap(P[0][i], P[1][i], false, false);
        const auto b = __builtin_amdgcn_permlane32_swap(P[2][i], P[3][i], false, false);
        L[i] = a[0]; L[2 + i] = a[1]; H[i] = b[0]; H[2 + i] = b[1];
    }
    lo = __builtin_bit_cast(bf16x8, L);
    hi = __builtin_bit_cast(bf16x8, H);
}
// The identity's 16 x 32 halves as B operands
__device__ __forceinline__ bf16x8 identity(int c, int h, int half) {
    bf16x8 v;
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = (__bf16)(c == 16 * half + 8 * h + j ? 1.0f : 0.0f);
    return v;
}
// tile (lane = row) -> lane = feature c, rows 8q + 4h + t in elements 4q + t
__device__ __forceinline__ f32x16 transpose_tile(const bf16x8 &lo, const bf16x8 &hi, int c, int h) {
    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(lo, identity(c, h, 0), acc, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(hi, identity(c, h, 1), acc, 0, 0, 0);
}
// k block u of a transposed tile (16 rows): exact bf16 values, their upper halves
__device__ __forceinline__ u32x4 fragment(const f32x16 &t, int u) {
    u32x4 v;
#pragma unroll
    for (int i = 0; i < 4; ++i)
        v[i] = __builtin_amdgcn_perm(__float_as_uint(t[8 * u + 2 * i + 1]), __float_as_uint(t[8 * u + 2 * i]), 0x07060302u);
    return v;
}
// fragments of feature tile nt of a 32-row block (`out`, scalar): two k blocks of 16 rows, 16 B
// per lane each.  Global stores with a scalar base: after a buffer store with a scalar
// offset the compiler lets the next instruction overwrite the data registers, and under
// load stores then wrote the new values.
__device__ __forceinline__ void store_fragments(__bf16 *out, int nt, int lane, const f32x16 &t) {
#pragma unroll
    for (int u = 0; u < 2; ++u) *(u32x4 *)((char *)out + (unsigned)((nt * 2 + u) * 1024 + lane * 16)) = fragment(t, u);
}
// tile nt of a 256x256 product from staged weight rows (row 0 of `w` is row 0 of the tile's half)
__device__ __forceinline__ f32x16 train_tile(const __bf16 *w, int nt, int c, int h, const bf16x8 (&H)[16]) {
    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
    const __bf16 *row = w + (32 * nt + c) * kRowPad + 8 * h;
#pragma unroll
    for (int kb = 0; kb < 16; ++kb)
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*(const bf16x8 *)(row + 16 * kb), H[kb], acc, 0, 0, 0);
    return acc;
}
// pre-activations of layer 1's tile nt: b1 + the chain over the inputs
__device__ __forceinline__ f32x16 layer1_tile(const TrainLds &S, int nt, int c, int h, const float (&xf)[7]) {
    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = S.b[32 * nt + 8 * (r >> 2) + 4 * h + (r & 3)];
#pragma unroll
    for (int k = 0; k < 7; ++k)
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(S.w1[(2 * k + h) * kNH + 32 * nt + c], xf[k], acc, 0, 0, 0);
    return acc;
}
// Asynchronous copy of 128 rows of a weight, from row r0, into the LDS image (stage_half_async
// with scalar row addresses, which take no vector registers)
__device__ __forceinline__ void stage_train(const __bf16 *W, __bf16 *wl, int r0, int wv, int lane) {
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void *)W, (short)0, kNH * kNH * 2, 0x00020000);
    if (lane < 32) {
#pragma unroll 1   // (unrolled, its row addresses would take 64 scalar registers)
        for (int i = 0; i < 128 / kTrainWaves; ++i) {
            const int row = r0 + 128 / kTrainWaves * wv + i;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void *)(wl + row * kRowPad), 16, lane * 16, row * kNH * 2, 0, 0);
        }
    }
}

__global__ __launch_bounds__(64 * kTrainWaves) void k_train_rows(TrainArgs a) {
    static_assert(kNL == 3 && kNIN == 14 && kNOUT == 4 && kNH == 256, "the layer sequence is written out");
    extern __shared__ __attribute__((aligned(16))) char smem[];
    TrainLds &S = *(TrainLds *)smem;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), h = lane >> 5, c = lane & 31;
    const int row0 = ((int)blockIdx.x * kTrainWaves + wv) * 32;
    const bool active = row0 < a.rows;   // rows is a multiple of 32: whole waves
    const int row = min(row0, a.rows - 32) + c, rb = row0 / 32;
    __bf16 *wA = S.w, *wB = S.w + 128 * kRowPad;
    for (int i = threadIdx.x; i < kNIN * kNH; i += 64 * kTrainWaves) S.w1[i] = a.W1[i];
    for (int i = threadIdx.x; i < kNH; i += 64 * kTrainWaves) {
        S.b[i] = a.b1[i];
        S.b[kNH + i] = a.b2[i];
        S.b[2 * kNH + i] = a.b3[i];
        S.w5[i] = make_float4(a.W5[4 * i], a.W5[4 * i + 1], a.W5[4 * i + 2], a.W5[4 * i + 3]);
    }
    float xf[7];
#pragma unroll
    for (int k = 0; k < 7; ++k) xf[k] = a.X[(size_t)row * kXS + 2 * k + h];
    __syncthreads();
    stage_train(a.w2t, wA, 0, wv, lane);
    stage_train(a.w2t, wA, 128, wv, lane);
    const float *b2 = S.b + kNH, *b3 = S.b + 2 * kNH;

    bf16x8 H1[16], H2[16];
#pragma unroll
    for (int nt = 0; nt < 8; ++nt) {   // layer 1
        const f32x16 z = layer1_tile(S, nt, c, h, xf);
        float v[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) v[r] = act(z[r]);
        tile_to_bf16(v, H1[2 * nt], H1[2 * nt + 1]);
        const f32x16 t = transpose_tile(H1[2 * nt], H1[2 * nt + 1], c, h);
        if (active) store_fragments(a.h1 + (size_t)rb * 32 * kNH, nt, lane, t);
    }
    wait_all_and_sync();
    auto forward_tile = [&](const float *bias, int nt, const bf16x8 (&In)[16], bf16x8 &lo, bf16x8 &hi) {
        const f32x16 z = train_tile(S.w, nt, c, h, In);
        float v[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) v[r] = act(z[r] + bias[32 * nt + 8 * (r >> 2) + 4 * h + (r & 3)]);
        tile_to_bf16(v, lo, hi);
    };
#pragma unroll
    for (int nt = 0; nt < 8; ++nt) {   // layer 2
        if (nt == 4) {
            wait_all_and_sync();
            stage_train(a.w3t, wA, 0, wv, lane);
        }
        forward_tile(b2, nt, H1, H2[2 * nt], H2[2 * nt + 1]);
        const f32x16 t = transpose_tile(H2[2 * nt], H2[2 * nt + 1], c, h);
        if (active) store_fragments(a.h2 + (size_t)rb * 32 * kNH, nt, lane, t);
    }
    wait_all_and_sync();
    stage_train(a.w3t, wA, 128, wv, lane);
    float dyf[2];   // this lane's half of the output gradients
    float *part5 = a.part5 + (size_t)rb * kPart5;
    {
        bf16x8 H3[16];
#pragma unroll
        for (int nt = 0; nt < 8; ++nt) {   // layer 3
            if (nt == 4) wait_all_and_sync();
            forward_tile(b3, nt, H2, H3[2 * nt], H3[2 * nt + 1]);
        }
        // layer 5: 4-input chains, then the tree of a 64-lane butterfly (chain L = features 4L ..
        // 4L + 3 with L + 32, 16, 8, 4, 2, 1); L = 4 kb + 2h + j
        float y[2][4];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            float s[16][4];
#pragma unroll
            for (int kb = 0; kb < 16; ++kb) {
#pragma unroll
                for (int o = 0; o < 4; ++o) s[kb][o] = 0.f;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float hv = (float)H3[kb][4 * j + q];
                    const float4 w = S.w5[16 * kb + 8 * h + 4 * j + q];
                    s[kb][0] = fmaf(hv, w.x, s[kb][0]);
                    s[kb][1] = fmaf(hv, w.y, s[kb][1]);
                    s[kb][2] = fmaf(hv, w.z, s[kb][2]);
                    s[kb][3] = fmaf(hv, w.w, s[kb][3]);
                }
                // combine as soon as the partners of a level are there
                if (kb >= 8) {
#pragma unroll
                    for (int o = 0; o < 4; ++o) s[kb - 8][o] += s[kb][o];
                }
            }
#pragma unroll
            for (int off = 4; off > 0; off >>= 1)
#pragma unroll
                for (int kb = 0; kb < off; ++kb)
#pragma unroll
                    for (int o = 0; o < 4; ++o) s[kb][o] += s[kb + off][o];
#pragma unroll
            for (int o = 0; o < 4; ++o) y[j][o] = s[0][o] + __shfl_xor(s[0][o], 32, 64);
        }
        const float inv = 1.0f / ((float)a.rows * kNOUT);
        float d[5];
        d[4] = 0.f;
#pragma unroll
        for (int o = 0; o < 4; ++o) {
            const float e = (y[0][o] + y[1][o]) + a.b5[o] - a.T[(size_t)row * kNOUT + o];
            d[o] = 2.0f * e * inv;
            d[4] += e * e;
        }
        dyf[0] = h ? d[1] : d[0];
        dyf[1] = h ? d[3] : d[2];
        if (h == 0) S.dy[wv][c] = make_float4(d[0], d[1], d[2], d[3]);
        __builtin_amdgcn_wave_barrier();
        // dW5 = H3^T dY over this wave's rows on the bf16 matrix cores: dY is exactly the sum of
        // three bf16 numbers, columns o, 4 + o and 8 + o of the right operand, whose products
        // add up in FP32; db5 and the loss
        bf16x8 dyb[2];
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const float v = ((const float *)&S.dy[wv][8 * (2 * u + (j >> 2)) + 4 * h + (j & 3)])[c & 3];
                const __bf16 hi = (__bf16)v, mid = (__bf16)(v - (float)hi), lo = (__bf16)((v - (float)hi) - (float)mid);
                dyb[u][j] = c < 4 ? hi : c < 8 ? mid : c < 12 ? lo : (__bf16)0.0f;
            }
#pragma unroll
        for (int nt = 0; nt < 8; ++nt) {
            const f32x16 t = transpose_tile(H3[2 * nt], H3[2 * nt + 1], c, h);
            f32x16 g;
#pragma unroll
            for (int r = 0; r < 16; ++r) g[r] = 0.0f;
#pragma unroll
            for (int u = 0; u < 2; ++u)
                g = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, fragment(t, u)), dyb[u], g, 0, 0, 0);
            float w[16];
#pragma unroll
            for (int r = 0; r < 16; ++r) {   // columns o + (4 + o) + (8 + o) (row_shl by 4 and by 8 lanes)
                const int v = __float_as_int(g[r]);
                w[r] = g[r] + (__int_as_float(__builtin_amdgcn_update_dpp(0, v, 0x104, 0xf, 0xf, true)) +
                               __int_as_float(__builtin_amdgcn_update_dpp(0, v, 0x108, 0xf, 0xf, true)));
            }
            if (active && c < 4) {
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    *(float4 *)(part5 + kNH * c + 32 * nt + 8 * q + 4 * h) =
                        make_float4(w[4 * q], w[4 * q + 1], w[4 * q + 2], w[4 * q + 3]);
            }
        }
#pragma unroll
        for (int o = 0; o < 5; ++o) {
#pragma unroll
            for (int off = 16; off > 0; off >>= 1) d[o] += __shfl_xor(d[o], off, 64);
            if (active && lane == 0) part5[kNH * kNOUT + o] = o < 4 ? d[o] : d[o] * inv;
        }
    }
    bf16x8 D3[16];
#pragma unroll
    for (int nt = 0; nt < 8; ++nt) {   // dZ3 = (dY W5^T) act'(Z3), Z3 again
        if (nt == 4) {
            wait_all_and_sync();
            stage_train(a.w3b, wA, 0, wv, lane);
        }
        const f32x16 z = train_tile(S.w, nt, c, h, H2);
        f32x16 g;   // dY W5^T, an FMA chain over the outputs
#pragma unroll
        for (int r = 0; r < 16; ++r) g[r] = 0.0f;
#pragma unroll
        for (int k = 0; k < 2; ++k)
            g = __builtin_amdgcn_mfma_f32_32x32x2f32(((const float *)&S.w5[32 * nt + c])[2 * k + h], dyf[k], g, 0, 0, 0);
        float v[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) v[r] = g[r] * dact(z[r] + b3[32 * nt + 8 * (r >> 2) + 4 * h + (r & 3)]);
        tile_to_bf16(v, D3[2 * nt], D3[2 * nt + 1]);
        const f32x16 t = transpose_tile(D3[2 * nt], D3[2 * nt + 1], c, h);
        if (active) store_fragments(a.d3 + (size_t)rb * 32 * kNH, nt, lane, t);
    }
    bf16x8 D2[16];
#pragma unroll
    for (int half = 0; half < 2; ++half) {   // dZ2 = (dZ3 W3^T) act'(Z2), Z2 again
        wait_all_and_sync();
        if (half == 1) stage_train(a.w3b, wA - 128 * kRowPad, 128, wv, lane);
        stage_train(a.w2t, wB - 128 * half * kRowPad, 128 * half, wv, lane);
        wait_all_and_sync();
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int nt = 4 * half + i;
            const f32x16 z = train_tile(wB, i, c, h, H1), p = train_tile(wA, i, c, h, D3);
            float v[16];
#pragma unroll
            for (int r = 0; r < 16; ++r) v[r] = p[r] * dact(z[r] + b2[32 * nt + 8 * (r >> 2) + 4 * h + (r & 3)]);
            tile_to_bf16(v, D2[2 * nt], D2[2 * nt + 1]);
            const f32x16 t = transpose_tile(D2[2 * nt], D2[2 * nt + 1], c, h);
            if (active) store_fragments(a.d2 + (size_t)rb * 32 * kNH, nt, lane, t);
        }
    }
    wait_all_and_sync();
    stage_train(a.w2b, wA, 0, wv, lane);
    stage_train(a.w2b, wA, 128, wv, lane);
    wait_all_and_sync();
    // dZ1 = (dZ2 W2^T) act'(Z1), Z1 again, FP32; dW1 and db1 (input 14 is 1) over this wave's
    // rows: dZ1 through LDS, 64 features at a time, FP32 products on the matrix cores.  The
    // transposes go where the first half of the weight was; a row's float4 e is at
    // e ^ (4 (row % 4) + row / 4 % 4), which spreads writes and reads over the banks.
    float xa[8];
    const int m = lane & 15, k4 = lane >> 4;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const float x = m < kNIN ? a.X[(size_t)(min(row0, a.rows - 32) + 4 * k + k4) * kXS + m] : m == kNIN ? 1.0f : 0.0f;
        xa[k] = active ? x : 0.0f;
    }
    float *tw = (float *)S.w + wv * (32 * 64);
    f32x4 dw[16];
#pragma unroll
    for (int half = 0; half < 2; ++half) {
        float g1[4][16];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const f32x16 z = layer1_tile(S, 4 * half + i, c, h, xf), p = train_tile(S.w, 4 * half + i, c, h, D2);
#pragma unroll
            for (int r = 0; r < 16; ++r) g1[i][r] = p[r] * dact(z[r]);
        }
        if (half == 0) __syncthreads();   // every wave is done with the first half
#pragma unroll
        for (int pair = 0; pair < 2; ++pair) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float (&g)[16] = g1[2 * pair + i];
                    *(float4 *)(tw + c * 64 + 4 * ((8 * i + 2 * q + h) ^ (4 * (c & 3) + ((c >> 2) & 3)))) =
                        make_float4(g[4 * q], g[4 * q + 1], g[4 * q + 2], g[4 * q + 3]);
                }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int n = 0; n < 4; ++n) {
                f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int k = 0; k < 8; ++k)   // row 4 k + k4, feature 16 n + m
                    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(
                        xa[k], tw[(4 * k + k4) * 64 + 4 * ((4 * n + (m >> 2)) ^ (4 * k4 + (k & 3))) + (m & 3)], acc, 0, 0, 0);
                dw[8 * half + 4 * pair + n] = acc;
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
    }
    __syncthreads();
    float *ws = (float *)S.w;   // [wave][16][256]
#pragma unroll
    for (int n = 0; n < 16; ++n)
#pragma unroll
        for (int r = 0; r < 4; ++r) ws[(wv * 16 + 4 * k4 + r) * kNH + 16 * n + m] = dw[n][r];
    __syncthreads();
    for (int e = threadIdx.x; e < 15 * kNH; e += 64 * kTrainWaves) {
        float sum = 0.f;
#pragma unroll
        for (int w = 0; w < kTrainWaves; ++w) sum += ws[w * 16 * kNH + e];
        a.part1[(size_t)blockIdx.x * 15 * kNH + e] = sum;
    }
}

// dW = H^T dZ of layers 2 (blockIdx.z 0) and 3 over a range of 32-row blocks, one
// 128 x 128 tile per workgroup (blockIdx.y), 64 x 64 per wave, straight from the
// fragments; db = the column sums of dZ as products with ones.  A tile's fragments are
// read by two waves of a workgroup and two workgroups, which share an XCD's L2 (the
// range is blockIdx.x, a multiple of 8 of them where there are that many).
__global__ __launch_bounds__(256) void k_train_dw(const __bf16 *h1, const __bf16 *d2, const __bf16 *h2, const __bf16 *d3,
                                                  int nrb, float *__restrict__ part, float *__restrict__ partb) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, h = lane >> 5, c = lane & 31;
    const __bf16 *A = blockIdx.z ? h2 : h1, *B = blockIdx.z ? d3 : d2;
    const int mt = (blockIdx.y >> 1) * 4 + (w >> 1) * 2, nt = (blockIdx.y & 1) * 4 + (w & 1) * 2;
    const int ns = gridDim.x, rb0 = (int)((long long)nrb * blockIdx.x / ns), rb1 = (int)((long long)nrb * (blockIdx.x + 1) / ns);
    const bool bias = mt == 0;
    f32x16 acc[2][2], sum[2];
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[0][0][r] = acc[0][1][r] = acc[1][0][r] = acc[1][1][r] = sum[0][r] = sum[1][r] = 0.0f;
    bf16x8 ones;
#pragma unroll
    for (int j = 0; j < 8; ++j) ones[j] = (__bf16)1.0f;
    struct Frag {
        bf16x8 a[2][2], b[2][2];   // [tile][k block]
    };
    auto load = [&](int rb) {
        Frag f;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                f.a[i][u] = *(const bf16x8 *)(A + ((((size_t)rb * 8 + mt + i) * 2 + u) * 64 + lane) * 8);
                f.b[i][u] = *(const bf16x8 *)(B + ((((size_t)rb * 8 + nt + i) * 2 + u) * 64 + lane) * 8);
            }
        return f;
    };
    Frag f0 = load(rb0), f1 = load(min(rb0 + 1, rb1 - 1));
    for (int rb = rb0; rb < rb1; ++rb) {
        const Frag f = f0;
        f0 = f1;
        f1 = load(min(rb + 2, rb1 - 1));
#pragma unroll
        for (int u = 0; u < 2; ++u) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.a[i][u], f.b[j][u], acc[i][j], 0, 0, 0);
            if (bias) {
#pragma unroll
                for (int j = 0; j < 2; ++j) sum[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ones, f.b[j][u], sum[j], 0, 0, 0);
            }
        }
    }
    const size_t split = (size_t)blockIdx.z * ns + blockIdx.x;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                part[split * kNH * kNH + (size_t)(32 * (mt + i) + 8 * (r >> 2) + 4 * h + (r & 3)) * kNH + 32 * (nt + j) + c] = acc[i][j][r];
    if (bias && h == 0) {
#pragma unroll
        for (int j = 0; j < 2; ++j) partb[split * kNH + 32 * (nt + j) + c] = sum[j][0];
    }
}

// Gradient e (and, behind the parameters, the loss) = the sum of its partials, with 4 threads
// per value (16 for the waves' partials, of which there are 8 times as many as of workgroups),
// up to 16 loads in flight each: 24 us with 16 threads per value everywhere, 18 so.
// Parameters: W1, b1 (partials of workgroups), W2, b2, W3, b3 (of row ranges), W5, b5, loss (of waves).
constexpr int kRedL1 = 15 * kNH, kRedLH = kNH * kNH + kNH, kRed5 = kRedL1 + kNG * kRedLH, kRedN = kRed5 + kNH * kNOUT + kNOUT;
__global__ __launch_bounds__(256) void k_train_reduce(const float *__restrict__ part1, int nwg, const float *__restrict__ part,
                                                      const float *__restrict__ partb, int ns, const float *__restrict__ part5,
                                                      int nwave, float *__restrict__ g, float *__restrict__ loss) {
    static_assert(kRed5 % 64 == 0, "a workgroup's values have one kind of partials");
    __shared__ float s[256];
    const bool waves = blockIdx.x >= kRed5 / 64;
    const int E = waves ? 16 : 64, S = 256 / E, x = threadIdx.x % E, k0 = threadIdx.x / E;
    const int e = waves ? kRed5 + ((int)blockIdx.x - kRed5 / 64) * 16 + x : (int)blockIdx.x * 64 + x;
    const float *p = part1 + e;
    int count = nwg;
    size_t stride = kRedL1;
    if (waves) {
        const int i = e - kRed5;   // W5 as [output][256] there
        p = part5 + (i < kNH * kNOUT ? (i % kNOUT) * kNH + i / kNOUT : i);
        count = nwave;
        stride = kPart5;
    } else if (e >= kRedL1) {
        const int L = (e - kRedL1) / kRedLH, i = (e - kRedL1) % kRedLH;
        count = ns;
        stride = i < kNH * kNH ? kNH * kNH : kNH;
        p = (i < kNH * kNH ? part + i : partb + (i - kNH * kNH)) + (size_t)L * ns * stride;
    }
    float v = 0.f;
    if (e <= kRedN) {
        int k = k0;
        for (; k + 15 * S < count; k += 16 * S) {
            float y[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) y[i] = p[(k + i * S) * stride];
#pragma unroll
            for (int i = 0; i < 16; ++i) v += y[i];
        }
        for (; k < count; k += S) v += p[k * stride];
    }
    s[threadIdx.x] = v;
    __syncthreads();
    if (k0 == 0 && e <= kRedN) {
        for (int k = 1; k < S; ++k) v += s[k * E + x];
        if (e < kRedN) g[e] = v;
        else *loss = v;
    }
}

// Weights of the fused kernel from the FP32 parameters: layer 1 (+ bias in
// column 14) split into bf16 hi/lo, layer 5 into FP16 hi/lo, the hidden
// weights as FP16 [out][in] and their biases packed.
__global__ __launch_bounds__(256) void k_prep_fused(const float *__restrict__ W1, const float *__restrict__ b1,
                                                    const float *__restrict__ W5, const float *__restrict__ Wh0,
                                                    const float *__restrict__ bh0, size_t bstride, __bf16 *a1h,
                                                    __bf16 *a1l, _Float16 *wt, _Float16 *a5h, _Float16 *a5l,
                                                    float *bh) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < kNH * 16) {
        const int nn = i / 16, k = i % 16;
        const float v = k < kNIN ? W1[k * kNH + nn] : (k == kNIN ? b1[nn] : 0.0f);
        const __bf16 vh = (__bf16)v;
        a1h[i] = vh;
        a1l[i] = (__bf16)(v - (float)vh);
    } else if (i < kNH * 16 + kNOUT * kNH) {
        const int j = i - kNH * 16, o = j / kNH, k = j % kNH;
        const float v = W5[k * kNOUT + o];
        const _Float16 vh = (_Float16)v;
        a5h[j] = vh;
        a5l[j] = (_Float16)(v - (float)vh);
    } else if (i < kNH * 16 + kNOUT * kNH + kNG * kNH) {
        const int j = i - kNH * 16 - kNOUT * kNH;
        bh[j] = bh0[(size_t)(j / kNH) * bstride + j % kNH];
    } else if (i < kNH * 16 + kNOUT * kNH + kNG * kNH + kNG * kNH * kNH) {
        const int j = i - kNH * 16 - kNOUT * kNH - kNG * kNH;   // layer L, output n, input k
        const int L = j / (kNH * kNH), n = (j / kNH) % kNH, k = j % kNH;
        wt[j] = (_Float16)Wh0[(size_t)L * bstride + (size_t)k * kNH + n];
    }
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
hipError_t gemm_act(const __bf16 *A, const __bf16 *B, int M, int N, int K, const float *bias, __bf16 *hout, hipStream_t st) {
    if (M % 128 || N % 128 || K % 32) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_gemm_act, dim3(N / 128, M / 128), dim3(256), 0, st, A, B, M, N, K, bias, hout);
    return hipGetLastError();
}

static unsigned blocks(size_t n) { return (unsigned)((n + 255) / 256); }

hipError_t layer1_fwd(const float *X, const float *W1, const float *b1, int rows, __bf16 *H1, hipStream_t st) {
    hipLaunchKernelGGL(k_layer1_fwd, dim3(blocks((size_t)rows * kNH)), dim3(256), 0, st, X, W1, b1, rows, H1);
    return hipGetLastError();
}
hipError_t layer5(const __bf16 *H4, const float *W5, const float *b5, int rows, float *Y, hipStream_t st) {
    hipLaunchKernelGGL(k_layer5, dim3((rows + 63) / 64), dim3(256), 0, st, H4, W5, b5, rows, Y);
    return hipGetLastError();
}
hipError_t adam(float *p, const float *g, float *m, float *v, int n, float lr, float b1, float b2,
                float eps, float c1, float c2, hipStream_t st) {
    hipLaunchKernelGGL(k_adam, dim3(blocks(n)), dim3(256), 0, st, p, g, m, v, n, lr, b1, b2, eps, c1, c2);
    return hipGetLastError();
}
hipError_t to_bf16(const float *W, __bf16 *Wb, __bf16 *Wt, hipStream_t st) {
    hipLaunchKernelGGL(k_to_bf16, dim3(blocks(kNH * kNH)), dim3(256), 0, st, W, Wb, Wt);
    return hipGetLastError();
}
hipError_t make_rows(const FeatSet &fs, const float4 *S4, const float4 *S1, const float *E, const float *E1, int ns,
                     unsigned long long seed, float *X, float *Tg, const TargetNorm &tn, hipStream_t st) {
    const int n = ns + fs.SW * fs.SH;
    hipLaunchKernelGGL(k_make_rows, dim3(blocks(n)), dim3(256), 0, st, fs, S4, S1, E, E1, ns, seed, X, Tg, tn);
    return hipGetLastError();
}
hipError_t code_rows(const FeatSet &fs, const unsigned *codes, int n, const float4 *S1, const float *E1, float *X,
                     hipStream_t st) {
    hipLaunchKernelGGL(k_code_rows, dim3(blocks(n)), dim3(256), 0, st, fs, codes, n, S1, E1, X);
    return hipGetLastError();
}
hipError_t target_stats(const float *Tg, size_t n, double *out, hipStream_t st) {
    hipLaunchKernelGGL(k_target_stats, dim3(1024), dim3(256), 0, st, Tg, n, out);
    return hipGetLastError();
}
hipError_t norm_targets(float *Tg, size_t n, const TargetNorm &tn, hipStream_t st) {
    hipLaunchKernelGGL(k_norm_targets, dim3(blocks(n)), dim3(256), 0, st, Tg, n, tn);
    return hipGetLastError();
}
hipError_t gather(const float *Xa, const float *Ta, size_t n, int B, unsigned long long seed, float *X,
                  float *Tg, hipStream_t st) {
    hipLaunchKernelGGL(k_gather, dim3(blocks(B)), dim3(256), 0, st, Xa, Ta, n, B, seed, X, Tg);
    return hipGetLastError();
}
hipError_t relerr(const float *a, const float *b, size_t n, int stride, int ncomp, float floorv,
                  unsigned *out, hipStream_t st) {
    hipLaunchKernelGGL(k_relerr, dim3(blocks(n)), dim3(256), 0, st, a, b, n, stride, ncomp, floorv, out);
    return hipGetLastError();
}
hipError_t absmax(const float *a, size_t n, int stride, int ncomp, unsigned *out, hipStream_t st) {
    hipLaunchKernelGGL(k_absmax, dim3(blocks(n)), dim3(256), 0, st, a, n, stride, ncomp, out);
    return hipGetLastError();
}

}  // namespace sg
}  // namespace atmo

namespace atmo {
namespace sg {
constexpr int kFusedNW = 8;
int fused_rows_per_block() { return 32 * kFusedNW; }
hipError_t prep_fused(const float *W1, const float *b1, const float *W5, const float *Wh0, const float *bh0,
                      size_t bstride, __bf16 *a1h, __bf16 *a1l, _Float16 *wt, _Float16 *a5h, _Float16 *a5l,
                      float *bh, hipStream_t st) {
    const int n = kNH * 16 + kNOUT * kNH + kNG * kNH + kNG * kNH * kNH;
    hipLaunchKernelGGL(k_prep_fused, dim3(blocks(n)), dim3(256), 0, st, W1, b1, W5, Wh0, bh0, bstride, a1h, a1l,
                       wt, a5h, a5l, bh);
    return hipGetLastError();
}
// Kernels that take more dynamic LDS than the default limit: raised once per device.
static hipError_t raise_lds(const void *kernel, size_t bytes, unsigned long long &done) {
    static std::mutex mu;
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= 64) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lk(mu);
    if (!(done & (1ull << dev))) {
        e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
        if (e != hipSuccess) return e;
        done |= 1ull << dev;
    }
    return hipSuccess;
}

// Row ranges of k_train_dw: at least 4 blocks of 32 rows each, at most 64 (512 workgroups)
static int dw_ranges(int rows) { return std::max(1, std::min(64, rows / 128)); }
size_t train_scratch(int rows) {
    const size_t nwg = (rows + 255) / 256, ns = dw_ranges(rows);
    return sizeof(float) * (nwg * 15 * kNH + (size_t)(rows / 32) * kPart5 + 2 * ns * ((size_t)kNH * kNH + kNH));
}
hipError_t train_pass(TrainArgs a, float *scratch, float *g, float *loss, hipStream_t st) {
    if (a.rows <= 0 || a.rows % 32) return hipErrorInvalidValue;
    const int nwg = (a.rows + 255) / 256, ns = dw_ranges(a.rows), nrb = a.rows / 32;
    a.part5 = scratch;   // 16-byte stores
    a.part1 = a.part5 + (size_t)nrb * kPart5;
    float *part = a.part1 + (size_t)nwg * 15 * kNH, *partb = part + (size_t)2 * ns * kNH * kNH;
    static unsigned long long done = 0;
    hipError_t e = raise_lds((const void *)k_train_rows, sizeof(TrainLds), done);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_train_rows, dim3(nwg), dim3(64 * kTrainWaves), sizeof(TrainLds), st, a);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    hipLaunchKernelGGL(k_train_dw, dim3(ns, 4, 2), dim3(256), 0, st, a.h1, a.d2, a.h2, a.d3, nrb, part, partb);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    hipLaunchKernelGGL(k_train_reduce, dim3(kRed5 / 64 + (kRedN + 1 - kRed5 + 15) / 16), dim3(256), 0, st, a.part1, nwg, part, partb, ns,
                       a.part5, nrb, g, loss);
    return hipGetLastError();
}
hipError_t mlp_infer(const InferSet *sets, int nsets, int ntiles, int maxrows, const FusedWeights &fw, const TargetNorm &tn,
                     hipStream_t st) {
    if (nsets <= 0 || ntiles <= 0) return hipSuccess;
    int dev = 0, cus = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (e != hipSuccess) return e;
    for (int i = 0; i < nsets; i += 65535)   // grid limit in y
        hipLaunchKernelGGL(k_infer_rows, dim3(blocks(maxrows), std::min(nsets - i, 65535)), dim3(256), 0, st, sets + i);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    // one workgroup per CU (its LDS holds no second one)
    hipLaunchKernelGGL(k_mlp_infer<kFusedNW>, dim3(std::min(ntiles, std::max(cus, 1))), dim3(64 * kFusedNW), 0, st, sets,
                       nsets, ntiles, fw, tn);
    return hipGetLastError();
}
}  // namespace sg
}  // namespace atmo
