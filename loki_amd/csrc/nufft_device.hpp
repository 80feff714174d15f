// Chunk spectra and their interpolation: sum_k x_k exp(-2 pi i u (k - C)) of a
// chunk of 2C samples at any frequency u (turns per sample) from one FFT of the
// chunk and a few neighbouring spectral values.
//
// The chunk is divided by the transform of a Kaiser-Bessel window, transformed
// at twice its length (M = 4C points, k centred on C), and the value at u is
// the window-weighted sum of the 9 spectral points nearest to u M.  With 9
// points and twofold oversampling the interpolation's own error is 6e-9 of
// the chunk's norm (rms over the samples; 5e-8 for a sample at the chunk's
// edge), a tenth of FP32's rounding.  Both tables are polynomials, fitted to
// the window I0(b sqrt(1 - (2z/9)^2)), b = 0.995 * 9 pi * 0.75: the division
// in FP64 (3e-11), the weights in FP32 (1.3e-10 before rounding).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace loki_amd::kern {

constexpr int kSpecTaps      = 9;
constexpr int kSpecPad       = kSpecTaps / 2;  // spectral points beyond 0 and M/2
constexpr uint32_t kSpecMaxC = 2048;           // largest chunk (samples)

/// Records of one chunk's spectrum: points -4 .. M/2 + 4 as (Re E, Im E, Re V,
/// Im V), then the plain sums of both series as two doubles.
constexpr __host__ __device__ uint32_t spec_points(uint32_t m) { return m / 2 + 2 * kSpecPad + 1; }
constexpr __host__ __device__ uint32_t spec_stride(uint32_t m) { return spec_points(m) + 1; }

/// Reciprocal of the window's transform at sample k - C, x = ((k - C) / C)^2.
__device__ __forceinline__ double spec_inv_window(double x) {
    double p = 1.02698849514126780e-04;
    p = fma(p, x, 8.72249744134022918e-05);
    p = fma(p, x, 1.39855582892778481e-03);
    p = fma(p, x, 5.57122765249004875e-03);
    p = fma(p, x, 2.41942390123512166e-02);
    p = fma(p, x, 8.89443227673964026e-02);
    p = fma(p, x, 2.74695177249138223e-01);
    p = fma(p, x, 6.66153100903862150e-01);
    p = fma(p, x, 1.12790203238278064e+00);
    return fma(p, x, 9.99999999968185782e-01);
}

/// Even and odd parts of the window about point d, w(s - d) = E_d(s^2) + s O_d(s^2),
/// as polynomials in s^2 (|s| <= 1/2).
constexpr int kSpecDeg = 4;
__device__ constexpr float kSpecEven[kSpecPad + 1][kSpecDeg + 1] = {
    {4.097066473e-01F, -2.083281511e-01F, 5.045674281e-02F, -7.753501785e-03F, 8.101804419e-04F},
    {2.448597608e-01F, -1.051982073e-03F, -1.914012523e-02F, 4.811598407e-03F, -6.162238416e-04F},
    {4.807334798e-02F, 8.947632490e-02F, -1.393384355e-02F, -3.179588528e-04F, 2.512792429e-04F},
    {2.206964057e-03F, 1.552704906e-02F, 7.236012929e-03F, -9.047692722e-04F, -3.157867915e-05F},
    {6.603917400e-06F, 2.126500059e-04F, 6.098640552e-04F, 2.880512778e-04F, -1.204746299e-05F}};
__device__ constexpr float kSpecOdd[kSpecPad + 1][kSpecDeg + 1] = {
    {0.0F, 0.0F, 0.0F, 0.0F, 0.0F},
    {2.552360722e-01F, -8.674909089e-02F, 1.350685297e-02F, -1.246088800e-03F, 6.994109597e-05F},
    {1.088337421e-01F, 2.067225515e-02F, -9.329157141e-03F, 1.229546623e-03F, -8.125434403e-05F},
    {8.956326233e-03F, 1.452936225e-02F, 1.011406669e-03F, -5.101239540e-04F, 4.719417646e-05F},
    {5.688209364e-05F, 4.539484141e-04F, 5.305207828e-04F, 7.666968630e-05F, -1.480554840e-05F}};

/// D-th derivative (0, 1 or 2) of a polynomial of degree kSpecDeg at q.
template <int D>
__device__ __forceinline__ float spec_poly(const float (&c)[kSpecDeg + 1], float q) {
    float p = 0.0F;
#pragma unroll
    for (int i = kSpecDeg; i >= D; --i) {
        float k = c[i];
        if constexpr (D >= 1) {
            k *= static_cast<float>(i);
        }
        if constexpr (D >= 2) {
            k *= static_cast<float>(i - 1);
        }
        p = i == kSpecDeg ? k : fmaf(p, q, k);
    }
    return p;
}

/// Window weights of the points c - 4 .. c + 4 for a position s from point c
/// (|s| <= 1/2).
__device__ __forceinline__ void spec_weights(float s, float (&w)[kSpecTaps]) {
    const float q = s * s;
    w[kSpecPad]   = spec_poly<0>(kSpecEven[0], q);
#pragma unroll
    for (int d = 1; d <= kSpecPad; ++d) {
        const float e   = spec_poly<0>(kSpecEven[d], q);
        const float o   = spec_poly<0>(kSpecOdd[d], q);
        w[kSpecPad + d] = fmaf(s, o, e);
        w[kSpecPad - d] = fmaf(-s, o, e);
    }
}

/// First (w1) and second (w2) derivatives of the weights in s: they give the
/// chunk's sums of x_k (k - C) and x_k (k - C)^2 from the same points.
__device__ __forceinline__ void spec_weights_d(float s, float (&w1)[kSpecTaps],
                                               float (&w2)[kSpecTaps]) {
    const float q = s * s;
    const float t = 2.0F * s;
#pragma unroll
    for (int d = 0; d <= kSpecPad; ++d) {
        const float e1 = spec_poly<1>(kSpecEven[d], q);
        const float e2 = fmaf(4.0F * q, spec_poly<2>(kSpecEven[d], q), 2.0F * e1);
        const float o0 = spec_poly<0>(kSpecOdd[d], q);
        const float o1 = spec_poly<1>(kSpecOdd[d], q);
        const float a  = fmaf(2.0F * q, o1, o0);
        const float b  = s * fmaf(4.0F * q, spec_poly<2>(kSpecOdd[d], q), 6.0F * o1);
        w1[kSpecPad + d] = fmaf(t, e1, a);
        w2[kSpecPad + d] = e2 + b;
        if (d > 0) {
            w1[kSpecPad - d] = fmaf(t, e1, -a);
            w2[kSpecPad - d] = e2 - b;
        }
    }
}

/// Position of frequency u (turns per sample, u >= 0) on an M-point spectrum:
/// the record of the first weighted point, the offset from the middle one and
/// whether the value is the conjugate of the interpolated one (u folded to
/// [0, 1/2]: the series are real).  Every point lies in -4 .. M/2 + 4.
__device__ __forceinline__ uint32_t spec_position(double u, uint32_t m, float& s, bool& conj) {
    u -= floor(u);
    conj             = u > 0.5;
    const double pos = (conj ? 1.0 - u : u) * static_cast<double>(m);
    const double c   = rint(pos);
    s                = static_cast<float>(pos - c);
    return static_cast<uint32_t>(c);
}

// Over a chunk of half length D around tau_c a candidate's phase is phi_c + f_c d +
// a_c d^2 / 2 + fddot d^3 / 6.  The spectra give the straight part exactly and
// the quadratic one to first order; the candidate goes this way when, at the
// highest harmonic and anywhere in the series, the quadratic part stays below
// 2e-4 turns (its dropped square: 8e-7 rad at the ends of such a chunk) and
// the cubic one below 1e-7 turns.  A NaN is not below.
constexpr double kMaxQuadTurns  = 2e-4;
constexpr double kMaxCubicTurns = 1e-7;

/// Candidates (f, fdot, fddot) that may take spectra of m points over a series
/// of nsamps; theta null: the spectra are wanted in any case.
struct SpecUsers {
    const double* theta;
    uint32_t ncand, top;  ///< top: highest harmonic
    uint32_t m;
    uint64_t nsamps;
    double tsamp, t_ref;
};

__device__ __forceinline__ bool spectral_ok(const double* th, const SpecUsers& u) {
    const double d  = 0.25 * static_cast<double>(u.m) * u.tsamp;
    const double t0 = -u.t_ref;
    const double t1 = (static_cast<double>(u.nsamps) * u.tsamp) - u.t_ref;
    const double a  = fmax(fabs(th[1] + th[2] * t0), fabs(th[1] + th[2] * t1));
    const double n  = static_cast<double>(u.top);
    return n * a * d * d * 0.5 <= kMaxQuadTurns &&
           n * fabs(th[2]) * d * d * d / 6.0 <= kMaxCubicTurns && fabs(th[0]) < 1e15;
}

/// The chunk's (E, V) values from the 9 records at `p`.
__device__ __forceinline__ float4 spec_value(const float4* p, const float (&w)[kSpecTaps]) {
    float4 a = make_float4(0.0F, 0.0F, 0.0F, 0.0F);
#pragma unroll
    for (int i = 0; i < kSpecTaps; ++i) {
        const float4 v = p[i];
        a.x = fmaf(w[i], v.x, a.x);
        a.y = fmaf(w[i], v.y, a.y);
        a.z = fmaf(w[i], v.z, a.z);
        a.w = fmaf(w[i], v.w, a.w);
    }
    return a;
}

}  // namespace loki_amd::kern
