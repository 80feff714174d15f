// FFTs of sample chunks (nufft_device.hpp) and the Fourier brute fold from them.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "device.hpp"
#include "kernels.hpp"
#include "nufft_device.hpp"
#include "merge_device.hpp"

namespace loki_amd::kern {
namespace {

struct cplx {
    double x, y;
};

__device__ __forceinline__ cplx cmul(cplx a, cplx b) {
    return {fma(a.x, b.x, -(a.y * b.y)), fma(a.x, b.y, a.y * b.x)};
}

// ---------------------------------------------------------------------------
// Chunk spectra
// ---------------------------------------------------------------------------
// A workgroup transforms one chunk of both series: M = 2^LG points of the
// real, window-divided samples as an H = M/2-point complex FFT per series
// (even samples real, odd ones imaginary; the two series never mix, so a NaN
// of one stays in it), FP64 in LDS, radix 4 with a last radix-2 pass where
// log2 H is odd.  The points are rounded to FP32 once, when they are written.
// FP64 costs little here: 2^22 samples x 2 are 5e8 complex operations of a
// step that interpolates 2.4e8 values, and the sums over the samples are then
// better than any FP32 order of them.
template <int LG> struct SpecShape {
    static constexpr int kH       = 1 << (LG - 1);             // complex points per series
    static constexpr int kQ       = kH / 4;                    // radix-4 butterflies per series
    static constexpr int kThreads = kQ >= 256 ? 512 : (kQ >= 32 ? 2 * kQ : 64);
    static constexpr int kLanes   = kThreads / 2;              // lanes per series
    static constexpr int kPer     = (kQ + kLanes - 1) / kLanes;
};

template <int LG>
__global__ void __launch_bounds__(SpecShape<LG>::kThreads)
k_chunk_spectra(const float* __restrict__ ts_e, const float* __restrict__ ts_v, uint64_t seglen,
                uint32_t nchunk, uint64_t q0, float4* __restrict__ spec, SpecUsers users) {
    using S          = SpecShape<LG>;
    constexpr int M  = 1 << LG;
    constexpr int H  = S::kH;
    constexpr int C  = M / 4;   // half a chunk
    constexpr int T  = S::kThreads;
    constexpr int TL = S::kLanes;
    constexpr int kFine = M < 64 ? M : 64;
    __shared__ cplx buf[2][H];
    __shared__ cplx t1[M / kFine], t2[kFine];  // exp(-2 pi i (64 a + b) / M) = t1[a] t2[b]
    __shared__ double red[2][T / 64 > 0 ? T / 64 : 1];

    const uint64_t q   = q0 + blockIdx.x;
    const uint64_t seg = q / nchunk;
    const uint64_t k0  = (q % nchunk) * (2 * C);
    const uint32_t len = static_cast<uint32_t>(min(static_cast<uint64_t>(2 * C), seglen - k0));
    const int tid      = static_cast<int>(threadIdx.x);
    // nothing to do if no candidate reads the spectra; mostly the first one does
    if (users.theta != nullptr && !spectral_ok(users.theta, users)) {
        bool any = false;
        for (uint32_t c = threadIdx.x; c < users.ncand && !any; c += T) {
            any = spectral_ok(users.theta + 3 * static_cast<uint64_t>(c), users);
        }
        if (__syncthreads_or(any) == 0) {
            return;
        }
    }
    const int side     = tid / TL;  // 0: e, 1: v
    const int lane     = tid % TL;
    const float* x     = (side == 0 ? ts_e : ts_v) + seg * seglen + k0;

    for (int i = tid; i < M / kFine + kFine; i += T) {
        const bool fine = i >= M / kFine;
        const double a  = fine ? static_cast<double>(i - M / kFine) / M
                               : static_cast<double>(i) * kFine / M;
        double sn, cs;
        sincospi(2.0 * a, &sn, &cs);
        (fine ? t2[i - M / kFine] : t1[i]) = {cs, -sn};
    }
    // point n holds y[2n] + i y[2n+1], y[(k - C) mod M] = x_k / window
    double sum = 0.0;
    for (int n = lane; n < H; n += TL) {
        double v[2] = {0.0, 0.0};
        const int d0 = n < H / 2 ? 2 * n : 2 * n - M;  // k - C of the even sample
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int k = d0 + j + C;
            if (k >= 0 && k < static_cast<int>(len)) {
                const double r = static_cast<double>(d0 + j) / C;
                const double s = static_cast<double>(x[k]);
                sum += s;
                v[j] = s * spec_inv_window(r * r);
            }
        }
        buf[side][n] = {v[0], v[1]};
    }
    // plain sums: lanes of one series fill whole waves (or half of one wave)
    constexpr int kSumLanes = TL < 64 ? TL : 64;
    for (int o = kSumLanes / 2; o > 0; o >>= 1) {
        sum += __shfl_xor(sum, o);
    }
    if (lane % kSumLanes == 0) {
        red[side][lane / kSumLanes] = sum;
    }
    __syncthreads();

    auto twiddle = [&](int i) { return cmul(t1[i / kFine], t2[i % kFine]); };
    cplx* b = buf[side];
#pragma unroll
    for (int ns = 1; ns * 4 <= H; ns *= 4) {
        cplx v[S::kPer][4];
#pragma unroll
        for (int p = 0; p < S::kPer; ++p) {
            const int j = lane + p * TL;
            if (j < S::kQ) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    v[p][r] = b[j + r * S::kQ];
                }
                if (ns > 1) {
                    const cplx w1 = twiddle((j % ns) * (M / (4 * ns)));
                    const cplx w2 = cmul(w1, w1);
                    v[p][1] = cmul(v[p][1], w1);
                    v[p][2] = cmul(v[p][2], w2);
                    v[p][3] = cmul(v[p][3], cmul(w1, w2));
                }
                const cplx a0 = {v[p][0].x + v[p][2].x, v[p][0].y + v[p][2].y};
                const cplx a1 = {v[p][0].x - v[p][2].x, v[p][0].y - v[p][2].y};
                const cplx a2 = {v[p][1].x + v[p][3].x, v[p][1].y + v[p][3].y};
                const cplx a3 = {v[p][1].y - v[p][3].y, v[p][3].x - v[p][1].x};  // -i (v1 - v3)
                v[p][0] = {a0.x + a2.x, a0.y + a2.y};
                v[p][1] = {a1.x + a3.x, a1.y + a3.y};
                v[p][2] = {a0.x - a2.x, a0.y - a2.y};
                v[p][3] = {a1.x - a3.x, a1.y - a3.y};
            }
        }
        __syncthreads();
#pragma unroll
        for (int p = 0; p < S::kPer; ++p) {
            const int j = lane + p * TL;
            if (j < S::kQ) {
                const int o = (j / ns) * ns * 4 + j % ns;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    b[o + r * ns] = v[p][r];
                }
            }
        }
        __syncthreads();
    }
    if constexpr ((LG - 1) % 2 == 1) {
        for (int j = lane; j < H / 2; j += TL) {
            const cplx a = b[j];
            const cplx c = cmul(b[j + H / 2], twiddle(2 * j));
            b[j]         = {a.x + c.x, a.y + c.y};
            b[j + H / 2] = {a.x - c.x, a.y - c.y};
        }
        __syncthreads();
    }
    // Y_p = (Z_p + Z*_{H-p}) / 2 - i w^p (Z_p - Z*_{H-p}) / 2, w = exp(-2 pi i / M)
    float4* out = spec + q * spec_stride(M);
    for (int i = tid; i < static_cast<int>(spec_points(M)); i += T) {
        const int p  = (i - kSpecPad + M) % M;
        const int z0 = p % H;
        const int z1 = (H - z0) % H;
        const cplx w = twiddle(p);
        double y[4];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const cplx a = buf[s][z0];
            const cplx c = buf[s][z1];
            const cplx e = {0.5 * (a.x + c.x), 0.5 * (a.y - c.y)};
            const cplx o = cmul({0.5 * (a.y + c.y), -0.5 * (a.x - c.x)}, w);
            y[2 * s]     = e.x + o.x;
            y[2 * s + 1] = e.y + o.y;
        }
        out[i] = make_float4(static_cast<float>(y[0]), static_cast<float>(y[1]),
                             static_cast<float>(y[2]), static_cast<float>(y[3]));
    }
    if (tid == 0) {
        double s[2] = {0.0, 0.0};
        for (int j = 0; j < TL / kSumLanes; ++j) {
            s[0] += red[0][j];
            s[1] += red[1][j];
        }
        *reinterpret_cast<double2*>(out + spec_points(M)) = make_double2(s[0], s[1]);
    }
}

// ---------------------------------------------------------------------------
// Brute fold
// ---------------------------------------------------------------------------
struct SpecFoldArgs {
    const float4* spec;
    float2* fold;
    const double* freqs;
    uint32_t nfreqs, nbf, nseg, nchunk, m;
    uint32_t segs_per_block, nblk_out;
    double tsamp, t_ref;
};

/// exp(-2 pi i d) for an FP64 angle d in turns: sincospi of the FP32 head of
/// d's fraction and a first-order correction for its tail.
__device__ __forceinline__ float2 turns(double d) {
    d -= floor(d);
    d              = d > 0.5 ? d - 1.0 : d;
    const float hi = static_cast<float>(d);
    const float lo = static_cast<float>(d - static_cast<double>(hi));
    float sn, cs;
    sincospif(2.0F * hi, &sn, &cs);
    const float dl = 6.28318530717958647692F * lo;
    return make_float2(fmaf(-dl, sn, cs), -fmaf(dl, cs, sn));
}

constexpr int kFoldThreads = 512;

// fold[s, i, q, m] at frequency u = m f_i tsamp of every segment's chunks.  A
// lane owns OUTS (frequency, harmonic) pairs and keeps their weights in
// registers over segs_per_block segments, whose spectra (33 KB at 2048
// samples) pass through LDS.  The 8 lanes of a group take 8 neighbouring
// frequencies of one harmonic: their positions on the spectrum are at most two
// points apart, so a group's 16-byte LDS reads are spread over the banks, and
// a wave's writes are runs of 8 harmonics of a row.
// 2^22 samples in 2048 segments, 1888 frequencies, 32 harmonics (2.0 GB
// written): 0.80 ms, plus 0.09 ms for the spectra and their sums, where the
// matrix-core DFT took 19.9 + 0.29 ms (2.0e12 flop).  LDS reads bound it: 9
// points of 16 bytes per value of both series.
// TURN: the chunk's centre is not at t_ref (or there are several chunks), and
// each value is turned by the phase of its chunk's centre.
// Harmonic 0 is the segment's plain sum, the same for every frequency: the
// chunks' FP64 sums are added in FP64 and rounded once.
template <int OUTS, bool TURN>
__global__ void __launch_bounds__(kFoldThreads)
k_spectra_fold(SpecFoldArgs a) {
    extern __shared__ float4 sp[];
    __shared__ double s_dc[2];  // FP64 registers for it would cost a workgroup per CU
    const uint32_t blk  = xcd_remap(blockIdx.x, gridDim.x);
    const uint32_t ob   = blk % a.nblk_out;
    const uint64_t seg0 = static_cast<uint64_t>(blk / a.nblk_out) * a.segs_per_block;
    const uint32_t npt  = spec_stride(a.m);
    const uint32_t ngrp = ((a.nfreqs + 7) / 8) * a.nbf;

    float w[OUTS][kSpecTaps];
    uint32_t first[OUTS], fi[OUTS], hm[OUTS];
    bool conj[OUTS], valid[OUTS];
#pragma unroll
    for (int o = 0; o < OUTS; ++o) {
        const uint32_t t = (ob * OUTS + o) * kFoldThreads + threadIdx.x;
        const uint32_t g = t / 8;
        fi[o]            = (g / a.nbf) * 8 + t % 8;
        hm[o]            = g % a.nbf;
        valid[o]         = g < ngrp && fi[o] < a.nfreqs;
        const double ft  = a.freqs[valid[o] ? fi[o] : 0] * a.tsamp;
        float s;
        first[o] = spec_position((ft - floor(ft)) * static_cast<double>(hm[o]), a.m, s, conj[o]);
        spec_weights(s, w[o]);
    }
    const auto* sums    = reinterpret_cast<const double*>(sp + (npt - 1));  // of the staged chunk
    const uint64_t seg1 = min(seg0 + a.segs_per_block, static_cast<uint64_t>(a.nseg));
    for (uint64_t seg = seg0; seg < seg1; ++seg) {
        float4 acc[OUTS];
#pragma unroll
        for (int o = 0; o < OUTS; ++o) {
            acc[o] = make_float4(0.0F, 0.0F, 0.0F, 0.0F);
        }
        for (uint32_t c = 0; c < a.nchunk; ++c) {
            __syncthreads();  // the previous chunk's readers are done
            const float4* src = a.spec + (seg * a.nchunk + c) * npt;
            for (uint32_t i = threadIdx.x; i < npt; i += kFoldThreads) {
                sp[i] = src[i];
            }
            __syncthreads();
            if constexpr (TURN) {
                if (a.nchunk > 1 && threadIdx.x < 2) {
                    s_dc[threadIdx.x] = c == 0 ? sums[threadIdx.x] : s_dc[threadIdx.x] + sums[threadIdx.x];
                }
            }
#pragma unroll
            for (int o = 0; o < OUTS; ++o) {
                float4 v = spec_value(sp + first[o], w[o]);
                v.y      = conj[o] ? -v.y : v.y;
                v.w      = conj[o] ? -v.w : v.w;
                if constexpr (TURN) {
                    const double k  = static_cast<double>(c) * (a.m / 2) + (a.m / 4);
                    const double ph = a.freqs[valid[o] ? fi[o] : 0] * ((k * a.tsamp) - a.t_ref);
                    const float2 z  = turns((ph - floor(ph)) * static_cast<double>(hm[o]));
                    v = make_float4(fmaf(v.x, z.x, -(v.y * z.y)), fmaf(v.x, z.y, v.y * z.x),
                                    fmaf(v.z, z.x, -(v.w * z.y)), fmaf(v.z, z.y, v.w * z.x));
                }
                if constexpr (TURN) {
                    acc[o].x += v.x;
                    acc[o].y += v.y;
                    acc[o].z += v.z;
                    acc[o].w += v.w;
                } else {  // the only chunk
                    acc[o] = hm[o] == 0 ? make_float4(static_cast<float>(sums[0]), 0.0F,
                                                      static_cast<float>(sums[1]), 0.0F)
                                        : v;
                }
            }
        }
        if constexpr (TURN) {
            const double* dc = sums;  // the only chunk's
            if (a.nchunk > 1) {
                __syncthreads();  // s_dc is complete
                dc = s_dc;
            }
#pragma unroll
            for (int o = 0; o < OUTS; ++o) {
                if (hm[o] == 0) {
                    acc[o] = make_float4(static_cast<float>(dc[0]), 0.0F,
                                         static_cast<float>(dc[1]), 0.0F);
                }
            }
        }
#pragma unroll
        for (int o = 0; o < OUTS; ++o) {
            if (valid[o]) {
                float2* row = a.fold + ((seg * a.nfreqs + fi[o]) * 2) * a.nbf + hm[o];
                row[0]      = make_float2(acc[o].x, acc[o].y);
                row[a.nbf]  = make_float2(acc[o].z, acc[o].w);
            }
        }
    }
}

template <int OUTS>
void launch_fold(const SpecFoldArgs& a, bool turn, hipStream_t s) {
    const uint64_t nblk =
        static_cast<uint64_t>(a.nblk_out) * ((a.nseg + a.segs_per_block - 1) / a.segs_per_block);
    LOKI_REQUIRE(nblk < (1ULL << 31), "Fourier brute fold grid too large");
    const size_t lds = spec_stride(a.m) * sizeof(float4);
    if (turn) {
        k_spectra_fold<OUTS, true><<<static_cast<uint32_t>(nblk), kFoldThreads, lds, s>>>(a);
    } else {
        k_spectra_fold<OUTS, false><<<static_cast<uint32_t>(nblk), kFoldThreads, lds, s>>>(a);
    }
}

template <int LG>
void launch_spectra(const float* e, const float* v, uint64_t seglen, uint32_t nchunk, uint64_t n,
                    float4* spec, const SpecUsers& users, hipStream_t s) {
    constexpr uint64_t kMaxGrid = 1ULL << 30;
    for (uint64_t q0 = 0; q0 < n; q0 += kMaxGrid) {
        const auto g = static_cast<uint32_t>(std::min(kMaxGrid, n - q0));
        k_chunk_spectra<LG><<<g, SpecShape<LG>::kThreads, 0, s>>>(e, v, seglen, nchunk, q0, spec,
                                                          users);
    }
}

}  // namespace

SpectraShape spectra_shape(uint64_t seglen) {
    SpectraShape sh{};
    uint32_t c = 64;
    while (c < kSpecMaxC && c < seglen) {
        c *= 2;
    }
    sh.m      = 2 * c;
    sh.nchunk = (seglen + c - 1) / c;
    return sh;
}

namespace {

/// Bytes of one segment's spectra.
uint64_t segment_bytes(uint64_t seglen) {
    const auto sh = spectra_shape(seglen);
    return sh.nchunk * spec_stride(sh.m) * sizeof(float4);
}

}  // namespace

uint64_t spectra_bytes(uint64_t nseg, uint64_t seglen, uint64_t max_bytes) {
    const uint64_t one = segment_bytes(seglen);
    return std::min(nseg, std::max<uint64_t>(max_bytes / one, 1)) * one;
}

void chunk_spectra(const float* ts_e, const float* ts_v, uint64_t nseg, uint64_t seglen,
                   const SpectraShape& sh, void* spec, hipStream_t s, const SpecUsers* users) {
    const uint64_t n = nseg * sh.nchunk;
    auto* out        = static_cast<float4*>(spec);
    LOKI_REQUIRE(sh.nchunk < (1ULL << 32), "chunk spectra: segment too long");
    const auto nc = static_cast<uint32_t>(sh.nchunk);
    const SpecUsers u = users != nullptr ? *users : SpecUsers{};
    switch (sh.m) {
    case 128: launch_spectra<7>(ts_e, ts_v, seglen, nc, n, out, u, s); break;
    case 256: launch_spectra<8>(ts_e, ts_v, seglen, nc, n, out, u, s); break;
    case 512: launch_spectra<9>(ts_e, ts_v, seglen, nc, n, out, u, s); break;
    case 1024: launch_spectra<10>(ts_e, ts_v, seglen, nc, n, out, u, s); break;
    case 2048: launch_spectra<11>(ts_e, ts_v, seglen, nc, n, out, u, s); break;
    default: launch_spectra<12>(ts_e, ts_v, seglen, nc, n, out, u, s); break;
    }
}

namespace {

/// Time the spectra save over the matrix cores, in us, without their fixed costs.
/// Fitted to segments of 64 to 256 samples: a matrix-core fold takes 2.0 ps per
/// (sample, frequency) for its twiddles and 0.15-0.17 ps per harmonic beyond (the
/// first 18 share a tile with their neighbours up to 33), 0.7 of it from 128
/// samples; the FFTs 7 ns per chunk (of c samples, padding included) and 6 ps per
/// sample (2^23 samples: 0.94, 0.51, 0.29 ms for segments of 64, 128 and 256).
double spectra_gain_us(uint64_t nseg, uint32_t seglen, uint32_t nfreqs, uint32_t nbf) {
    const auto sh   = spectra_shape(seglen);
    const double n  = static_cast<double>(nseg) * seglen;
    const double c  = sh.m / 2.0;
    const double pad = c * static_cast<double>(sh.nchunk) / seglen;
    const double mc = (2.0 + 0.17 * std::min(nbf, 18U) + 0.146 * (nbf > 33 ? nbf - 33.0 : 0.0)) *
                      (seglen < 128 ? 1.0 : 0.7);
    return 1e-6 * n * (mc * nfreqs - (7000.0 / c + 6.0) * pad);
}

}  // namespace

// The spectra cost the same for any number of frequencies, the matrix cores 2 K
// per value.  Level 0 of a plan, matrix cores against spectra, us:
//   2^17 samples, segments of 64: 48 frequencies, 16 bins 28 / 35; 64 frequencies,
//     64 bins 46 / 53; 96 frequencies, 4 bins 41 / 33, 64 bins 61 / 53
//   2^23 samples, segments of 64: 48 frequencies, 16 bins 1425 / 1003
//   2^17 samples, segments of 128: 48 frequencies, 16 bins 35 / 23, 64 bins 38 / 26
//   2^23 samples, segments of 128: 32 frequencies, 16 bins 742 (spectra about 500)
//   2^23 samples, segments of 2048: 48 frequencies, 16 bins 446 / 148
//   2^23 samples, segments of 8192: 2 frequencies, 16 bins 1672 / 145 (the matrix
//     cores have too few rows)
// A one-off call allocates the spectra, 25 us and more:
//   2^17 samples, segments of 128: 64 frequencies, 64 bins 50 / 81, 48, 256 bins 120 / 99
//   2^20 samples, segments of 128: 48 frequencies, 16 bins 117 / 131, 64 bins 184 / 143
//   2^17 samples, segments of 256: 64 frequencies, 64 bins 52 / 67, 96 70 / 68
bool spectra_fold_better(uint64_t nseg, uint32_t seglen, uint32_t nfreqs, uint32_t nbins,
                         bool one_off) {
    if (seglen < 64 || (nfreqs < 48 && seglen < 4096)) {
        return false;
    }
    if (seglen > 256 || (!one_off && (seglen >= 128 || nfreqs >= 96))) {
        return true;
    }
    const double least = !one_off ? 40.0 : (seglen <= 128 ? 65.0 : 40.0);
    return spectra_gain_us(nseg, seglen, nfreqs, nbins / 2 + 1) >= least;
}

void brute_fold_spectra(const float* ts_e, const float* ts_v, uint64_t nseg, uint32_t seglen,
                        const double* freqs_dev, uint32_t nfreqs, uint32_t nbins, double tsamp,
                        double t_ref, float2* fold, void* spec, uint64_t spec_bytes,
                        hipStream_t s) {
    LOKI_REQUIRE(nbins >= 2 && nbins <= 256, "Fourier brute fold: nbins must be in [2, 256]");
    LOKI_REQUIRE(seglen >= 1 && nfreqs >= 1, "Fourier brute fold: empty input");
    LOKI_REQUIRE(nseg >= 1 && 2 * nseg < (1ULL << 31), "Fourier brute fold: too many segments");
    const auto sh         = spectra_shape(seglen);
    const uint64_t fit    = spec_bytes / segment_bytes(seglen);
    LOKI_REQUIRE(fit >= 1, "Fourier brute fold: workspace below one segment's spectra");
    const uint64_t passes = (nseg + fit - 1) / fit;
    const uint64_t slab   = (nseg + passes - 1) / passes;
    SpecFoldArgs a{};
    a.spec   = static_cast<const float4*>(spec);
    a.freqs  = freqs_dev;
    a.nfreqs = nfreqs;
    a.nbf    = nbins / 2 + 1;
    a.nchunk = static_cast<uint32_t>(sh.nchunk);
    a.m      = sh.m;
    a.tsamp  = tsamp;
    a.t_ref  = t_ref;
    const uint64_t lanes = static_cast<uint64_t>((nfreqs + 7) / 8) * 8 * a.nbf;
    LOKI_REQUIRE(lanes < (1ULL << 31), "Fourier brute fold grid too large");
    const bool turn = sh.nchunk > 1 || (static_cast<double>(sh.m / 4) * tsamp) - t_ref != 0.0;
    // Four outputs per lane read each staged spectrum for 2048 values; one
    // where that leaves fewer than two workgroups per CU.
    constexpr uint32_t kOuts   = 4;
    constexpr uint64_t kBlocks = 512;
    const bool wide = (lanes + kOuts * kFoldThreads - 1) / (kOuts * kFoldThreads) * slab >= kBlocks;
    const uint32_t per = kFoldThreads * (wide ? kOuts : 1);
    a.nblk_out         = static_cast<uint32_t>((lanes + per - 1) / per);
    for (uint64_t s0 = 0; s0 < nseg; s0 += slab) {
        const uint64_t n = std::min(slab, nseg - s0);
        a.nseg           = static_cast<uint32_t>(n);
        a.fold           = fold + s0 * nfreqs * 2 * a.nbf;
        // segments per workgroup: the weights (~60 operations per value) are
        // shared by them, as long as four workgroups per CU remain
        a.segs_per_block =
            static_cast<uint32_t>(std::clamp<uint64_t>(n * a.nblk_out / (4 * kBlocks), 1, 16));
        chunk_spectra(ts_e + s0 * seglen, ts_v + s0 * seglen, n, seglen, sh, spec, s);
        if (wide) {
            launch_fold<kOuts>(a, turn, s);
        } else {
            launch_fold<1>(a, turn, s);
        }
    }
}

}  // namespace loki_amd::kern
