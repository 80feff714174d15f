// Fused return to the time domain and boxcar S/N of the last Fourier-domain
// level: the inverse real DFT (fft_cuda.cu:357-448, 1/n normalised) of each
// final fold row runs on the matrix cores as [rows x (re, im of nbins/2+1
// harmonics)] x [(re, im) x nbins] (v_mfma_f32_16x16x4f32), the profile
// p = e / sqrt(v) is formed from the accumulators, and the S/N of
// score.cpp:95-172 is taken from a per-lane prefix sum.  The time-domain final fold
// (2 * nbins floats per trial) is never written.
//
// One wave owns 64 consecutive trials: 8 MFMA tiles of 8 trials (16 rows:
// trial-major, e before v), then one lane per trial for the prefix sum and the
// width maxima.  Neither memory (0.40 ms at the copy rate for 3.87e6 trials of 64
// bins and 10 widths) nor the matrix cores (0.43 ms) nor the vector unit (0.28 ms)
// bounds it alone; the waits between them do, so:
//  - the A operands come straight from the rows into registers, one tile ahead,
//    with the harmonics ordered for float2 loads (the basis is permuted alike);
//    staged through LDS instead: 1.40 ms;
//  - the basis stays in registers (read from the LDS table for each tile before);
//  - the prefix sum stays in registers and every width has its own code with
//    compile-time offsets, 1.5 operations per bin; widths from the LDS row with the
//    rest alike: 1.38 ms.
// 0.92 ms at that size; 1.83 ms with staged tiles, basis and widths from LDS and the
// general division sequences.  Two waves per SIMD: a third needs 168 registers,
// which spill (0.12 ms slower).
#include <hip/hip_runtime.h>

#include <cfloat>
#include <cmath>
#include <utility>

#include "kernels.hpp"
#include "score_device.hpp"

namespace loki_amd::kern {
namespace {

using f32x4 = float __attribute__((ext_vector_type(4)));

constexpr int kWaveTrials = 64;
constexpr int kTileTrials = 8;

__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int NB> struct IrsGeom {
    static constexpr int kNh  = NB / 2 + 1;
    static constexpr int kRow = 2 * kNh;     // floats per component row
    static constexpr int kF2  = NB / 8;      // float2 loads per lane and tile
    static constexpr int kKs  = 2 * kF2 + 1; // K steps of 4
    static constexpr int kNt  = NB / 16;     // N tiles of 16 bins
};

/// Inverse real DFT basis entry B[k][n] (k = 2h + {0: re, 1: im}):
/// c_h cos(2 pi h n / NB) and -c_h sin(2 pi h n / NB), c_h = 1/NB for h = 0
/// and h = NB/2 (whose imaginary parts are ignored), 2/NB otherwise, 0 for
/// the padding k >= nbins + 2.  tw[t] = (cos, sin)(2 pi t / NB).
template <int NB>
__device__ __forceinline__ float irdft_basis(const float2* tw, int k, int n) {
    constexpr int kRow = IrsGeom<NB>::kRow;
    const int h        = k >> 1;
    const bool edge    = h == 0 || h == NB / 2;
    const bool imag    = (k & 1) != 0;
    const float c      = (k >= kRow || (imag && edge)) ? 0.0F
                         : edge                        ? 1.0F / static_cast<float>(NB)
                                                       : 2.0F / static_cast<float>(NB);
    const float2 w     = tw[(h * n) & (NB - 1)];
    return c * (imag ? -w.y : w.x);
}

/// max_j (psum[j + W] - psum[j]) of the circular prefix sum, psum[i] for i >=
/// NB being psum[i - NB] + psum[NB - 1].
template <int NB, int W>
__device__ __forceinline__ float window_max_fixed(const float (&ps)[NB]) {
    float ma = -FLT_MAX, mb = -FLT_MAX;
#pragma unroll
    for (int j = 0; j < NB; ++j) {
        const float hi = (j + W < NB) ? ps[(j + W) % NB] : ps[(j + W - NB) % NB] + ps[NB - 1];
        if ((j & 2) == 0) {
            ma = __builtin_fmaxf(ma, hi - ps[j]);
        } else {
            mb = __builtin_fmaxf(mb, hi - ps[j]);
        }
    }
    return __builtin_fmaxf(ma, mb);
}

template <int NB, int... Ws>
__device__ __forceinline__ float window_max_reg(std::integer_sequence<int, Ws...>,
                                                const float (&ps)[NB], uint32_t w) {
    float r = 0.0F;
    (void)((w == static_cast<uint32_t>(Ws + 1) ? (r = window_max_fixed<NB, Ws + 1>(ps), true)
                                               : false) ||
           ...);
    return r;
}

template <int NB, bool FINDMAX, bool EXACT>
__global__ void __launch_bounds__(64, 2)
k_irfft_score(const float* __restrict__ fold, uint64_t ntrials, WidthTable wt, uint32_t stride,
              float* __restrict__ scores, FilterOut fo) {
    using G = IrsGeom<NB>;
    extern __shared__ float lds[];
    float* __restrict__ prow = lds;  // [64][stride]
    auto* tw = reinterpret_cast<float2*>(prow + ((kWaveTrials * stride + 1) & ~1U));  // [NB]
    const int lane = static_cast<int>(threadIdx.x);
    const int mrow = lane & 15;   // A row / D column within the tile
    const int kq   = lane >> 4;   // A column / D row group
    for (int t = lane; t < NB; t += 64) {
        double sn, cs;
        sincospi(2.0 * static_cast<double>(t) / static_cast<double>(NB), &sn, &cs);
        tw[t] = make_float2(static_cast<float>(cs), static_cast<float>(sn));
    }
    wave_sync();
    // this lane's basis values, one register each (68 at 64 bins) for the whole
    // kernel; opaque, or they would be formed again for every tile
    float basis[G::kKs][G::kNt];
#pragma unroll
    for (int ks = 0; ks < G::kKs; ++ks) {
#pragma unroll
        for (int nt = 0; nt < G::kNt; ++nt) {
            const int k   = ks + 1 == G::kKs ? NB + kq : 8 * (ks >> 1) + 2 * kq + (ks & 1);
            basis[ks][nt] = irdft_basis<NB>(tw, k, 16 * nt + mrow);
            asm volatile("" : "+v"(basis[ks][nt]));
        }
    }
    const uint64_t ngroups = (ntrials + kWaveTrials - 1) / kWaveTrials;
    // A operands of one tile (8 trials from trial c), straight from the rows: K
    // step 2i + j takes harmonic component 8i + 2 kq + j, so that a lane reads
    // float2s; the last step is the real part of harmonic NB/2 in lane group 0.
    // Zeros for trials past the end.
    float2 pre[G::kF2];
    float pre_last = 0.0F;
    auto load_tile = [&](uint64_t c) {
        const bool live = c + static_cast<uint64_t>(mrow >> 1) < ntrials;
        const float* __restrict__ r =
            fold + (live ? 2 * c + static_cast<uint64_t>(mrow) : 0) * G::kRow;
#pragma unroll
        for (int i = 0; i < G::kF2; ++i) {
            const float2 v = *reinterpret_cast<const float2*>(r + 8 * i + 2 * kq);
            pre[i].x       = live ? v.x : 0.0F;
            pre[i].y       = live ? v.y : 0.0F;
        }
        const float v = r[NB];
        pre_last      = live && kq == 0 ? v : 0.0F;
    };
    load_tile(static_cast<uint64_t>(blockIdx.x) * kWaveTrials);
    for (uint64_t grp = blockIdx.x; grp < ngroups; grp += gridDim.x) {
        const uint64_t c0 = grp * kWaveTrials;
#pragma unroll 1
        for (int t = 0; t < kWaveTrials / kTileTrials; ++t) {
            float a[G::kKs];
#pragma unroll
            for (int i = 0; i < G::kF2; ++i) {
                a[2 * i]     = pre[i].x;
                a[2 * i + 1] = pre[i].y;
            }
            a[G::kKs - 1] = pre_last;
            // the next tile, of this group or of the wave's next one, comes in
            // while the matrix cores run and the widths are taken
            load_tile(t + 1 < kWaveTrials / kTileTrials
                          ? c0 + static_cast<uint64_t>(t + 1) * kTileTrials
                          : c0 + static_cast<uint64_t>(gridDim.x) * kWaveTrials);
            f32x4 acc[G::kNt];
#pragma unroll
            for (int nt = 0; nt < G::kNt; ++nt) {
                acc[nt] = f32x4{0.0F, 0.0F, 0.0F, 0.0F};
            }
#pragma unroll
            for (int ks = 0; ks < G::kKs; ++ks) {
#pragma unroll
                for (int nt = 0; nt < G::kNt; ++nt) {
                    acc[nt] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[ks], basis[ks][nt], acc[nt], 0,
                                                                  0, 0);
                }
            }
            // D rows 4*kq + v: trial 2*kq + v/2 of the tile, component v % 2
            const int tr = t * kTileTrials + 2 * kq;
            float* __restrict__ prow0 = prow + tr * stride + mrow;
            float* __restrict__ prow1 = prow0 + stride;
            if constexpr (EXACT) {
                // two accumulators at a time: one range check for the short
                // correctly rounded sequences
#pragma unroll
                for (int nt = 0; nt < G::kNt; nt += 2) {
                    const int nu   = nt + 1 < G::kNt ? nt + 1 : nt;
                    const float4 p = normalise4_exact(
                        make_float4(acc[nt][0], acc[nt][2], acc[nu][0], acc[nu][2]),
                        make_float4(acc[nt][1], acc[nt][3], acc[nu][1], acc[nu][3]));
                    prow0[16 * nt] = p.x;
                    prow1[16 * nt] = p.y;
                    if (nu != nt) {
                        prow0[16 * nu] = p.z;
                        prow1[16 * nu] = p.w;
                    }
                }
            } else {
#pragma unroll
                for (int nt = 0; nt < G::kNt; ++nt) {
                    prow0[16 * nt] = normalise<false>(acc[nt][0], acc[nt][1]);
                    prow1[16 * nt] = normalise<false>(acc[nt][2], acc[nt][3]);
                }
            }
        }
        wave_sync();  // the rows are complete
        const uint64_t c = c0 + static_cast<uint64_t>(lane);
        if (c < ntrials) {
            float* __restrict__ row = prow + lane * stride;
            float ps[NB];
            float acc = 0.0F;
#pragma unroll
            for (int j = 0; j < NB; ++j) {
                acc   = (j == 0) ? row[0] : acc + row[j];
                ps[j] = acc;
            }
            const float sum = ps[NB - 1];
            float best      = -FLT_MAX;
            for (uint32_t iw = 0; iw < wt.n; ++iw) {
                // opaque once per width: otherwise the maxima of all NB - 1
                // widths are formed ahead of the loop
#pragma unroll
                for (int j = 0; j < NB; ++j) {
                    asm volatile("" : "+v"(ps[j]));
                }
                // every width's window with compile-time offsets, picked by a
                // scalar branch on the wave-uniform width
                const float dmax = window_max_reg<NB>(std::make_integer_sequence<int, NB - 1>{},
                                                      ps, wt.w[iw]);
                const float snr = ((wt.h[iw] + wt.b[iw]) * dmax) - (wt.b[iw] * sum);
                if constexpr (FINDMAX) {
                    best = (best < snr) ? snr : best;
                } else if (fo.count != nullptr) {
                    filter_emit(fo, snr > fo.threshold, static_cast<uint32_t>(c * wt.n + iw),
                                snr);
                } else {
                    scores[c * wt.n + iw] = snr;
                }
            }
            if constexpr (FINDMAX) {
                if (fo.count != nullptr) {
                    filter_emit(fo, best > fo.threshold, static_cast<uint32_t>(c), best);
                } else {
                    scores[c] = best;
                }
            }
        }
        wave_sync();  // rows are rewritten by the next group
    }
}

template <int NB, bool FINDMAX, bool EXACT>
void launch_irs(const float2* fold, uint64_t ntrials, const WidthTable& wt, float* scores,
                const FilterOut& fo, hipStream_t s) {
    using G = IrsGeom<NB>;
    const uint32_t stride = NB + 1;  // odd: conflict-free per-lane rows
    const size_t lds = (((static_cast<size_t>(kWaveTrials) * stride + 1) & ~size_t{1}) + 2 * NB) *
                       sizeof(float);
    LOKI_REQUIRE(lds <= 65536, "irfft+score: LDS row too long");
    const uint64_t ngroups = (ntrials + kWaveTrials - 1) / kWaveTrials;
    const uint64_t nblocks = ngroups < 8192 ? ngroups : 8192;
    k_irfft_score<NB, FINDMAX, EXACT><<<static_cast<uint32_t>(nblocks), 64, lds, s>>>(
        reinterpret_cast<const float*>(fold), ntrials, wt, stride, scores, fo);
}

template <int NB>
void dispatch_irs(const float2* fold, uint64_t ntrials, const WidthTable& wt, float* scores,
                  bool find_max, bool exact, const FilterOut& fo, hipStream_t s) {
    if (find_max) {
        return exact ? launch_irs<NB, true, true>(fold, ntrials, wt, scores, fo, s)
                     : launch_irs<NB, true, false>(fold, ntrials, wt, scores, fo, s);
    }
    return exact ? launch_irs<NB, false, true>(fold, ntrials, wt, scores, fo, s)
                 : launch_irs<NB, false, false>(fold, ntrials, wt, scores, fo, s);
}

}  // namespace

bool irfft_score_supported(uint32_t nbins) { return nbins == 16 || nbins == 32 || nbins == 64; }

void irfft_score(const float2* fold, uint64_t ntrials, uint32_t nbins, const WidthTable& wt,
                 float* scores, bool find_max, bool exact, hipStream_t s, const FilterOut* fo) {
    LOKI_REQUIRE(irfft_score_supported(nbins), "irfft+score: nbins must be 16, 32 or 64");
    if (ntrials == 0) {
        return;
    }
    const FilterOut f = fo != nullptr ? *fo : FilterOut{};
    if (fo != nullptr) {
        LOKI_REQUIRE(fo->count != nullptr, "score filter: null counter");
        LOKI_REQUIRE(ntrials * (find_max ? 1U : wt.n) <= 0xFFFFFFFFULL,
                     "score filter: trial index exceeds 32 bits");
    }
    switch (nbins) {
    case 16: return dispatch_irs<16>(fold, ntrials, wt, scores, find_max, exact, f, s);
    case 32: return dispatch_irs<32>(fold, ntrials, wt, scores, find_max, exact, f, s);
    default: return dispatch_irs<64>(fold, ntrials, wt, scores, find_max, exact, f, s);
    }
}

}  // namespace loki_amd::kern
