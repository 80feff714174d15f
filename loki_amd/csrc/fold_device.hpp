// Device code of the time brute fold shared by the fold kernels
// (k_brutefold.hip) and the batch's persistent kernel (k_tree.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "grid.hpp"
#include "kernels.hpp"
#include "storage.hpp"

namespace loki_amd::kern {
namespace {

constexpr int kFoldBlock = 256;
constexpr int kPairsBlk  = 2048;  // (freq, bin) pairs per fold block
constexpr int kLdsSamps  = 4096;  // segments up to this length are staged in LDS

// One lane per (segment, freq, bin) pair; consecutive lanes are consecutive
// bins, so list reads and output writes are contiguous.  USE_LDS: the
// segment's samples are staged in the LDS arrays s_e and s_v (kLdsSamps
// floats each, seglen <= kLdsSamps; longer segments take the run path).
// TO: stored element type of the fold (float, or _Float16 / __bf16 with each
// FP32 sum multiplied by `scale` before rounding).
template <bool USE_LDS, typename TO>
__device__ __forceinline__ void bf_fold_block(uint32_t bid, const float* __restrict__ ts_e,
                                              const float* __restrict__ ts_v, uint32_t seglen,
                                              uint32_t nfreqs, uint32_t nbins,
                                              uint32_t blocks_per_seg,
                                              const uint32_t* __restrict__ list,
                                              const uint64_t* __restrict__ base_f,
                                              const uint32_t* __restrict__ counts,
                                              TO* __restrict__ fold, float scale,
                                              float* __restrict__ s_e,
                                              float* __restrict__ s_v) {
    const uint64_t seg   = bid / blocks_per_seg;
    const uint32_t pbase = (bid % blocks_per_seg) * kPairsBlk;
    const uint32_t npair = nfreqs * nbins;
    const float* __restrict__ ge = ts_e + seg * seglen;
    const float* __restrict__ gv = ts_v + seg * seglen;
    if constexpr (USE_LDS) {
        for (uint32_t k = threadIdx.x; k < seglen; k += kFoldBlock) {
            s_e[k] = ge[k];
            s_v[k] = gv[k];
        }
        __syncthreads();
    }
    const float* __restrict__ e = USE_LDS ? s_e : ge;
    const float* __restrict__ v = USE_LDS ? s_v : gv;
    const uint32_t pend = min(pbase + static_cast<uint32_t>(kPairsBlk), npair);
    for (uint32_t p = pbase + threadIdx.x; p < pend; p += kFoldBlock) {
        const uint32_t f   = p / nbins;
        const uint32_t b   = p - f * nbins;
        const uint32_t cnt = counts[p];
        const uint32_t* __restrict__ lst = list + base_f[f] + b;
        float se = 0.0F;
        float sv = 0.0F;
        uint32_t k = 0;
        for (; k + 4 <= cnt; k += 4) {
            const uint32_t i0 = lst[static_cast<uint64_t>(k) * nbins];
            const uint32_t i1 = lst[static_cast<uint64_t>(k + 1) * nbins];
            const uint32_t i2 = lst[static_cast<uint64_t>(k + 2) * nbins];
            const uint32_t i3 = lst[static_cast<uint64_t>(k + 3) * nbins];
            const float e0 = e[i0], e1 = e[i1], e2 = e[i2], e3 = e[i3];
            const float v0 = v[i0], v1 = v[i1], v2 = v[i2], v3 = v[i3];
            se = se + e0;
            sv = sv + v0;
            se = se + e1;
            sv = sv + v1;
            se = se + e2;
            sv = sv + v2;
            se = se + e3;
            sv = sv + v3;
        }
        for (; k < cnt; ++k) {
            const uint32_t i = lst[static_cast<uint64_t>(k) * nbins];
            se = se + e[i];
            sv = sv + v[i];
        }
        TO* __restrict__ out = fold + (seg * nfreqs + f) * 2 * nbins;
        if constexpr (std::is_same_v<TO, float>) {
            out[b]         = se;
            out[nbins + b] = sv;
        } else {
            out[b]         = narrow1<TO>(se * scale);
            out[nbins + b] = narrow1<TO>(sv * scale);
        }
    }
}

// ---------------------------------------------------------------------------
// Long segments: bucket sums over contiguous runs, no lists.
// For one frequency the unwrapped bin U(k) (grid::unwrapped_bin) is
// non-decreasing in the sample index k, so bin b's samples are the runs
// [K(u), K(u + 1)) for u = b (mod nbins), K(u) = min{k : U(k) >= u}.  Each lane
// finds its run boundaries from an analytic estimate corrected against the
// exact U (a binary search if the estimate is far off) and sums the runs in
// ascending k: the same elements in the same order as the bucket list.
// ---------------------------------------------------------------------------
__device__ __forceinline__ int64_t u_at(uint32_t k, double tsamp, double t_ref, double f,
                                        uint32_t nbins) {
    const double t = (static_cast<double>(k) * tsamp) - t_ref;
    return grid::unwrapped_bin(t, f, nbins);
}

/// Per-frequency constants of run_bound: k_est(u) = (u - 1/2) A + B with
/// A = 1 / (nbins f tsamp) samples per bin and B = t_ref / tsamp, and the bound
/// eta (in bins) on the rounding of U(k) against nbins (k tsamp - t_ref) f:
/// the FP32 conversion and +0.5F of the bin ((2 nbins + 1/2) 2^-24) plus the
/// FP64 evaluation of the phase (3 * 2^-53 (n tsamp + |t_ref|) f nbins).
struct RunGeom {
    double f, A, B, eta_len;
};

__device__ __forceinline__ RunGeom run_geom(double f, uint32_t n, double tsamp, double t_ref,
                                            uint32_t nbins) {
    RunGeom g;
    g.f             = f;
    const double nb = static_cast<double>(nbins);
    g.A             = 1.0 / (nb * f * tsamp);
    g.B             = t_ref / tsamp;
    const double eta = ((2.0 * nb) + 0.5) * 0x1p-24 +
                       3.0 * 0x1p-53 * ((static_cast<double>(n) * tsamp) + fabs(t_ref)) * f * nb;
    g.eta_len       = eta * g.A;  // in samples
    return g;
}

/// K(u) = min{k in [0, n] : U(k) >= u} (n if none).  U(k) >= u exactly when
/// nbins (k tsamp - t_ref) f >= u - 1/2 up to eta bins, i.e. k >= k_est(u) up to
/// eta * A samples; when k_est is farther than 4x that (plus its own FP64
/// rounding) from an integer, K = ceil(k_est) needs no check.  Otherwise the
/// estimate is corrected against the exact U (a binary search if it is far).
__device__ __forceinline__ uint32_t run_bound(int64_t u, uint32_t n, double tsamp, double t_ref,
                                              const RunGeom& g, uint32_t nbins) {
    const double est = ((static_cast<double>(u) - 0.5) * g.A) + g.B;
    if (est > 0.0 && est < static_cast<double>(n)) {
        const double fr = est - floor(est);
        const double m  = (4.0 * g.eta_len) + 16.0 * 0x1p-53 * (est + 2.0 * fabs(g.B)) + 1e-9;
        if (fr > m && fr < 1.0 - m) {
            return static_cast<uint32_t>(ceil(est));
        }
    }
    const double f = g.f;
    uint32_t k = 0;
    if (est >= static_cast<double>(n)) {
        k = n;
    } else if (est > 0.0) {
        k = static_cast<uint32_t>(ceil(est));
        k = k > n ? n : k;
    }
    for (int it = 0; it < 4 && k > 0 && u_at(k - 1, tsamp, t_ref, f, nbins) >= u; ++it) {
        --k;
    }
    for (int it = 0; it < 4 && k < n && u_at(k, tsamp, t_ref, f, nbins) < u; ++it) {
        ++k;
    }
    const bool lo_ok = k == 0 || u_at(k - 1, tsamp, t_ref, f, nbins) < u;
    const bool hi_ok = k == n || u_at(k, tsamp, t_ref, f, nbins) >= u;
    if (lo_ok && hi_ok) {
        return k;
    }
    uint32_t lo = 0, hi = n;  // invariant: answer in [lo, hi]
    while (lo < hi) {
        const uint32_t mid = lo + (hi - lo) / 2;
        if (u_at(mid, tsamp, t_ref, f, nbins) >= u) {
            hi = mid;
        } else {
            lo = mid + 1;
        }
    }
    return lo;
}

// A block owns NF frequencies of one segment with all their bins; their running
// sums live in LDS, and per chunk of samples the block deals the (frequency,
// bin) units that have samples in the chunk -- for each frequency the bins of
// the unwrapped range [U(c0), U(c1 - 1)] -- out to the lanes.  A unit adds all
// runs of its bin inside the chunk to the bin's running sum in ascending
// sample order, so every bucket is the same ordered FP32 sum as the bucket
// list's.  The next chunk is on its way into registers, and its units are
// counted by the last wave, while the units of this one are added.
//
// VALU and LDS bound it together (256 series of 2^18 to 2^22 samples, 2.6e11
// (sample, frequency) pairs, 59 ms: 5.8 lane-instructions per pair, two of them
// the adds, 39 ms of single-issue VALU, and 25 ms a CU of bank conflicts between
// the lanes' runs).  1024 pairs per block leave five blocks on a CU (26 KB of LDS,
// 86 registers); 24 series of 2^18 to 2^21 samples, 1.3e10 pairs, take 4.0 ms, and
// took 5.3 ms with 4096 pairs (three blocks), every boundary by run_bound and the
// staging unhidden.  Chunks of 4096 samples keep more lanes busy
// where a launch is too small to fill the chip (2^20 samples, 403 frequencies,
// 0.5-2 Hz: 0.18 against 0.20 ms, 0.49 ms before; 2^17 samples 0.03 against 0.21
// ms before); they hold three blocks of 64 bins on a CU (43 KB; four by their 102
// registers) and cost a larger launch (the batch above: 4.6 ms).
constexpr int kUnitChunk      = 2048;  // samples staged per chunk
constexpr int kUnitChunkSmall = 4096;  // ... where all blocks are resident at once
constexpr uint32_t kUnitPairs = 1024;  // (frequency, bin) pairs per block
constexpr int kUnitMaxNF      = 64;    // frequencies per block (one wave counts their units)

/// What a block keeps per frequency; the chunk's part twice, in turn.
struct UnitChunk {
    double est;        ///< estimated start of bin ulo, from the chunk's first sample
    int64_t ulo, uhi;  ///< unwrapped bins of the chunk's first and last sample
    uint32_t cnt, b0;  ///< units in the chunk, bin of the first
};
struct UnitFreq {
    RunGeom g;
    double sure;  ///< 1/2 less the estimates' error bound (samples)
    UnitChunk c[2];
};

/// LDS of a block of nf frequencies.
inline size_t unit_lds_bytes(uint32_t nf, uint32_t nbins, int chunk) {
    return static_cast<size_t>(chunk) * sizeof(float2) +
           nf * (nbins * sizeof(float2) + sizeof(UnitFreq)) + 2 * sizeof(uint32_t);
}

/// First sample of the chunk at or after the beginning of bin ulo + i: the
/// smallest integer not below est + i A unless that is too close to an
/// integer to tell (run_bound's margin, so the same value), then run_bound.
template <int CHUNK>
__device__ __forceinline__ uint32_t unit_start(const UnitFreq& q, const UnitChunk& c, double i,
                                               uint32_t c0, uint32_t c1, uint32_t seglen,
                                               double tsamp, double t_ref, uint32_t nbins) {
    const double est = fma(i, q.g.A, c.est);
    const double up  = ceil(est);
    if (fabs((up - est) - 0.5) < q.sure && est < static_cast<double>(CHUNK)) {
        const auto k = static_cast<uint32_t>(fmax(up, 0.0));
        return min(k, c1 - c0);
    }
    const uint32_t k =
        run_bound(c.ulo + static_cast<int64_t>(i), seglen, tsamp, t_ref, q.g, nbins);
    return min(max(k, c0), c1) - c0;
}

template <typename TO, int CHUNK = kUnitChunk>
__device__ __forceinline__ void bf_units_block(uint32_t bid, const float* __restrict__ ts_e,
                                               const float* __restrict__ ts_v, uint32_t seglen,
                                               uint32_t nfreqs, uint32_t nbins,
                                               uint32_t blocks_per_seg,
                                               const double* __restrict__ freqs, double tsamp,
                                               double t_ref, TO* __restrict__ fold, float scale) {
    constexpr int kPre = CHUNK / kFoldBlock;  // samples a lane stages per chunk
    extern __shared__ __align__(16) unsigned char s_mem[];
    const uint32_t NF  = (nfreqs + blocks_per_seg - 1) / blocks_per_seg;
    auto* s_ev         = reinterpret_cast<float2*>(s_mem);  // [CHUNK], 16-byte aligned
    auto* acc          = s_ev + CHUNK;                   // [NF][nbins]
    auto* fq           = reinterpret_cast<UnitFreq*>(acc + NF * nbins);  // [NF]
    auto* ncol         = reinterpret_cast<uint32_t*>(fq + NF);  // [2]: most units of a frequency
    const uint64_t seg = bid / blocks_per_seg;
    const uint32_t f0  = (bid % blocks_per_seg) * NF;
    if (f0 >= nfreqs) {
        return;
    }
    const uint32_t nf  = min(NF, nfreqs - f0);
    const float* __restrict__ ge = ts_e + seg * seglen;
    const float* __restrict__ gv = ts_v + seg * seglen;
    const int64_t nb    = nbins;
    const uint32_t tid  = threadIdx.x;
    const uint32_t lane = tid % 64;
    const bool counter  = tid / 64 == kFoldBlock / 64 - 1;  // the counting wave
    for (uint32_t i = tid; i < nf * nbins; i += kFoldBlock) {
        acc[i] = make_float2(0.0F, 0.0F);
    }
    auto count = [&](uint32_t c0, uint32_t turn) {
        const uint32_t c1 = min(c0 + static_cast<uint32_t>(CHUNK), seglen);
        uint32_t cnt      = 0;
        if (lane < nf) {
            const RunGeom g  = fq[lane].g;
            const int64_t lo = u_at(c0, tsamp, t_ref, g.f, nbins);
            const int64_t hi = u_at(c1 - 1, tsamp, t_ref, g.f, nbins);
            cnt              = hi < lo ? 0U : static_cast<uint32_t>(min(hi - lo + 1, nb));
            UnitChunk& c     = fq[lane].c[turn];
            c.est            = (((static_cast<double>(lo) - 0.5) * g.A) + g.B) - c0;
            c.ulo            = lo;
            c.uhi            = hi;
            c.cnt            = cnt;
            c.b0             = static_cast<uint32_t>(((lo % nb) + nb) % nb);
        }
        for (int o = 32; o > 0; o >>= 1) {
            cnt = max(cnt, static_cast<uint32_t>(__shfl_xor(static_cast<int>(cnt), o)));
        }
        if (lane == 0) {
            ncol[turn] = cnt;
        }
    };
    float pe[kPre], pv[kPre];
    auto fetch = [&](uint32_t c0) {
#pragma unroll
        for (int i = 0; i < kPre; ++i) {
            const uint32_t k = c0 + tid + i * kFoldBlock;
            pe[i]            = k < seglen ? ge[k] : 0.0F;
            pv[i]            = k < seglen ? gv[k] : 0.0F;
        }
    };
    fetch(0);
    if (counter) {
        if (lane < nf) {
            const RunGeom g = run_geom(freqs[f0 + lane], seglen, tsamp, t_ref, nbins);
            fq[lane].g      = g;
            fq[lane].sure   = 0.5 - ((4.0 * g.eta_len) + 1e-9 +
                                   32.0 * 0x1p-53 * (static_cast<double>(seglen) + 2.0 * fabs(g.B)));
        }
        count(0, 0);
    }
    uint32_t turn = 0;
    for (uint32_t c0 = 0; c0 < seglen; c0 += CHUNK, turn ^= 1U) {
        const uint32_t c1 = min(c0 + static_cast<uint32_t>(CHUNK), seglen);
        __syncthreads();  // the previous chunk's units are done with s_ev, this one's counted
#pragma unroll
        for (int i = 0; i < kPre; ++i) {
            s_ev[tid + i * kFoldBlock] = make_float2(pe[i], pv[i]);
        }
        __syncthreads();
        if (c1 < seglen) {
            fetch(c1);
            if (counter) {
                count(c1, turn ^ 1U);
            }
        }
        const uint32_t cols = ncol[turn];
        const float inv     = 1.0F / static_cast<float>(cols);
        for (uint32_t t = tid; t < nf * cols; t += kFoldBlock) {
            // t / cols: below 2^16, where the rounded product is off by less than half
            const uint32_t fi  = static_cast<uint32_t>((static_cast<float>(t) + 0.5F) * inv);
            const uint32_t i   = t - fi * cols;
            const UnitFreq& q  = fq[fi];
            const UnitChunk& c = q.c[turn];
            if (i >= c.cnt) {
                continue;
            }
            const uint32_t b = c.b0 + i;
            float2* slot     = acc + fi * nbins + (b >= nbins ? b - nbins : b);
            float ae = slot->x, av = slot->y;
            double u = static_cast<double>(i);
            for (int64_t ui = c.ulo + i; ui <= c.uhi; ui += nb, u += static_cast<double>(nbins)) {
                uint32_t k = unit_start<CHUNK>(q, c, u, c0, c1, seglen, tsamp, t_ref, nbins);
                const uint32_t z =
                    unit_start<CHUNK>(q, c, u + 1.0, c0, c1, seglen, tsamp, t_ref, nbins);
                if ((k & 1U) != 0 && k < z) {  // align to a sample pair
                    const float2 x = s_ev[k];
                    ae = ae + x.x;
                    av = av + x.y;
                    ++k;
                }
                // 16-byte reads of two (e, v) pairs (fewer LDS instructions, and 8 lanes
                // per LDS pass instead of 16), 16 samples per step, then 8, then one by
                // one: every sample is still added in ascending order
                const uint32_t npair = k < z ? (z - k) / 2 : 0;
                const auto* __restrict__ p = reinterpret_cast<const float4*>(s_ev) +
                                              (k < z ? k / 2 : 0);
                const float4* const pend = p + npair;
                for (; p + 8 <= pend; p += 8) {
                    float4 y[8];
#pragma unroll
                    for (int w = 0; w < 8; ++w) {
                        y[w] = p[w];
                    }
#pragma unroll
                    for (int w = 0; w < 8; ++w) {
                        ae = ae + y[w].x;
                        av = av + y[w].y;
                        ae = ae + y[w].z;
                        av = av + y[w].w;
                    }
                }
                if (p + 4 <= pend) {
                    float4 y[4];
#pragma unroll
                    for (int w = 0; w < 4; ++w) {
                        y[w] = p[w];
                    }
#pragma unroll
                    for (int w = 0; w < 4; ++w) {
                        ae = ae + y[w].x;
                        av = av + y[w].y;
                        ae = ae + y[w].z;
                        av = av + y[w].w;
                    }
                    p += 4;
                }
                for (; p < pend; ++p) {
                    const float4 y = *p;
                    ae = ae + y.x;
                    av = av + y.y;
                    ae = ae + y.z;
                    av = av + y.w;
                }
                k += 2 * npair;
                if (k < z) {  // an odd last sample
                    const float2 x = s_ev[k];
                    ae = ae + x.x;
                    av = av + x.y;
                }
            }
            *slot = make_float2(ae, av);
        }
    }
    __syncthreads();
    for (uint32_t i = tid; i < nf * nbins; i += kFoldBlock) {
        const uint32_t fi    = i / nbins;
        const uint32_t b     = i - fi * nbins;
        TO* __restrict__ out = fold + (seg * nfreqs + f0 + fi) * 2 * nbins;
        if constexpr (std::is_same_v<TO, float>) {
            out[b]         = acc[i].x;
            out[nbins + b] = acc[i].y;
        } else {
            out[b]         = narrow1<TO>(acc[i].x * scale);
            out[nbins + b] = narrow1<TO>(acc[i].y * scale);
        }
    }
}

}  // namespace
}  // namespace loki_amd::kern
