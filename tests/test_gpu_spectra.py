"""The Fourier brute fold from chunk spectra, at the sizes where it can go wrong.

One segment of K samples is cut into power-of-two chunks of 64 to 2048 samples (the last one
zero-padded); each chunk's FP64 FFT is rounded to FP32 once and interpolated with 9 FP32
weights.  Per value the errors are the rounding of the points and weights (each <= u = 2^-24
relative, at most 9 terms whose absolute sum is below 3 times the chunk's L1 norm: the window's
reciprocal is <= 3.2, the weights sum to 1), the 9 FP32 accumulations and the interpolation's own
6e-8 per sample at worst: 3 L1 (2u + 9u) + L1 u < 35 u L1 at the very worst; the parts add at
random, so the bound asserted is 8 u L1 per chunk sum, and one more u per chunk added in FP32.
"""

from __future__ import annotations

import numpy as np
import pytest

from test_gpu_parity import _series

pytestmark = pytest.mark.gpu

TSAMP = 64e-6
U = 2.0**-24


@pytest.mark.parametrize(("seglen", "nseg", "nbins", "nfreqs", "t_ref"), [
    # the smallest chunks, which a one-off fold takes where there is enough work
    (64, 5500, 16, 96, 0.0),
    (65, 5400, 16, 97, 65 * TSAMP / 2),
    (100, 3500, 50, 99, 0.0021),
    (256, 2600, 2, 64, 0.0),
    # less work: the matrix cores, the same bound
    (64, 5, 16, 48, 0.0),
    (65, 3, 64, 57, 65 * TSAMP / 2),    # zero-padded to 128, centre not at t_ref
    (100, 7, 50, 63, 0.0021),
    (256, 1, 2, 200, 0.0),             # harmonics 0 and 1 only
    (2048, 2, 64, 49, 2048 * TSAMP / 2),   # one full chunk centred on t_ref (no turn)
    (2048, 33, 256, 51, 0.0),
    (2049, 2, 63, 64, 0.0),             # a second chunk of one sample
    (5000, 3, 32, 1, 0.16),
    (16384, 2, 128, 11, 0.0),
    (1024, 700, 64, 301, 1024 * TSAMP / 2),  # several segments per workgroup, ragged outputs
])
def test_fold_from_spectra_within_bound(oracle, seglen, nseg, nbins, nfreqs, t_ref):
    from loki_amd import libculoki

    nsamps = seglen * nseg
    ts_e, ts_v = _series(nsamps, seed=seglen + nbins)
    # up to and beyond the sampling rate at the highest harmonics
    freqs = np.linspace(1.7, 400.0, nfreqs)
    got = libculoki.fold.compute_brute_fold_fourier_cuda(ts_e, ts_v, freqs, seglen, nbins, TSAMP,
                                                         t_ref)
    nbf = nbins // 2 + 1
    k = np.arange(seglen) * TSAMP - t_ref
    x = np.stack([ts_e.reshape(nseg, seglen), ts_v.reshape(nseg, seglen)], 1).astype(np.float64)
    got = got.reshape(nseg, nfreqs, 2, nbf).astype(np.complex128)
    l1 = np.abs(x).sum(axis=2)[:, :, None]
    bound = (8.0 + -(-seglen // 2048)) * U * l1
    worst = 0.0
    for i, f in enumerate(freqs):
        ph = f * k
        w = np.exp(-2j * np.pi * np.outer(ph - np.floor(ph), np.arange(nbf)))
        err = np.abs(got[:, i] - x @ w)
        worst = max(worst, float((err / l1).max() / U))
        assert np.all(err <= bound), (i, float((err / l1).max() / U))
    print(f"K={seglen} nbins={nbins}: max error {worst:.2f} u of the L1 norm")
    assert np.all(got[..., 0].imag == 0)


@pytest.mark.parametrize(("seglen", "nseg", "nfreqs", "t_ref"), [
    (2048, 3, 50, 0.0),          # one chunk
    (2049, 5, 64, 0.0),          # two, the second of one sample
    (65536, 4, 51, 1.7),         # 32
    (1 << 20, 2, 3, 0.0),        # 512
])
def test_harmonic_zero_is_rounded_once(seglen, nseg, nfreqs, t_ref):
    """Harmonic 0 is the segment's sum in FP64, rounded once to FP32: within u = 2^-24 of it
    and the FP64 sum's own error, at most seglen 2^-53 of the L1 norm."""
    from loki_amd import libculoki

    rng = np.random.default_rng(seglen)
    n = seglen * nseg
    ts_e = (3.0 + rng.standard_normal(n)).astype(np.float32)
    ts_v = (1000.0 + 20.0 * rng.standard_normal(n)).astype(np.float32)
    freqs = np.linspace(0.7, 90.0, nfreqs)
    got = libculoki.fold.compute_brute_fold_fourier_cuda(ts_e, ts_v, freqs, seglen, 16, TSAMP,
                                                         t_ref).reshape(nseg, nfreqs, 2, 9)
    x = np.stack([ts_e.reshape(nseg, seglen), ts_v.reshape(nseg, seglen)], 1).astype(np.longdouble)
    want = x.sum(axis=2).astype(np.float64)[:, None]
    l1 = np.abs(x).sum(axis=2).astype(np.float64)[:, None]
    err = np.abs(got[..., 0].real.astype(np.float64) - want)
    assert np.all(err <= U * np.abs(want) + seglen * 2.0**-53 * l1), float((err / want).max() / U)
    assert np.all(got[..., 0].imag == 0)


def test_series_do_not_mix():
    """A NaN in ts_e stays out of the variance rows and of the other segments, and variances
    twelve decades above the samples leave them exact."""
    from loki_amd import libculoki

    seglen, nseg, nbins = 512, 4, 32
    rng = np.random.default_rng(5)
    e = rng.standard_normal(seglen * nseg).astype(np.float32)
    v = np.full(seglen * nseg, 1.0e12, np.float32)
    freqs = np.linspace(20.0, 60.0, 50)

    def fold(a, b):
        return libculoki.fold.compute_brute_fold_fourier_cuda(
            a, b, freqs, seglen, nbins, TSAMP, 0.0).reshape(nseg, freqs.size, 2, nbins // 2 + 1)

    plain = fold(e, np.ones_like(v))
    assert np.array_equal(fold(e, v)[:, :, 0], plain[:, :, 0])
    bad = e.copy()
    bad[seglen + 3] = np.nan
    got = fold(bad, np.ones_like(v))
    assert np.isnan(got[1, :, 0]).all()
    keep = np.ones(nseg, bool)
    keep[1] = False
    assert np.array_equal(got[:, :, 1], plain[:, :, 1])
    assert np.array_equal(got[keep], plain[keep])


def test_passes_of_segments_equal_one():
    """A standalone fold whose spectra exceed its 64 MiB workspace runs in several passes over
    the segments: the same bits as folding each part of the series by itself."""
    from loki_amd import libculoki

    seglen, nbins = 1000, 16
    nseg = 3 * 4000 + 7  # 16.6 kB of spectra per segment
    rng = np.random.default_rng(3)
    e = rng.standard_normal(seglen * nseg, dtype=np.float32)
    v = (0.5 + rng.random(seglen * nseg)).astype(np.float32)
    freqs = np.linspace(10.0, 90.0, 49)

    def fold(lo, hi):
        return np.asarray(libculoki.fold.compute_brute_fold_fourier_cuda(
            e[lo * seglen: hi * seglen], v[lo * seglen: hi * seglen], freqs, seglen, nbins, TSAMP,
            0.0)).reshape(hi - lo, -1)

    whole = fold(0, nseg)
    for lo, hi in ((0, 2500), (2500, 6001), (6001, 9500), (9500, nseg)):
        assert np.array_equal(whole[lo:hi], fold(lo, hi))


@pytest.mark.parametrize(("nsamps", "lims", "bseg", "extra"), [
    # levels larger than the spectra (65 MiB): no memory beyond the presized workspace
    (2**22, [(20.0, 60.0)], 2048, 0),
    # eight frequencies of long segments, levels of 0.3 MiB: the spectra (16.6 MiB) are kept
    (2**20, [(1.0, 1.02)], 65536, 17),
])
def test_spectra_take_the_partner_buffer(nsamps, lims, bseg, extra):
    import torch

    from loki_amd import libculoki, libloki

    cfg = libloki.configs.PulsarSearchConfig(
        nsamps=nsamps, tsamp=TSAMP, nbins=64, eta=1.0, param_limits=np.array(lims),
        use_fourier=True, bseg_brute=bseg)
    e = torch.randn(nsamps, device="cuda")
    v = torch.ones(nsamps, device="cuda")
    plan = libculoki.ffa.FFACOMPLEXCUDA(cfg, 0).plan
    ws = libculoki.ffa.FFAWorkspaceCUDA(device_id=0, buffer_bytes=8 * int(plan.buffer_size),
                                        coord_bytes=16 * int(plan.coord_size))
    ffa = libculoki.ffa.FFACOMPLEXCUDA(cfg, 0, workspace=ws)
    fold = torch.empty(int(plan.buffer_size), dtype=torch.complex64, device="cuda")
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    ffa.execute_device(e.data_ptr(), v.data_ptr(), fold.data_ptr(), fold.numel(), 0)
    torch.cuda.synchronize()
    took = (before - torch.cuda.mem_get_info()[0]) / 2**20
    # the plan's frequencies and row terms, and the allocator's granularity: a few MiB
    assert extra - 1 <= took <= extra + 16, took
