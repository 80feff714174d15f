"""The run path of the time brute fold (segments over 4096 samples) against the oracle, bit for
bit, in both of its forms: launches whose blocks are resident at once (chunks of 4096 samples, few
frequencies per block where there are few) and larger ones (chunks of 2048), with 1024 (frequency,
bin) pairs per block, up to 2048 where a chunk holds few of them."""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TSAMP = 64e-6


@pytest.mark.parametrize(("seglen", "nseg", "nbins", "nfreqs", "f_lo", "f_hi", "t_ref"), [
    (4097, 1, 64, 1, 0.5, 0.5, 0.0),          # one block, a second chunk of one sample
    (8192, 3, 64, 37, 0.5, 2.0, 0.0),         # runs of hundreds of samples
    (5000, 9, 50, 41, 1.0, 30.0, 0.16),       # bins not a power of two, negative unwrapped bins
    (16384, 16, 32, 60, 2.0, 10.0, 1.3),
    (6000, 5, 17, 19, 20.0, 9000.0, 0.0),     # many cycles per chunk, runs of one sample or none
    (4100, 70, 1000, 3, 0.3, 0.7, 0.0),       # two frequencies per block, then one
    (4100, 9, 1024, 5, 300.0, 900.0, 0.0),    # one
    (8192, 300, 64, 120, 3.0, 12.0, 0.0),     # over 1024 blocks
    (4608, 1200, 128, 9, 5.0, 40.0, 0.147),   # over 1024 blocks, a chunk of 512 samples
    (4608, 256, 512, 9, 0.3, 1.0, 0.0),       # 768 blocks of 2048 pairs: all resident
    (4608, 257, 512, 9, 0.3, 1.0, 0.0),       # 771: small chunks
    (5000, 1024, 8, 3, 40.0, 90.0, 0.0),      # 1024 blocks, four a CU
    (10000, 900, 5, 300, 0.01, 800.0, 0.0),   # five bins, cycles from 20 samples to the segment
])
def test_long_segments_bit_exact(oracle, seglen, nseg, nbins, nfreqs, f_lo, f_hi, t_ref):
    from loki_amd import libculoki

    rng = np.random.default_rng(seglen + nbins)
    n = seglen * nseg
    ts_e = rng.standard_normal(n, dtype=np.float32)
    ts_v = (0.5 + rng.random(n)).astype(np.float32)
    freqs = np.linspace(f_lo, f_hi, nfreqs)
    rng.shuffle(freqs)  # the fold takes frequencies in any order
    got = libculoki.fold.compute_brute_fold_time_cuda(ts_e, ts_v, freqs, seglen, nbins, TSAMP,
                                                      t_ref)
    want = oracle.brute_fold_time(ts_e, ts_v, freqs, seglen, nbins, TSAMP, t_ref)
    np.testing.assert_array_equal(got, want)
