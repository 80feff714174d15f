"""Fourier merge passes of one, two and three levels against the FP64 oracle.

Sizes are chosen so that the pass plan (from the top level down: three levels where four
segments per lane fill the card, else two, one where a level is left over or the grid grows)
reaches each kernel: power-of-two and other nbins, accel and freq-only records, 4, 2 and 1
segments per lane.  Bound: a few ulp of |tail| + |head| per level, 1e-5 of the oracle row's
norm after all of them, the bound of tests/test_gpu_fourier.py.
"""

from __future__ import annotations

import numpy as np
import pytest

from test_gpu_fourier import _row_check
from test_gpu_parity import TSAMP, _series

pytestmark = pytest.mark.gpu

CASES = {
    # name: (nsamps, nbins, limits, bseg_brute); above it: passes from the top level down, as
    # levels x segments per lane
    # 2x1, 3x4, 1x4
    "accel_64": (2**18, 64, [(-500.0, 500.0), (8.0, 260.0)], 4096),
    # 1x1, 1x2, 2x2, 2x2, 1x2
    "accel_50_grows": (2**18, 50, [(-5000.0, 5000.0), (8.0, 230.0)], 2048),
    # 2x1, 3x4, 1x4
    "freq_64": (2**18, 64, [(5.0, 150.0)], 4096),
    # 2x1, 2x2, 1x2
    "freq_50": (2**18, 50, [(5.0, 150.0)], 8192),
    # 2x1, 3x4, 2x4
    "freq_50_deep": (2**18, 50, [(5.0, 230.0)], 2048),
}
# the level each pass ends at, as the timing records give it
PASS_ENDS = {
    "accel_64": [1, 4, 6],
    "accel_50_grows": [1, 3, 5, 6, 7],
    "freq_64": [1, 4, 6],
    "freq_50": [1, 3, 5],
    "freq_50_deep": [2, 5, 7],
}


@pytest.mark.parametrize("name", list(CASES))
def test_fourier_passes_within_bound(oracle, name):
    from loki_amd import libculoki, libloki
    from oracle.plan import SearchConfig

    nsamps, nbins, lims, bseg = CASES[name]
    cfg = libloki.configs.PulsarSearchConfig(
        nsamps=nsamps, tsamp=TSAMP, nbins=nbins, eta=1.0, param_limits=np.array(lims),
        use_fourier=True, bseg_brute=bseg)
    ocfg = SearchConfig(nsamps, TSAMP, nbins, 1.0, lims, use_fourier=True, bseg_brute=bseg)
    ts_e, ts_v = _series(nsamps, seed=31)
    ffa = libculoki.ffa.FFACOMPLEXCUDA(cfg, device_id=0)
    ffa.set_timing(True)
    got = np.zeros(ffa.plan.buffer_size, dtype=np.complex64)
    ffa.execute(ts_e, ts_v, got)
    assert [level for kind, level, _ in ffa.timings() if kind == "merge"] == PASS_ENDS[name]
    # one pass per level: the same bits
    ffa.set_two_level_merges(False)
    single = np.zeros_like(got)
    ffa.execute(ts_e, ts_v, single)
    assert [level for kind, level, _ in ffa.timings() if kind == "merge"] == \
        list(range(1, int(ffa.plan.n_levels)))
    size = int(ffa.plan.fold_size)
    np.testing.assert_array_equal(got[:size].view(np.float32), single[:size].view(np.float32))
    want, _ = oracle.compute_ffa(ts_e, ts_v, ocfg, fourier=True)
    _row_check(got[: ffa.plan.fold_size], want, nbins // 2 + 1, 1e-5, name)


@pytest.mark.parametrize("name", ["accel_64", "freq_64"])
def test_fused_scores_of_a_ragged_trial_count(name):
    """The fused return + S/N against the separate one, both within 1e-4 + 1e-5 |S/N| of the
    exact values, where the last tile and the last wave's rows are not full."""
    from loki_amd import libculoki, libloki

    nsamps, nbins, lims, bseg = CASES[name]
    cfg = libloki.configs.PulsarSearchConfig(
        nsamps=nsamps, tsamp=TSAMP, nbins=nbins, eta=1.0, param_limits=np.array(lims),
        use_fourier=True, bseg_brute=bseg)
    ts_e, ts_v = _series(nsamps, seed=32)
    widths = np.array([1, 2, 7, 31, 63], dtype=np.uint64)
    ffa = libculoki.ffa.FFACOMPLEXCUDA(cfg, device_id=0)
    got = np.asarray(ffa.scores(ts_e, ts_v, widths, False)).ravel()
    assert (got.size // widths.size) % 8 != 0
    ffa.set_fused(False)
    want = np.asarray(ffa.scores(ts_e, ts_v, widths, False)).ravel()
    assert np.all(np.abs(got - want) <= 2 * (1e-4 + 1e-5 * np.abs(want)))
