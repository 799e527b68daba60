"""Statistics of column-major accumulators do not depend on the PRN batch.

The reduction of a column-major accumulator adds FP64 partials of column chunks,
so its chunks have to follow from the search alone: a plan whose workspace holds
one PRN at a time and one that holds all give the same statistics, bit for bit
(rotation search of 2000 bins, sign search of two data bits), and so does a plan
of one PRN.
"""
import numpy as np
import pytest

from acquisition import plan_acquire
from acquisition._native import ELTYPE
from acquisition.estimators import GlobalMeanNoiseEstimator, OppositeRowNoiseEstimator
from acquisition.systems import E1Like, GPSL1CA

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("est", [OppositeRowNoiseEstimator(), GlobalMeanNoiseEstimator()])
@pytest.mark.parametrize("sysm,fs,kw", [
    (E1Like(), 1e6, dict(min_doppler_coverage=9000.0, num_coherently_integrated_code_periods=25)),
    (GPSL1CA(), 2.1e6, dict(min_doppler_coverage=6900.0, num_coherently_integrated_code_periods=40))])
def test_batches_give_the_same_statistics(sysm, fs, kw, est, monkeypatch):
    raw = []
    for gb, prns in (("32", [1, 2, 3, 4]), ("0.001", [1, 2, 3, 4]), ("32", [1])):
        monkeypatch.setenv("FMDBZP_WORKSPACE_GB", gb)
        plan = plan_acquire(sysm, fs, prns, num_noncoherent_accumulations=1,
                            noise_estimator=est, **kw)
        try:
            assert plan.native.column_kernel() in ("k_column_rot2000", "k_column_sign")
            n = kw["num_coherently_integrated_code_periods"] * plan.samples_per_code
            # one step of noise that grows over the samples: powers spread widely enough that FP64 sums round
            sig = np.random.default_rng(7).standard_normal((n, 2)) * np.logspace(-3, 0, n)[:, None] ** 2
            sig = sig.astype(np.float32).view(np.complex64).ravel()
            st = plan.native.acquire(sig.ctypes.data, ELTYPE["cf32"], n, 0.0, list(range(len(prns))), 0)
            raw.append([bytes(s) for s in st])
        finally:
            plan.close()
    assert raw[0] == raw[1]
    assert raw[0][0] == raw[2][0]
