"""Coherent periods of the full-period correlation.

Its fold over the coherent periods costs their square and sums one by one, so
searches of more than 32 periods (pilots without data bits and rotation) keep
to the tile. At both sides of that limit and far beyond: the kernels of a call,
and the statistics against the FP64 oracle. The tile path stays within 2.5e-7
of the peak there; the bar is 4e-7 (the sequential fold reaches 4.9e-7 at 2000
periods), 1e-6 for the mean noise.
"""
import numpy as np
import pytest

import oracle
from acquisition import acquire_, plan_acquire
from acquisition._native import ELTYPE
from acquisition.signals import generate_test_signal
from acquisition.systems import SeededCodeSystem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ncoh,cov,full", [(32, 2000.0, True), (33, 2000.0, False), (200, 1500.0, False),
                                           (2000, 400.0, False)])
def test_many_periods_keep_to_the_tile(ncoh, cov, full):
    sysm = SeededCodeSystem("pilot", 1023, 1.023e6, 1575.42e6, 1, 0x5EED0B01)
    prns = [3, 5]
    plan = plan_acquire(sysm, 2.048e6, prns, min_doppler_coverage=cov, num_coherently_integrated_code_periods=ncoh)
    sig = generate_test_signal(sysm, 3, num_samples=ncoh * 2048, sampling_freq=2.048e6, interm_freq=0.0, doppler=130.0,
                               code_phase=321.5, CN0=45, seed=0x5EED0F20 + ncoh)["signal"].astype(np.complex64)
    try:
        assert ("_full" in plan.native.call_kernels(ELTYPE["cf32"], 2)) == full
        res = acquire_(plan, sig, prns)
        _, osurf = oracle.acquire(plan, sig, [0, 1], surfaces=True, bits=64)
        for r, o in zip(res, osurf):
            e = r.engine_stats
            assert abs(e["peak"] - o.max()) <= 4e-7 * o.max()
            assert abs(e["peak"] - o[e["row"], e["col"]]) <= 4e-7 * o.max()
            mean = o[(e["row"] + o.shape[0] // 2) % o.shape[0]].astype(np.float64).mean()
            assert abs(e["noise"] / mean - 1) <= 1e-6
    finally:
        plan.close()
