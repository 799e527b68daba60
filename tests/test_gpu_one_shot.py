"""`acquire` (plan and search in one call) takes the form with the smaller sum.

Code spectra of the full-period correlation are plan data, which a plan of one
call pays for each time: up to four steps, and with surfaces, `acquire` builds
the plan without them. The kernels of its plans, and its results against a kept
plan's: the same place, powers to the bar of tests/test_gpu_full_corr.py.
"""
import numpy as np
import pytest

from acquisition import GPSL1CA, acquire, acquire_, plan_acquire
from acquisition import _native
from acquisition._native import ELTYPE
from acquisition.signals import generate_test_signal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nnc,store,full", [(1, False, False), (4, False, False), (5, False, True), (5, True, False)])
def test_plans_of_one_call(nnc, store, full, monkeypatch):
    made = []
    create = _native.NativePlan.create.__func__

    def record(cls, plan):
        native = create(cls, plan)
        made.append(native.call_kernels(ELTYPE["cf32"], 2))
        return native

    fs, prns = 4e6, [7, 12]
    sig = generate_test_signal(GPSL1CA(), 7, num_samples=nnc * 8000, sampling_freq=fs, interm_freq=0.0, doppler=1730.0,
                               code_phase=411.3, CN0=52, seed=0x5EED0F31)["signal"].astype(np.complex64)
    kw = dict(num_coherently_integrated_code_periods=2, num_noncoherent_accumulations=nnc)
    plan = plan_acquire(GPSL1CA(), fs, prns, **kw)
    try:
        kept = acquire_(plan, sig, prns)
    finally:
        plan.close()
    monkeypatch.setattr(_native.NativePlan, "create", classmethod(record))
    once = acquire(GPSL1CA(), sig, fs, prns, store_power_bins=store, **kw)
    assert len(made) == 1 and ("_full" in made[0]) == full
    a, b = once[0], kept[0]
    assert (a.code_phase, a.carrier_doppler) == (b.code_phase, b.carrier_doppler)
    assert abs(a.engine_stats["peak"] / b.engine_stats["peak"] - 1) <= 1e-5
    assert abs(a.noise_power / b.noise_power - 1) <= 1e-6
