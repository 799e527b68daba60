"""tile_precision "auto" takes the full-period correlation before the FP16 tile.

Integer samples at 160 bins: statistics-only calls of an "auto" plan are those of
an "fp32" plan, bit for bit, through both entry points; calls with surfaces keep
the FP16 tile.
"""
import numpy as np
import pytest

from acquisition import GPSL1CA, plan_acquire
from acquisition._native import ELTYPE, FLAG_DEVICE_SIGNAL, FLAG_STORE_SURFACES
from acquisition.device import DeviceArray

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fs,kind", [(16.368e6, "i16"), (4e6, "ci8")])
def test_auto_runs_the_faster_exact_form(fs, kind):
    n = 2 * 10 * int(fs / 1e3)
    shape = (n,) if kind == "i16" else (n, 2)
    sig = np.random.default_rng(3).integers(-100, 100, shape).astype(np.int16 if kind == "i16" else np.int8)
    dev = DeviceArray(sig)
    raw = []
    try:
        for prec in ("fp32", "auto", "fp16"):
            plan = plan_acquire(GPSL1CA(), fs, [1, 2, 3], num_coherently_integrated_code_periods=10,
                                num_noncoherent_accumulations=2, tile_precision=prec)
            try:
                assert plan.num_doppler_bins == 160
                name = plan.native.call_kernels(ELTYPE[kind], 3)
                assert ("_full" in name) == (prec != "fp16") and ("fp16" in name) == (prec == "fp16")
                assert ("fp16" in plan.native.call_kernels(ELTYPE[kind], 3, FLAG_STORE_SURFACES)) == (prec != "fp32")
                a = plan.native.acquire(dev.ptr, ELTYPE[kind], n, fs / 4, [0, 1, 2], FLAG_DEVICE_SIGNAL)
                b = plan.native.acquire_noalloc(dev.ptr, ELTYPE[kind], n, fs / 4, [0, 1, 2])
                raw.append([bytes(memoryview(x).cast("B")) for x in (a, b)])
            finally:
                plan.close()
    finally:
        dev.free()
    assert raw[0][0] == raw[0][1] == raw[1][0] == raw[1][1]
    assert raw[2][0] == raw[2][1] != raw[0][0]
