"""Full-period correlation (statistics-only calls of simple-path plans).

A Doppler row is one circular correlation of the code period (k_full_corr,
runtime radices; k_full31_corr, the multiples of 31 samples with matrix-core
31-point DFTs) instead of the coherent tile and its column transform. Both are
compared with the tile path of the same search (`tile_path` plans) at the edges
of their radix plans: powers of two (padded LDS), odd and prime-power periods,
radices 7, 11, 13, 22 and 25, odd column counts, one and several noncoherent
steps with drift, one and several coherent periods (an odd row count among
them), sample types with an IF, both noise estimators, one PRN and a batch.

Both paths are FP32 transforms of the same search, each within a few 1e-7 of
the FP64 result relative to the row's power. The bar: 1e-5 of the peak for the
peak and its four neighbours, 1e-6 for the mean noise, the same peak cell (the
searched PRN is present, so its peak stands clear of every other cell).
"""
import numpy as np
import pytest

from acquisition import GPSL1CA, acquire_
from acquisition import _native
from acquisition.estimators import GlobalMeanNoiseEstimator, OppositeRowNoiseEstimator
from acquisition.plan import _plan_host
from acquisition.signals import generate_test_signal

pytestmark = pytest.mark.gpu


def _plan(fs, prns, tile, **kw):
    plan = _plan_host(GPSL1CA(), fs, prns, **kw)
    plan.tile_path = tile
    plan.native = _native.NativePlan.create(plan)
    return plan


def _signal(fs, n, if_hz, kind, seed):
    g = generate_test_signal(GPSL1CA(), 7, num_samples=n, sampling_freq=fs, interm_freq=if_hz, doppler=1730.0,
                             code_phase=411.3, CN0=52, seed=seed)["signal"]
    g = g / np.std(g)
    if kind == "i16":
        return np.rint(1000 * g.real).astype(np.int16)
    if kind == "ci8":
        q = np.stack([g.real, g.imag], axis=1)
        return np.clip(np.rint(30 * q), -127, 127).astype(np.int8)
    return g.astype(np.complex64)


def _check(fs, coh, nnc, *, kind="cf32", if_hz=0.0, prns=(7, 12), est=OppositeRowNoiseEstimator(), cov=7000.0):
    prns = list(prns)
    kw = dict(num_coherently_integrated_code_periods=coh, num_noncoherent_accumulations=nnc, noise_estimator=est,
              min_doppler_coverage=cov)
    stats = []
    for tile in (True, False):
        plan = _plan(fs, prns, tile, **kw)
        try:
            sig = _signal(fs, plan.samples_per_code * coh * nnc, if_hz, kind, 0x5EED0F11)
            plan.native.set_timing(True)
            stats.append([r.engine_stats for r in acquire_(plan, sig, prns, interm_freq=if_hz)])
            # the tile path runs the block correlation, the full path does not
            assert (plan.native.kernel_times()["corr_tile"][1] > 0) == tile
        finally:
            plan.close()
    for p, a, b in zip(prns, *stats):
        scale = a["peak"]
        err = max(abs(x - y) for x, y in zip([a["peak"]] + a["nbr"], [b["peak"]] + b["nbr"])) / scale
        print(f"{fs / 1e6} MHz coh {coh} nnc {nnc} prn {p}: {err:.1e} of the peak, noise {b['noise'] / a['noise'] - 1:.1e}")
        if p == 7:
            assert (a["row"], a["col"]) == (b["row"], b["col"])
            assert err <= 1e-5
        assert abs(b["peak"] / a["peak"] - 1) <= 1e-5
        if (a["row"], a["col"]) == (b["row"], b["col"]):
            assert abs(b["noise"] / a["noise"] - 1) <= 1e-6 and a["noise_cells"] == b["noise_cells"]


@pytest.mark.parametrize("spc", [2048, 2500, 3125, 3375, 4000, 5000, 5250, 5500, 6500, 6144, 9000, 10000, 12500,
                                 15000, 16384, 20000])
def test_runtime_radices_match_the_tile_path(spc):
    _check(spc * 1e3, 1, 1)
    _check(spc * 1e3, 2, 3)


@pytest.mark.parametrize("spc", [2046, 2790, 3069, 4092, 5115, 5456, 6138, 8184, 10230, 16368])
def test_multiples_of_31_match_the_tile_path(spc):
    _check(spc * 1e3, 1, 1)
    _check(spc * 1e3, 3, 4)


@pytest.mark.parametrize("fs,coh,nnc,kw", [
    (4.092e6, 10, 2, dict(kind="i16", if_hz=1.023e6)), (4e6, 10, 2, dict(kind="i16", if_hz=1e6)),
    (5.115e6, 11, 2, dict(kind="ci8", if_hz=38400.0)), (5e6, 20, 2, dict(kind="ci8")),
    (4e6, 4, 2, dict(est=GlobalMeanNoiseEstimator())), (4.092e6, 4, 1, dict(est=GlobalMeanNoiseEstimator())),
    (2.046e6, 5, 40, dict(prns=(7,))), (2.048e6, 5, 40, dict(prns=(7,))), (2.5e6, 1, 2, dict(prns=range(1, 33))),
    (16.368e6, 10, 8, dict(cov=5000.0)), (3.375e6, 3, 2, dict(cov=3000.0))])
def test_options_match_the_tile_path(fs, coh, nnc, kw):
    _check(fs, coh, nnc, **kw)
