"""Block correlation on in-place transforms (k_corr_fc).

The sizes that the runtime-radix k_corr_tile ran with one transform per pass:
above 2048 points, or with a prime radix above 5 in a middle stage. F 686
(2 7^3), 2744, 3000, 4096 (padded LDS), 5600 and 6480, with few and many column
blocks (one and several workgroups per row), one and two steps, FP32 tiles and
the FP16 tile (F 3136): surfaces against the FP32 oracle
(src/coherent_integration.jl:136-171), to the bar of tests/parity.py.
"""
import numpy as np
import pytest

import oracle
from acquisition import GPSL1CA, acquire_, plan_acquire
from acquisition.signals import generate_test_signal
from parity import check_prn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("spc,nb,F,ncoh,nnc", [(5115, 15, 686, 1, 2), (16368, 12, 2744, 1, 1), (16368, 11, 3000, 2, 1),
                                              (16384, 8, 4096, 1, 2), (8370, 3, 5600, 2, 2), (6480, 2, 6480, 4, 1),
                                              (27900, 10, 5600, 1, 1)])
def test_in_place_correlation_matches_the_oracle(spc, nb, F, ncoh, nnc):
    sysm = GPSL1CA()
    fs = spc * 1e3
    g = generate_test_signal(sysm, 7, num_samples=spc * ncoh * nnc, sampling_freq=fs, interm_freq=0.0, doppler=300.0,
                             code_phase=333.25, CN0=50, seed=0x5EED0D20 + F)
    sig = g["signal"].astype(np.complex64)
    cov = max(1.0, (nb - 2 / ncoh) / 2 * 1e3 - 1.0)
    plan = plan_acquire(sysm, fs, [7, 12], min_doppler_coverage=cov, num_coherently_integrated_code_periods=ncoh,
                        num_noncoherent_accumulations=nnc)
    try:
        assert (plan.num_blocks, plan.fft_size) == (nb, F)
        res = acquire_(plan, sig, [7, 12], subsample_interpolation=True, store_power_bins=True)
        ores, osurf = oracle.acquire(plan, sig, [0, 1], subsample_interpolation=True, surfaces=True)
        for j, p in enumerate([7, 12]):
            check_prn(res[j], ores[j], osurf[j], res[j].power_bins, interp=True, label=f"F {F} prn {p}",
                      fp64_surface=lambda j=j: oracle.acquire(plan, sig, [0, 1], surfaces=True, bits=64)[1][j])
    finally:
        plan.close()


def test_fp16_tile_behind_the_in_place_correlation():
    """GPS L1 C/A at 25 MHz, N_coh 10, ndop 160 (bs 1562 has no nb 16; 25.088 MHz: bs 1568, F 3136 = 2^6 7^2)."""
    fs, sysm = 25.088e6, GPSL1CA()
    g = generate_test_signal(sysm, 7, num_samples=2 * 250880, sampling_freq=fs, interm_freq=0.0, doppler=300.0,
                             code_phase=333.25, CN0=50, seed=0x5EED0D30)["signal"]
    sig = np.rint(200 * np.stack([g.real, g.imag], axis=1) / np.std(g)).astype(np.int16)
    out = []
    for prec in ("fp32", "fp16"):
        plan = plan_acquire(sysm, fs, [7], num_coherently_integrated_code_periods=10, num_noncoherent_accumulations=2,
                            tile_precision=prec)
        try:
            assert plan.num_doppler_bins == 160 and plan.fft_size == 3136
            out.append(np.array(acquire_(plan, sig, [7], store_power_bins=True)[0].power_bins, copy=True))
        finally:
            plan.close()
    a, b = out
    # the bar of the FP16 tile (tests/test_gpu_mixed.py)
    assert np.abs(a - b).max() <= 2e-3 * a.max()
    m = a >= 1e-3 * a.max()
    assert (np.abs(a - b)[m] / a[m]).max() <= 2e-2 and not np.array_equal(a, b)
