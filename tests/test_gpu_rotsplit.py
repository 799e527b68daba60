"""Direct rotation search of few Doppler rows (k_column_rotsplit).

L5-like pilots (10-chip secondary code) over one and two secondary periods
(N_coh 10 and 20) at every compiled row length (nb 4-13, 15, 16, 20, 22), odd
and even (LDS padding), with 32 and 16 columns per workgroup, a ragged last
workgroup, and two noncoherent steps: surfaces and statistics against the FP32
oracle (src/noncoherent_integration.jl:183-297), to the bar of tests/parity.py.
"""
import numpy as np
import pytest

import oracle
from acquisition import acquire_, plan_acquire
from acquisition.signals import generate_test_signal
from acquisition.systems import L5Like
from parity import check_prn

pytestmark = pytest.mark.gpu

ROWS = [(600e3, (4, 5, 6, 8, 10, 12, 15, 20)), (819e3, (7, 9, 13)), (528e3, (11, 16, 22))]


@pytest.mark.parametrize("ncoh", [10, 20])
@pytest.mark.parametrize("fs,nb", [(fs, nb) for fs, nbs in ROWS for nb in nbs])
def test_every_row_length_matches_the_oracle(fs, nb, ncoh):
    sysm = L5Like()
    spc = int(fs / 1e3)
    n = 2 * ncoh * spc
    g = generate_test_signal(sysm, 3, num_samples=n, sampling_freq=fs, interm_freq=0.0, doppler=430.0,
                             code_phase=4321.5, CN0=58, seed=0x5EED0D10 + nb)
    sig = g["signal"].astype(np.complex64)
    # the smallest coverage whose block count is nb
    cov = (nb - 2 / ncoh) / 2 * 1e3 - 1.0
    plan = plan_acquire(sysm, fs, [3, 5], min_doppler_coverage=cov, num_coherently_integrated_code_periods=ncoh,
                        num_noncoherent_accumulations=2)
    try:
        assert plan.num_blocks == nb and plan.native.column_kernel() == f"k_column_rotsplit<{ncoh},{nb}>"
        res = acquire_(plan, sig, [3, 5], store_power_bins=True)
        ores, osurf = oracle.acquire(plan, sig, [0, 1], surfaces=True)
        for j, p in enumerate([3, 5]):
            check_prn(res[j], ores[j], osurf[j], res[j].power_bins, label=f"nb {nb} N_coh {ncoh} prn {p}",
                      fp64_surface=lambda j=j: oracle.acquire(plan, sig, [0, 1], surfaces=True, bits=64)[1][j])
    finally:
        plan.close()
