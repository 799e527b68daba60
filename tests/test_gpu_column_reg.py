"""Column stage of few Doppler rows in registers (k_column_reg).

L1 C/A at every compiled row count (4 to 32), block sizes around the workgroup
width of 256 columns, one and two noncoherent steps: surfaces and statistics
against the FP32 oracle (src/noncoherent_integration.jl:482-592), to the bar of
tests/parity.py.
"""
import numpy as np
import pytest

import oracle
from acquisition import acquire_, plan_acquire
from acquisition.signals import generate_test_signal
from acquisition.systems import GPSL1CA
from parity import check_prn

pytestmark = pytest.mark.gpu

ROWS = (4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 15, 16, 18, 20, 21, 22, 24, 25, 30, 32)


@pytest.mark.parametrize("rows,bs,nnc", [(n, (255, 256, 257, 1023 // n + 1)[i % 4], 1 + i % 2)
                                         for i, n in enumerate(ROWS)])
def test_every_row_count_matches_the_oracle(rows, bs, nnc):
    sysm = GPSL1CA()
    ncoh = 2 if rows >= 30 else 1
    nb = rows // ncoh
    spc = nb * bs
    fs = spc * 1e3
    g = generate_test_signal(sysm, 3, num_samples=nnc * ncoh * spc, sampling_freq=fs, interm_freq=0.0, doppler=430.0,
                             code_phase=321.5, CN0=55, seed=0x5EED0D30 + rows)
    sig = g["signal"].astype(np.complex64)
    cov = (nb - 2 / ncoh) / 2 * 1e3 - 1.0  # the smallest coverage whose block count is nb
    plan = plan_acquire(sysm, fs, [3, 5], min_doppler_coverage=cov, num_coherently_integrated_code_periods=ncoh,
                        num_noncoherent_accumulations=nnc)
    try:
        assert (plan.num_blocks, plan.block_size, plan.num_doppler_bins) == (nb, bs, rows)
        assert plan.native.column_kernel() == f"k_column_reg<{rows}>"
        res = acquire_(plan, sig, [3, 5], store_power_bins=True)
        ores, osurf = oracle.acquire(plan, sig, [0, 1], surfaces=True)
        for j, p in enumerate([3, 5]):
            check_prn(res[j], ores[j], osurf[j], res[j].power_bins, label=f"rows {rows} bs {bs} prn {p}",
                      fp64_surface=lambda j=j: oracle.acquire(plan, sig, [0, 1], surfaces=True, bits=64)[1][j])
    finally:
        plan.close()
