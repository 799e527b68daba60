"""Data-bit search of two 20-period bits (k_column_bitsplit).

L1 C/A over 40 code periods at every compiled row length (nb 10, 11, 12, 15,
16, 20, 22; the last two take one parity of bins per pass), with whole and
ragged column blocks (bs 16 to 66), one to four bit-edge offsets and one or
two noncoherent steps: surfaces and statistics against the FP32 oracle
(src/noncoherent_integration.jl:62-181), to the bar of tests/parity.py.
"""
import numpy as np
import pytest

import oracle
from acquisition import acquire_, plan_acquire
from acquisition.signals import generate_test_signal
from acquisition.systems import GPSL1CA
from parity import check_prn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb,bs,edges,nnc", [(10, 66, 1, 1), (11, 31, 2, 2), (12, 17, 4, 1), (15, 16, 2, 2),
                                             (16, 33, 5, 1), (20, 32, 2, 2), (22, 31, 4, 2)])
def test_every_row_length_matches_the_oracle(nb, bs, edges, nnc):
    sysm = GPSL1CA()
    spc = nb * bs
    fs = spc * 1e3
    n = nnc * 40 * spc
    g = generate_test_signal(sysm, 3, num_samples=n, sampling_freq=fs, interm_freq=0.0, doppler=430.0,
                             code_phase=321.5, CN0=52, seed=0x5EED0D20 + nb)
    sig = g["signal"].astype(np.complex64)
    cov = (nb - 2 / 40) / 2 * 1e3 - 1.0  # the smallest coverage whose block count is nb
    plan = plan_acquire(sysm, fs, [3, 5], min_doppler_coverage=cov, num_coherently_integrated_code_periods=40,
                        bit_edge_search_steps=edges, num_noncoherent_accumulations=nnc)
    try:
        assert (plan.num_blocks, plan.block_size, plan.num_data_bits) == (nb, bs, 2)
        assert plan.native.column_kernel() == f"k_column_bitsplit<{nb}>"
        res = acquire_(plan, sig, [3, 5], store_power_bins=True)
        ores, osurf = oracle.acquire(plan, sig, [0, 1], surfaces=True)
        for j, p in enumerate([3, 5]):
            check_prn(res[j], ores[j], osurf[j], res[j].power_bins, label=f"nb {nb} edges {edges} prn {p}",
                      fp64_surface=lambda j=j: oracle.acquire(plan, sig, [0, 1], surfaces=True, bits=64)[1][j])
    finally:
        plan.close()
