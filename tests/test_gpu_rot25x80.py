"""Direct rotation search at 25 periods of 80 rows (k_column_rot25 at 80 rows).

E1-like pilots (25-chip secondary code, 4 ms codes) with 80 blocks of 49 to 52
samples, so that the last workgroup of three code columns holds one to three of
them, over one and two noncoherent steps: surfaces and statistics against the
FP32 oracle (src/noncoherent_integration.jl:183-297), to the bar of
tests/parity.py.
"""
import numpy as np
import pytest

import oracle
from acquisition import acquire_, plan_acquire
from acquisition.signals import e1like_scene
from acquisition.systems import E1Like
from parity import check_prn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bs,nnc", [(49, 1), (50, 2), (51, 1), (52, 2)])
def test_ragged_columns_match_the_oracle(bs, nnc):
    sysm = E1Like()
    fs = bs * 80 / 4e-3
    sc = e1like_scene(n_periods=25, nnc=nnc, fs=fs, nprn=4, npresent=2, cn0_range=(46.0, 48.0), system=sysm)
    p0 = sc.present[0]
    prns = [p0, 1 if p0 != 1 else 4]
    plan = plan_acquire(sysm, sc.sampling_freq, prns, min_doppler_coverage=9000.0,
                        num_coherently_integrated_code_periods=25, num_noncoherent_accumulations=nnc)
    try:
        assert (plan.num_blocks, plan.block_size, plan.num_doppler_bins) == (80, bs, 2000)
        assert plan.native.column_kernel() == "k_column_rot2000"
        sig = sc.signal.astype(np.complex64)
        res = acquire_(plan, sig, prns, store_power_bins=True)
        ores, osurf = oracle.acquire(plan, sig, [0, 1], surfaces=True)
        for j, p in enumerate(prns):
            check_prn(res[j], ores[j], osurf[j], res[j].power_bins, label=f"bs {bs} steps {nnc} prn {p}",
                      fp64_surface=lambda j=j: oracle.acquire(plan, sig, [0, 1], surfaces=True, bits=64)[1][j])
    finally:
        plan.close()
