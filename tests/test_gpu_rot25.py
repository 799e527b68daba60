"""Rotation search at 25 periods of 50 and 100 rows (k_column_rot25) where the
last workgroup of five or two code columns is ragged.

E1-like pilots (25-chip secondary code, 4 ms codes) with odd block sizes, as one
window and in code-column chunks that cut a workgroup's columns: statistics, and
the surfaces of the whole window, against the FP32 oracle
(src/noncoherent_integration.jl:183-297), to the bar of tests/parity.py.
"""
import numpy as np
import pytest

import oracle
from acquisition import acquire_, plan_acquire
from acquisition.signals import e1like_scene
from acquisition.systems import E1Like
from parity import check_prn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("chunk", [0, 333])
@pytest.mark.parametrize("nb,bs,cov,nnc", [(50, 101, 6000.0, 2), (50, 103, 6000.0, 1), (100, 51, 12000.0, 2)])
def test_ragged_columns_match_the_oracle(nb, bs, cov, nnc, chunk, monkeypatch):
    sysm = E1Like()
    fs = bs * nb / 4e-3
    sc = e1like_scene(n_periods=25, nnc=nnc, fs=fs, nprn=4, npresent=2, cn0_range=(46.0, 48.0), system=sysm)
    p0 = sc.present[0]
    prns = [p0, 1 if p0 != 1 else 4]
    if chunk:
        monkeypatch.setenv("FMDBZP_CHUNK_COLS", str(chunk))
    plan = plan_acquire(sysm, sc.sampling_freq, prns, min_doppler_coverage=cov,
                        num_coherently_integrated_code_periods=25, num_noncoherent_accumulations=nnc)
    try:
        assert (plan.num_blocks, plan.block_size, plan.num_doppler_bins) == (nb, bs, 25 * nb)
        sig = sc.signal.astype(np.complex64)
        res = acquire_(plan, sig, prns, store_power_bins=not chunk)
        ores, osurf = oracle.acquire(plan, sig, [0, 1], surfaces=True)
        for j, p in enumerate(prns):
            check_prn(res[j], ores[j], None if chunk else osurf[j], None if chunk else res[j].power_bins,
                      label=f"nb {nb} bs {bs} steps {nnc} chunk {chunk} prn {p}",
                      fp64_surface=None if chunk else
                      lambda j=j: oracle.acquire(plan, sig, [0, 1], surfaces=True, bits=64)[1][j])
    finally:
        plan.close()
