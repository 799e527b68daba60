"""Which kernels a call runs (fmdbzp_plan_call_kernels), and the rotation
kernels that k_column_rot25 left in use.

k_column_rot25 runs the searches of 25 periods at 50, 80, 100, 250 and 500 rows,
as one window and in code-column chunks; the matrix-core form keeps its own.
k_column_rot2000 serves 2000 bins of other period counts (20 x 100 and 16 x 125
here), k_column_rotbig 25 periods of 10 rows: surfaces and statistics of both
against the FP32 oracle (src/noncoherent_integration.jl:183-297), to the bar of
tests/parity.py.
"""
import numpy as np
import pytest

import oracle
from acquisition import GPSL1CA, acquire_, plan_acquire
from acquisition._native import ELTYPE, FLAG_STORE_SURFACES, EngineError
from acquisition.signals import e1like_scene
from acquisition.systems import E1Like, L5Like, SeededCodeSystem
from parity import check_prn

pytestmark = pytest.mark.gpu

CF32 = ELTYPE["cf32"]


@pytest.mark.parametrize("nb,bs,cov,chunk", [(50, 101, 6000.0, 0), (50, 101, 6000.0, 333), (80, 50, 9000.0, 0),
                                             (100, 51, 12000.0, 0), (250, 16, 31000.0, 700), (500, 8, 62000.0, 700)])
def test_25_periods_run_k_column_rot25(nb, bs, cov, chunk, monkeypatch):
    if chunk:
        monkeypatch.setenv("FMDBZP_CHUNK_COLS", str(chunk))
    plan = plan_acquire(E1Like(), bs * nb / 4e-3, [1], min_doppler_coverage=cov,
                        num_coherently_integrated_code_periods=25)
    try:
        assert (plan.num_blocks, plan.num_doppler_bins) == (nb, 25 * nb)
        assert plan.native.call_kernels(CF32, 1).split()[1] == f"k_column_rot25<{nb}>"
    finally:
        plan.close()


@pytest.mark.parametrize("L,nb,bs", [(20, 100, 41), (16, 125, 33), (25, 10, 409)])
def test_earlier_rotation_kernels_match_the_oracle(L, nb, bs):
    sysm = SeededCodeSystem("pilot", 4092, 1.023e6, 1575.42e6, L, 0x5EED0A00 + L, boc=True)
    fs = nb * bs / 4e-3
    sc = e1like_scene(seed=0x5EED0A01, n_periods=L, nnc=2, fs=fs, nprn=4, npresent=2, cn0_range=(46.0, 48.0),
                      system=sysm)
    prns = [sc.present[0], next(p for p in sc.prns if p not in sc.present)]
    cov = (nb - 2 / L) / 2 * fs / (nb * bs) - 1.0  # the smallest coverage whose block count is nb
    plan = plan_acquire(sysm, fs, prns, min_doppler_coverage=cov, num_coherently_integrated_code_periods=L,
                        num_noncoherent_accumulations=2)
    try:
        assert (plan.num_blocks, plan.block_size, plan.num_secondary_rotations) == (nb, bs, L)
        want = "k_column_rotbig<64,25>" if L == 25 else "k_column_rot2000"
        assert plan.native.call_kernels(CF32, 2).split()[1] == want
        sig = sc.signal.astype(np.complex64)
        res = acquire_(plan, sig, prns, store_power_bins=True)
        ores, osurf = oracle.acquire(plan, sig, [0, 1], surfaces=True)
        for j, p in enumerate(prns):
            check_prn(res[j], ores[j], osurf[j], res[j].power_bins, label=f"{want} {L} x {nb} prn {p}",
                      fp64_surface=lambda j=j: oracle.acquire(plan, sig, [0, 1], surfaces=True, bits=64)[1][j])
    finally:
        plan.close()


def test_names_follow_samples_and_flags():
    kw = dict(num_coherently_integrated_code_periods=10, num_noncoherent_accumulations=2)
    plan = plan_acquire(GPSL1CA(), 16.368e6, [1, 2], tile_precision="auto", **kw)
    try:
        q = plan.native.call_kernels
        assert q(CF32, 2) == "k_full31_corr<512>"
        assert q(CF32, 2, FLAG_STORE_SURFACES) == "k_corr_tile<2,true,2048> k_column_c160_pair<32,512>"
        want = "k_corr_tile<2,true,2048,fp16> k_column_c160_pair<32,512,fp16>"
        assert q(ELTYPE["i16"], 2, FLAG_STORE_SURFACES) == want
        with pytest.raises(EngineError, match="eltype"):
            q(99, 1)
        with pytest.raises(EngineError, match="nreq"):
            q(CF32, 0)
    finally:
        plan.close()
    plan = plan_acquire(E1Like(), 1e6, [1], tile_precision="mfma", min_doppler_coverage=10000.0,
                        num_coherently_integrated_code_periods=25)
    try:
        assert plan.native.call_kernels(CF32, 1).split()[1] == "k_column_rotmma<4,1,4>"
    finally:
        plan.close()
    plan = plan_acquire(L5Like(), 30.69e6, [1], min_doppler_coverage=5000.0)
    try:
        assert plan.native.call_kernels(CF32, 1) == "k_corr_fc<256> k_column_reg<15>"
    finally:
        plan.close()
