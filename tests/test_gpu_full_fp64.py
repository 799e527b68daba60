"""Statistics of statistics-only calls against the FP64 oracle.

Peak, its four neighbours and the mean noise of the full-period correlation
(31-axis form at 2046, 5115, 6138 and 16368 samples per code, radices at 5000,
6500 and 16384) and of periods that fall back to the tile (7161 = 7 1023, 4250),
with one and several steps, an IF and drift, against the oracle's FP64 surface
(src/acquire.jl:335-385). A transform of n points rounds by about 2^-24 sqrt(log2 n)
of the row's rms, a power by twice that, 4e-7 of the peak here; the bar is 2e-6 of
the peak, and 1e-6 for the mean noise.
"""
import numpy as np
import pytest

import oracle
from acquisition import GPSL1CA, acquire_, plan_acquire
from acquisition._native import ELTYPE, full_period_form
from acquisition.signals import generate_test_signal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("spc,coh,nnc,if_hz", [(2046, 1, 1, 0.0), (5115, 4, 3, 38400.0), (6138, 2, 2, 0.0),
                                               (16368, 3, 4, 0.0), (5000, 10, 2, 38400.0), (6500, 1, 1, 0.0),
                                               (16384, 2, 3, 0.0), (7161, 2, 2, 0.0), (4250, 2, 2, 0.0)])
def test_statistics_match_the_fp64_oracle(spc, coh, nnc, if_hz):
    fs, prns = spc * 1e3, [7, 12, 21]
    plan = plan_acquire(GPSL1CA(), fs, prns, num_coherently_integrated_code_periods=coh,
                        num_noncoherent_accumulations=nnc)
    sig = generate_test_signal(GPSL1CA(), 7, num_samples=spc * coh * nnc, sampling_freq=fs, interm_freq=if_hz,
                               doppler=1730.0, code_phase=411.3, CN0=52, seed=0x5EED0F41 + spc)["signal"]
    sig = sig.astype(np.complex64)
    try:
        form = full_period_form(spc, plan.num_blocks, coh, nnc, 3)
        kernel = plan.native.call_kernels(ELTYPE["cf32"], 3)
        assert kernel.startswith({"axis31": "k_full31_corr<", "radix": "k_full_corr<", "": "k_corr_"}[form])
        assert (form == "") == (spc in (7161, 4250))
        res = acquire_(plan, sig, prns, interm_freq=if_hz)
        _, osurf = oracle.acquire(plan, sig, [0, 1, 2], if_hz=if_hz, surfaces=True, bits=64)
        worst = 0.0
        for r, o in zip(res, osurf):
            o, e = np.asarray(o, dtype=np.float64), r.engine_stats
            n, row, col = o.shape[0], e["row"], e["col"]
            want = [o[row, col], o[row, (col - 1) % spc], o[row, (col + 1) % spc], o[(row - 1) % n, col],
                    o[(row + 1) % n, col]]
            err = max(abs(x - y) for x, y in zip([e["peak"]] + list(e["nbr"]), want)) / o.max()
            worst = max(worst, err, o.max() / o[row, col] - 1)
            assert abs(e["noise"] / o[(row + n // 2) % n].mean() - 1) <= 1e-6
        print(f"{kernel} {spc}: {worst:.1e} of the peak")
        assert worst <= 2e-6
    finally:
        plan.close()
