"""`fmdbzp_prn_results` against the scalar formulas (src/acquire.jl:9-13,
:544-671) evaluated with numpy Float32 scalars: bit for bit, over ordinary
peaks, equal and zero neighbours (zero denominators), zero, negative,
infinite and NaN powers, and every block geometry of a code period."""
import ctypes
import math

import numpy as np
import pytest

from acquisition import _native
from acquisition.acquire import _RESULT_DTYPE, fmdbzp_column_to_tau, jl_mod, parabolic_interp

f32 = np.float32
SPECIAL = [0.0, -0.0, -1.0, 1.0, math.inf, -math.inf, math.nan, 1e-42, 3e38]


def reference(q, spc, nb, bs, fs, fc, length, tcoh, spacing, interp):
    peak, noise = f32(q.peak_power), f32(q.noise_power)
    with np.errstate(all="ignore"):
        signal = peak - noise
        ptn = (signal + noise) / noise
        ratio = float(signal / noise)
        cn0 = 10 * math.log10(ratio / tcoh / 1.0) if ratio > 0 else (-math.inf if ratio == 0 else math.nan)
        delay = fmdbzp_column_to_tau(q.peak_col % spc, nb, bs)
        phase, offset = jl_mod(-delay * fc / fs, length), 0.0
        if interp:
            sq = np.sqrt(noise)
            if max(f32(q.code_left), f32(q.code_right)) > sq:
                frac = parabolic_interp(q.code_left, peak, q.code_right)
                if isinstance(frac, np.float32):
                    # an infinite parabola offset: Python's fmod raises where C's gives NaN
                    x = float(-f32(f32(delay) + frac)) * fc / fs
                    phase = jl_mod(x, length) if math.isfinite(x) else math.nan
            if max(f32(q.dop_left), f32(q.dop_right)) > sq:
                offset = float(parabolic_interp(q.dop_left, peak, q.dop_right)) * spacing
    return cn0, phase, offset, ptn


@pytest.mark.parametrize("nb,bs", [(1, 2046), (16, 250), (20, 250), (11, 2790)])
@pytest.mark.parametrize("interp", [0, 1])
def test_results_equal_the_scalar_formulas(nb, bs, interp):
    rng = np.random.default_rng(nb * 7 + interp)
    spc, n = nb * bs, 2000
    fs, fc, length, tcoh, spacing = spc * 1e3, 1.023e6, 1023, 4e-3, 1e3 / 3
    stats = (_native.PrnStats * n)()
    for i, q in enumerate(stats):
        p = rng.uniform(1, 1e3)
        v = [p, rng.uniform(1e-3, 2) * p, *(rng.uniform(0, 1, 4) * p)]
        if i % 4 == 0:
            v[rng.integers(6)] = SPECIAL[rng.integers(len(SPECIAL))]
        if i % 7 == 0:
            v[2] = v[3] = v[4] = v[5] = v[0]
        q.peak_power, q.noise_power, q.code_left, q.code_right, q.dop_left, q.dop_right = v
        q.peak_row, q.peak_col = 0, int(rng.integers(3 * spc))
    out = np.empty(n, dtype=_RESULT_DTYPE)
    _native.prn_results(stats, n, spc, nb, bs, fs, fc, length, tcoh, spacing, interp, out.ctypes.data)
    for q, got in zip(stats, out):
        want = reference(q, spc, nb, bs, fs, fc, length, tcoh, spacing, interp)
        have = (got["cn0_dbhz"], got["code_phase"], got["doppler_offset"], got["peak_to_noise"])
        assert np.array_equal(np.array(want, dtype=np.float64), np.array(have, dtype=np.float64), equal_nan=True)


def test_bad_arguments_are_refused():
    lib, stats, out = _native.lib(), (_native.PrnStats * 1)(), (_native.PrnResult * 1)()
    args = (4000, 16, 250, 4e6, 1.023e6, 1023.0, 1e-3, 1e3, 0)
    assert lib.fmdbzp_prn_results(None, 1, *args, ctypes.addressof(out)) == -1
    assert lib.fmdbzp_prn_results(ctypes.addressof(stats), 1, *args, None) == -1
    assert lib.fmdbzp_prn_results(ctypes.addressof(stats), 1, 0, *args[1:], ctypes.addressof(out)) == -1
    assert lib.fmdbzp_prn_results(None, 0, *args, None) == 0
