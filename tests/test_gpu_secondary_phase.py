"""Secondary-code phase kernel (fmdbzp_secondary_phase) at the edges of its chunks.

The kernel runs the periods of a request in chunks of 64 samples, with instances
for up to 16, 32 and 64 periods, so its edges are chunk remainders (spc = 2046,
2048, 2500), one period, 32, 33 and 64 periods, and requests of different length in one launch.
On white noise the rotations' scores lie close together, so a wrong or missing
sample moves the best one. The bar: the oracle's rotation
(src/acquire.jl:503-538), exactly: the kernel keeps the order of operations.
"""
import numpy as np
import pytest

import oracle
from acquisition import GPSL1CA, plan_acquire
from acquisition._native import ELTYPE

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fs,lengths,kind", [(2.046e6, (1, 2, 10), "cf32"), (2.048e6, (25, 32), "ci16"),
                                             (2.5e6, (33, 64, 7, 25), "cf32"), (2.046e6, (63,), "i16")])
def test_secondary_phase_matches_the_oracle(fs, lengths, kind):
    rng = np.random.default_rng(int(fs) + len(lengths))
    plan = plan_acquire(GPSL1CA(), fs, [1])
    spc = plan.samples_per_code
    n = max(lengths) * spc
    if kind == "cf32":
        sig = (rng.standard_normal(n) + 1j * rng.standard_normal(n)).astype(np.complex64)
    elif kind == "ci16":
        sig = rng.integers(-500, 500, (n, 2)).astype(np.int16)
    else:
        sig = rng.integers(-500, 500, n).astype(np.int16)
    items, want = [], []
    for i, L in enumerate(lengths):
        code = rng.choice(np.array([-1, 1], np.int8), spc)
        sec = rng.choice(np.array([-1, 1], np.int8), L)
        dop = 731.25 * (i + 1) - 1500.0
        items.append((code, sec, dop))
        want.append(oracle.secondary_phase(sig, spc, L, fs, 0.0, dop, code, sec))
    try:
        got = plan.native.secondary_phase(sig.ctypes.data, ELTYPE[kind], n, 0.0, 0, items)
    finally:
        plan.close()
    assert got == want
