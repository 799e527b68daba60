"""Which code periods the full-period correlation serves (CPU only).

`fmdbzp_full_period_form` states the engine's rule: a period of 31 a b samples
with coprime stage radices a and b, or one without a prime factor above 13 and
small enough for one LDS buffer; at most 32 coherent periods, 4 GiB of code
spectra, and more than a few rows where the period is long.
"""
import time

import pytest

from acquisition._native import EngineError, full_period_form


def test_multiples_of_the_chip_rate():
    forms = {k: full_period_form(1023 * k, 16, 10, 8, 32) for k in range(1, 25)}
    assert {k for k, f in forms.items() if f == "axis31"} == {2, 3, 4, 5, 6, 8, 10, 16}
    assert {k for k, f in forms.items() if f == "radix"} == set()  # 31 is no radix


@pytest.mark.parametrize("spc,form", [
    (2048, "radix"), (2500, "radix"), (3125, "radix"), (4000, "radix"), (5250, "radix"), (6500, "radix"),
    (5000, "radix"), (16384, "radix"), (20000, "radix"), (2790, "axis31"), (5456, "axis31"), (12400, "axis31"),
    (4250, ""),     # 17
    (25000, ""),    # beyond LDS
    (30690, ""), (100000, ""), (70000, ""),
    (1000003, "")])
def test_other_periods(spc, form):
    for nnc in (1, 4):
        assert full_period_form(spc, 20, 2, nnc, 8) == form


def test_limits():
    assert full_period_form(4000, 16, 32, 1, 8) == "radix" and full_period_form(4000, 16, 33, 1, 8) == ""
    # 8 bytes x 20000 x 1600 bins: 16 PRNs within 4 GiB, 17 beyond
    assert full_period_form(20000, 80, 20, 1, 16) == "radix" and full_period_form(20000, 80, 20, 1, 17) == ""
    assert full_period_form(4000, 2**31 - 1, 32, 1, 2**31 - 1) == ""
    # few rows of more than 15360 samples
    assert full_period_form(20000, 16, 1, 8, 1) == "" and full_period_form(20000, 16, 1, 8, 3) == "radix"
    assert full_period_form(16368, 16, 1, 1, 1) == "" and full_period_form(16368, 16, 1, 2, 1) == "axis31"
    assert full_period_form(15000, 20, 1, 1, 1) == "radix"


def test_planning_is_quick_at_highly_composite_periods():
    """A plan's stages are chosen at its creation, a matter of 0.4 ms in all:
    every ordered product of radices took 0.84 ms at 20160 points."""
    best = 1.0
    for _ in range(30):
        t0 = time.perf_counter()
        assert full_period_form(20160, 16, 1, 1, 32) == "radix"
        best = min(best, time.perf_counter() - t0)
    assert best < 0.3e-3


@pytest.mark.parametrize("at", range(5))
def test_sizes_must_be_positive(at):
    args = [4000, 16, 1, 1, 1]
    args[at] = 0
    with pytest.raises(EngineError, match="positive"):
        full_period_form(*args)
