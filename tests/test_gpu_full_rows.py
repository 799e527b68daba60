"""Calls of few Doppler rows at long code periods run on the tile.

A row of the full-period correlation is one workgroup, so with few rows of more
than 15360 samples the tile's kernels are the faster ones. At the edges of that
rule (rows over all PRNs of the call, samples per code, steps, the 31-axis
form): the kernels of the call, and for those on the tile the statistics of a
`tile_path` plan, bit for bit.
"""
import numpy as np
import pytest

from acquisition import GPSL1CA
from acquisition import _native
from acquisition._native import ELTYPE
from acquisition.plan import _plan_host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("spc,cov,nprn,nnc,tile", [
    (20000, 7000.0, 1, 1, True), (20000, 7000.0, 1, 8, True), (20000, 7000.0, 2, 1, False), (20000, 7000.0, 2, 3, True),
    (20000, 7000.0, 3, 3, False), (20000, 2500.0, 3, 1, True), (16384, 7000.0, 1, 2, True), (15000, 7000.0, 1, 2, False),
    (16368, 7000.0, 1, 1, True), (16368, 7000.0, 1, 2, False), (16368, 7000.0, 2, 1, False)])
def test_few_rows_take_the_tile(spc, cov, nprn, nnc, tile):
    sig = np.random.default_rng(spc + nnc).standard_normal((nnc * spc, 2)).astype(np.float32).view(np.complex64).ravel()
    raw = []
    for force in (False, True):
        plan = _plan_host(GPSL1CA(), spc * 1e3, [1, 2, 3], min_doppler_coverage=cov, num_noncoherent_accumulations=nnc)
        plan.tile_path = force
        plan.native = _native.NativePlan.create(plan)
        try:
            on_tile = "_full" not in plan.native.call_kernels(ELTYPE["cf32"], nprn)
            assert on_tile == (tile or force), plan.num_doppler_bins
            stats = plan.native.acquire(sig.ctypes.data, ELTYPE["cf32"], len(sig), 0.0, list(range(nprn)), 0)
            raw.append(bytes(memoryview(stats).cast("B")))
        finally:
            plan.close()
    assert (raw[0] == raw[1]) or not tile
