"""Memory of the full-period correlation's plans.

The code spectra (8 bytes x samples per code x Doppler bins x PRNs) have a fixed
limit of 4 GiB, so which path a search takes does not depend on the memory that
happens to be free: 16 PRNs of 1600 bins at 20 MHz (4.1 GB) are within it, 17
are not. And a plan holds the tile from its creation, so that no later call can
fail for want of it.
"""
import numpy as np
import pytest
import torch

from acquisition import GPSL1CA, acquire_, plan_acquire
from acquisition._native import ELTYPE

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nprn,full", [(16, True), (17, False)])
def test_spectra_have_a_fixed_limit(nprn, full):
    plan = plan_acquire(GPSL1CA(), 20e6, list(range(1, nprn + 1)), min_doppler_coverage=35000.0,
                        num_coherently_integrated_code_periods=20)
    try:
        assert plan.num_doppler_bins == 1600
        assert ("_full" in plan.native.call_kernels(ELTYPE["cf32"], nprn)) == full
    finally:
        plan.close()


def test_surfaces_need_no_tile_allocation():
    """32 PRNs of 160 bins at 16.368 MHz: the two tiles of a plan are 1.35 GB. A
    call with surfaces after one without may allocate its staging (10.5 MB)."""
    prns = list(range(1, 33))
    plan = plan_acquire(GPSL1CA(), 16.368e6, prns, num_coherently_integrated_code_periods=10,
                        num_noncoherent_accumulations=2)
    sig = torch.zeros(2 * 163680, dtype=torch.complex64, device="cuda")
    try:
        assert "_full" in plan.native.call_kernels(ELTYPE["cf32"], 32)
        acquire_(plan, sig, prns)
        before = torch.cuda.mem_get_info()[0]
        r = acquire_(plan, sig, [1], store_power_bins=True)[0]
        assert np.asarray(r.power_bins).shape == (160, 16368)
        assert before - torch.cuda.mem_get_info()[0] < 200e6
    finally:
        plan.close()
