"""The engine cost model predicts the kernels that calls run (CPU only).

Where the full-period correlation serves a geometry, `predict_step` uses its
coefficients, elsewhere those of the tile's two kernels; a fit recovers known
full-period coefficients; and the in-place block correlation is a variant of
its own, by the engine's rule on the radix sequence.
"""
import numpy as np
import pytest

from acquisition.recommend import GpuCostModel, _corr_variant, _full_work

MODEL = GpuCostModel(corr={"generic": (6e-6, 8.0e-14), "fc": (1e-5, 3e-13)}, column={"generic": (5e-6, 1.5e-12, 6.0e-14)},
                     nprn=8, full={"radix": (7e-6, 1e-11, 3e-13, 2e-9), "axis31": (4e-6, 2e-11, 2e-13, 1e-8)})


@pytest.mark.parametrize("spc,nb,F,ncoh,form", [(10000, 16, 1250, 5, "radix"), (16368, 16, 2048, 10, "axis31"),
                                                (9207, 27, 686, 1, ""), (20460, 20, 2048, 1, ""), (10000, 16, 1250, 33, "")])
def test_step_follows_the_form(spc, nb, F, ncoh, form):
    ndop = nb * ncoh
    tile = sum(MODEL.predict_launches(spc, nb, F, ndop)) / 8
    full = float(np.dot(MODEL.full[form], _full_work(spc, ndop, 8))) / 8 if form else None
    assert MODEL.predict_step(spc, nb, F, ndop) == pytest.approx(full if form else tile, rel=1e-12)
    without = GpuCostModel(MODEL.corr, MODEL.column, 8)
    assert without.predict_step(spc, nb, F, ndop) == pytest.approx(tile, rel=1e-12)


def test_fit_recovers_full_period_coefficients():
    pts = [dict(spc=spc, nb=nb, F=0, ndop=nb * c, nprn=n, form=form,
                step_s=float(np.dot(MODEL.full[form], _full_work(spc, nb * c, n))))
           for form, spcs in (("radix", (2048, 4000, 10000, 20000)), ("axis31", (2046, 5115, 10230, 16368)))
           for spc in spcs for nb, c in ((16, 1), (16, 10)) for n in (2, 8, 32)]
    fit = GpuCostModel.fit(pts)
    assert fit.corr == {} and fit.column == {}
    for k, v in MODEL.full.items():
        np.testing.assert_allclose(fit.full[k], v, rtol=1e-6)


@pytest.mark.parametrize("F,variant", [(500, "f500"), (2048, "f2048"), (2500, "f2500"), (4000, "generic"), (1250, "generic"),
                                       (504, "generic"), (700, "generic"), (686, "fc"), (2744, "fc"), (3000, "fc"),
                                       (4096, "fc"), (980, "fc"), (1000, "generic")])
def test_in_place_correlation_is_its_own_variant(F, variant):
    assert _corr_variant(F) == variant


def test_recorded_table_ranks_by_the_path_that_calls_run():
    """16.368 MHz, 160 bins, 32 PRNs: a step of the full-period kernel took
    2.00 / 8 ms in the benchmark's search, of the tile's kernels 0.47 ms."""
    m = GpuCostModel.mi355x()
    assert 32 * m.predict_step(16368, 16, 2048, 160) == pytest.approx(0.25e-3, rel=0.4)
    assert sum(m.predict_launches(16368, 16, 2048, 160)) == pytest.approx(0.467e-3, rel=0.15)
