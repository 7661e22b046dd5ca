"""A planned or captured batch that is run on later spectra than those it was planned with."""
import numpy as np
import pytest

from test_gpu_rows import FORMS, Spectra, check, database, reference, spectra

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("replay", [False, True])
@pytest.mark.parametrize("form", sorted(FORMS))
def test_later_spectra_of_higher_charges(orc, form, replay):
    """Planned with fragment charges 1 and 2 only, run on the same rows with charges up to 4 (and
    5, which is not generated): the scores of each form, within its bound, and the rankings."""
    from hfx_amd import pipeline as pl

    hdb = database(pl, 3001, seed=21)
    x, lens, zmax, mass = spectra(pl, hdb, 90, 2112, seed=22)
    assert set(zmax) == {1, 2, 3, 4, 5}
    sp = Spectra(pl, x, lens, np.minimum(zmax, 2), mass)
    bs = pl.BatchSearch(pl.Ctx(0), pl.DeviceDB(hdb), sp, eps=3.0, topn=5)
    bs.set_precision({"fp32": bs.FP32_SPARSE, "bf16": bs.BF16X2_DENSE, "i8": bs.I8X3_DENSE}[form])
    bs.run()
    if replay:
        bs.capture()
    for z in (zmax, np.minimum(zmax, 2), zmax[::-1].copy()):
        sp.t_zmax.upload(z.astype(np.uint32))
        pl.sync()
        bs.replay() if replay else bs.run()
        ref, exact, scale = reference(orc, hdb, x, lens, z, mass, 5)
        check(orc, bs.results(keep_scores=True), ref, exact, scale, x, *FORMS[form])
