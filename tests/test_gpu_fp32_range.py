"""FP32 scores where one bin dwarfs the others: the small ones count with all of their 24 bits, as
in a sum of 32-bit products."""
import numpy as np
import pytest

from test_gpu_rows import FORMS, Spectra, check, database, reference, spectra

pytestmark = pytest.mark.gpu


# ratios of 2^14 and 2^22, which the fixed point holds, and of 2^35, which it does not
@pytest.mark.parametrize("large,small", [(100.0, 1e-2), (2e4, 1e-2), (2e6, 1e-4)])
@pytest.mark.parametrize("path", ["batch", "sparse"])
def test_small_values_beside_a_large_one(orc, path, large, small):
    from hfx_amd import pipeline as pl

    hdb = database(pl, 100003, seed=51, longest=20)
    x, lens, zmax, mass = spectra(pl, hdb, 4000 if path == "sparse" else 60, 1100, seed=52)
    x = np.where(x != 0, np.random.default_rng(53).uniform(0.5 * small, small, x.shape), 0.0)
    x[:, 60] = large
    x = x.astype(np.float32)
    ref, exact, scale = reference(orc, hdb, x, lens, zmax, mass, 5)
    ctx, db, sp = pl.Ctx(0), pl.DeviceDB(hdb), Spectra(pl, x, lens, zmax, mass)
    if path == "batch":
        bs = pl.BatchSearch(ctx, db, sp, eps=3.0, topn=5)
        bs.run()
        res = bs.results(keep_scores=True)
    else:
        assert ref["num"].sum() > 1_000_000
        res = pl.PlainSearch(ctx, db, sp, eps=3.0, topn=5).run(keep_scores=True)
    # sum w|x| over the bins that a candidate touches, so the large one only where it is touched
    check(orc, res, ref, exact, scale, x, *FORMS["fp32"])
