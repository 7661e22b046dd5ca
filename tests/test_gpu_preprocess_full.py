"""Preprocessing of spectra with a peak in every bin: values that add up past 2^17, beside values of
2^-13 and a little more, whose sums are not exact in FP64 in any order."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("full", [0.6, 0.64, 0.66, 1.0])  # of 4,096 bins; 2,621 at 50 are 2^17
def test_sums_around_the_largest_that_are_exact(orc, full):
    from hfx_amd import pipeline

    rng = np.random.default_rng(int(100 * full))
    specs = []
    for k in range(8):
        mz = np.arange(2.0, 4020.0 - 7 * k, 0.5).astype(np.float32)
        inten = np.ones(len(mz), np.float32)
        small = np.repeat(rng.random((len(mz) + 1) // 2) >= full, 2)[:len(mz)]
        # 50 sqrt(i) in [2^-13, 2^-12), with all of their 24 bits
        inten[small] = ((2.0**-13 * rng.uniform(1.0, 2.0, small.sum()) / 50.0) ** 2).astype(np.float32)
        specs.append((mz, inten))
    off = np.concatenate([[0], np.cumsum([len(m) for m, _ in specs])]).astype(np.uint32)
    mz, inten = (np.concatenate(v) for v in zip(*specs))
    pcr, z = np.full(len(specs), 3000.0, np.float32), np.full(len(specs), 2.0, np.float32)
    X, ln, st = orc.preprocess_batch(pcr, z, mz, inten, off, 4096, 1)
    sp = pipeline.DeviceSpectra(pipeline.Ctx(0), pcr, z, mz, inten, off, 4096, mean_mode=1)
    assert (st == 0).all() and (sp.lengths() == ln).all() and ln.max() > 4000
    assert (sp.x().view(np.uint32) == X.view(np.uint32)).all()
