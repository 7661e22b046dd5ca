"""Preprocessing where the compacted window sums can go wrong: lengths at the edges of 64-bin
chunks, every bin holding a peak, hardly any, the longest spectra.  Bit-exact to the oracle in
both mean modes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def spectrum(rng, length, fill):
    """A spectrum of `length` bins (length = 75 + cut-off, a multiple of ten in m/z) with a
    share `fill` of its bins holding a peak."""
    cut = (length - 75) // 10 * 10
    n = max(1, int(cut * fill))
    mz = np.sort(np.concatenate([rng.uniform(2.0, cut, n), [cut + 0.5]])).astype(np.float32)
    inten = rng.lognormal(3.0, 2.5, len(mz)).astype(np.float32)
    inten[rng.random(len(mz)) < 0.05] = 0.0
    return mz, inten


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("stride", [192, 2112, 4096])
def test_window_sums_over_peaks_only(orc, stride, mode):
    from hfx_amd import pipeline

    rng = np.random.default_rng(stride + mode)
    lens = [85, 125, 126, 127, 128, 129, 185, 192, stride - 1, stride]
    specs = [spectrum(rng, n, f) for n in lens for f in (0.003, 0.1, 3.0)]
    off = np.concatenate([[0], np.cumsum([len(m) for m, _ in specs])]).astype(np.uint32)
    mz, inten = (np.concatenate(v) for v in zip(*specs))
    pcr = rng.uniform(1500.0, 4000.0, len(specs)).astype(np.float32)
    z = np.full(len(specs), 2.0, np.float32)
    X, ln, st = orc.preprocess_batch(pcr, z, mz, inten, off, stride, mode)
    sp = pipeline.DeviceSpectra(pipeline.Ctx(0), pcr, z, mz, inten, off, stride, mean_mode=mode)
    assert (sp.status() == st).all() and (sp.lengths() == ln).all()
    assert (st == 0).any()
    assert (sp.x().view(np.uint32) == X.view(np.uint32)).all()
