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


@pytest.mark.parametrize("stride", [320, 2304, 2368, 4096])
def test_intensities_of_any_ratio(orc, stride):
    """Values too small beside their region's largest for exact sums, and spectra of both kinds side by side: the FP64 sums in either order, bit for bit."""
    from hfx_amd import pipeline

    rng = np.random.default_rng(stride)
    specs = []
    for k in range(12):
        mz, inten = spectrum(rng, stride - 3 * k, 0.3)
        if k % 3 == 1:
            inten = (inten * np.float32(10.0) ** rng.uniform(-14, 3, len(inten))).astype(np.float32)
        if k % 3 == 2:
            # on the line: 50 sqrt(i / max) = 2^-13 and its neighbours
            line = np.float32((2.0**-13 / 50.0) ** 2)
            inten[:] = 1.0
            inten[1::7] = line
            inten[2::7] = np.nextafter(line, np.float32(0.0))
        specs.append((mz, inten))
    off = np.concatenate([[0], np.cumsum([len(m) for m, _ in specs])]).astype(np.uint32)
    mz, inten = (np.concatenate(v) for v in zip(*specs))
    pcr = np.full(len(specs), 3000.0, np.float32)
    z = np.full(len(specs), 2.0, np.float32)
    X, ln, st = orc.preprocess_batch(pcr, z, mz, inten, off, stride, 1)
    sp = pipeline.DeviceSpectra(pipeline.Ctx(0), pcr, z, mz, inten, off, stride, mean_mode=1)
    assert (st == 0).all() and (sp.lengths() == ln).all()
    assert (sp.x().view(np.uint32) == X.view(np.uint32)).all()
