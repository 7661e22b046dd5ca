"""What the tuner writes to HFX_TUNE_CACHE, and what a batch takes from it."""
import pytest

from test_gpu_rows import Spectra, database, spectra

pytestmark = pytest.mark.gpu


def lg(v):
    return max(int(v), 1).bit_length() - 1


@pytest.mark.parametrize("stride", [1200, 2300])  # through rows, and past their longest
def test_the_fp32_form_tunes_what_it_runs(orc, tmp_path, monkeypatch, stride):
    from hfx_amd import pipeline as pl

    path = tmp_path / "tune.txt"
    monkeypatch.setenv("HFX_TUNE_CACHE", str(path))
    hdb = database(pl, 8000, seed=91)  # (the tuner keeps shapes for the process: another one each)
    ctx, db = pl.Ctx(0), pl.DeviceDB(hdb)
    sp = Spectra(pl, *spectra(pl, hdb, 48 if stride < 2176 else 100, stride, seed=92))
    b = pl.BatchSearch(ctx, db, sp, eps=3.0, topn=5)
    b.run()
    before, first = b.info(), b.results(keep_scores=True).scores
    cfg = b.autotune()
    after = b.info()
    key = f"{lg(after['spectra'])} {lg(after['scores'])} {after['levels']}"
    lines = path.read_text().splitlines()
    if stride <= 2176:
        # the ion-list kernel's launch shape was not timed, and is left alone
        assert cfg == tuple(before[k] for k in ("G", "C", "threads"))
        assert f"fp32 {key} {after['chunk']}" in lines
        assert not any(v.startswith(f"sparse {key} ") for v in lines)
        path.write_text(f"fp32 {key} 2048\nint8 {key} 256\nfp32 {key} 99999\n")
        monkeypatch.setenv("HFX_TUNE_CACHE", str(path) + "x")   # another path, then this one anew
        pl.BatchSearch(ctx, db, sp, eps=3.0, topn=5)
        monkeypatch.setenv("HFX_TUNE_CACHE", str(path))
        c = pl.BatchSearch(ctx, db, sp, eps=3.0, topn=5)
        assert c.info()["chunk"] == 2048
        c.set_precision(c.I8X3_DENSE)
        assert c.info()["chunk"] == 256
        c.run()      # a third of what a round of the waves takes
        c.set_precision(c.FP32_SPARSE)
        assert c.info()["chunk"] == 2048
        c.run()
        assert (c.results(keep_scores=True).scores == first).all()
    else:
        assert f"sparse {key} {cfg[0]} {cfg[1]} {cfg[2]}" in lines
        assert not any(v.startswith(f"fp32 {key} ") for v in lines)
    assert (b.results(keep_scores=True).scores == first).all() or stride > 2176
