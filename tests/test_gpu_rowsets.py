"""The theoretical rows that the indexes of one database share: what a batch adds to the device's
memory, and whose rows it reads."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_rows import Spectra, database, reference, spectra

pytestmark = pytest.mark.gpu


def free(pl):
    from hfx_amd import check, lib

    pl.sync()
    a, b = C.c_size_t(), C.c_size_t()
    check(lib().hfx_mem_info(C.byref(a), C.byref(b)), "hfx_mem_info")
    return a.value


def batch(pl, ctx, db, sp, form):
    forms = pl.PepIndex.IONS if form == "FP32_SPARSE" else pl.PepIndex.LADDER
    ix = pl.PepIndex(ctx, db, forms=forms)
    bs = pl.BatchSearch(ctx, db, sp, eps=3.0, topn=5, index=ix)
    bs.set_precision(getattr(bs, form))
    bs.run()
    return bs


def test_indexes_of_one_database_hold_one_copy_of_its_rows(orc):
    from hfx_amd import pipeline as pl

    hdb = database(pl, 200_000, seed=3, longest=12)
    x, lens, zmax, mass = spectra(pl, hdb, 40, 2112, seed=4)
    zmax = np.minimum(zmax, 2)
    ctx = pl.Ctx(0)
    dbs = [pl.DeviceDB(hdb) for _ in range(2)]   # the same contents at two places
    sp = Spectra(pl, x, lens, zmax, mass)
    rows = 2 * ((200_000 + 15) // 16) * 9 * 1024  # two charge levels of nine KiB a tile
    batch(pl, ctx, dbs[0], sp, "I8X3_DENSE")      # comes and goes: code and scratch are loaded
    start = free(pl)
    held = [batch(pl, ctx, dbs[0], sp, "I8X3_DENSE")]
    want = held[0].results(keep_scores=True).scores
    first = free(pl)
    assert start - first > rows
    for k in range(4):
        held.append(batch(pl, ctx, dbs[k % 2], sp, "I8X3_DENSE"))
        assert np.array_equal(held[-1].results(keep_scores=True).scores, want)
    later = free(pl)
    assert (first - later) / 4 < start - first - 0.9 * rows   # what is an index's own
    # the last one gone, the rows are too
    while held:
        held.pop()
    assert free(pl) >= start - (8 << 20)


@pytest.mark.parametrize("form", ["FP32_SPARSE", "BF16X2_DENSE", "I8X3_DENSE"])
def test_another_database_at_the_same_address_has_its_own_rows(orc, form):
    """The first database's index and batch stay alive while its buffers are given other
    peptides of the same number: an index built then reads those."""
    from hfx_amd import pipeline as pl

    one, two = database(pl, 5000, seed=11), database(pl, 5000, seed=12)
    db = pl.DeviceDB(one)
    x, lens, zmax, mass = spectra(pl, two, 30, 2112, seed=13)
    sp, ctx = Spectra(pl, x, lens, zmax, mass), pl.Ctx(0)
    old = batch(pl, ctx, db, sp, form)
    other = pl.DeviceDB(two)
    for name in ("t_ions", "t_r", "t_tc", "t_tn", "t_mass", "t_idx", "t_rsorted"):
        a, b = getattr(db, name), getattr(other, name)
        assert a.nbytes >= b.nbytes
        a.upload(pl.host(b, np.uint8, b.nbytes).copy())
    pl.sync()
    ref, exact, scale = reference(orc, two, x, lens, zmax, mass, 5)
    res = batch(pl, ctx, db, sp, form).results(keep_scores=True)
    assert (res.num == ref["num"]).all()
    for s in range(len(res.top_cnt)):
        c = int(res.top_cnt[s])
        assert res.top_pos[s, :c].tolist() == ref["top_pos"][s, :c].tolist()
        assert (res.top_exact[s, :c] == orc.fx_to_double(ref["top_fx"][s, :c])).all()
    # scores of every candidate, not the exact re-scores alone: within the widest form's bound
    bound = (2.0**-16 + 210 * 2.0**-24) * scale + np.repeat(np.abs(x).max(1), res.num) * 50 * 8000 / 8355711
    assert (np.abs(res.scores - exact) <= bound + 1e-6).all()
    assert old.index is not None


def test_rows_go_where_memory_is_short_and_come_back(orc):
    """An allocation that cannot be had (a PiB) takes the rows that no batch uses, and those that
    hfx_xcorr_sparse keeps; batches and calls after it write them again."""
    from hfx_amd import lib
    from hfx_amd import pipeline as pl

    hdb = database(pl, 100_003, seed=14, longest=20)
    x, lens, zmax, mass = spectra(pl, hdb, 4000, 600, seed=15)
    ctx, db, sp = pl.Ctx(0), pl.DeviceDB(hdb), Spectra(pl, x, lens, np.minimum(zmax, 2), mass)
    index = pl.PepIndex(ctx, db)

    def run(b):
        b.run()
        return b.results(keep_scores=True).scores

    b = pl.BatchSearch(ctx, db, sp, eps=3.0, topn=5, index=index)
    plain = pl.PlainSearch(ctx, db, sp, eps=3.0, topn=5)
    want, score = run(b), plain.run(keep_scores=True).scores
    rows = 2 * ((100_003 + 15) // 16) * 9 * 1024
    for _ in range(2):
        full = free(pl)
        p = C.c_void_p()
        assert lib().hfx_malloc(C.byref(p), 1 << 50) != 0
        assert free(pl) - full > (rows if b is None else 0)   # the plain call's; the idle set's too
        if b is not None:
            assert np.array_equal(run(b), want)               # a batch keeps the rows it uses
            b = None
        assert np.array_equal(plain.run(keep_scores=True).scores, score)
    again = pl.BatchSearch(ctx, db, sp, eps=3.0, topn=5, index=index)
    assert np.array_equal(run(again), want)
