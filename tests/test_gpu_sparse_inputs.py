"""hfx_xcorr_sparse over enough pairs that theoretical rows are taken, with what a call may leave
out: precursor masses, the begin of an empty window, anything between the spectra's scores."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_rows import FORMS, Spectra, check, database, reference, spectra

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def search(orc):
    from hfx_amd import pipeline as pl

    hdb = database(pl, 100_003, seed=31, longest=20)
    x, lens, zmax, mass = spectra(pl, hdb, 5000, 1400, seed=32)
    mass[::7] = -5000.0   # empty windows
    ref, exact, scale = reference(orc, hdb, x, lens, zmax, mass, 5)
    assert ref["num"].sum() > 1_000_000 and (ref["num"][::7] == 0).all()
    return hdb, x, lens, zmax, mass, ref, exact, scale


@pytest.mark.parametrize("what", ["no masses", "any begin", "gaps", "fewer peptides"])
def test_sparse_through_rows_reads_only_what_it_is_given(search, what):
    from hfx_amd import HfxSpectra, check as ok, lib
    from hfx_amd import pipeline as pl

    hdb, x, lens, zmax, mass, ref, exact, scale = search
    ctx, db, sp = pl.Ctx(0), pl.DeviceDB(hdb), Spectra(pl, x, lens, zmax, mass)
    begin, num = ref["begin"].astype(np.uint32), ref["num"].astype(np.uint32)
    S, total = len(num), int(num.sum())
    off = np.concatenate([[0], np.cumsum(num, dtype=np.uint64)]).astype(np.uint64)
    d = sp.desc
    if what == "no masses":
        d = HfxSpectra(d.d_x, d.x_stride, d.d_len, d.d_zmax, None, d.num_spec)
    if what == "any begin":
        begin = np.where(num == 0, np.uint32(0xfffffff0), begin)
    if what == "gaps":
        off = off + 5 * np.arange(S + 1, dtype=np.uint64)
    dd = type(db.desc)(*[getattr(db.desc, f) for f, _ in db.desc._fields_])
    if what == "fewer peptides":   # the windows say where the candidates are
        dd.num_pep = 70_000
    t = [pl.dev(v) for v in (off, begin, num)]
    out = pl.dev(np.full(int(off[-1]), 12345.0, np.float32))
    ok(lib().hfx_xcorr_sparse(ctx.h, out.p, *[b.p for b in t], total, C.byref(dd), C.byref(d),
                              None), "hfx_xcorr_sparse")
    pl.sync()
    got = pl.host(out, np.float32, int(off[-1]))
    n = num.astype(np.int64)
    mine = np.repeat(off[:-1].astype(np.int64) - (np.cumsum(n) - n), n) + np.arange(total)
    bound = FORMS["fp32"][0] * scale + 1e-6 + 2.0**-24 * np.abs(exact)
    assert (np.abs(got[mine] - exact) <= bound).all()
    rest = np.ones(len(got), bool)
    rest[mine] = False
    assert (got[rest] == 12345.0).all()


def test_batch_with_masses_that_are_not_numbers(search, orc):
    from hfx_amd import pipeline as pl

    hdb, x, lens, zmax, mass, *_ = search
    x, lens, zmax, mass = x[:200], lens[:200], zmax[:200], mass[:200].copy()
    bs = {}
    for name, odd in (("nan", np.nan), ("empty", -5000.0)):
        mass[::3] = odd
        b = bs[name] = pl.BatchSearch(pl.Ctx(0), pl.DeviceDB(hdb), Spectra(pl, x, lens, zmax, mass), 3.0, 5)
        b.run()
        assert sorted(b.order()) == list(range(200))
    # every window but those of NaN, whose two bounds are where the search leaves them
    ref, exact, scale = reference(orc, hdb, x, lens, zmax, mass, 5)
    check(orc, bs["empty"].results(keep_scores=True), ref, exact, scale, x, *FORMS["fp32"])
    got, want = bs["nan"].results(), bs["empty"].results()
    keep = np.arange(200) % 3 != 0
    for a, b in ((got.top_pos, want.top_pos), (got.top_exact, want.top_exact)):
        live = keep[:, None] & (np.arange(5) < want.top_cnt[:, None])
        assert (a[live] == b[live]).all()
