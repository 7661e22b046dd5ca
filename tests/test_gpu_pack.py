"""The packed sparse scorer: the same bits whatever the size of the call (and with it the tiles
its candidates are dealt in), within the FP32 bound of the exact scores; and the line past which
hfx_xcorr_sparse takes rows instead."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_rows import Spectra, database, reference, spectra

pytestmark = pytest.mark.gpu


def scores(pl, L, ctx, db, hdb, sp, S, noalloc):
    P = len(hdb.r)
    num = np.full(S, P, np.uint32)
    off = np.arange(S + 1, dtype=np.uint64) * P
    t = [pl.dev(v) for v in (off, np.zeros(S, np.uint32), num)]
    out = pl.empty(4 * S * P)
    args = (pl.ptr(out), *[pl.ptr(v) for v in t], S * P, C.byref(db.desc), C.byref(sp.desc), None)
    if noalloc:
        pl.check(L.hfx_xcorr_sparse_noalloc(*args), "hfx_xcorr_sparse_noalloc")
    else:
        pl.check(L.hfx_xcorr_sparse(ctx.h, *args), "hfx_xcorr_sparse")
    pl.sync()
    return pl.host(out, np.float32, S * P).reshape(S, P)


# 23,985 and 24,600 pairs; 159,900 and 160,515; 999,990 and 1,000,605: 16, 32, 64 or 128
# candidates a tile
def test_tiles_of_any_size_give_the_same_bits(orc):
    import hfx_amd
    from hfx_amd import pipeline as pl

    L = hfx_amd.lib()
    hdb = database(pl, 615, seed=21)
    x, lens, zmax, mass = spectra(pl, hdb, 1627, 2112, seed=22)
    ctx, db = pl.Ctx(0), pl.DeviceDB(hdb)
    first = None
    for S in (1, 39, 40, 260, 261, 1626, 1627):
        sp = Spectra(pl, x[:S], lens[:S], zmax[:S], mass[:S])
        got = scores(pl, L, ctx, db, hdb, sp, S, True)
        if first is None:
            first = got
        elif S == 39:
            assert np.array_equal(got[:1], first)
            first = got
        else:
            assert np.array_equal(got[:39], first), S
    # against the exact scores
    ref, exact, scale = reference(orc, hdb, x[:39], lens[:39], zmax[:39], mass[:39], 5, eps=1e6)
    assert (ref["num"] == 615).all()
    assert (np.abs(first.ravel() - exact) <= 80 * 2.0**-24 * scale + 1e-6).all()


# 617 tiles: rows pay from about 420,000 pairs on
@pytest.mark.parametrize("S", [30, 41, 42, 43, 44, 60])
def test_either_side_of_the_rows(orc, S):
    import hfx_amd
    from hfx_amd import pipeline as pl

    L = hfx_amd.lib()
    hdb = database(pl, 9871, seed=23)
    x, lens, zmax, mass = spectra(pl, hdb, S, 2112, seed=24)
    ctx, db = pl.Ctx(0), pl.DeviceDB(hdb)
    sp = Spectra(pl, x, lens, zmax, mass)
    got = scores(pl, L, ctx, db, hdb, sp, S, False).ravel()
    ref, exact, scale = reference(orc, hdb, x, lens, zmax, mass, 5, eps=1e6)
    assert (np.abs(got - exact) <= 80 * 2.0**-24 * scale + 1e-6).all()
