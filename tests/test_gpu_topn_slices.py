"""hfx_topn over part of the spectra of a search, whose scores start past the first and leave room
between the spectra, and over rows whose stride passes the longest spectrum."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_rows import Spectra, database, reference, spectra

pytestmark = pytest.mark.gpu

N = 5


@pytest.fixture(scope="module")
def env(orc):
    from hfx_amd import pipeline as pl

    hdb = database(pl, 30011, seed=41, longest=30)
    rows = spectra(pl, hdb, 40, 1500, seed=42)
    ref, exact, _ = reference(orc, hdb, *rows, N, eps=60.0)   # windows past the re-score list
    return pl, pl.Ctx(0), pl.DeviceDB(hdb), rows, ref, exact.astype(np.float32)


def topn(pl, ctx, db, sp, S, args, total, rel0):
    from hfx_amd import check, lib

    t = [pl.empty(4 * S * N), pl.empty(8 * S * N), pl.empty(4 * S * N), pl.empty(4 * S), pl.empty(4 * S)]
    scores, off, begin, num = args
    check(lib().hfx_topn_rel(ctx.h, *[b.p for b in t], N, 0, rel0, 0.0, scores, off, total, begin, num,
                             C.byref(db.desc), C.byref(sp), None), "hfx_topn_rel")
    pl.sync()
    return (pl.host(t[0], np.uint32, S * N).reshape(S, N), pl.host(t[1], np.float64, S * N).reshape(S, N),
            pl.host(t[3], np.uint32, S), pl.host(t[4], np.uint32, S))


def same(orc, got, ref, a, b):
    pos, ex, cnt, _ = got
    assert (cnt == ref["top_cnt"][a:b]).all()
    for k in range(a, b):
        c = int(cnt[k - a])
        assert pos[k - a, :c].tolist() == ref["top_pos"][k, :c].tolist()
        assert (ex[k - a, :c] == orc.fx_to_double(ref["top_fx"][k, :c])).all()


@pytest.mark.parametrize("rel0", [80 * 2.0**-24, 0.5])  # a short band; the exact route for all
@pytest.mark.parametrize("gap", [0, 7])
def test_part_of_a_search(env, orc, gap, rel0):
    from hfx_amd import HfxSpectra

    pl, ctx, db, rows, ref, scores = env
    sp = Spectra(pl, *rows)
    off = ref["off"].astype(np.uint64)
    S = sp.num_spec
    wide = np.zeros(len(scores) + gap * (S + 1), np.float32)
    for k in range(S):
        o = int(off[k])
        wide[o + gap * k:int(off[k + 1]) + gap * k] = scores[o:int(off[k + 1])]
    t_sc, t_off = pl.dev(wide), pl.dev(off + np.uint64(gap) * np.arange(S + 1, dtype=np.uint64))
    t_b, t_n = pl.dev(ref["begin"].astype(np.uint32)), pl.dev(ref["num"].astype(np.uint32))
    d = sp.desc
    for a, b in ((0, S), (13, 29), (S - 1, S)):
        part = HfxSpectra(d.d_x + 4 * a * d.x_stride, d.x_stride, d.d_len + 4 * a, d.d_zmax + 4 * a,
                          d.d_mass + 4 * a, b - a)
        got = topn(pl, ctx, db, part, b - a, (t_sc.p, t_off.p + 8 * a, t_b.p + 4 * a, t_n.p + 4 * a),
                   int(ref["num"][a:b].sum()), rel0)
        same(orc, got, ref, a, b)
        assert rel0 < 0.1 or b - a == 1 or got[3].any()   # some took the exact route


def test_rows_of_a_longer_stride(env, orc):
    pl, ctx, db, (x, lens, zmax, mass), ref, scores = env
    long = np.zeros((len(x), 9000), np.float32)
    long[:, :x.shape[1]] = x
    sp = Spectra(pl, long, lens, zmax, mass)
    t = [pl.dev(v) for v in (scores, ref["off"].astype(np.uint64), ref["begin"].astype(np.uint32),
                             ref["num"].astype(np.uint32))]
    for rel0 in (80 * 2.0**-24, 0.5):
        got = topn(pl, ctx, db, sp.desc, len(x), [b.p for b in t], len(scores), rel0)
        same(orc, got, ref, 0, len(x))
