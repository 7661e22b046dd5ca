"""Top-N where its ways part: selections from the lanes' largest scores and by radix, windows read
once and twice, lists a wave re-scores alone and lists shared out, bands past the list, fewer
candidates than N, long peptides, uncommon scores.  The ranking must be the oracle's whatever the
stated error bound makes of the band."""
import numpy as np
import pytest

from test_gpu_rows import Spectra, database, reference, spectra

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tenv(orc):
    from hfx_amd import pipeline as pl

    hdb = database(pl, 60007, seed=11, longest=30)
    x, lens, zmax, mass = spectra(pl, hdb, 48, 2112, seed=12)
    mass[:4] = hdb.r.max() + np.array([2.0, 2.9, 500.0, 2.0], np.float32)  # few candidates, none
    ctx = pl.Ctx(0)
    db, sp = pl.DeviceDB(hdb), Spectra(pl, x, lens, zmax, mass)
    ref = {eps: reference(orc, hdb, x, lens, zmax, mass, 64, eps)[0] for eps in (3.0, 250.0)}
    assert ref[3.0]["num"].min() == 0 and 0 < np.median(ref[3.0]["num"]) < 6144
    assert ref[250.0]["num"].max() > 6144
    return dict(pl=pl, ctx=ctx, db=db, sp=sp, ref=ref, rows=(x, lens, zmax, mass))


def check(orc, s, ref, N):
    from hfx_amd import pipeline as pl

    S = s.sp.num_spec
    cnt = pl.host(s.t_cnt, np.uint32, S)
    pos = pl.host(s.t_pos, np.uint32, S * N).reshape(S, N)
    ex = pl.host(s.t_exact, np.float64, S * N).reshape(S, N)
    f32 = pl.host(s.t_f32, np.float32, S * N).reshape(S, N)
    sc = pl.host(s.t_scores, np.float32, s.total)
    assert (cnt == np.minimum(ref["num"], N)).all()
    assert len(s.short()) == 0
    for k in range(S):
        c = int(cnt[k])
        assert pos[k, :c].tolist() == ref["top_pos"][k, :c].tolist(), k
        assert (ex[k, :c] == orc.fx_to_double(ref["top_fx"][k, :c])).all(), k
        assert (f32[k, :c] == sc[int(ref["off"][k]) + pos[k, :c].astype(np.int64)]).all(), k


@pytest.mark.parametrize("eps", [3.0, 250.0])
@pytest.mark.parametrize("N,margin", [(1, 0), (5, 0), (6, 1), (10, 0), (32, 0), (32, 1), (64, 64)])
def test_every_way_gives_the_same_ranking(tenv, orc, eps, N, margin):
    pl = tenv["pl"]
    s = pl.PlainSearch(tenv["ctx"], tenv["db"], tenv["sp"], eps=eps, topn=N, margin=margin)
    s.window()
    s.score()
    flagged = []
    # the FP32 bound, then wider ones: bands of a few, tens, hundreds, the whole window
    for rel0 in (80 * 2.0**-24, 1e-4, 1e-3, 1e-2, 0.5):
        s.t_cnt.zero()
        s.select_rel(rel0)
        check(orc, s, tenv["ref"][eps], N)
        flagged.append(len(s.flagged()))
    assert flagged == sorted(flagged)  # a wider bound, a wider band
    assert flagged[-1] > 0 or eps < 10


@pytest.mark.parametrize("N", [15, 16, 17])
def test_exact_windows_by_rounds_and_by_radix(tenv, orc, N):
    """Windows scored exactly as a whole: up to sixteen places by rounds of the best, more by radix.
    The two meet here, and the top N is the oracle's on both sides."""
    pl = tenv["pl"]
    s = pl.PlainSearch(tenv["ctx"], tenv["db"], tenv["sp"], eps=250.0, topn=N)
    s.window()
    s.score()
    s.t_cnt.zero()
    s.select_rel(0.5)
    check(orc, s, tenv["ref"][250.0], N)
    assert len(s.flagged()) > 0


@pytest.mark.parametrize("S", [4096, 4097])
def test_lists_shared_out_whole_and_in_halves(tenv, S):
    """Many spectra re-score longer runs a wave: each copy of a spectrum has the ranking of the
    first."""
    pl = tenv["pl"]
    which = np.arange(S) % 48
    sp = Spectra(pl, *(a[which] for a in tenv["rows"]))
    s = pl.PlainSearch(tenv["ctx"], tenv["db"], sp, eps=3.0, topn=40)
    s.window()
    s.score()
    s.select_rel(1e-3)
    assert len(s.short()) == 0
    ref = tenv["ref"][3.0]
    cnt = pl.host(s.t_cnt, np.uint32, S)
    pos = pl.host(s.t_pos, np.uint32, S * 40).reshape(S, 40)
    assert (cnt == np.minimum(ref["num"], 40)[which]).all()
    for k in range(S):
        assert pos[k, :cnt[k]].tolist() == ref["top_pos"][which[k], :cnt[k]].tolist(), k


@pytest.mark.parametrize("S", [255, 700])
def test_many_spectra_on_the_exact_route(tenv, S):
    """The list of flagged spectra in one turn of its workgroup and in several."""
    pl = tenv["pl"]
    which = np.arange(S) % 48
    sp = Spectra(pl, *(a[which] for a in tenv["rows"]))
    s = pl.PlainSearch(tenv["ctx"], tenv["db"], sp, eps=250.0, topn=5)
    s.window()
    s.score()
    s.select_rel(0.5)
    assert len(s.short()) == 0 and (len(s.flagged()) > 256) == (S == 700)
    ref = tenv["ref"][250.0]
    pos = pl.host(s.t_pos, np.uint32, S * 5).reshape(S, 5)
    for k in range(S):
        c = min(int(ref["num"][which[k]]), 5)
        assert pos[k, :c].tolist() == ref["top_pos"][which[k], :c].tolist(), k


@pytest.mark.parametrize("N", [5, 40])
def test_scores_with_infinities_keep_their_order(tenv, orc, N):
    """The selection follows the scores' total order: with -inf in most places the finite ones
    are ranked, exactly."""
    pl = tenv["pl"]
    ref = tenv["ref"][3.0]
    s = pl.PlainSearch(tenv["ctx"], tenv["db"], tenv["sp"], eps=3.0, topn=N)
    s.window()
    sc = np.full(s.total, -np.inf, np.float32)
    off = ref["off"].astype(np.int64)
    for k in range(s.sp.num_spec):
        c = int(min(ref["num"][k], 64))
        sc[off[k] + ref["top_pos"][k, :c].astype(np.int64)] = orc.fx_to_double(ref["top_fx"][k, :c])
    s.t_scores.upload(sc)
    s.select()
    check(orc, s, ref, N)
