"""Scores through theoretical rows (hfx_rows.hip) where they can go wrong: databases that end
inside a tile of sixteen, long and residue-free peptides, peaks past either end of a row, rows of
one group and of the longest stride, every fragment charge, spectra whose values do not fit 32-bit
fixed point (they keep the FP32 kernel), and strides past the rows'."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LETTERS = np.frombuffer(b"ACDEFGHIKLMNPQRSTVWY", np.uint8)


def database(pl, npep, seed, longest=70):
    """npep peptides of 0..longest ladder positions (a few of 200) over random residues."""
    rng = np.random.default_rng(seed)
    seq = LETTERS[rng.integers(0, 20, 6000)]
    mass = pl.mass_table()
    n = rng.integers(0, longest + 1, npep)
    n[rng.random(npep) < 0.01] = 200
    tc = rng.integers(0, len(seq) - 201, npep).astype(np.uint32)
    cs = np.concatenate([[0.0], np.cumsum(mass[seq - 65].astype(np.float64))])
    r = (cs[tc + n + 1] - cs[tc]).astype(np.float32)
    return pl.HostDB(seq, r, tc, (tc + n).astype(np.uint32), mass)


class Spectra:
    """Preprocessed rows given directly, with lengths, fragment charges and window centres."""

    def __init__(self, pl, x, lens, zmax, mass):
        from hfx_amd import HfxSpectra

        self.num_spec, self.x_stride = x.shape
        self.zmax, self.mass = zmax.astype(np.uint32), mass.astype(np.float32)
        self.keep = [pl.dev(v) for v in (x.astype(np.float32), lens.astype(np.uint32), self.zmax,
                                         self.mass)]
        self.t_x, self.t_len, self.t_zmax, self.t_mass = self.keep
        self.desc = HfxSpectra(self.t_x.p, self.x_stride, self.t_len.p, self.t_zmax.p,
                               self.t_mass.p, self.num_spec)


def spectra(pl, hdb, S, stride, seed):
    rng = np.random.default_rng(seed)
    lens = rng.integers(min(85, stride), stride + 1, S)
    lens[:3] = stride, stride - 1, max(stride // 2, 1)
    x = rng.normal(0.0, 0.3, (S, stride))
    hit = rng.random((S, stride)) < 0.08
    x[hit] = rng.uniform(1.0, 50.0, hit.sum())
    x[np.arange(stride)[None, :] >= lens[:, None]] = 0.0
    zmax = rng.choice([1, 2, 3, 4, 5], S, p=[0.3, 0.3, 0.2, 0.15, 0.05])
    mass = hdb.r[rng.integers(0, len(hdb.r), S)]
    return x.astype(np.float32), lens, zmax, mass


def reference(orc, hdb, x, lens, zmax, mass, topn, eps=3.0):
    idx, _ = orc.sort_idx(hdb.r)
    args = (orc.prepare_ions(hdb.ions), hdb.r, hdb.tc, hdb.tn, hdb.mass, idx)
    kw = dict(want_all=True, nthreads=8)
    m = mass.astype(np.float32)
    ref = orc.search_plain(*args, x, lens.astype(np.uint32), zmax.astype(np.uint32), m, eps, topn, **kw)
    scale = orc.search_plain(*args, np.abs(x), lens.astype(np.uint32), zmax.astype(np.uint32), m, eps,
                             topn, **kw)
    n = int(ref["off"][-1])
    return ref, orc.fx_to_double(ref["all_fx"])[:n], orc.fx_to_double(scale["all_fx"])[:n]


def check(orc, res, ref, exact, scale, x, rel, absq=0.0):
    """|score - exact| <= rel * sum w|x| + absq * max|x| * 50 per non-zero bin (at most one a
    ladder position, charge and peak: 10 * 200 * 4); the same ranking."""
    assert (res.num == ref["num"]).all()
    big = np.repeat(np.abs(x).max(1), res.num)
    bound = rel * scale + absq * big * 50 * 8000 + 1e-6 + 2.0**-24 * np.abs(exact)
    assert (np.abs(res.scores - exact) <= bound).all()
    assert (res.top_cnt == ref["top_cnt"]).all()
    for s in range(len(res.top_cnt)):
        c = int(res.top_cnt[s])
        assert res.top_pos[s, :c].tolist() == ref["top_pos"][s, :c].tolist()
        assert (res.top_exact[s, :c] == orc.fx_to_double(ref["top_fx"][s, :c])).all()


# one FP32 sum of a candidate's bins; the quantum of each digit form
FORMS = {"fp32": (80 * 2.0**-24, 0.0), "bf16": (2.0**-16 + 210 * 2.0**-24, 0.0),
         "i8": (0.0, 1.0 / 8355711)}


@pytest.mark.parametrize("npep,stride", [(1, 2112), (16, 2176), (1021, 100), (4099, 2112), (4096, 700)])
@pytest.mark.parametrize("form", sorted(FORMS))
def test_batch_rows_match_the_oracle(orc, form, npep, stride):
    from hfx_amd import pipeline as pl

    hdb = database(pl, npep, seed=npep)
    x, lens, zmax, mass = spectra(pl, hdb, 70, stride, seed=stride)
    ref, exact, scale = reference(orc, hdb, x, lens, zmax, mass, 5)
    ctx = pl.Ctx(0)
    db, sp = pl.DeviceDB(hdb), Spectra(pl, x, lens, zmax, mass)
    bs = pl.BatchSearch(ctx, db, sp, eps=3.0, topn=5)
    bs.set_precision({"fp32": bs.FP32_SPARSE, "bf16": bs.BF16X2_DENSE, "i8": bs.I8X3_DENSE}[form])
    bs.run()
    first = bs.results(keep_scores=True)
    check(orc, first, ref, exact, scale, x, *FORMS[form])
    bs.capture()
    for _ in range(3):
        bs.replay()
        assert np.array_equal(bs.results(keep_scores=True).scores, first.scores)


def test_sparse_scores_through_rows_and_wide_spectra(orc):
    """hfx_xcorr_sparse over enough pairs that rows are taken; some spectra hold a value that
    dwarfs the rest, or one that is not finite, and are scored in FP32 all the same."""
    from hfx_amd import pipeline as pl

    hdb = database(pl, 100003, seed=5, longest=20)
    x, lens, zmax, mass = spectra(pl, hdb, 4000, 2112, seed=6)
    x[7, 40], x[8, 0] = 3e5, -1e6   # 50 x 2^36 within the oracle's 64 bits
    odd = np.array([100, 101, 102])
    clean = x.copy()
    clean[odd] = 0.0
    ref, exact, scale = reference(orc, hdb, clean, lens, zmax, mass, 5)
    n = ref["num"]
    assert n.sum() > 1_000_000
    x[odd[0], 3], x[odd[1], 4], x[odd[2], 5] = np.inf, -np.inf, np.nan
    ctx = pl.Ctx(0)
    db = pl.DeviceDB(hdb)
    s = pl.PlainSearch(ctx, db, Spectra(pl, x, lens, zmax, mass), eps=3.0, topn=5)
    s.window()
    s.score()
    pl.sync()
    got = pl.host(s.t_scores, np.float32, s.total).astype(np.float64)
    keep = ~np.repeat(np.isin(np.arange(len(n)), odd), n)
    bound = 80 * 2.0**-24 * scale + 1e-6
    off = np.repeat(np.arange(len(n)), n)[keep & ~(np.abs(got - exact) <= bound)]
    assert len(off) == 0, np.unique(off)
    # the plain kernel's own answer for the others, NaN where it has one
    o = ref["off"].astype(np.int64)
    for k in odd:
        one = pl.PlainSearch(ctx, db, Spectra(pl, x[k:k + 1], lens[k:k + 1], zmax[k:k + 1],
                                              mass[k:k + 1]), eps=3.0, topn=5)
        one.window()
        one.score()
        pl.sync()
        want = pl.host(one.t_scores, np.float32, one.total)
        assert np.array_equal(got[o[k]:o[k + 1]].astype(np.float32), want, equal_nan=True)


def test_strides_past_the_rows_keep_the_ion_lists(orc):
    from hfx_amd import pipeline as pl

    hdb = database(pl, 2000, seed=8)
    x, lens, zmax, mass = spectra(pl, hdb, 40, 2300, seed=9)
    ref, exact, scale = reference(orc, hdb, x, lens, zmax, mass, 5)
    bs = pl.BatchSearch(pl.Ctx(0), pl.DeviceDB(hdb), Spectra(pl, x, lens, zmax, mass), eps=3.0,
                        topn=5)
    bs.run()
    check(orc, bs.results(keep_scores=True), ref, exact, scale, x, *FORMS["fp32"])
