"""Mass windows, prefix sums and the enumeration of modified peptides at the sizes where
their kernels change steps.  Whole numbers throughout: identical to NumPy's searches and
sums, and to the CPU oracle."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lib():
    import hfx_amd
    from hfx_amd import pipeline

    return pipeline, hfx_amd.lib()


def _bounds(rs, lo, hi):
    return np.searchsorted(rs, lo, "left"), np.searchsorted(rs, hi, "right")


# a wave probes 64 parts of what is left, a thread seven
@pytest.mark.parametrize("n", [1, 2, 7, 8, 9, 63, 64, 65, 127, 4095, 4096, 4097, 262145])
def test_windows(lib, n):
    import hfx_amd

    pl, L = lib
    rng = np.random.default_rng(n)
    r = np.round(rng.uniform(400, 3000, n), 1).astype(np.float32)   # many equal
    idx = np.argsort(r, kind="stable").astype(np.uint32)
    rs = r[idx]
    S = 150
    mass = np.concatenate([rng.uniform(300, 3100, S - 4), rs[[0, -1]], [-1e9, 1e9]]).astype(np.float32)
    eps = np.float32(0.3)
    ctx = pl.Ctx(0)
    t = dict(r=pl.dev(r), idx=pl.dev(idx), rs=pl.dev(rs), mass=pl.dev(mass))
    b, e = _bounds(rs, mass - eps, mass + eps)
    delta = np.array([0.0, 15.9949, 79.9663, -40.0] * 17, np.float32)   # more than a wave's lanes
    M = len(delta)
    t["delta"] = pl.dev(delta)
    for srt in (True, False):
        db = hfx_amd.HfxDb()
        db.d_r, db.d_idx_sorted, db.num_pep = pl.ptr(t["r"]), pl.ptr(t["idx"]), n
        db.d_r_sorted = pl.ptr(t["rs"]) if srt else None
        ob, on = pl.empty(4 * S), pl.empty(4 * S)
        pl.check(L.hfx_window(ctx.h, pl.ptr(ob), pl.ptr(on), C.byref(db), pl.ptr(t["mass"]), S,
                              float(eps), None), "hfx_window")
        w = [pl.empty(4 * S * M) for _ in range(3)] + [pl.empty(4 * S)]
        pl.check(L.hfx_mod_windows(ctx.h, *[pl.ptr(v) for v in w], C.byref(db), pl.ptr(t["mass"]), S,
                                   pl.ptr(t["delta"]), M, float(eps), None), "hfx_mod_windows")
        pl.sync()
        assert (pl.host(ob, np.uint32, S) == b).all() and (pl.host(on, np.uint32, S) == e - b).all()
        lo = (mass - eps)[:, None] - delta
        hi = (mass + eps)[:, None] - delta
        mb, me = _bounds(rs, lo, hi)
        num = me - mb
        assert (pl.host(w[0], np.uint32, S * M).reshape(S, M) == mb).all()
        assert (pl.host(w[1], np.uint32, S * M).reshape(S, M) == me).all()
        assert (pl.host(w[2], np.uint32, S * M).reshape(S, M) == np.cumsum(num, 1) - num).all()
        assert (pl.host(w[3], np.uint32, S) == num.sum(1)).all()
    # the reference's call, one spectrum
    v = [pl.empty(4 * M) for _ in range(3)]
    total = L.findBeginEnd_f(*[pl.ptr(x) for x in v], pl.ptr(t["r"]), pl.ptr(t["idx"]), n,
                             pl.ptr(t["delta"]), M, float(mass[0]), float(eps))
    assert total == num[0].sum()
    assert (pl.host(v[0], np.uint32, M) == mb[0]).all() and (pl.host(v[1], np.uint32, M) == me[0]).all()


# one workgroup with 1, 4 or 16 counts a thread, then tiles of 8192
@pytest.mark.parametrize("n", [1, 63, 64, 1024, 1025, 4095, 4096, 4097, 16384, 16385, 32767, 32768,
                               40961, 300007])
def test_scan_offsets(lib, n):
    pl, L = lib
    rng = np.random.default_rng(n)
    cnt = rng.integers(0, 2 ** 32, n + 1, dtype=np.uint64).astype(np.uint32)
    ctx = pl.Ctx(0)
    for first in (0, 1):      # counts and offsets at any multiple of their size
        c = cnt[first:first + n]
        tc, to = pl.dev(cnt), pl.empty(8 * (n + 3))
        pl.check(L.hfx_scan_offsets(ctx.h, pl.ptr(to) + 8 * first, pl.ptr(tc) + 4 * first, n, None),
                 "hfx_scan_offsets")
        pl.sync()
        got = pl.host(to, np.uint64, n + 2)[first:first + n + 1]
        assert (got == np.concatenate([[0], np.cumsum(c.astype(np.uint64))]).astype(np.uint64)).all()


# positions around a word of 64, modable acids with a kernel of their own (4) and without
@pytest.mark.parametrize("npep,var", [(1, "S"), (63, "ST"), (64, "MSTY"), (65, "MSTY"), (700, "MSTYK"),
                                      (5000, "MSTY"), (3000, "M")])
def test_enumeration(lib, orc, npep, var):
    pl, L = lib
    rng = np.random.default_rng(npep + len(var))
    mi = pl.mod_info({a: 10.0 + 7.3 * i for i, a in enumerate(var)}, 4)
    M, na = mi.num_mod, mi.num_ma
    seq = rng.choice(np.frombuffer(b"ACDEFGHIKLMNPQRSTVWYSTSTM", np.uint8), 20 * npep + 60)
    tc = rng.integers(0, 20 * npep, npep).astype(np.uint32)
    tn = (tc + rng.integers(5, 45, npep)).astype(np.uint32)
    r = np.sort(rng.uniform(400, 3000, npep)).astype(np.float32)
    idx = rng.permutation(npep).astype(np.uint32)
    ions = orc.prepare_ions(seq, mi.ma)
    S = 9
    b = rng.integers(0, npep + 1, (S, M)).astype(np.uint32)
    e = np.minimum(npep, b + rng.integers(0, min(npep, 400) + 1, (S, M))).astype(np.uint32)
    e[3] = b[3]
    b[4], e[4] = 0, npep
    num = (e - b).astype(np.uint32)
    sc = (np.cumsum(num, 1) - num).astype(np.uint32)
    scan = np.concatenate([[0], np.cumsum(num.sum(1))]).astype(np.uint32)
    total = int(scan[-1])
    want = orc.find_modable_peptides(scan, total, ions, tc, tn, idx, b.ravel(), e.ravel(), sc.ravel(),
                                     mi.mod_ma_count, mi.ma)
    t = [pl.dev(v) for v in (scan, ions, tc, tn, idx, b.ravel(), e.ravel(), sc.ravel(),
                             mi.mod_ma_count.reshape(-1), np.frombuffer(mi.ma, np.uint8), mi.mod_sum)]
    o = [pl.empty(4 * max(total, 1)), pl.empty(4 * max(total, 1)), pl.empty(4 * max(total, 1) * na),
         pl.empty(4 * S)]
    nv = L.findModablePeptides(*[pl.ptr(x) for x in o], pl.ptr(t[0]), S, total, pl.ptr(t[1]),
                               *[pl.ptr(x) for x in t[2:9]], M, pl.ptr(t[9]), na)
    assert nv == want[0]
    for buf, ref, k in zip(o, want[1:], (nv, nv, nv * na, S)):
        assert (pl.host(buf, np.uint32, k) == np.asarray(ref).ravel()[:k]).all()
    if nv == 0:
        return
    pep, pmod, pcnt = want[1:4]
    nmp, cnum, comb = orc.calc_total_mod_cands(mi.mod_ma_count, pep, pmod, pcnt, na)
    tn_, tcomb = pl.empty(4 * nv), pl.empty(4 * nv * na)
    assert nmp == L.calcTotalModCands(pl.ptr(tn_), pl.ptr(tcomb), pl.ptr(t[8]), pl.ptr(o[0]),
                                      pl.ptr(o[1]), pl.ptr(o[2]), nv, M, na)
    assert (pl.host(tn_, np.uint32, nv) == cnum).all()
    assert (pl.host(tcomb, np.uint32, nv * na) == np.asarray(comb).ravel()).all()
    gen = orc.prepare_gen_mod(mi.mod_sum, pep, pmod, cnum, nmp)
    tm = [pl.empty(4 * nmp) for _ in range(5)]
    lu = L.prepareGenMod(*[pl.ptr(x) for x in tm], pl.ptr(t[10]), pl.ptr(o[0]), pl.ptr(o[1]),
                         pl.ptr(tn_), nv, nmp)
    assert lu == gen[0]
    for buf, ref in zip(tm, gen[1:]):
        assert (pl.host(buf, np.uint32, nmp) == ref).all()
    tu = pl.empty(4 * max(lu, 1))
    L.genModCands(pl.ptr(tu), pl.ptr(t[8]), pl.ptr(tm[3]), pl.ptr(tm[2]), pl.ptr(tm[4]), pl.ptr(o[1]),
                  pl.ptr(o[2]), pl.ptr(tcomb), nmp, na)
    pl.sync()
    ref = orc.gen_mod_cands(lu, mi.mod_ma_count, gen[4], gen[3], gen[5], pmod, pcnt, comb, na)
    assert (pl.host(tu, np.uint32, lu) == ref).all()


def test_rows_without_modified_peptides(lib):
    """prepareGenMod over rows of no modified peptides, few and more than a workgroup's."""
    pl, L = lib
    rng = np.random.default_rng(11)
    for n, hi in ((1, 5000), (3000, 2), (400, 60), (20000, 3)):
        cnt = np.where(rng.random(n) < 0.5, 0, rng.integers(0, hi, n)).astype(np.uint32)
        cnt[n // 2] = 5001
        total = int(cnt.sum())
        mod = rng.integers(0, 3, n).astype(np.uint32)
        pep = rng.integers(0, 1000, n).astype(np.uint32)
        msum = np.array([1, 2, 3], np.uint32)
        t = [pl.dev(v) for v in (msum, pep, mod, cnt)]
        o = [pl.empty(4 * total) for _ in range(5)]
        lu = L.prepareGenMod(*[pl.ptr(x) for x in o], *[pl.ptr(x) for x in t], n, total)
        row = np.repeat(np.arange(n), cnt)
        ref = [pep[row], mod[row], np.arange(total) - (np.cumsum(cnt) - cnt)[row], row,
               np.cumsum(msum[mod[row]]) - msum[mod[row]]]
        assert lu == msum[mod[row]].sum()
        for k, buf in enumerate(o):
            assert (pl.host(buf, np.uint32, total) == ref[k]).all(), (n, k)
