"""Modified ladders past what one word of masks holds: peptides with more than fifteen residues of
a modable acid and sites among the last of them, and one to seven modable acids (masks of sixteen
to nine bits).  FP32 scores within 1e-4 of the exact score relative to max(|exact|, 100); rankings
and exact scores identical to the CPU oracle."""
import numpy as np
import pytest

from test_gpu_rows import Spectra

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("var", ["S", "ST", "MSTY", "KMSTY", "KMQSTY", "KMNQSTY"])
def test_many_residues_of_an_acid(orc, var):
    from hfx_amd import pipeline as pl

    rng = np.random.default_rng(len(var))
    mi = pl.mod_info({a: 8.0 + 5.25 * i for i, a in enumerate(var)}, 3)
    # runs of few letters, most of them modable
    seq = rng.choice(np.frombuffer((var[0] * 6 + var[-1] * 4 + var + "AGL").encode(), np.uint8), 3000)
    mass = pl.mass_table()
    P = 60
    n = rng.integers(6, 62, P)
    n[:6] = 18, 30, 45, 60, 62, 63
    tc = rng.integers(0, len(seq) - 70, P).astype(np.uint32)
    tn = (tc + n).astype(np.uint32)
    cs = np.concatenate([[0.0], np.cumsum(mass[seq - 65].astype(np.float64))])
    r = (cs[tc + n + 1] - cs[tc]).astype(np.float32)
    ctx = pl.Ctx(0)
    db = pl.DeviceDB(pl.HostDB(seq, r, tc, tn, mass), ma=mi.ma)
    S, stride = 6, 2112
    x = np.where(rng.random((S, stride)) < 0.1, rng.uniform(1, 50, (S, stride)),
                 rng.normal(0, 0.3, (S, stride))).astype(np.float32)
    lens = np.full(S, stride)
    zmax = np.array([1, 2, 3, 4, 2, 1])
    centre = r[[0, 1, 2, 3, 4, 5]] + mi.mod_delta[rng.integers(0, mi.num_mod, S)]
    sp = Spectra(pl, x, lens, zmax, centre.astype(np.float32))
    sp.mass = centre.astype(np.float32)
    ms = pl.ModSearch(ctx, db, sp, mi, eps=3.0, topn=5)
    res = ms.run(keep_scores=True)
    idx, _ = orc.sort_idx(r)
    ions = orc.prepare_ions(seq, mi.ma)
    ref = orc.search_mods(ions, r, tc, tn, mass, idx, mi.ma, mi.ma_mass, mi.mod_ma_count, mi.mod_sum,
                          mi.mod_delta, x, lens.astype(np.uint32), zmax.astype(np.uint32), sp.mass,
                          3.0, 5)
    assert (np.diff(res.mp_off).astype(np.uint32) == ref["spec_num_mpep"]).all()
    st = res.stages
    far = 0
    for s in range(S):
        a, b = int(res.mp_off[s]), int(res.mp_off[s + 1])
        for i in rng.choice(np.arange(a, b), size=min(60, b - a), replace=False) if b > a else []:
            p, m = int(st["mp_pep"][i]), int(st["mp_mod"][i])
            u0, k = int(st["mp_scan"][i]), int(mi.mod_sum[m])
            far += int((st["unrank"][u0:u0 + k] >= 15).any())
            w = orc.mpeaks_dense(ions, int(tc[p]), int(tn[p]), r[p], mass, int(zmax[s]), stride,
                                 mi.mod_ma_count[m], mi.mod_delta[m], mi.ma, mi.ma_mass,
                                 st["unrank"][u0:u0 + k])
            ex = orc.fx_to_double(orc.score_fx(w, x[s]))
            assert abs(float(res.scores[i]) - ex) <= 1e-4 * max(abs(ex), 100.0), (s, i)
    assert far > 0
    assert (res.top_cnt == ref["top_cnt"]).all()
    for s in range(S):
        c = int(res.top_cnt[s])
        assert res.top_pos[s, :c].tolist() == ref["top_pos"][s, :c].tolist(), s
        assert (res.top_exact[s, :c] == orc.fx_to_double(ref["top_fx"][s, :c])).all()
