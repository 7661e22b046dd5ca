"""findModablePeptides where the bits of all modifications at once would take too much memory."""
import numpy as np
import pytest

from test_gpu_rows import database
from test_gpu_rowsets import free

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("max_ma", [3, 6, 7])   # 65, 3,002 and 8,007 modifications
def test_many_modifications_of_a_large_database(orc, max_ma):
    from hfx_amd import lib
    from hfx_amd import pipeline as pl

    P = 200_000
    hdb = database(pl, P, seed=71, longest=12)
    mi = pl.mod_info({a: 10.0 + 1.37 * k for k, a in enumerate("ACDEGKLMST")}, max_ma)
    db = pl.DeviceDB(hdb)
    idx = db.idx_sorted()
    mass = np.sort(hdb.r)[[150_000, 195_000]].astype(np.float32)
    S, M, na = 2, mi.num_mod, mi.num_ma
    assert na == 10
    w = [orc.find_begin_end(hdb.r, idx, mi.mod_delta, m, 0.02) for m in mass]
    b, e, sc = (np.concatenate([v[k] for v in w]).astype(np.uint32) for k in range(3))
    cand = np.array([v[3] for v in w], np.uint32)
    scan = np.concatenate([[0], np.cumsum(cand)]).astype(np.uint32)
    total = int(scan[-1])
    t = {k: pl.dev(v) for k, v in dict(b=b, e=e, sc=sc, scan=scan, cnt=mi.mod_ma_count.astype(np.uint32),
                                       ma=np.frombuffer(mi.ma, np.uint8)).items()}
    out = [pl.empty(4 * total), pl.empty(4 * total), pl.empty(4 * total * na), pl.empty(4 * S)]
    before = free(pl)
    nv = lib().findModablePeptides(*[o.p for o in out], t["scan"].p, S, total, db.t_ions.p, db.t_tc.p,
                                   db.t_tn.p, db.t_idx.p, t["b"].p, t["e"].p, t["sc"].p, t["cnt"].p, M,
                                   t["ma"].p, na)
    # 64 MiB of bits and ranks and 40 bytes a position, a quarter more as scratch grows, and once
    # more what the windows take; 195,000 positions and 8,007 modifications at once take 290 MB
    assert before - free(pl) <= 1.25 * ((64 << 20) + 40 * P + 12 * S * M) + (8 << 20)
    want = orc.find_modable_peptides(scan, total, orc.prepare_ions(hdb.ions), hdb.tc, hdb.tn, idx, b, e,
                                     sc, mi.mod_ma_count, mi.ma)
    assert nv == want[0] > 0
    assert (pl.host(out[0], np.uint32, nv) == want[1]).all()
    assert (pl.host(out[1], np.uint32, nv) == want[2]).all()
    assert (pl.host(out[2], np.uint32, nv * na) == np.asarray(want[3]).reshape(-1)[:nv * na]).all()
    assert (pl.host(out[3], np.uint32, S) == want[4][:S]).all()
