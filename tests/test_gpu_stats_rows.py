"""E-value fits at the sizes where their kernel's paths meet, and SP ion matches of
top-N lists for every row length that has a kernel of its own, against the CPU oracle.

Whole numbers are identical; alpha and beta are FP64 sums over the same histogram in
another order: within 1e-9 relative (absolute 1e-9 near zero).
"""
import ctypes as C

import numpy as np
import pytest

from test_gpu_stats import _check_fits, _fit_direct

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lib():
    import hfx_amd
    from hfx_amd import pipeline

    return pipeline, hfx_amd.lib()


# keys (x - min - 4000) / 350: the counts are kept 16, 8, 4, 2 and once each up to 64, 128,
# 256, 512 and 1024 keys, then by ranges of 1024
@pytest.mark.parametrize("keys", [1, 60, 64, 70, 127, 200, 256, 400, 600, 1000, 1023, 1024, 1100,
                                  5000])
def test_evalue_fit_key_spreads(lib, orc, keys):
    rng = np.random.default_rng(keys)
    top = 4000.0 + 350.0 * keys
    segs = []
    for n in (64, 1023, 1024, 1025, 6143, 6144, 6145, 9001):
        x = (top * rng.beta(2.0, 3.0, n) - 900.0).astype(np.float32)
        x[rng.integers(n)], x[rng.integers(n)] = -900.0, top - 900.0 - 1.0
        # on the edges of bins
        k = rng.integers(0, n, n // 8)
        x[k] = (np.rint(x[k] / 350.0) * 350.0 - 901.0).astype(np.float32)
        segs.append(x)
    _check_fits(orc, _fit_direct(*lib, segs), segs)
    # two sets: the second starts anywhere, and both hold partial chunks
    cut = [int(rng.integers(0, len(x) + 1)) for x in segs]
    _check_fits(orc, _fit_direct(*lib, [x[:c] for x, c in zip(segs, cut)],
                                 [x[c:] for x, c in zip(segs, cut)]), segs)


def test_evalue_fit_large_values(lib, orc):
    """Scores whose FP32 quotients err by more than a bin."""
    rng = np.random.default_rng(3)
    segs = [(1e9 + rng.integers(0, 2000, 3000) * 64.0).astype(np.float32),
            (-3e7 + rng.normal(0, 9e4, 5000)).astype(np.float32)]
    _check_fits(orc, _fit_direct(*lib, segs), segs)


@pytest.mark.parametrize("stride,N", [(768, 5), (769, 1), (1536, 16), (2176, 17), (2305, 5),
                                      (3072, 40), (3073, 17)])
def test_sp_ions_topn_row_lengths(lib, orc, small_workload, stride, N):
    import hfx_amd

    pl, L = lib
    w = small_workload
    rng = np.random.default_rng(stride + N)
    S, P = 9, len(w["r"])
    ctx = pl.Ctx(0)
    db = pl.DeviceDB(pl.HostDB(ions=w["prot"].seq, r=w["r"], tc=w["tc"], tn=w["tn"],
                               mass=w["mass"]))
    X = np.where(rng.random((S, stride)) < 0.4, np.abs(rng.normal(0, 1, (S, stride))), 0.0)
    X[1] = np.round(X[1] * 3) / 3                   # ties at the 200th value
    X[2] = (rng.random(stride) < 0.9) * 0.5         # all of them
    X[3] = -1.0
    X = X.astype(np.float32)
    lens = rng.integers(stride // 2, stride + 1, S).astype(np.uint32)
    lens[4], lens[5] = 0, stride
    zmax = rng.integers(0, 5, S).astype(np.uint32)
    begin = rng.integers(0, P - 400, S).astype(np.uint32)
    pos = rng.integers(0, 400, (S, N)).astype(np.uint32)
    cnt = rng.integers(0, N + 1, S).astype(np.uint32)
    cnt[:3] = N
    t = [pl.dev(v) for v in (X, lens, zmax, np.zeros(S, np.float32), pos, cnt, begin)]
    desc = hfx_amd.HfxSpectra(pl.ptr(t[0]), stride, pl.ptr(t[1]), pl.ptr(t[2]), pl.ptr(t[3]), S)
    outs = [pl.empty(4 * S * N) for _ in range(3)]
    pl.check(L.hfx_sp_ions_topn(ctx.h, *[pl.ptr(o) for o in outs], pl.ptr(t[4]), pl.ptr(t[5]),
                                pl.ptr(t[6]), N, C.byref(db.desc), C.byref(desc), 1, None),
             "hfx_sp_ions_topn")
    pl.sync()
    got = [pl.host(o, np.uint32, S * N).reshape(S, N) for o in outs]
    idx, ions = db.idx_sorted(), orc.prepare_ions(w["prot"].seq)
    matched = 0
    for s in range(S):
        flags = orc.extract_peaks(X[s, :lens[s]])
        for k in range(N):
            if k >= cnt[s]:
                assert [int(g[s, k]) for g in got] == [0, 0, 0]
                continue
            p = int(idx[int(begin[s]) + int(pos[s, k])])
            want = orc.match_ions(ions, int(w["tc"][p]), int(w["tn"][p]), w["r"][p], w["mass"],
                                  int(zmax[s]), flags)
            assert tuple(int(g[s, k]) for g in got) == want, (s, k)
            matched += want[0] + want[1]
    assert matched > 0
