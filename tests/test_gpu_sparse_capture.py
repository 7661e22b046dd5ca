"""hfx_xcorr_sparse under a caller's capture: the graph outlives the theoretical rows that calls
outside it keep in the context."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_rows import FORMS, Spectra, database, reference, spectra

pytestmark = pytest.mark.gpu


def free_rows(pl):
    """What a shortage of memory does: an allocation that cannot be had takes the rows back."""
    from hfx_amd import lib

    p = C.c_void_p()
    assert lib().hfx_malloc(C.byref(p), 1 << 50) != 0


def test_a_graph_and_larger_calls_afterwards(orc):
    from hfx_amd import check, lib
    from hfx_amd import pipeline as pl

    hdb = database(pl, 100_003, seed=101, longest=20)
    x, lens, zmax, mass = spectra(pl, hdb, 6000, 600, seed=102)
    ref, exact, scale = reference(orc, hdb, x, lens, zmax, mass, 5)
    ctx, db, sp = pl.Ctx(0), pl.DeviceDB(hdb), Spectra(pl, x, lens, zmax, mass)
    t = [pl.dev(ref["off"].astype(np.uint64)), pl.dev(ref["begin"].astype(np.uint32)),
         pl.dev(ref["num"].astype(np.uint32))]

    def score(out, S, stream):
        d = type(sp.desc)(sp.desc.d_x, sp.desc.x_stride, sp.desc.d_len, sp.desc.d_zmax, sp.desc.d_mass, S)
        check(lib().hfx_xcorr_sparse(ctx.h, out.p, *[b.p for b in t], int(ref["off"][S]), C.byref(db.desc),
                                     C.byref(d), stream), "hfx_xcorr_sparse")

    half = 3000
    n = int(ref["off"][half])
    assert n > 600_000   # rows are taken outside a capture
    out, big = pl.empty(4 * n), pl.empty(4 * int(ref["off"][-1]))
    score(big, 6000, None)   # the tile table, 12 bytes a spectrum, is there for the largest call
    score(out, half, None)
    pl.sync()
    hip, s, g, run = C.CDLL("libamdhip64.so"), pl.Stream(), C.c_void_p(), C.c_void_p()
    assert hip.hipStreamBeginCapture(C.c_void_p(s.p), 1) == 0   # hipStreamCaptureModeThreadLocal
    score(out, half, s.p)
    assert hip.hipStreamEndCapture(C.c_void_p(s.p), C.byref(g)) == 0
    assert hip.hipGraphInstantiate(C.byref(run), g, None, None, C.c_size_t(0)) == 0
    bound = FORMS["fp32"][0] * scale + 1e-6 + 2.0**-24 * np.abs(exact)
    for _ in range(3):
        score(big, 6000, None)
        free_rows(pl)
        pl.sync()
        out.zero()
        pl.sync()
        assert hip.hipGraphLaunch(run, C.c_void_p(s.p)) == 0
        pl.sync()
        got = pl.host(out, np.float32, n)
        assert (np.abs(got - exact[:n]) <= bound[:n]).all()
        got = pl.host(big, np.float32, len(exact))
        assert (np.abs(got - exact) <= bound).all()
    assert hip.hipGraphExecDestroy(run) == 0 and hip.hipGraphDestroy(g) == 0
