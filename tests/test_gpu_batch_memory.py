"""What a batch takes of the device's memory, and when."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_rows import Spectra, database, spectra
from test_gpu_rowsets import free

pytestmark = pytest.mark.gpu

S = 16000


@pytest.fixture(scope="module")
def env():
    from hfx_amd import pipeline as pl

    hdb = database(pl, 20_000, seed=61, longest=12)
    x, lens, zmax, mass = spectra(pl, hdb, 200, 1024, seed=62)
    x, lens, zmax, mass = (np.tile(v, (S // 200,) + (1,) * (v.ndim - 1)) for v in (x, lens, np.minimum(zmax, 3), mass))
    return pl, pl.Ctx(0), pl.DeviceDB(hdb), Spectra(pl, x, lens, zmax, mass)


@pytest.mark.parametrize("form", ["FP32_SPARSE", "BF16X2_DENSE", "I8X3_DENSE"])
def test_a_plan_takes_what_required_bytes_says(env, form):
    from hfx_amd import check, lib

    pl, ctx, db, sp = env
    index = pl.PepIndex(ctx, db)

    def batch():
        b = pl.BatchSearch(ctx, db, sp, eps=3.0, topn=5, index=index)
        b.set_precision(getattr(b, form))
        b.run()
        return b

    first = batch()   # keeps the rows
    b = batch()       # and the allocator's pools are warm
    before = free(pl)
    del b
    took = free(pl) - before
    n = C.c_uint64()
    check(lib().hfx_batch_required_bytes(S, first.info()["scores"], 5, db.num_pep,
                                         getattr(first, form), C.byref(n)), "hfx_batch_required_bytes")
    # some thirty allocations, each rounded up to the driver's 2 MiB at most
    assert took <= n.value + (60 << 20)


@pytest.mark.parametrize("form", ["FP32_SPARSE", "BF16X2_DENSE", "I8X3_DENSE"])
def test_no_run_allocates_after_an_index_is_attached(env, form):
    from hfx_amd import check, lib

    pl, ctx, db, sp = env
    pl.BatchSearch(ctx, db, sp, eps=3.0, topn=5, index=pl.PepIndex(ctx, db)).run()  # code is loaded
    b = pl.BatchSearch(ctx, db, sp, eps=3.0, topn=5)
    b.set_precision(getattr(b, form))
    index = pl.PepIndex(ctx, db)
    check(lib().hfx_batch_use_index(b.h, index.h), "hfx_batch_use_index")
    before = free(pl)
    b.run()
    b.stream.sync()
    assert free(pl) == before
