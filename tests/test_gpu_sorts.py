"""The stable sorts at the sizes where the way they are done changes, and the row product at
remainders of its steps."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 63, 64, 65, 383, 384, 385, 1023, 1024, 1025, 2049, 8191, 8192, 8193, 12289, 16384,
         16385, 100003]


def order_key(f):
    """Total order of the float bits: -0 before +0, as a radix sort has it."""
    u = f.view(np.uint32)
    return np.where(u & 0x80000000, ~u, u | np.uint32(0x80000000))


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("ties", [False, True])
def test_sorts_are_stable_at_every_size(n, ties):
    import hfx_amd
    from hfx_amd import pipeline as pl

    L = hfx_amd.lib()
    rng = np.random.default_rng(n + ties)
    keys = rng.normal(0, 1000, n).astype(np.float32)
    if ties:
        keys = rng.choice(np.array([-np.inf, -3.5, -0.0, 0.0, 1e-40, 2.0, np.inf, 7e8], np.float32), n)
    vals = rng.permutation(n).astype(np.uint32)
    up = np.argsort(order_key(keys), kind="stable")
    down = np.argsort(~order_key(keys), kind="stable")
    for name, o, index in (("sort_b40c_f", up, False), ("sort_val_f", up, False),
                           ("sort_rf", down, False), ("sort_idx_f", up, True),
                           ("sort_idx_rf", down, True)):
        k, v = pl.dev(keys), pl.dev(vals)
        if index:
            getattr(L, name)(k.p, v.p, n, 7)
        else:
            getattr(L, name)(k.p, v.p, n)
        pl.sync()
        want = o.astype(np.uint32) + 7 if index else vals[o]
        assert np.array_equal(pl.host(v, np.uint32, n), want), name
        assert np.array_equal(pl.host(k, np.uint32, n), keys[o].view(np.uint32)), name


@pytest.mark.parametrize("n", [1, 63, 64, 511, 512, 513, 1471, 2065])
def test_row_products(n):
    """|y - exact| <= (n / 64 + 7) roundings of a lane's sum and the lanes' tree."""
    import hfx_amd
    from hfx_amd import pipeline as pl

    rng = np.random.default_rng(n)
    m = 37
    A, x = rng.normal(0, 1, (m, n)).astype(np.float32), rng.normal(0, 1, n).astype(np.float32)
    ta, tx, ty = pl.dev(A), pl.dev(x), pl.empty(4 * m)
    hfx_amd.lib().mvm_ff(None, ty.p, ta.p, tx.p, m, n)
    pl.sync()
    a, b = A.astype(np.float64), x.astype(np.float64)
    bound = (n / 64 + 8) * 2.0**-23 * (np.abs(a) @ np.abs(b))
    assert (np.abs(pl.host(ty, np.float32, m) - a @ b) <= bound).all()
