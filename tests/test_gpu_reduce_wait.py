"""Reductions hand their results to the host through marked memory: results of
any bit pattern arrive, the mark's own included, and no slot keeps a value of
an earlier reduction, whatever the counts and lengths that follow each other."""
import ctypes

import numpy as np
import pytest

from hiplib import package

pytestmark = pytest.mark.gpu
MARK = 0xFFF8DEAD5EEDC0DE


@pytest.fixture(scope="module")
def pk():
    return package()


@pytest.fixture(scope="module")
def ctx(pk):
    c = pk.Context()
    yield c
    c.close()


@pytest.mark.parametrize("n", [1, 511, 1025, 70000])
def test_any_result_arrives(pk, ctx, n):
    one = pk.Vector.from_numpy(ctx, np.ones(n))
    for bits in (MARK, 0x7FF8000000000000, 0x7FF0000000000000, 0xFFF0000000000000, 0x8000000000000000):
        a = np.zeros(n)
        a.view(np.uint64)[n // 2] = bits
        x = pk.Vector.from_numpy(ctx, a)
        got = pk.lib().N_VDotProd(x.h, one.h)
        want = a[n // 2]
        assert np.isnan(got) if np.isnan(want) else got == want
        d = (ctypes.c_double * 9)(*[7.0] * 9)
        Y = (ctypes.c_void_p * 9)(*[getattr(one.h, "value", one.h)] * 9)
        assert pk.lib().N_VDotProdMulti(9, x.h, Y, d) == 0
        assert all(np.isnan(v) if np.isnan(want) else v == want for v in d)


def test_results_of_alternating_reductions(pk, ctx):
    """Whole numbers, so that every order of summation gives the same value."""
    rng = np.random.default_rng(3)
    vecs = {}
    for n in (1, 300, 5000, 200000):
        a = rng.integers(-4, 5, (17, n)).astype(float)
        vecs[n] = (a, a @ a.T, [pk.Vector.from_numpy(ctx, v) for v in a])
    for _ in range(400):
        n = int(rng.choice(list(vecs)))
        a, dots, vs = vecs[n]
        i, m = int(rng.integers(17)), int(rng.choice([1, 2, 3, 5, 8, 9, 16, 17]))
        ids = rng.integers(0, 17, m)
        Y = (ctypes.c_void_p * m)(*[getattr(vs[j].h, "value", vs[j].h) for j in ids])
        d = (ctypes.c_double * m)()
        assert pk.lib().N_VDotProdMulti(m, vs[i].h, Y, d) == 0
        assert list(d) == [dots[i, j] for j in ids]
        assert pk.lib().N_VMaxNorm(vs[i].h) == np.abs(a[i]).max()
