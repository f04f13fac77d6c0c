"""The batch engine's register tiles on the GPU: the default batch must give
bitwise the states and the counts of the batch on marching tiles of one stage
per pass, at sides around the edges of a tile (128 columns by 64 or 32 rows,
104 by 42 or 10 of them owned where there is a halo), odd and even, both
boundary kinds in one batch, adaptive and fixed steps, with few tiles (32-row
tiles) and many (64-row ones), and over several sub-batches of 4M cells."""
import numpy as np
import pytest

from hiplib import package

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def pk():
    return package()


@pytest.fixture(scope="module")
def ctx(pk):
    c = pk.Context()
    yield c
    c.close()


def run(pk, ctx, plist, method, marching, fixed, tout):
    B = pk.Batch(ctx, plist, method)
    B.SetTolerances(1e-5, 1e-10)
    B.SetMaxNumSteps(100000)
    if marching:
        assert B.SetStagesPerPass(1) == 0
    if fixed:
        B.SetFixedStep(fixed)
    assert B.evolve(tout) == 0
    out = [(B.time(k), B.stats(k), B.solution(k)) for k in range(len(plist))]
    B.release()
    return out


def check(pk, ctx, plist, method, fixed, tout):
    a = run(pk, ctx, plist, method, False, fixed, tout)
    b = run(pk, ctx, plist, method, True, fixed, tout)
    for k, (x, y) in enumerate(zip(a, b)):
        assert x[0] == y[0] and x[1] == y[1], plist[k]
        assert np.isfinite(x[2]).all()
        np.testing.assert_array_equal(x[2], y[2], err_msg=str(plist[k]))


def prob(kind, nx, ny):
    k = 0.1 * (1 + (7 * nx + 3 * ny) % 40)
    return dict(kind=kind, nx=nx, ny=ny, kx=k, ky=4.2 - k, inhomogeneous=ny % 2 if kind == 0 else 0)


FEW = [(1, 128, 64), (1, 129, 64), (1, 128, 65), (1, 127, 32), (1, 126, 33), (1, 2, 2), (1, 3, 64), (0, 2, 3),
       (0, 104, 42), (0, 105, 43), (0, 77, 10), (0, 31, 11)]
MANY = [(1, 209, 421), (1, 208, 420), (1, 313, 85), (0, 209, 421), (0, 312, 419), (0, 130, 841), (1, 65, 1000)]


@pytest.mark.parametrize("fixed", [0.0, 4e-4])
@pytest.mark.parametrize("shapes", [FEW, MANY, [(1, 257, 129)]], ids=["few", "many", "one"])
@pytest.mark.parametrize("method", ["rkc", "rkl"])
def test_batch_tiles_are_bitwise(pk, ctx, method, shapes, fixed):
    check(pk, ctx, [prob(*s) for s in shapes], method, fixed, 4e-3)


def test_batch_tiles_over_sub_batches(pk, ctx):
    check(pk, ctx, [prob(1, 1501, 1000), prob(0, 1400, 1300), prob(1, 1600, 1203), prob(0, 40, 40)], "rkl", 1e-4, 3e-4)
