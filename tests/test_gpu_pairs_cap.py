"""Training pairs that never converge (an infinite ratio makes every residual NaN)
stop at the solver's cap of 20,000 iterations, by one compute unit per pair and,
for sides over 192, by a launch per iteration."""
import ctypes

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


@pytest.mark.parametrize("n", [4, 5, 193])
def test_iteration_cap(pk, ctx, n):
    r, e = pk.Vector(ctx, n=2 * n * n), pk.Vector(ctx, n=2 * n * n)
    its = ctypes.c_int()
    rc = pk.lib().LearnedPrec_MakeTrainingSetXY(2, n, float("inf"), 1.0, 1e-12, 1, pk.dptr_of(r), pk.dptr_of(e),
                                               ctypes.byref(its), ctx.h)
    assert rc == 1 and its.value == 20000
