"""The tuned shapes of a size are kept for problems of the same kernels: a
periodic problem with constant coefficients and one with varying ones run
different tile kernels and are tuned separately, a second one of either kind is
not tuned again.  Tuning times hundreds of launches (tens of milliseconds), a
look-up none."""
import time

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


def tune_ms(pk, ctx, inhomogeneous):
    G = pk.Problem(ctx, pk.CEDA_PERIODIC, nx=186, ny=114, inhomogeneous=inhomogeneous)
    t = time.perf_counter()
    assert G.autotune() == 0
    ms = (time.perf_counter() - t) * 1e3
    G.destroy()
    return ms


def test_constant_and_varying_coefficients_are_tuned_separately(pk, ctx):
    first = [tune_ms(pk, ctx, k) for k in (0, 1)]
    again = [tune_ms(pk, ctx, k) for k in (0, 1)]
    assert min(first) > 5.0 and max(again) < 1.0
