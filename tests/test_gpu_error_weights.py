"""Error weights and the STS error test of the vector path in fused kernels: the
step sequence and state must be bitwise those of the stage-table path, whose
error test is the separate kernel; a zero absolute tolerance keeps its check of
the weights; weights follow a change of tolerances between steps."""
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


def run(pk, ctx, kind, nx, ny, method, atol, fast, y0=None):
    G = pk.Problem(ctx, kind, nx=nx, ny=ny, kx=0.7, ky=1.9)
    I = pk.Integrator(G, method, G.initial() if y0 is None else G.vector(y0))
    I.ARKodeSStolerances(1e-4, atol)
    if fast:
        assert I.LSRKStepSetDiffusionFastPath(G.h, 0) == 0
    out = []
    for k in range(8):
        if k == 4 and atol > 0.0:
            I.ARKodeSStolerances(1e-6, 10.0 * atol)
        flag, t = I.evolve(1.0, pk.ARK_ONE_STEP)
        out.append((flag, t))
        if flag:
            break
    y, s = I.y.get(), I.stats()
    I.free()
    return out, y, {k: s[k] for k in ("nst", "attempts", "nfe", "netf", "stage_max")}


@pytest.mark.parametrize("method", ["rkc", "rkl"])
@pytest.mark.parametrize("kind,nx,ny", [(1, 2, 2), (1, 31, 33), (1, 64, 64), (0, 45, 30), (0, 128, 100)])
def test_vector_path_equals_stage_table_path(pk, ctx, kind, nx, ny, method):
    a = run(pk, ctx, kind, nx, ny, method, 1e-10, False)
    b = run(pk, ctx, kind, nx, ny, method, 1e-10, True)
    assert a[0] == b[0] and a[2] == b[2]
    np.testing.assert_array_equal(a[1], b[1])


def test_zero_absolute_tolerance(pk, ctx):
    y0 = np.full(30 * 30, 2.0)
    out, y, _ = run(pk, ctx, 0, 30, 30, "rkc", 0.0, False, y0)
    assert all(flag == 0 for flag, _ in out) and np.isfinite(y).all()
    y0[17] = 0.0  # a weight of 1 / 0
    out, _, _ = run(pk, ctx, 0, 30, 30, "rkc", 0.0, False, y0)
    assert out[0][0] == -22
