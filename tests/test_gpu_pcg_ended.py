"""Fused PCG solves that end inside a batch of enqueued iterations: after a long
solve the next one is enqueued at that length and ends early in it.  Whatever
the batches, the iterate, the iteration counts and the step are bitwise those
of a solver that has no previous solve."""
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


def integrator(pk, G, y0, t0, dt, precond):
    I = pk.Integrator(G, "dirk", y0, t0=t0, ls="cg", maxl=20000, precond=precond)
    I.ARKodeSetFixedStep(dt)
    I.ARKodeSetLinear(1)
    I.ARKodeSetLSRelativeTolerance(1e-9)
    I.analytic_jtimes()
    assert I.fused_pcg() == 0
    return I


@pytest.mark.parametrize("precond", [True, False, "mg"])
@pytest.mark.parametrize("kind,nx,ny,inh", [(1, 700, 600, 0), (0, 301, 211, 1), (0, 64, 40, 0)])
def test_end_inside_a_batch(pk, ctx, kind, nx, ny, inh, precond):
    if precond == "mg" and kind == 0 and nx % 2:
        pytest.skip("the periodic hierarchy takes even sides")
    G = pk.Problem(ctx, kind, nx=nx, ny=ny, inhomogeneous=inh)
    lam, _ = G.dom_eig()
    long, short = 400.0 / abs(lam), 2.0 / abs(lam)
    for rep in range(3):
        A = integrator(pk, G, G.vector(0.5 + np.random.default_rng(rep).random(G.n)), 0.0, long, precond)
        assert A.evolve(1e3, pk.ARK_ONE_STEP)[0] == 0
        A.ARKodeSetFixedStep(short)  # from the step after the next one on
        flag, t = A.evolve(1e3, pk.ARK_ONE_STEP)
        assert flag == 0
        before = A.stats()
        B = integrator(pk, G, A.y, t, short, precond)
        flag, ta = A.evolve(1e3, pk.ARK_ONE_STEP)
        assert flag == 0
        flag, tb = B.evolve(1e3, pk.ARK_ONE_STEP)
        assert flag == 0 and ta == tb
        a, b = A.stats(), B.stats()
        for k in ("nli", "npsolve", "njtimes"):
            if k in a:
                assert a[k] - before[k] == b[k], k
        assert b["nli"] < before["nli"]
        np.testing.assert_array_equal(A.y.get(), B.y.get())
        A.free()
        B.free()
