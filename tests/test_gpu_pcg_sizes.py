"""The fused PCG against the N_Vector PCG where its kernels change: grids below
one workgroup, around the count from which workgroups come in eights and the
cap of 1,024, odd and even rows; constant coefficients (z formed from r),
variable ones (z stored by the update), none and a callback; repeated solves,
whose batches follow the previous solve's length."""
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


def run(pk, ctx, kind, nx, ny, inh, precond, fused, reltol):
    G = pk.Problem(ctx, kind, nx=nx, ny=ny, kx=1.0, ky=0.7, inhomogeneous=inh)
    lam, _ = G.dom_eig()
    dt = 40.0 / abs(lam)
    I = pk.Integrator(G, "dirk", G.vector(0.5 + np.random.default_rng(nx + ny).random(G.n)), ls="cg", maxl=20000,
                      precond=precond)
    I.ARKodeSetFixedStep(dt)
    if reltol:
        I.ARKodeSetLSRelativeTolerance(reltol)
    I.analytic_jtimes()
    if fused:
        assert I.fused_pcg() == 0
    flag, _ = I.evolve(3 * dt)
    out = flag, I.y.get(), I.stats()
    I.free()
    return out


# 2 x 2 up to one workgroup; 7, 8 and 9 workgroups of 512 pairs; over 1,024
@pytest.mark.parametrize("kind,nx,ny", [(1, 2, 2), (0, 2, 3), (1, 31, 17), (0, 32, 16), (1, 112, 64), (0, 128, 64), (1, 130, 70),
                                        (0, 129, 33), (1, 1100, 1000)])
@pytest.mark.parametrize("precond", [True, False, "mg"])
def test_sizes(pk, ctx, kind, nx, ny, precond):
    if precond == "mg" and kind == 0 and (nx % 2 or ny % 2):
        pytest.skip("the periodic hierarchy takes even sides")
    for inh in ((0, 1) if kind == 0 else (0,)):
        for reltol in ((1e-9, 0.0) if nx * ny < 100000 else (1e-6,)):
            a = run(pk, ctx, kind, nx, ny, inh, precond, False, reltol)
            b = run(pk, ctx, kind, nx, ny, inh, precond, True, reltol)
            assert a[0] == b[0] == 0
            assert a[2]["nni"] == b[2]["nni"] and abs(a[2]["nli"] - b[2]["nli"]) <= max(2, 0.01 * a[2]["nli"])
            # both stop at the same tolerance of the same system (as the other fused PCG tests bound them)
            assert np.abs(a[1] - b[1]).max() <= 1e-10 * np.abs(a[1]).max(), (inh, reltol)
