"""The multigrid cycle on register tiles at the edges of the tiles (128
columns, 32 or 64 rows less the halo), of the levels that run in one
workgroup and of the sweep counts that run on tiles: bitwise the oracle's
cycle, also into its own input vector and with unaligned vectors."""
import ctypes

import numpy as np
import pytest

import oracle_lib as O
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


KINDS = {1: ("MMS_DIRICHLET", "MMS"), 0: ("CEDA_PERIODIC", "CEDA")}

# one tile; one column or row past a tile; several of both; more rows than
# columns; the tall tiles (R = 4) of a level with over 256 of them; the
# single-workgroup levels at their limit and a coarsest level too large for it
SHAPES = [(1, 128, 32), (1, 129, 33), (1, 127, 21), (1, 64, 300), (1, 250, 41), (1, 1100, 1501), (1, 32, 32),
          (1, 33, 33), (1, 2000, 3), (0, 128, 64), (0, 260, 96), (0, 118, 500), (0, 1200, 1504), (0, 32, 32), (0, 66, 50)]


@pytest.mark.parametrize("kind,nx,ny", SHAPES)
def test_cycle_is_bitwise(pk, ctx, kind, nx, ny):
    gamma = 1e-3
    kw = dict(nx=nx, ny=ny, kx=1.0, ky=0.4, inhomogeneous=1 - kind)
    G = pk.Problem(ctx, getattr(pk, KINDS[kind][0]), **kw)
    P = O.OracleProblem(getattr(O, KINDS[kind][1]), **kw)
    r = np.random.default_rng(nx + ny).standard_normal(P.n)
    R, Z = G.vector(r), G.vector()
    for relax, nu in [(2, 2)] if nx * ny > 100000 else [(2, 2), (3, 1), (2, 0), (2, 4), (3, 5)]:
        assert G.mg_options(relax, nu) == 0 and G.mg_psetup(gamma) == 0
        ref = P.mg_apply(gamma, r, relax, nu)[0]
        for _ in range(2):  # a replay after other work on the same buffers
            assert G.mg_psolve(R, Z) == 0
            np.testing.assert_array_equal(Z.get(), ref, err_msg=f"{relax} {nu}")
        np.testing.assert_array_equal(R.get(), r)
    assert G.mg_psolve(R, R) == 0  # into its own input
    np.testing.assert_array_equal(R.get(), ref)


def test_unaligned_vectors(pk, ctx):
    nx, ny, gamma = 140, 70, 1e-3
    G = pk.Problem(ctx, pk.MMS_DIRICHLET, nx=nx, ny=ny)
    P = O.OracleProblem(O.MMS, nx=nx, ny=ny)
    r = np.random.default_rng(3).standard_normal(P.n)
    pools = [pk.Vector(ctx, n=P.n + 1) for _ in range(2)]
    pools[0].set(np.concatenate([[0.0], r]))

    def shifted(v):  # an N_Vector 8 bytes into an allocation
        at = ctypes.cast(pk.lib().N_VGetDeviceArrayPointer(v.h), ctypes.c_void_p).value + 8
        return pk.Vector(ctx, handle=pk.lib().N_VMake_HipNative(P.n, ctypes.c_void_p(at), ctx.h))

    R, Z = (shifted(v) for v in pools)
    assert G.mg_psetup(gamma) == 0 and G.mg_psolve(R, Z) == 0
    np.testing.assert_array_equal(pools[1].get()[1:], P.mg_apply(gamma, r)[0])
