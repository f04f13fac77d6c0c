"""Register-tile passes on the GPU: the fused path on tiles must give bitwise the
trajectory of the fused path with one kernel per stage, for every tile shape,
at grid sides around the edges of a tile, its halo and its lanes, odd and even,
both boundary kinds, adaptive and fixed steps."""
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


def solve(pk, ctx, kind, nx, ny, method, tile, fixed, steps=6):
    """A few steps of up to about 30 stages from a rough state."""
    G = pk.Problem(ctx, kind, nx=nx, ny=ny, kx=1.3, ky=0.6, inhomogeneous=1 if kind == 0 and fixed else 0)
    G.autotune(1)
    assert G.set_config(2, 0, 32, 0) == 0  # one kernel per stage, no tiles
    if tile:
        assert G.set_tile(*tile) == 0 and G.get_tile() == tile
    rng = np.random.default_rng(nx * 31 + ny)
    y0 = G.vector(0.5 + rng.random(G.n))
    lam, _ = G.dom_eig()
    h = 20.0 ** 2 / (2.0 * abs(lam))
    I = pk.Integrator(G, method, y0)
    I.ARKodeSStolerances(1e-2, 1e-3)
    if fixed:
        I.ARKodeSetFixedStep(h)
        I.LSRKStepSetDomEigSafetyFactor(2.0)
    else:
        I.ARKodeSetInitStep(h)
    assert I.LSRKStepSetDiffusionFastPath(G.h, 1) == 0
    for _ in range(steps):
        flag, t = I.evolve(1e3, pk.ARK_ONE_STEP)
        assert flag == 0
    y, s = I.y.get(), I.stats()
    I.free()
    assert np.isfinite(y).all()
    return t, y, {k: s[k] for k in ("nst", "attempts", "nfe", "stage_max")}


# K up to the deepest pass; tiles of 4 to 64 rows
TILES = [(1, 1, 4), (3, 1, 16), (4, 2, 8), (8, 2, 16), (5, 4, 12), (10, 4, 16), (12, 4, 16), (7, 4, 5)]
# within one strip and row block, at their edges, over several of both
SHAPES = [(1, 128, 64), (1, 127, 65), (1, 130, 63), (1, 300, 200), (1, 129, 33), (1, 2, 2), (1, 64, 7),
          (0, 128, 64), (0, 77, 65), (0, 301, 131), (0, 2, 3), (0, 256, 30)]


@pytest.mark.parametrize("kind,nx,ny", SHAPES)
def test_tile_passes_are_bitwise(pk, ctx, kind, nx, ny):
    for method, fixed in (("rkc", False), ("rkl", True)):
        base = solve(pk, ctx, kind, nx, ny, method, None, fixed)
        for tile in TILES:
            G = pk.Problem(ctx, kind, nx=nx, ny=ny)
            ok = G.set_tile(*tile) == 0
            rows = tile[1] * tile[2]
            # a tile needs a row inside its halo, unless it holds the whole domain
            assert ok == (rows > 2 * (tile[0] + 1) or (kind == 1 and ny <= rows))
            if not ok:
                continue
            got = solve(pk, ctx, kind, nx, ny, method, tile, fixed)
            assert got[0] == base[0] and got[2] == base[2], (method, tile)
            np.testing.assert_array_equal(got[1], base[1], err_msg=f"{method} {tile}")


def test_tile_shapes_are_checked(pk, ctx):
    G = pk.Problem(ctx, pk.MMS_DIRICHLET, nx=200, ny=200)
    for bad in ((13, 4, 16), (-1, 4, 16), (4, 3, 16), (4, 8, 8), (4, 4, 17), (4, 4, 0), (8, 1, 16)):
        assert G.set_tile(*bad) == -1, bad
    assert G.set_tile(8, 4, 16) == 0 and G.get_tile() == (8, 4, 16)
    assert G.set_config(2, 4, 16, 0) == 0 and G.get_tile() == (0, 0, 0)
    assert G.set_tile(8, 4, 16) == 0 and G.set_tile(0) == 0 and G.get_tile() == (0, 0, 0)
