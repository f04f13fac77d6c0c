"""Which kernels a batch runs on after its tile options were set: a chosen number
of stages per pass or of thin-phase rows stays in force when the tile height is
set back to automatic, and a tile height alone is taken back by it.  The
launches of the step groups tell the routes apart."""
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


def launches(pk, ctx, *calls):
    B = pk.Batch(ctx, [dict(kind=1, nx=60, ny=50), dict(kind=1, nx=41, ny=70)], "rkl")
    B.SetTolerances(1e-5, 1e-10)
    for name, *args in calls:
        assert getattr(B, name)(*args) == 0
    assert B.evolve(1e-3) == 0
    out = B.groups(), B.algorithmic_bytes()
    B.release()
    return out


def test_tile_height_set_back_to_automatic(pk, ctx):
    tiles = launches(pk, ctx)
    one = launches(pk, ctx, ("SetStagesPerPass", 1))
    thin = launches(pk, ctx, ("SetThinPhases", 0, 1))
    rows = launches(pk, ctx, ("SetTileRows", 8))
    assert len({tiles, one, thin}) == 3 and rows != tiles
    assert launches(pk, ctx, ("SetStagesPerPass", 1), ("SetTileRows", 0)) == one
    assert launches(pk, ctx, ("SetThinPhases", 0, 1), ("SetTileRows", 0)) == thin
    assert launches(pk, ctx, ("SetTileRows", 0), ("SetStagesPerPass", 1)) == one
    assert launches(pk, ctx, ("SetTileRows", 8), ("SetTileRows", 0)) == tiles
    assert launches(pk, ctx, ("SetStagesPerPass", 1), ("SetTileRows", 8), ("SetTileRows", 0)) == one
