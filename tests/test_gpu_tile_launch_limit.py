"""Register tiles on grids so tall that a tile shape would need 2^32 threads or
more in one launch: such a shape is refused, the tuning passes over it, and the
fused path still runs, with the result of one kernel per stage."""
import pytest

from hiplib import package

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def pk():
    return package()


@pytest.fixture()
def ctx(pk):
    c = pk.Context()
    yield c
    c.close()


def test_shapes_past_the_limit_are_refused(pk, ctx):
    # tiles of five wavefronts with a row each that own one row: 320 threads a row
    assert 320 * 13421772 < 2 ** 32 <= 320 * 13421773
    for ny, rc in ((13421772, 0), (13421773, -1)):
        G = pk.Problem(ctx, pk.MMS_DIRICHLET, nx=2, ny=ny)
        assert G.set_tile(1, 1, 5) == rc
        assert G.get_tile() == ((1, 1, 5) if rc == 0 else (0, 0, 0))
        assert G.set_tile(1, 4, 16) == 0  # 60 rows
        G.destroy()


def test_tuning_passes_over_them(pk, ctx):
    # tiles of twelve wavefronts with a row each for three stages own four rows
    nx, ny = 2, 23000000
    assert 768 * (ny // 4) >= 2 ** 32
    G = pk.Problem(ctx, pk.MMS_DIRICHLET, nx=nx, ny=ny)
    assert G.set_tile(3, 1, 12) == -1
    lam, _ = G.dom_eig()
    out = []
    for tuned in (True, False):
        if tuned:
            assert G.autotune(1) == 0
        else:
            assert G.set_config(2, 0, 32, 0) == 0
        I = pk.Integrator(G, "rkl", G.initial())
        I.ARKodeSetFixedStep(15.0 ** 2 / (2.0 * abs(lam)))
        assert I.LSRKStepSetDiffusionFastPath(G.h, 0) == 0
        flag, t = I.evolve(1.0, pk.ARK_ONE_STEP)
        assert flag == 0
        out.append(I.y)
        I.free()
    L = pk.lib()
    assert L.N_VMaxNorm(out[0].h) > 0.5
    L.N_VLinearSum(1.0, out[0].h, -1.0, out[1].h, out[1].h)
    assert L.N_VMaxNorm(out[1].h) == 0.0
