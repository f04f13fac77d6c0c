"""The multigrid cycle forms its quotients from reciprocals: bitwise the oracle's
divisions also for huge entries, signed zeros and infinite or NaN ones, on the
tiles and in the single-workgroup levels (on a single level an infinity stays
one: there is no residual to make a NaN of it), and within the last bits of it for
entries near and below the smallest normal number."""
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


def special(name, n):
    rng = np.random.default_rng(11)
    v = rng.standard_normal(n)
    if name == "tiny":  # around 2^-970, below which a residual of a quotient underflows
        return v * np.exp2(rng.integers(-1000, -940, n).astype(float))
    if name == "subnormal":
        return v * 1e-310
    if name == "huge":
        return v * 1e300
    if name == "negative zeros":
        return np.where(v < 0.5, -0.0, v)
    v[n // 3] = np.inf
    if name == "both infinities":
        v[n // 2] = -np.inf
    if name == "nan":
        v[n // 4] = np.nan
    return v


NAMES = ["tiny", "subnormal", "huge", "negative zeros", "infinite", "both infinities", "nan"]
# a quotient is off by at most two units of the smallest subnormal or of its
# last place; a residual multiplies them by twice the diagonal (up to 165
# here), the other operations average them
QUANTA = 1e4 * 5e-324


@pytest.mark.parametrize("name", NAMES)
@pytest.mark.parametrize("kind,nx,ny,gamma", [(1, 200, 150, 1e-3), (1, 31, 30, 1e-3), (0, 256, 64, 1e-3),
                                              (0, 32, 32, 0.1), (1, 5, 5, 1e-3)])
def test_special_values(pk, ctx, kind, nx, ny, gamma, name):
    kw = dict(nx=nx, ny=ny, kx=1.0, ky=0.4, inhomogeneous=1 - kind)
    G = pk.Problem(ctx, pk.MMS_DIRICHLET if kind else pk.CEDA_PERIODIC, **kw)
    P = O.OracleProblem(O.MMS if kind else O.CEDA, **kw)
    r = special(name, P.n)
    with np.errstate(all="ignore"):
        ref = P.mg_apply(gamma, r, 2, 2)[0]
    Z = G.vector()
    assert G.mg_options(2, 2) == 0 and G.mg_psetup(gamma) == 0 and G.mg_psolve(G.vector(r), Z) == 0
    z = Z.get()
    if name in ("tiny", "subnormal"):
        assert np.abs(z - ref).max() <= 1e-12 * np.abs(ref).max() + QUANTA
        return
    nan = np.isnan(ref)
    np.testing.assert_array_equal(np.isnan(z), nan)
    np.testing.assert_array_equal(z[~nan].view(np.int64), ref[~nan].view(np.int64))
