"""Training pairs at the sides where their solver changes: p in LDS with 256,
512 and 1,024 threads, p in memory, the per-iteration kernel; odd and even
sides, more iterations than one launch runs, anisotropic operators."""
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


def apply_a(u, rx, ry):
    v = np.pad(u, ((0, 0), (1, 1), (1, 1)))
    return (u - rx * (v[:, 1:-1, :-2] + v[:, 1:-1, 2:] - 2.0 * u) - ry * (v[:, :-2, 1:-1] + v[:, 2:, 1:-1] - 2.0 * u))


@pytest.mark.parametrize("n,rx,ry", [(2, 5.0, 5.0), (3, 5.0, 1.0), (63, 40.0, 40.0), (64, 40.0, 3.0), (65, 40.0, 40.0),
                                     (90, 60.0, 60.0), (91, 60.0, 9.0), (127, 80.0, 80.0), (128, 3000.0, 3000.0),
                                     (129, 90.0, 90.0), (192, 4000.0, 500.0), (193, 100.0, 100.0)])
def test_pairs_solve_their_system(pk, ctx, n, rx, ry):
    ns, tol = 5, 1e-10
    R, E, its, rc = pk.training_set(ctx, ns, n, rx, reltol=tol, seed=7, ratio_y=ry)
    assert rc == 0 and its >= 1
    r, e = (v.get().reshape(ns, n, n) for v in (R, E))
    res = np.linalg.norm((apply_a(e, rx, ry) - r).reshape(ns, -1), axis=1)
    # the recurrence's residual reaches tol; the true one follows it to the
    # rounding of A e, eps * |A| |e| <= 2.2e-16 * (1 + 8 max(r)) |e| per cell
    eps = 2.2e-16 * (1.0 + 8.0 * max(rx, ry)) * np.linalg.norm(e.reshape(ns, -1), axis=1)
    assert (res <= 1.01 * tol * np.linalg.norm(r.reshape(ns, -1), axis=1) + 4.0 * eps).all()
    if n in (128, 192):
        assert its > 256  # more than one launch
    # the same pairs again, and as the first of a smaller set
    R2, E2, its2, _ = pk.training_set(ctx, 2, n, rx, reltol=tol, seed=7, ratio_y=ry)
    np.testing.assert_array_equal(R2.get().reshape(2, n, n), r[:2])
    np.testing.assert_array_equal(E2.get().reshape(2, n, n), e[:2])
