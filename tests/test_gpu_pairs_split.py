"""Training pairs at the sides where the solver keeps the first 18 * 1024 cells
of p in LDS and the others in memory: all of p still in LDS (135), the first
cells outside (136, 137), borders inside a thread's odd and even units, the
largest side."""
import numpy as np
import pytest

from hiplib import package

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,rx,ry", [(130, 900.0, 900.0), (135, 900.0, 90.0), (136, 90.0, 900.0), (137, 900.0, 900.0),
                                     (143, 20.0, 700.0), (160, 900.0, 300.0), (191, 900.0, 900.0)])
def test_split_pairs_solve_their_system(n, rx, ry):
    pk = package()
    ctx = pk.Context()
    ns, tol = 300, 1e-10  # more pairs than CUs
    R, E, its, rc = pk.training_set(ctx, ns, n, rx, reltol=tol, seed=5, ratio_y=ry)
    assert rc == 0 and its >= 1
    r, e = (v.get().reshape(ns, n, n) for v in (R, E))
    v = np.pad(e, ((0, 0), (1, 1), (1, 1)))
    ae = e - rx * (v[:, 1:-1, :-2] + v[:, 1:-1, 2:] - 2.0 * e) - ry * (v[:, :-2, 1:-1] + v[:, 2:, 1:-1] - 2.0 * e)
    res = np.linalg.norm((ae - r).reshape(ns, -1), axis=1)
    # the recurrence's residual reaches tol; the true one follows it to the
    # rounding of A e, eps * |A| |e| <= 2.2e-16 * (1 + 8 max(r)) |e| per cell
    eps = 2.2e-16 * (1.0 + 8.0 * max(rx, ry)) * np.linalg.norm(e.reshape(ns, -1), axis=1)
    assert (res <= 1.01 * tol * np.linalg.norm(r.reshape(ns, -1), axis=1) + 4.0 * eps).all()
    ctx.close()
