"""Weight gradients of the learned network against the oracle, layer by layer, at
the edges of the kernel's tasks: rows of fewer or one more pixel than a
16-pixel block, chains shorter and one longer than a task's eight rows, a
dilation above the grid's height, one image and several."""
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


# products of BF16 numbers summed in FP32 on both sides in another order: 1e-6;
# an activation that rounds the other way in BF16 moves its products by 2^-8,
# as rarely as in the whole-gradient tests, whose bound is 1e-2.  A missing or
# doubled border row or column of these small images is 1/ny or 1/nx: over 3e-2.
TOL = 1e-2


@pytest.mark.parametrize("sym,dil", [(True, (1, 3, 9, 27)), (True, (2,)), (False, (1, 1, 1, 1)), (False, (3, 5))])
@pytest.mark.parametrize("nb,nx,ny", [(1, 16, 8), (3, 15, 9), (1, 17, 30), (2, 31, 17), (5, 5, 3)])
def test_weight_gradients_match_oracle(pk, ctx, sym, dil, nb, nx, ny):
    ratio = 25.0
    scale = 1.0 / (1.0 + 4.0 * ratio)
    net = pk.LearnedPrec(ctx, dil, symmetric=sym)
    rng = np.random.default_rng(nx * 100 + ny)
    p = (0.2 * rng.standard_normal(net.nparams)).astype(np.float32)
    net.set_params(p)
    p = net.params()
    net.set_output_scale(scale)
    r, e = rng.standard_normal(nb * nx * ny), rng.standard_normal(nb * nx * ny)
    # e.r > 0 in every image: r = e plus noise
    r = e + 0.3 * r
    R, E = pk.Vector.from_numpy(ctx, r), pk.Vector.from_numpy(ctx, e)
    _, g = net.loss_grad(nb, nx, ny, ratio, R, E)
    _, ref, _ = O.lp_lossgrad(dil, p, scale, nb, nx, ny, ratio, r, e, emu=1, **({"sym": True} if sym else {}))
    off = 0
    for l in range(len(dil)):
        cin, cout = (1 if l == 0 else 16), (1 if l == len(dil) - 1 and not sym else 16)
        for n in (cout * cin * 9, cout):
            a, b = g[off:off + n], ref[off:off + n]
            assert np.linalg.norm(a - b) <= TOL * np.linalg.norm(b), (l, n)
            off += n
    net.release()
