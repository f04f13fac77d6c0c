"""Weight gradients where one channel of a hidden layer overflows to infinity at a
few pixels, one of them in the last column of rows that end inside a 16-pixel
block: the following ReLU drops what the convolutions make of them, so only the
gradients of the weights that read that channel may be non-finite; all others
are the oracle's."""
import numpy as np
import pytest

import oracle_lib as O
from hiplib import package

pytestmark = pytest.mark.gpu

BAD = 3  # the channel that overflows
# as in the layer-by-layer gradient tests: BF16 activations that round the other way
TOL = 1e-2


@pytest.fixture(scope="module")
def pk():
    return package()


@pytest.fixture(scope="module")
def ctx(pk):
    c = pk.Context()
    yield c
    c.close()


@pytest.mark.parametrize("dil", [(1, 1, 1), (1, 2, 1)])
@pytest.mark.parametrize("nx,ny", [(40, 20), (33, 18), (48, 9)])
def test_infinite_activations_stay_in_their_channel(pk, ctx, nx, ny, dil):
    nb, ratio, scale = 2, 5.0, 1.0 / 21.0
    net = pk.LearnedPrec(ctx, dil)
    rng = np.random.default_rng(nx)
    W = [(0.2 * rng.standard_normal((co, ci, 3, 3)), np.zeros(co)) for co, ci in ((16, 1), (16, 16), (1, 16))]
    W[0][0][BAD] = 0.0
    W[0][0][BAD, 0, 1, 1] = 1e38
    W[1][0][:, BAD] = 0.0
    net.set_params(np.concatenate([np.concatenate([w.ravel(), b]) for w, b in W]).astype(np.float32))
    p = net.params()
    net.set_output_scale(scale)
    r = rng.uniform(0.5, 1.0, (nb, ny, nx))
    r[0, 3, nx - 1] = r[0, ny - 1, 5] = r[1, 4, 17] = 8.0  # 8e38 after the first layer
    e = 0.1 * r * rng.uniform(0.8, 1.2, r.shape)
    r, e = r.ravel(), e.ravel()
    loss, g = net.loss_grad(nb, nx, ny, ratio, pk.Vector.from_numpy(ctx, r), pk.Vector.from_numpy(ctx, e))
    with np.errstate(all="ignore"):
        ref_loss, ref, _ = O.lp_lossgrad(dil, p, scale, nb, nx, ny, ratio, r, e, emu=1)
    assert np.isfinite(ref_loss) and abs(loss - ref_loss) <= TOL * abs(ref_loss)
    off = 0
    for l, (w, b) in enumerate(W):
        reads_bad = np.zeros(w.shape, bool)
        if l == 1:
            reads_bad[:, BAD] = True
        a, c = g[off:off + w.size].reshape(w.shape)[~reads_bad], ref[off:off + w.size].reshape(w.shape)[~reads_bad]
        assert np.isfinite(c).all() and np.isfinite(a).all(), l
        assert np.linalg.norm(a - c) <= TOL * np.linalg.norm(c), l
        off += w.size
        a, c = g[off:off + b.size], ref[off:off + b.size]
        assert np.linalg.norm(a - c) <= TOL * np.linalg.norm(c), l
        off += b.size
    net.release()
