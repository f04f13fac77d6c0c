"""The sine fields of the training pairs at the edges of the synthesis' 64 x 64
tiles and 16-deep steps.  A mode's coefficient depends on the seed, the sample
and the mode alone and every sample holds the modes up to |k| = 4, so the sine
transform of a field must give the same low coefficients at every side, and
none beyond |k| = n."""
import numpy as np
import pytest

from hiplib import package

pytestmark = pytest.mark.gpu


def coefficients(pk, ctx, n, nsamp=5):
    """Sine coefficients of the even (not operator-applied) samples, and the
    bound on their rounding: a field is two sums of n products, each sum wrong
    by at most n eps of its terms' magnitudes, as are the two of the transform
    here, which scales a field error by at most (2 n / (n + 1))^2 < 4."""
    R, _, _, rc = pk.training_set(ctx, nsamp, n, 1.0, reltol=1e-3, seed=11)
    assert rc == 0
    r = R.get().reshape(nsamp, n, n)[::2]
    k = np.arange(1, n + 1)
    S = np.sin(np.pi * np.outer(k, k) / (n + 1))
    c = (S @ r @ S) * (2.0 / (n + 1)) ** 2
    tol = 4.0 * 4.0 * n * 2.2e-16 * np.abs(c).sum(axis=(1, 2))
    return c, tol


@pytest.mark.parametrize("n", [4, 5, 15, 16, 17, 48, 63, 64, 65, 80, 127, 128, 129, 193])
def test_low_modes_do_not_depend_on_the_side(n):
    pk = package()
    ctx = pk.Context()
    ref, rtol = coefficients(pk, ctx, 33)
    c, tol = coefficients(pk, ctx, n)
    m = min(n, 4)
    k = np.arange(1, n + 1)
    kk = np.sqrt(k[:, None] ** 2 + k[None, :] ** 2)
    low = kk[:m, :m] <= 4.0
    for a, b, t, u in zip(c, ref, tol, rtol):
        assert (np.abs(a[:m, :m] - b[:m, :m])[low] <= t + u).all()
        assert (np.abs(b[:m, :m])[low] > 100 * (t + u)).any()
        assert (np.abs(a)[kk > n] <= t).all()
    ctx.close()
