"""The fused error weights and STS error test against the vector operations they
stand for: a run whose vectors carry a replaced operation (a forwarding callback
in their operations table) forms weights, error vector and norm by the single
operations, and must take the same steps to the same state.  The weighted norm
is reduced in the same tree and the weights and error are formed by the same
operations per entry, so the two are bitwise equal."""
import ctypes

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


ABS, WRMSNORM = 16, 21  # positions in the operations table


def replace(pk, v, slot, calls):
    """Puts a callback that forwards to the operation into v's table; its clones
    copy the table."""
    ops = ctypes.cast(v.h, ctypes.POINTER(ctypes.c_void_p))[1]
    table = ctypes.cast(ops, ctypes.POINTER(ctypes.c_void_p))
    types = {ABS: ctypes.CFUNCTYPE(None, ctypes.c_void_p, ctypes.c_void_p),
             WRMSNORM: ctypes.CFUNCTYPE(ctypes.c_double, ctypes.c_void_p, ctypes.c_void_p)}
    native = types[slot](table[slot])

    def forward(*args):
        calls.append(slot)
        return native(*args)

    cb = types[slot](forward)
    table[slot] = ctypes.cast(cb, ctypes.c_void_p).value
    return cb  # alive as long as the vectors


def run(pk, ctx, kind, nx, ny, method, slot):
    G = pk.Problem(ctx, kind, nx=nx, ny=ny, kx=0.7, ky=1.9)
    y0 = G.vector(0.5 + np.random.default_rng(nx + ny).random(G.n))
    calls = []
    keep = replace(pk, y0, slot, calls) if slot else None
    I = pk.Integrator(G, method, y0)
    I.ARKodeSStolerances(1e-4, 1e-9)
    if method == "dirk":
        I.analytic_jtimes()
    out = []
    for k in range(8):
        if k == 4:
            I.ARKodeSStolerances(1e-6, 1e-8)
        out.append(I.evolve(1.0, pk.ARK_ONE_STEP))
        assert out[-1][0] == 0
    y, s = I.y.get(), I.stats()
    I.free()
    I.y.release()
    y0.release()
    del keep
    return out, y, {k: s[k] for k in ("nst", "attempts", "nfe", "netf", "stage_max", "nli")}, calls


@pytest.mark.parametrize("method", ["rkc", "rkl", "dirk"])
@pytest.mark.parametrize("kind,nx,ny", [(1, 2, 2), (1, 31, 33), (1, 200, 130), (0, 45, 30), (0, 128, 100)])
def test_fused_error_test_equals_the_operations(pk, ctx, kind, nx, ny, method):
    a = run(pk, ctx, kind, nx, ny, method, None)
    assert not a[3]
    for slot in (ABS, WRMSNORM):
        b = run(pk, ctx, kind, nx, ny, method, slot)
        assert len(b[3]) >= 8  # at least one a step
        assert a[0] == b[0] and a[2] == b[2]
        np.testing.assert_array_equal(a[1], b[1])
