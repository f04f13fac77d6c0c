"""A batch's vectors and tables share device allocations: batches made and
released in any order keep their states, their memory is given back, a creation
that fails half-way gives back what it took, and batches on several threads do
not disturb each other."""
import threading

import numpy as np
import pytest
import torch

from hiplib import package

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def pk():
    return package()


def plist(n, side):
    # sides up to 1500: a vector of 18 MB is allocated by itself
    return [dict(kind=1, nx=side + 7 * k, ny=side, kx=0.2 + 0.1 * k, ky=1.0) for k in range(n)]


def solve(B, n, tout):
    B.SetTolerances(1e-5, 1e-10)
    assert B.evolve(tout) == 0
    return [B.solution(k) for k in range(n)]


def free_mb():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0] / 2 ** 20


@pytest.mark.parametrize("n,side", [(1, 2), (40, 60), (3, 1500)])
def test_release_order_and_memory(pk, n, side):
    ctx = pk.Context()
    tout = 1e-4
    want = solve(pk.Batch(ctx, plist(n, side), "rkc"), n, tout)  # released by the collector
    import gc
    gc.collect()
    before = free_mb()
    a, b, c = (pk.Batch(ctx, plist(n, side), "rkc") for _ in range(3))
    got = [solve(b, n, tout)]
    b.release()
    d = pk.Batch(ctx, plist(n, side), "rkc")
    got.append(solve(a, n, tout))
    a.release()
    got += [solve(c, n, tout), solve(d, n, tout)]
    d.release()
    c.release()
    for g in got:
        for x, y in zip(g, want):
            np.testing.assert_array_equal(x, y)
    assert free_mb() > before - 8
    ctx.close()


def test_failed_creation_gives_memory_back(pk):
    ctx = pk.Context()
    bad = plist(30, 200) + [dict(kind=1, nx=1, ny=5)]
    before = free_mb()
    for _ in range(3):
        with pytest.raises(Exception):
            pk.Batch(ctx, bad, "rkc")
    assert free_mb() > before - 8
    ctx.close()


def test_threads(pk):
    out = {}

    def work(t):
        ctx = pk.Context()
        for r in range(3):
            B = pk.Batch(ctx, plist(12, 50 + t), "rkl")
            out[t, r] = solve(B, 12, 1e-3)
            B.release()
        ctx.close()

    ts = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for t in range(4):
        for r in range(1, 3):
            for x, y in zip(out[t, 0], out[t, r]):
                np.testing.assert_array_equal(x, y)
