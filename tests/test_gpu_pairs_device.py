"""Training pairs whose solves need more LDS per workgroup than the default, on
every device of the process in turn: the kernel's attribute belongs to a device."""
import ctypes

import numpy as np
import pytest
import torch

from hiplib import package

pytestmark = pytest.mark.gpu


def test_pairs_on_every_device():
    pk = package()
    n, out = 100, []
    try:
        for dev in range(torch.cuda.device_count()):
            torch.cuda.set_device(dev)
            ctx = pk.Context()
            r, e = pk.Vector(ctx, n=n * n), pk.Vector(ctx, n=n * n)
            its = ctypes.c_int()
            rc = pk.lib().LearnedPrec_MakeTrainingSetXY(1, n, 50.0, 20.0, 1e-12, 3, pk.dptr_of(r), pk.dptr_of(e),
                                                       ctypes.byref(its), ctx.h)
            assert rc == 0
            out.append((r.get(), e.get(), its.value))
            r.release()
            e.release()
            ctx.close()
    finally:
        torch.cuda.set_device(0)
    for o in out[1:]:
        assert o[2] == out[0][2]
        np.testing.assert_array_equal(o[0], out[0][0])
        np.testing.assert_array_equal(o[1], out[0][1])
