"""A call refused for want of memory leaves no error behind: the next calls on the
context work, and give what they gave before."""
import ctypes as C
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
K0 = 2 * math.pi / 0.1


def test_calls_after_a_failed_allocation(dm):
    ctx = dm.Context()
    m = dm.make_rect_plate(0.3, 0.3, 30, 30, ctx=ctx)
    r = dm.build_rwg(m)
    Z = dm.assemble_Z_efie(m, r, K0, device=True)
    x = np.arange(r.nedges) + 1j
    y = Z.matmul(x)
    nomega = int(400e9 / (48 * r.nedges))  # radiation vectors beyond the device's memory
    rhat = np.tile([0.0, 0.0, 1.0], (nomega, 1))
    for _ in range(2):
        rc = dm.lib().dm_radiation_vectors(ctx.h, r.h, rhat.ctypes.data_as(C.c_void_p), nomega, K0, 376.7, 3,
                                           x.ctypes.data_as(C.c_void_p))
        assert rc == dm.DM_ERR_MEMORY
        assert np.array_equal(Z.matmul(x), y)
        Z2 = dm.assemble_Z_efie(m, r, K0, device=True)
        assert np.allclose(Z2.matmul(x), y, rtol=1e-12, atol=1e-12 * np.abs(y).max())
