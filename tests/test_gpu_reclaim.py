"""A handle freed while products on it are still queued: its memory waits in the
context, and an allocation that does not fit gets it back for the device (an
allocation beyond the whole device, so that it fails either way)."""
import ctypes as C
import math

import numpy as np
import pytest

from test_gpu_host_path import _free_bytes
from test_zz_no_alloc import _hip

pytestmark = pytest.mark.gpu
K0 = 2 * math.pi / 0.1


def test_failed_allocation_returns_what_is_kept(dm):
    ctx = dm.Context()
    m = dm.make_rect_plate(34 / 120, 34 / 120, 34, 34, ctx=ctx)
    r = dm.build_rwg(m)
    n = r.nedges
    Z = dm.assemble_Z_efie(m, r, K0, forms=dm.DM_Z64P, device=True, max_output_bytes=None)
    assert 64 << 20 < 8 * n * n < 128 << 20
    hip = _hip()
    dx = C.c_void_p()
    assert hip.hipMalloc(C.byref(dx), 16 * n) == 0
    x = np.ones(n, complex)
    assert hip.hipMemcpy(dx, x.ctypes.data_as(C.c_void_p), x.nbytes, 1) == 0
    Z.matmul(x, form=dm.DM_Z64P)
    held = _free_bytes()
    for _ in range(3000):  # about 0.1 s of work
        dm._check(dm.lib().dm_apply_noalloc(ctx.h, Z.h, dm.DM_Z64P, 0, dx, dx))
    Z.free()
    nomega = int(400e9 / (48 * n))
    rhat = np.tile([0.0, 0.0, 1.0], (nomega, 1))
    rc = dm.lib().dm_radiation_vectors(ctx.h, r.h, rhat.ctypes.data_as(C.c_void_p), nomega, K0, 376.7, 3,
                                       x.ctypes.data_as(C.c_void_p))
    assert rc == dm.DM_ERR_MEMORY
    # (the failed call's own copy of the directions stays with the context)
    assert _free_bytes() - held + rhat.nbytes >= 8 * n * n
    assert hip.hipFree(dx) == 0
    hip.hipGetLastError()
