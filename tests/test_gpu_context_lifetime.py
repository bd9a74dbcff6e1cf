"""Handles outlive their context: freed after dm_destroy they give their memory
back, any other use of them is refused, and other contexts go on."""
import gc
import math

import numpy as np
import pytest

from test_gpu_host_path import _free_bytes

pytestmark = pytest.mark.gpu
K0 = 2 * math.pi / 0.1


def _handles(dm, ctx):
    m = dm.make_rect_plate(0.1, 0.1, 12, 12, ctx=ctx)
    r = dm.build_rwg(m)
    Z = dm.assemble_Z_efie(m, r, K0, forms=dm.DM_Z64 | dm.DM_Z64P, device=True)
    S = dm.NearFieldOperator(dm.build_nearfield_preconditioner(Z, m, r, 2.0 * float(np.mean(r.len))), Z)
    op = dm.matrixfree_efie_operator(m, r, K0)
    net = dm.MPNN(ctx=ctx)
    x = np.ones(r.nedges, complex)
    y = Z.matmul(x, form=dm.DM_Z64P)
    assert np.allclose(op @ x, y, rtol=1e-9, atol=1e-9 * np.abs(y).max())
    assert np.isfinite(S @ x).all()
    return m, r, Z, S, op, net


def test_handles_freed_after_their_context(dm):
    other = dm.Context()
    mo = dm.make_rect_plate(0.1, 0.1, 6, 6, ctx=other)
    Zo = dm.assemble_Z_efie(mo, dm.build_rwg(mo), K0, device=True)
    xo = np.arange(Zo.N) + 1j
    yo = Zo.matmul(xo)
    free0 = None
    for _ in range(3):
        ctx = dm.Context()
        m, r, Z, S, op, net = _handles(dm, ctx)
        ctx.close()
        with pytest.raises(ValueError, match="destroyed"):
            dm.build_rwg(m)
        with pytest.raises(ValueError, match="destroyed"):
            Z.to_numpy()
        for h in (net, S, Z, r, m):
            h.__del__()
        assert np.array_equal(Zo.matmul(xo), yo)
        free0 = free0 or _free_bytes()
    assert free0 - _free_bytes() <= 16 << 20


def test_handles_collected_in_any_order(dm):
    """A cycle: the collector runs the finalizers in an order of its own."""
    ctx = dm.Context()
    ring = [ctx, *_handles(dm, ctx)]
    ring.append(ring)
    del ctx, ring
    gc.collect()
