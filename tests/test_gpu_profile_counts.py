"""dm_profile_read counts launches: one per column of a product of a few columns,
whichever kernel serves it."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
K0 = 2 * math.pi / 0.1


@pytest.mark.parametrize("cells", [6, 33])  # one launch with gather and scatter inside, and apart
def test_products_are_counted_per_column(dm, cells):
    ctx = dm.Context()
    m = dm.make_rect_plate(cells / 120, cells / 120, cells, cells, ctx=ctx)
    r = dm.build_rwg(m)
    forms = dict(gemv_z64=dm.DM_Z64, gemv_z32=dm.DM_Z32, symv_z64=dm.DM_Z64P, symv_z32=dm.DM_Z32P)
    Z = dm.assemble_Z_efie(m, r, K0, forms=sum(forms.values()), device=True, max_output_bytes=None)
    X = np.ones((r.nedges, 5), complex)
    for form in forms.values():
        Z.matmul(X, form=form)  # the tuner's launches are behind
    ctx.profile(True)
    for name, form in forms.items():
        ctx.profile_reset()
        Z.matmul(X, form=form)
        Z.matmul(X[:, :2], form=form)
        assert ctx.profile_read(name)[0] == 7
