"""Dense LU of singular matrices: bases with zero coefficients give zero rows and
columns, which stay zero through the elimination, so the solve is refused and
names the first such column (in the library's own order) whatever panel kernel
holds it: up to 256, 512, 1024, 2048, 4096 rows in registers, more in memory."""
import math
import re

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
K0 = 2 * math.pi / 0.1


@pytest.fixture(scope="module")
def plate(dm):
    m = dm.make_rect_plate(0.4, 0.35, 38, 38)
    return m, dm.build_rwg(m)


def _refused_column(dm, plate, n, zero):
    """1-based column that the direct solve of the first n bases names when the
    bases `zero` have zero coefficients."""
    m, r = plate
    c = np.ones(n)
    c[list(zero)] = 0.0
    sub = dm.rwg_from_arrays(m, r.tplus[:n], r.tminus[:n], r.vplus_opp[:n], r.vminus_opp[:n], r.len[:n],
                             r.area_plus[:n], r.area_minus[:n], evert=r.evert[:n], coeff_plus=c, coeff_minus=c)
    Z = dm.assemble_Z_efie(m, sub, K0, forms=dm.DM_Z64, device=True, mesh_precheck=False, max_output_bytes=None)
    with pytest.raises(ValueError, match="dense LU: matrix is singular") as e:
        dm.solve_forward(Z, np.ones((n, 3), complex), solver="direct")
    Z.free()
    return int(re.search(r"zero pivot (\d+)", str(e.value)).group(1))


@pytest.mark.parametrize("n", [1, 40, 250, 500, 1000, 2048, 2081, 4096, 4130])
def test_singular_matrix_is_refused(dm, plate, n):
    # bases spread over the matrix: their columns are found one by one, ...
    some = sorted({0, 1 % n, 7 % n, 8 % n, n // 3, n // 2, (3 * n) // 4, n - 1})
    where = [_refused_column(dm, plate, n, [b]) for b in some]
    assert len(set(where)) == len(some) and min(where) >= 1 and max(where) <= n
    # ... the first of several is named, and a zero matrix fails at once
    for a in range(len(some) - 1):
        assert _refused_column(dm, plate, n, some[a:]) == min(where[a:])
    assert _refused_column(dm, plate, n, range(n)) == 1
