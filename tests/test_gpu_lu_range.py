"""Dense LU of matrices whose pivots' squared magnitudes are subnormal or
overflow: the EFIE matrix scales with eta0, here by a power of two, so that
|pivot|^2 is near 2^-1060 and near 2^1050.  The solution scales back exactly; the
bound is that of the unscaled solves (backward error 8 n u)."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
K0 = 2 * math.pi / 0.1


@pytest.mark.parametrize("cells,n", [((8, 5), 33), ((14, 9), 300), ((24, 22), 1057), ((38, 38), 4130)])
@pytest.mark.parametrize("power", [-530, 520])
def test_pivots_out_of_the_squares_range(dm, cells, n, power):
    m = dm.make_rect_plate(cells[0] / 96, cells[1] / 96, *cells)
    r = dm.build_rwg(m)
    sub = dm.rwg_from_arrays(m, r.tplus[:n], r.tminus[:n], r.vplus_opp[:n], r.vminus_opp[:n], r.len[:n],
                             r.area_plus[:n], r.area_minus[:n], evert=r.evert[:n])
    scale = 2.0 ** power
    Z = dm.assemble_Z_efie(m, sub, K0, eta0=dm.ETA0 * scale, forms=dm.DM_Z64, device=True, mesh_precheck=False,
                           max_output_bytes=None)
    A = Z.to_numpy() / scale
    squares = 2 * np.log2(np.abs(np.diag(A))) + 2 * power  # log2 |pivot candidate|^2
    assert np.all(squares < -1022) if power < 0 else np.all(squares > 1024)
    rng = np.random.default_rng(n)
    B = rng.standard_normal((n, 2)) + 1j * rng.standard_normal((n, 2))
    X = dm.solve_forward(Z, B, solver="direct") * scale
    err = np.linalg.norm(B - A @ X, axis=0) / (np.linalg.norm(A) * np.linalg.norm(X, axis=0))
    assert np.all(err <= 8 * n * 2.0 ** -53)
