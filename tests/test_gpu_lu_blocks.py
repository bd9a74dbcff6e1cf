"""Dense LU past the sizes whose right-hand side fits the LDS of the back
substitution (8192 rows), and right-hand sides beyond the block that is carried
through the factorization against the same ones carried."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
K0 = 2 * math.pi / 0.1
U = 2.0 ** -53


def _first_bases(dm, nx, ny, n):
    m = dm.make_rect_plate(nx / 96, ny / 96, nx, ny)
    r = dm.build_rwg(m)
    sub = dm.rwg_from_arrays(m, r.tplus[:n], r.tminus[:n], r.vplus_opp[:n], r.vminus_opp[:n], r.len[:n],
                             r.area_plus[:n], r.area_minus[:n], evert=r.evert[:n])
    return dm.assemble_Z_efie(m, sub, K0, forms=dm.DM_Z64, device=True, mesh_precheck=False, max_output_bytes=None)


def test_back_substitution_from_memory(dm):
    n = 8200
    Z = _first_bases(dm, 55, 52, n)
    A = Z.to_numpy()
    rng = np.random.default_rng(8)
    B = rng.standard_normal((n, 2)) + 1j * rng.standard_normal((n, 2))
    X = dm.solve_forward(Z, B, solver="direct")
    Z.free()
    err = np.linalg.norm(B - A @ X, axis=0) / (np.linalg.norm(A) * np.linalg.norm(X, axis=0))
    assert np.all(err <= 8 * n * U)


def test_later_blocks_agree_with_carried_columns(dm):
    """Both solutions have a backward error of 8 n u, so they differ by at most
    twice that times the condition number."""
    n = 97
    Z = _first_bases(dm, 8, 5, n)
    A = Z.to_numpy()
    rng = np.random.default_rng(5)
    B = rng.standard_normal((n, 1030)) + 1j * rng.standard_normal((n, 1030))
    X = dm.solve_forward(Z, B, solver="direct")[:, 1024:]
    Y = dm.solve_forward(Z, B[:, 1024:], solver="direct")
    cond = np.linalg.norm(A) * np.linalg.norm(np.linalg.inv(A), 2)
    assert np.all(np.linalg.norm(X - Y, axis=0) <= 16 * n * U * cond * np.linalg.norm(Y, axis=0))
