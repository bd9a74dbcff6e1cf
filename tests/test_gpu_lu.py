"""Dense LU at the edges of its panels, sub-panels and column blocks: the
register-resident panels hold up to 256, 512, 1024, 2048 and 4096 rows (beyond
that the panel stays in memory), panels are 32 columns, right-hand sides go
through the factorization in blocks of up to 1024.

Bound: a backward stable solve leaves ||b - A x|| <= c n u ||A||_F ||x|| with
u = 2^-53; c = 8 allows for the pivot growth of these matrices."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
K0 = 2 * math.pi / 0.1


@pytest.fixture(scope="module")
def plate(dm):
    m = dm.make_rect_plate(0.4, 0.35, 38, 38)
    return m, dm.build_rwg(m)


def _first_bases(dm, plate, n):
    """The matrix of the plate's first n bases (any n: no plate has every size)."""
    m, r = plate
    sub = dm.rwg_from_arrays(m, r.tplus[:n], r.tminus[:n], r.vplus_opp[:n], r.vminus_opp[:n], r.len[:n],
                             r.area_plus[:n], r.area_minus[:n], evert=r.evert[:n])
    return dm.assemble_Z_efie(m, sub, K0, forms=dm.DM_Z64, device=True, mesh_precheck=False, max_output_bytes=None)


@pytest.mark.parametrize("n,nrhs", [(1, 1), (7, 3), (8, 1), (31, 2), (32, 70), (33, 1), (65, 64), (256, 3), (257, 65),
                                    (512, 1), (513, 2), (1024, 1), (1057, 3), (2048, 2), (2081, 1), (4130, 2)])
def test_lu_backward_error(dm, plate, n, nrhs):
    Z = _first_bases(dm, plate, n)
    A = Z.to_numpy()
    rng = np.random.default_rng(n)
    B = rng.standard_normal((n, nrhs)) + 1j * rng.standard_normal((n, nrhs))
    X = dm.solve_forward(Z, B, solver="direct")
    err = np.linalg.norm(B - A @ X, axis=0) / (np.linalg.norm(A) * np.linalg.norm(X, axis=0))
    assert np.all(err <= 8 * n * 2.0 ** -53)


def test_lu_right_hand_sides_beyond_one_block(dm, plate):
    """1030 right-hand sides: the last six take the forward substitution of
    their own, and agree with the same ones solved first."""
    n, nrhs = 97, 1030
    Z = _first_bases(dm, plate, n)
    A = Z.to_numpy()
    rng = np.random.default_rng(5)
    B = rng.standard_normal((n, nrhs)) + 1j * rng.standard_normal((n, nrhs))
    X = dm.solve_forward(Z, B, solver="direct")
    err = np.linalg.norm(B - A @ X, axis=0) / (np.linalg.norm(A) * np.linalg.norm(X, axis=0))
    assert np.all(err <= 8 * n * 2.0 ** -53)
