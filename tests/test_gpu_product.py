"""Products of a few columns with a stored matrix against the same matrix on the
host, at the sizes where the kernel changes (one launch to 3072 unknowns, gather
+ product + scatter beyond) and around its strides (4 columns a workgroup, 512
rows a step, pairs of complex64 entries)."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
K0 = 2 * math.pi / 0.1


@pytest.mark.parametrize("nx,ny", [(1, 1), (2, 3), (5, 6), (12, 14), (13, 14), (18, 19), (31, 33), (32, 33)])
def test_few_columns_match_the_host_product(dm, nx, ny):
    """Each sum of N products in FP64 is within 4 N u of the sum of magnitudes
    (u = 2^-53), whatever its order; the host's is too."""
    m = dm.make_rect_plate(nx / 120, ny / 120, nx, ny)
    r = dm.build_rwg(m)
    n = r.nedges
    rng = np.random.default_rng(n)
    Z = dm.assemble_Z_efie(m, r, K0, forms=dm.DM_Z64 | dm.DM_Z32, device=True, max_output_bytes=None)
    X = rng.standard_normal((n, 3)) + 1j * rng.standard_normal((n, 3))
    for form in (dm.DM_Z64, dm.DM_Z32):
        A = Z.to_numpy(form=form).astype(np.complex128)
        for adjoint in (False, True):
            B = A.conj().T if adjoint else A
            bound = 8 * n * 2.0 ** -53 * (np.abs(B) @ np.abs(X))
            Y = Z.matmul(X, form=form, adjoint=adjoint)
            assert np.all(np.abs(Y - B @ X) <= bound)
            y = Z.matmul(X[:, 1], form=form, adjoint=adjoint)
            assert np.array_equal(y, Y[:, 1])


@pytest.mark.parametrize("nx,ny", [(1, 1), (5, 6), (7, 7), (13, 14), (31, 33)])
def test_packed_columns_match_the_host_product(dm, nx, ny):
    """The packed forms, whose reduction writes the caller's order itself: the same bound."""
    m = dm.make_rect_plate(nx / 120, ny / 120, nx, ny)
    r = dm.build_rwg(m)
    n = r.nedges
    rng = np.random.default_rng(n)
    Z = dm.assemble_Z_efie(m, r, K0, forms=dm.DM_Z64P | dm.DM_Z32P, device=True, max_output_bytes=None)
    X = rng.standard_normal((n, 2)) + 1j * rng.standard_normal((n, 2))
    for form in (dm.DM_Z64P, dm.DM_Z32P):
        A = Z.to_numpy(form=form).astype(np.complex128)
        for adjoint in (False, True):
            B = A.conj().T if adjoint else A
            bound = 8 * n * 2.0 ** -53 * (np.abs(B) @ np.abs(X))
            assert np.all(np.abs(Z.matmul(X, form=form, adjoint=adjoint) - B @ X) <= bound)
