"""Infinite inputs give the infinite outputs that the plain sums give, not NaN."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
K0 = 2 * math.pi / 0.1


@pytest.mark.parametrize("adjoint", [False, True])
def test_matrix_free_product_of_an_infinite_entry(dm, adjoint):
    """Every row gets one infinite term, entry (m, 3) of Z times it."""
    m = dm.make_rect_plate(0.08, 0.06, 9, 7)
    r = dm.build_rwg(m)
    Z = dm.assemble_Z_efie(m, r, K0)
    op = dm.matrixfree_efie_operator(m, r, K0)
    x = np.arange(1.0, r.nedges + 1) + 0.5j
    x[3] = complex(np.inf, 0.0)
    y = (op.adjoint() if adjoint else op) @ x
    col = Z[:, 3].conj() if adjoint else Z[:, 3]  # Z is symmetric
    assert np.array_equal(y.real, np.copysign(np.inf, col.real))
    assert np.array_equal(y.imag, np.copysign(np.inf, col.imag))
