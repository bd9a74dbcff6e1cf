"""Columns of the near-field sparse approximate inverse against numpy's least
squares on the same matrix and pattern, for support widths in and at the ends of
each workgroup size of the kernel that builds them (widest support 1, up to 39,
up to 59, up to 80; widths at and beside multiples of the 4 x 4 blocks)."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
K0 = 2 * math.pi / 0.1
CAP = 80


@pytest.mark.parametrize("form", ["z64", "z64p"])
@pytest.mark.parametrize("edges,lo,hi", [(0.01, 1, 1), (1.3, 5, 39), (1.6, 20, 39), (1.8, 40, 59), (2.0, 40, 59),
                                         (2.2, 60, 80), (2.4, 60, 80), (6.0, 80, 80)])
def test_columns_match_least_squares(dm, form, edges, lo, hi):
    """The columns come from the normal equations by Cholesky, whose error is of
    the order u kappa(A)^2 of the solution (Higham, Accuracy and Stability, ch.
    20), with a factor that grows with the dimensions: 80 u kappa^2 allowed."""
    p = dm.make_rect_plate(0.18, 0.15, 21, 18)
    xyz = p.xyz.copy()
    xyz[:, :2] += np.random.default_rng(3).normal(0, 0.05 * 0.18 / 21, (len(xyz), 2))
    m = dm.TriMesh(xyz, p.tri)
    r = dm.build_rwg(m)
    n = r.nedges
    f = dict(z64=dm.DM_Z64, z64p=dm.DM_Z64P)[form]
    Z = dm.assemble_Z_efie(m, r, K0, forms=f, device=True)
    A = Z.to_numpy(form=f)
    v = m.xyz[m.tri - 1].sum(axis=1)
    c = (v[r.tplus - 1] + v[r.tminus - 1]) / 6
    cut = edges * float(np.mean(r.len)) * 1.0000123
    S = dm.NearFieldOperator(dm.build_nearfield_preconditioner(Z, m, r, cut), Z)
    D = np.linalg.norm(c[:, None] - c[None], axis=2)
    width = np.minimum((D <= cut).sum(axis=0), CAP)
    assert lo <= width.max() <= hi
    for w in np.unique(width):  # one column of each width
        j = int(np.where(width == w)[0][-1])
        e = np.zeros(n, complex)
        e[j] = 1.0
        J = np.sort(np.argsort(D[j], kind="stable")[:w])
        I = np.where(D[j] <= max(1.6 * D[j][J].max(), 1e-300))[0]
        assert len(I) <= 512
        M = A[np.ix_(I, J)]
        ref, *_ = np.linalg.lstsq(M, (I == j).astype(complex), rcond=None)
        got = S @ e
        assert np.array_equal(np.nonzero(got)[0], J)
        tol = 80 * 2.0 ** -53 * np.linalg.cond(M) ** 2
        assert np.linalg.norm(got[J] - ref) <= tol * np.linalg.norm(ref)
