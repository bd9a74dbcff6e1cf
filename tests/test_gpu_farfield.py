"""Far fields at the edges of their two paths (up to eight currents straight from
the quadrature points, more through the transverse radiation vectors and the
matrix product in parts) against the radiation vectors times the currents.

Bound: both sides add n terms (a few thousand) in FP64 in different orders:
1e-13 of the result's norm."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
K0 = 2 * math.pi / 0.1


@pytest.fixture(scope="module")
def meshes(dm):
    out = {}
    for name, m in (("plate", dm.make_rect_plate(0.11, 0.2, 9, 14)), ("sphere", dm.make_icosphere(0.06, 3)),
                    ("two", dm.make_rect_plate(0.02, 0.01, 1, 1))):
        out[name] = (m, dm.build_rwg(m))
    return out


@pytest.mark.parametrize("name,order", [("plate", 3), ("sphere", 3), ("two", 3), ("plate", 1), ("sphere", 7)])
@pytest.mark.parametrize("ncur,ndir", [(1, 1), (3, 65), (4, 64), (5, 17), (8, 200), (9, 16), (9, 33), (65, 7), (130, 130)])
def test_farfield_paths(dm, meshes, name, order, ncur, ndir):
    m, r = meshes[name]
    rng = np.random.default_rng(ncur * 1000 + ndir)
    d = rng.standard_normal((ndir, 3))
    d[: min(ndir, 3)] = np.eye(3)[: min(ndir, 3)]  # along the axes, then any length
    cur = rng.standard_normal((r.nedges, ncur)) + 1j * rng.standard_normal((r.nedges, ncur))
    G = dm.radiation_vectors(m, r, d, K0, quad_order=order)
    want = (G @ cur).reshape((3, ndir, ncur), order="F")
    E = dm.farfield(m, r, d, K0, cur, quad_order=order)
    assert np.linalg.norm(E - want) <= 1e-13 * np.linalg.norm(want)
