"""Far fields on both sides of the lines between their three routes (all three
components of the radiation vectors, the transverse two, straight from the
quadrature points) against the radiation vectors times the currents.

Bound: both sides add 6 n products in FP64 in different orders, 4 sqrt(6 n) u for
independent roundings (u = 2^-53), and form phases of up to 30 radians from
coordinates rounded alike, 64 u."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
K0 = 2 * math.pi / 0.1


@pytest.fixture(scope="module")
def plate(dm):
    m = dm.make_rect_plate(58 / 120, 58 / 120, 58, 58)
    return m, dm.build_rwg(m)


def _bases(dm, plate, n):
    m, r = plate
    return m, dm.rwg_from_arrays(m, r.tplus[:n], r.tminus[:n], r.vplus_opp[:n], r.vminus_opp[:n], r.len[:n],
                                 r.area_plus[:n], r.area_minus[:n], evert=r.evert[:n])


@pytest.mark.parametrize("n,ndir", [(1, 3), (255, 40), (256, 40), (511, 70), (512, 70), (1200, 33), (1201, 33),
                                    (5859, 256), (5860, 256), (5900, 255), (9765, 1024), (9766, 1024), (9800, 1023)])
@pytest.mark.parametrize("ncur", [1, 4, 5, 8, 9])
def test_routes(dm, plate, n, ndir, ncur):
    m, r = _bases(dm, plate, n)
    assert r.nedges == n
    rng = np.random.default_rng(n + ncur)
    d = rng.standard_normal((ndir, 3))
    cur = rng.standard_normal((n, ncur)) + 1j * rng.standard_normal((n, ncur))
    G = dm.radiation_vectors(m, r, d, K0)
    want = (G @ cur).reshape((3, ndir, ncur), order="F")
    E = dm.farfield(m, r, d, K0, cur)
    assert np.linalg.norm(E - want) <= (4 * math.sqrt(6 * n) + 64) * 2.0 ** -53 * np.linalg.norm(want)
