"""The near-field pattern built on the device against brute force in numpy: the
counts, the mean radius and the capped columns for cutoffs that give short,
capped and complete lists, on a mesh smaller than the column cap, a sphere
(many equal distances), a graded plate (more bases within the first search
radius than a wave holds) and two far-apart plates (the search radius grows);
and the supports themselves through the preconditioner's columns."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
K0 = 2 * math.pi / 0.1
CAP = 80


def _plate(dm, nx, ny, lx, ly, seed=0, grade=1.0, shift=0.0):
    p = dm.make_rect_plate(lx, ly, nx, ny)
    xyz = p.xyz.copy()
    if grade != 1.0:
        xyz[:, 0] = lx * (xyz[:, 0] / lx + 0.5) ** grade
        xyz[:, 1] = ly * (xyz[:, 1] / ly + 0.5) ** grade
    else:
        xyz[:, :2] += np.random.default_rng(seed).normal(0, 0.05 * lx / nx, (len(xyz), 2))
    xyz[:, 2] += shift
    return xyz, p.tri


def _meshes(dm, name):
    if name == "small":
        return dm.TriMesh(*_plate(dm, 4, 4, 0.04, 0.04))
    if name == "plate":
        return dm.TriMesh(*_plate(dm, 21, 18, 0.18, 0.15))
    if name == "sphere":
        return dm.make_icosphere(0.05, 3)
    if name == "graded":
        return dm.TriMesh(*_plate(dm, 60, 60, 0.3, 0.3, grade=2.5))
    a, ta = _plate(dm, 5, 4, 0.05, 0.04)
    b, tb = _plate(dm, 5, 4, 0.05, 0.04, seed=1, shift=0.6)
    return dm.TriMesh(np.concatenate([a, b]), np.concatenate([ta, tb + len(a)]))


def _centres(m, r):
    v = m.xyz[m.tri - 1].sum(axis=1)
    return (v[r.tplus - 1] + v[r.tminus - 1]) / 6


@pytest.mark.parametrize("name", ["small", "plate", "sphere", "graded", "apart"])
@pytest.mark.parametrize("edges", [0.0, 0.7, 2.0, 4.0, 30.0])
def test_pattern_figures(dm, name, edges):
    m = _meshes(dm, name)
    r = dm.build_rwg(m)
    c = _centres(m, r)
    # cutoffs between the distances, so that rounding decides nothing
    cut = edges * float(np.mean(r.len)) * 1.0000123
    nnz, rad, cap, capped = dm.build_nearfield_preconditioner(None, m, r, cut).pattern_info(r)
    if cut == 0.0:
        cut = 2.5 * float(np.mean(r.len))  # 0: the library's default
    assert cap == CAP
    want, rsum, over = 0, 0.0, 0
    for j in range(r.nedges):
        d = np.sort(np.linalg.norm(c - c[j], axis=1))
        k = min(CAP, int((d <= cut).sum()))
        want += k
        rsum += d[k - 1]
        over += int(k == CAP and len(d) > CAP and d[CAP] <= cut)
    assert nnz == want and capped == over
    assert abs(rad - rsum / r.nedges) <= 1e-12 * max(rad, 1e-300)


def test_pattern_supports(dm):
    m = _meshes(dm, "plate")
    r = dm.build_rwg(m)
    Z = dm.assemble_Z_efie(m, r, K0, device=True)
    S = dm.NearFieldOperator(dm.build_nearfield_preconditioner(Z, m, r, 4.0 * float(np.mean(r.len))), Z)
    c = _centres(m, r)
    for j in (0, 17, r.nedges // 2, r.nedges - 1):
        e = np.zeros(r.nedges, complex)
        e[j] = 1.0
        d = np.linalg.norm(c - c[j], axis=1)
        near = np.argsort(d)[:CAP]
        near = near[d[near] <= 4.0 * float(np.mean(r.len))]
        assert np.array_equal(np.nonzero(S @ e)[0], np.sort(near))
