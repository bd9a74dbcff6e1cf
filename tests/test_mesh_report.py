"""mesh_resolution_report against the edges listed one by one, for meshes held in
any object with vertices and triangles: 32-bit indices whose edge keys pass 2^31,
and indices that no vertex has, which numpy's indexing refuses."""
from types import SimpleNamespace

import numpy as np
import pytest

from conftest import load_package


def _lengths(xyz, tri):
    e = {tuple(sorted((int(t[i]), int(t[(i + 1) % 3])))) for t in tri for i in range(3)}
    return np.sort([np.linalg.norm(xyz[a - 1] - xyz[b - 1]) for a, b in e])


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
@pytest.mark.parametrize("nv", [5, 100_000])
def test_report_of_plain_arrays(dtype, nv):
    rng = np.random.default_rng(nv)
    xyz = rng.standard_normal((nv, 3))
    tri = (nv - rng.permuted(np.tile(np.arange(min(nv, 40)), (30, 1)), axis=1)[:, :3]).astype(dtype)
    rep = load_package().mesh_resolution_report(SimpleNamespace(xyz=xyz, tri=tri), 3e9)
    want = _lengths(xyz, tri)
    assert rep["edge_min_m"] == pytest.approx(want[0], rel=1e-14)
    assert rep["edge_max_m"] == pytest.approx(want[-1], rel=1e-14)
    assert rep["edge_median_m"] == pytest.approx(np.median(want), rel=1e-14)


def test_report_refuses_what_no_vertex_has():
    xyz = np.zeros((4, 3))
    with pytest.raises(IndexError):
        load_package().mesh_resolution_report(SimpleNamespace(xyz=xyz, tri=np.array([[1, 2, 5]]), nv=4), 3e9)
