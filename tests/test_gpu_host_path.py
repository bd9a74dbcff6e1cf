"""Host side of a call: mesh checks against a plain restatement on random
triangle soups (duplicates, non-manifold edges, orientation conflicts,
repeated vertices), and what freed matrices leave in the context's cache."""
import collections
import ctypes as C
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
K0 = 2 * math.pi / 0.1


def _counts(xyz, tri):
    """(invalid, degenerate, duplicate, non-manifold, conflicts, boundary) as assert_mesh_quality counts them
    (area_tol_rel = 0: a zero area is degenerate)."""
    invalid = degenerate = duplicate = 0
    faces, edges = set(), collections.defaultdict(list)
    for t in tri:
        if len(set(t)) < 3:
            invalid += 1
            continue
        key = tuple(sorted(t))
        dup = key in faces
        duplicate += dup
        faces.add(key)
        a, b, c = xyz[t - 1]
        degenerate += not np.any(np.cross(b - a, c - a))
        if dup:
            continue
        for j in range(3):
            u, v = t[j], t[(j + 1) % 3]
            edges[min(u, v), max(u, v)].append(u < v)
    n = [len(e) for e in edges.values()]
    conflicts = sum(len(e) == 2 and e[0] == e[1] for e in edges.values())
    return invalid, degenerate, duplicate, sum(k > 2 for k in n), conflicts, sum(k == 1 for k in n)


@pytest.mark.parametrize("seed", range(8))
def test_mesh_check_counts(dm, seed):
    rng = np.random.default_rng(seed)
    nv = int(rng.integers(4, 60))
    tri = rng.integers(1, nv + 1, (int(rng.integers(3, 80)), 3))
    tri = np.concatenate([tri, tri[:2], tri[:1, ::-1]])
    xyz = rng.integers(0, 4, (nv, 3)).astype(float)  # coincident and collinear points
    want = _counts(xyz, tri)
    m = dm.TriMesh(xyz, tri)
    names = ("invalid triangles", "degenerate triangles", "duplicate triangles", "non-manifold edges",
             "orientation conflicts", "boundary edges")
    with pytest.raises(ValueError) as e:
        dm.assert_mesh_quality(m, allow_boundary=False, require_closed=True, area_tol_rel=0.0)
    for name, k in zip(names, want):
        assert (f"{k} {name}" in str(e.value)) if k else (name not in str(e.value)), (name, k, str(e.value))


def _free_bytes():
    """Free device memory, from the HIP runtime the library already loaded."""
    try:
        h = C.CDLL("libamdhip64.so.7")
    except OSError:
        h = C.CDLL("/opt/rocm/lib/libamdhip64.so")
    f, t = C.c_size_t(), C.c_size_t()
    assert h.hipMemGetInfo(C.byref(f), C.byref(t)) == 0
    return f.value


def test_freed_matrices_in_the_cache(dm):
    """Small freed matrices are reused (same entries as fresh ones), at most
    2 GiB of them stay, and a large one goes back to the device."""
    ctx = dm.Context(0)
    m = dm.make_rect_plate(0.3, 0.3, 30, 30, ctx=ctx)
    r = dm.build_rwg(m)
    asm = lambda forms=dm.DM_Z64: dm.assemble_Z_efie(m, r, K0, forms=forms, device=True, mesh_precheck=False,  # noqa: E731
                                                     max_output_bytes=None)
    z = asm()
    first = z.entries([0, 5, 9], [1, 5, 2639])
    z.free()
    free0 = _free_bytes()
    zs = [asm() for _ in range(24)]  # 24 x 113 MB
    for z in zs:
        assert np.allclose(z.entries([0, 5, 9], [1, 5, 2639]), first, rtol=1e-13, atol=0)
        z.free()
    assert free0 - _free_bytes() <= (2 << 30) + (64 << 20)
    big = dm.make_rect_plate(0.4, 0.4, 40, 40, ctx=ctx)
    rb = dm.build_rwg(big)
    zb = dm.assemble_Z_efie(big, rb, K0, device=True, mesh_precheck=False, max_output_bytes=None)  # 360 MB
    held = _free_bytes()
    zb.free()
    assert _free_bytes() - held >= 300 << 20
