"""The same call gives the same bits: stored matrices assembled again, in every form
(complex128 with the rules of up to three points, FP32 with every rule) and with
both workgroup sizes of the FP64 tiles, and the currents of a lockstep mixed solve
in contexts of their own, one of them without the tuner."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
K0 = 2 * math.pi / 0.1


SIDES = {"plate": (0.2, 0.15, 21, 17), "strip": (0.234, 0.15, 4, 30)}


def _mesh(dm, kind):
    if kind == "pieces":  # 10 x 11 squares apart: two triangles to a basis, 128 to a block
        at = np.array([[0, 0, 0], [1, 0, 0], [1, 1, 0], [0, 1, 0.0]])
        xyz = np.concatenate([0.01 * at + 0.013 * np.array([i, j, 0]) for i in range(10) for j in range(11)])
        tri = np.concatenate([4 * q + np.array([[1, 2, 3], [1, 3, 4]]) for q in range(110)])
        return dm.TriMesh(xyz, tri)
    return dm.make_rect_plate(*SIDES[kind]) if kind in SIDES else dm.make_icosphere(0.07, 3)


@pytest.mark.parametrize("kind", ["plate", "strip", "pieces", "sphere"])
@pytest.mark.parametrize("quad_order", [1, 3, 4, 7])
def test_matrices_repeat(dm, kind, quad_order):
    m = _mesh(dm, kind)
    r = dm.build_rwg(m)
    ctx = dm.default_context()
    saved = ctx.tune_get()
    for forms in (dm.DM_Z64, dm.DM_Z32, dm.DM_Z64P, dm.DM_Z32P, dm.DM_Z64P | dm.DM_Z32P | dm.DM_Z32_ROUNDED):
        if quad_order > 3 and forms not in (dm.DM_Z32, dm.DM_Z32P):
            continue
        single = [f for f in (dm.DM_Z64, dm.DM_Z32, dm.DM_Z64P, dm.DM_Z32P) if forms & f]
        want = None
        for threads in (1024, 512, 1024, 512):
            ctx.tune_set({f"asm/{w}/q{q}/{r.nedges}": threads for w in ("z64", "z64p", "z64p+z32") for q in (1, 3, 4, 7)})
            Z = dm.assemble_Z_efie(m, r, K0 * (1 - 0.01j), forms=forms, device=True, quad_order=quad_order)
            got = [Z.to_numpy(f) for f in single]
            Z.free()
            want = want or got
            assert all(np.array_equal(a, b) for a, b in zip(got, want))
    ctx.tune_set(saved)


@pytest.mark.parametrize("quad_order", [1, 3])
def test_matrices_of_many_meshes_repeat(dm, quad_order):
    """... and are those of each mesh alone."""
    ms = [dm.make_rect_plate(nx / 120, ny / 120, nx, ny) for nx, ny in ((3, 4), (21, 17), (9, 14), (12, 6))]
    ms += [_mesh(dm, "strip"), _mesh(dm, "pieces")]
    rs = [dm.build_rwg(m) for m in ms]
    for form in (dm.DM_Z64, dm.DM_Z32, dm.DM_Z64P, dm.DM_Z32P):
        a, b = ([z.to_numpy(form) for z in dm.assemble_Z_efie_multi(ms, rs, K0, forms=form, quad_order=quad_order)]
                for _ in range(2))
        alone = [dm.assemble_Z_efie(m, r, K0, forms=form, device=True, quad_order=quad_order).to_numpy(form)
                 for m, r in zip(ms, rs)]
        assert all(np.array_equal(x, y) and np.array_equal(x, z) for x, y, z in zip(a, b, alone))


def test_lockstep_solve_repeats(dm, monkeypatch):
    """7680 unknowns: more than one accumulation chunk of the bf16 product."""
    got = []
    for tune in ("0", "1", "1"):
        monkeypatch.setenv("DM_TUNE", tune)
        ctx = dm.Context()
        m = dm.make_icosphere(0.1, 4, ctx=ctx)
        r = dm.build_rwg(m)
        pw = dm.seeded_planewaves(K0, 24, np.random.default_rng(3))
        P = dm.build_nearfield_preconditioner(None, m, r, 2.0 * float(np.mean(r.len)))
        got.append(dm.solve_planewaves(m, r, K0, pw, "mixed", P, tol=1e-6, maxiter=300, relax=0.1)[0])
    assert all(np.array_equal(g, got[0]) for g in got[1:])
