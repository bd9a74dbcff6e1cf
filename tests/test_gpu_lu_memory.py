"""Many right-hand sides of a direct solve take a block's device memory, not all
columns': 100 000 columns of a small plate (146 MB) leave the context with less
than a third of that, and every block's solutions are right."""
import ctypes as C
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
K0 = 2 * math.pi / 0.1


def _free_bytes():
    try:
        h = C.CDLL("libamdhip64.so.7")
    except OSError:
        h = C.CDLL("/opt/rocm/lib/libamdhip64.so")
    f, t = C.c_size_t(), C.c_size_t()
    assert h.hipMemGetInfo(C.byref(f), C.byref(t)) == 0
    return f.value


def test_direct_solve_holds_a_block_of_columns(dm):
    ctx = dm.Context()
    m = dm.make_rect_plate(0.1, 0.1, 6, 6, ctx=ctx)
    r = dm.build_rwg(m)
    n, cols = r.nedges, 100_000
    Z = dm.assemble_Z_efie(m, r, K0, device=True)
    A = Z.to_numpy()
    rng = np.random.default_rng(2)
    B = rng.standard_normal((n, cols)) + 1j * rng.standard_normal((n, cols))
    dm.solve_forward(Z, B[:, :1], solver="direct")
    before = _free_bytes()
    X = dm.solve_forward(Z, B, solver="direct")
    assert before - _free_bytes() < B.nbytes / 3
    err = np.linalg.norm(B - A @ X, axis=0) / (np.linalg.norm(A) * np.linalg.norm(X, axis=0))
    assert np.all(err <= 8 * n * 2.0 ** -53)
