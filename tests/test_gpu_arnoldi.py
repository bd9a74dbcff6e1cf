"""Steps of the lockstep-batch Arnoldi kernels at the basis sizes where the
kernels change (one fused pass by 256 threads to 36 vectors, by 512 to 64, two
passes beyond) against GMRES written out in numpy."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
K0 = 2 * math.pi / 0.1


def gmres_steps(A, b, m):
    """The iterate of smallest residual over m Krylov steps (orthogonalised twice)."""
    n = b.size
    V = np.zeros((n, m + 1), complex)
    H = np.zeros((m + 1, m), complex)
    beta = np.linalg.norm(b)
    V[:, 0] = b / beta
    for j in range(m):
        w = A @ V[:, j]
        for _ in range(2):
            h = V[:, :j + 1].conj().T @ w
            w -= V[:, :j + 1] @ h
            H[:j + 1, j] += h
        H[j + 1, j] = np.linalg.norm(w)
        V[:, j + 1] = w / H[j + 1, j]
    e = np.zeros(m + 1, complex)
    e[0] = beta
    return V[:, :m] @ np.linalg.lstsq(H, e, rcond=None)[0]


@pytest.mark.parametrize("steps", [1, 36, 37, 64, 65])
def test_batched_steps_match_host_gmres(dm, steps):
    """After a fixed number of steps every column holds the smallest residual of
    its Krylov space.  The minimum is flat, so the residual norm of an iterate
    from a basis that is orthonormal to u = 1.1e-16 per step differs by about
    steps * N * u = 4e-12 of |b| from the host's; a lost or doubled term of one
    dot product changes it by that term's share, far above the 1e-9 asked."""
    m = dm.make_rect_plate(0.3, 0.26, 15, 13)
    r = dm.build_rwg(m)
    assert r.nedges % 64 and r.nedges > 512  # a ragged last chunk of rows
    Z = dm.assemble_Z_efie(m, r, K0, forms=dm.DM_Z64, device=True)
    rng = np.random.default_rng(20261205)
    V = rng.standard_normal((r.nedges, 9)) + 1j * rng.standard_normal((r.nedges, 9))
    X, st = dm.solve_gmres(Z, V, precond_side="right", tol=1e-14, maxiter=steps, batch=1,
                           check_gmres_convergence=False)
    assert st.niter == steps * 9
    Zh = Z.to_numpy()
    for c in range(9):
        ref = gmres_steps(Zh, V[:, c], steps)
        nb = np.linalg.norm(V[:, c])
        got, want = np.linalg.norm(V[:, c] - Zh @ X[:, c]) / nb, np.linalg.norm(V[:, c] - Zh @ ref) / nb
        assert abs(got - want) < 1e-9
