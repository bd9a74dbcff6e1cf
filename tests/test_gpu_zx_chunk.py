"""The accumulation chunk of the bf16 Z X is not chosen by a timer: at a size
where chunks of 8192 columns are as fast as chunks of 4096, every column count
takes 4096 (large products 8192), and the products are those of a context without
the tuner, bit for bit.  A loaded choice is still honoured."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
K0 = 2 * math.pi / 0.1


def test_chunk_is_fixed(dm, monkeypatch):
    ctx = dm.Context()
    m = dm.make_rect_plate(66 / 120, 64 / 120, 66, 64, ctx=ctx)
    r = dm.build_rwg(m)
    n = r.nedges
    assert 8192 < n < 16384
    Z = dm.assemble_Z_efie(m, r, K0, forms=dm.DM_Z64 | dm.DM_Z32 | dm.DM_Z32_ROUNDED, device=True, max_output_bytes=None)
    rng = np.random.default_rng(1)
    for cols in (16, 32, 64, 96, 128):
        X = rng.standard_normal((n, cols)) + 1j * rng.standard_normal((n, cols))
        monkeypatch.setenv("DM_TUNE", "0")
        want = Z.matmul(X, form=dm.DM_Z32)
        monkeypatch.delenv("DM_TUNE")
        assert np.array_equal(Z.matmul(X, form=dm.DM_Z32), want)
        assert ctx.tune_get()[f"zx/c64/{n}/{cols}"] == 4096
    ctx.tune_set({f"zx/c64/{n}/{cols}": 8192})
    assert not np.array_equal(Z.matmul(X, form=dm.DM_Z32), want)
    Z.free()


def test_chunk_of_large_products(dm, monkeypatch):
    """From n^2 columns = 3e10 on the chunk is 8192, with the tuner or without."""
    ctx = dm.Context()
    m = dm.make_rect_plate(80 / 120, 80 / 120, 80, 80, ctx=ctx)
    r = dm.build_rwg(m)
    n = r.nedges
    Z = dm.assemble_Z_efie(m, r, K0, forms=dm.DM_Z32, device=True, max_output_bytes=None)
    X = np.random.default_rng(2).standard_normal((n, 128)) + 0j
    for cols, chunk in ((64, 4096), (128, 8192)):
        assert (n * n * cols >= 3e10) == (chunk == 8192)
        monkeypatch.setenv("DM_TUNE", "0")
        want = Z.matmul(X[:, :cols], form=dm.DM_Z32)
        monkeypatch.delenv("DM_TUNE")
        assert np.array_equal(Z.matmul(X[:, :cols], form=dm.DM_Z32), want)
        assert ctx.tune_get()[f"zx/c64/{n}/{cols}"] == chunk
    Z.free()
