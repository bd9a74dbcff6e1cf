"""A large matrix freed right after its first assembly (the one that times the
tile kernel's launches) has given its memory back when the call returns."""
import math

import pytest

from test_gpu_host_path import _free_bytes

pytestmark = pytest.mark.gpu
K0 = 2 * math.pi / 0.1


def test_large_matrix_is_back_at_once(dm):
    ctx = dm.Context()
    for cells in range(40, 46):  # 4720 to 5985 unknowns, 360 MB to 570 MB
        m = dm.make_rect_plate(cells / 120, cells / 120, cells, cells, ctx=ctx)
        r = dm.build_rwg(m)
        Z = dm.assemble_Z_efie(m, r, K0, device=True, mesh_precheck=False, max_output_bytes=None)
        held = _free_bytes()
        Z.free()
        assert _free_bytes() - held >= 16 * r.nedges ** 2 - (8 << 20)
