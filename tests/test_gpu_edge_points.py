"""Field points exactly on interior edges of a uniformly magnetized mesh with
integer coordinates (tests/test_edge_points_host.py tells what is expected
there): one point, and waves of points along an edge, in both field forms and
both precisions."""
import ctypes

import numpy as np
import pytest

from radiacuda_amd import _native as N
from radiacuda_amd import rad
from tests.test_edge_points_host import MAG, STEP, TOL, body, edge_points, expected_H
from tests.test_mesh_host import LIB

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["tets", "hexes"])
def test_field_on_interior_edges(kind):
    print("case: edge points", kind, flush=True)
    by_dir = edge_points(kind)
    single = [x[len(x) // 2:len(x) // 2 + 1] for x in by_dir]
    # a line along an axis-parallel edge: the point's wave sees the other faces
    # of that line under no angle
    line = np.array([[STEP + STEP * (0.5 + k) / 64, STEP, STEP] for k in range(64)])
    sets = by_dir + single + [line]
    H0 = [expected_H(ctypes.CDLL(LIB), x) for x in sets]
    P, items = body(kind)
    M = np.tile(MAG, (len(items), 1))
    m = N.Model(P)
    assert m.field_form() == 2
    for x, h0 in zip(sets, H0):
        for fp32, prec in ((0, N.RH_FP64), (1, N.RH_MIXED)):
            H = m.field(M, x, precision=prec)[1]
            assert np.isfinite(H).all()
            assert np.abs(H - h0).max() <= TOL[fp32]
    # element by element no term cancels, and a point on an edge has no limit:
    # finite is what is promised
    m.set_field_form(1)
    for x in sets:
        for prec in (N.RH_FP64, N.RH_MIXED):
            B, H = m.field(M, x, precision=prec)[:2]
            assert np.isfinite(B).all() and np.isfinite(H).all()
    m.close()
    rad.UtiDelAll()
