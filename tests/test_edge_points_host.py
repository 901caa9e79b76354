"""Field points exactly on interior edges of a uniformly magnetized mesh with
integer coordinates: a face that holds the point has the solid-angle pair
(0, 0), whose angle is 0, and no net charge; the net edge weight cancels.  The
field there is that of the body's surface, finite and smooth (CPU, the kernels'
forms; tests/test_gpu_edge_points.py runs the kernels)."""
import numpy as np
import pytest

from radiacuda_amd import rad
from tests import models
from tests.test_device_forms_host import _blocks, _field
from tests.test_mesh_host import L  # noqa: F401

N, STEP = 3, 4.0
MAG = [0.3, -0.5, 0.8]


def body(kind):
    """A cube of 3 x 3 x 3 cells of 4 mm, as tetrahedra or hexahedra."""
    rad.UtiDelAll()
    if kind == "tets":
        ids = models.tet_mesh((N, N, N), STEP, jitter=0.0, M=MAG)
    else:
        ids = [models.hex_block([STEP * (i + 0.5) for i in c], np.full(3, STEP), MAG) for c in np.ndindex(N, N, N)]
    return models.packed(rad.ObjCnt(ids))


def edge_points(kind):
    """Quarter points of the edges that lie inside the cube, by direction."""
    dirs = [[1, 0, 0], [0, 1, 0], [0, 0, 1]]
    if kind == "tets":
        dirs += [[1, 1, 0], [1, 0, 1], [0, 1, 1], [1, 1, 1]]
    out = []
    for d in np.array(dirs, float):
        x = np.array([STEP * (np.array(c) + t * d) for c in np.ndindex(N, N, N) for t in (0.25, 0.5, 0.75)])
        out.append(x[np.all((x > 0) & (x < N * STEP), axis=1)])
    return out


def expected_H(lib, pts):
    """The same cube as one block."""
    rad.UtiDelAll()
    c = 0.5 * N * STEP
    P, _items = models.packed(rad.ObjRecMag([c, c, c], [N * STEP] * 3, MAG))
    H = _field(lib, "rhc_field", P, np.array([MAG]), pts)[1]
    rad.UtiDelAll()
    return H


# FP64: some 1,000 terms of order 1, each to a few units of 1.1e-16; FP32: the
# bound of the single-precision sweep
TOL = {0: 1e-12, 1: 2e-6}


@pytest.mark.parametrize("kind", ["tets", "hexes"])
def test_sweep_on_interior_edges(L, kind):  # noqa: F811
    pts = np.concatenate(edge_points(kind))
    H0 = expected_H(L, pts)
    P, items = body(kind)
    M = np.tile(MAG, (len(items), 1))
    for fp32, tol in TOL.items():
        _B, H = _field(L, "rhc_field_sweep", P, M, pts, fp32)
        assert np.isfinite(H).all()
        assert np.abs(H - H0).max() <= tol
    # an element's own block is finite on its edges as well
    assert np.isfinite(_blocks(L, P, len(items), pts)[0]).all()
    rad.UtiDelAll()
