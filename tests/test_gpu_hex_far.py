"""Hexahedra seen from both sides of the far form's limit: parallelepipeds and
frusta with their vertices and faces in any order, next to a polyhedron that is
none, with and without transform copies, inside and outside."""
import ctypes

import numpy as np
import pytest

from radiacuda_amd import _abi
from radiacuda_amd import _native as N
from radiacuda_amd import rad
from tests import models
from tests.test_mesh_host import LIB, dp

pytestmark = pytest.mark.gpu

CUBE = [[0, 0, 0], [1, 0, 0], [1, 1, 0], [0, 1, 0], [0, 0, 1], [1, 0, 1], [1, 1, 1], [0, 1, 1]]
FACES = [[0, 3, 2, 1], [4, 5, 6, 7], [0, 1, 5, 4], [1, 2, 6, 5], [2, 3, 7, 6], [3, 0, 4, 7]]


def _hex(rng, centre, shape, M):
    v = np.array(CUBE, dtype=float) - 0.5
    if shape == "skew":
        v = v @ (np.eye(3) + rng.uniform(-0.4, 0.4, (3, 3))).T
    elif shape == "frustum":  # all six faces stay planar
        v[:, :2] *= np.where(v[:, 2:] > 0, 0.4, 1.0)
    elif shape == "plate":
        v = v * [3.0, 2.0, 0.1]
    q, _r = np.linalg.qr(rng.normal(size=(3, 3)))
    order = rng.permutation(8)
    inv = np.argsort(order)
    faces = []
    for k in rng.permutation(6):
        f = np.roll([inv[i] + 1 for i in FACES[k]], rng.integers(4))
        faces.append([int(i) for i in (f if rng.integers(2) else f[::-1])])
    return rad.ObjPolyhdr(((v @ q.T) + centre)[order].tolist(), faces, list(M))


@pytest.mark.parametrize("shape", ["skew", "frustum", "plate"])
@pytest.mark.parametrize("sym", [False, True])
def test_field_of_hexahedra(shape, sym):
    print("case: hexahedra", shape, sym, flush=True)
    rng = np.random.default_rng(71)
    rad.UtiDelAll()
    centres = np.array([[6.0 * k, 0, 0] for k in range(19)])
    ids = [_hex(rng, c, shape, rng.uniform(-1, 1, 3)) for c in centres]
    # a triangular prism, which the sweep takes by the general form
    ids.insert(7, rad.ObjPolyhdr([[0, 9, 0], [1, 9, 0], [0, 10, 0], [0, 9, 2], [1, 9, 2], [0, 10, 2]],
                                 [[1, 2, 3], [4, 5, 6], [1, 2, 5, 4], [2, 3, 6, 5], [3, 1, 4, 6]], [0.3, 0.2, 0.5]))
    top = rad.ObjCnt(ids)
    if sym:
        rad.TrfZerPara(top, [0, 0, -8], [0.1, 0.2, 1])
    P, items = models.packed(top)
    M = rng.uniform(-1, 1, (len(items), 3))
    # near each element at 0.05 to 40 sizes, so that waves mix near and far
    pts = np.concatenate([centres[rng.integers(19, size=400)] + rng.normal(size=(400, 3)) *
                          rng.choice([0.05, 0.3, 1.0, 2.0, 3.0, 40.0], (400, 1)),
                          rng.uniform(-20, 130, (200, 3))])
    model = N.Model(P)
    # the host build of the general form (the oracle's own nudges near special
    # directions leave up to 6e-12 here, against either)
    desc, _keep = _abi.model_desc(P)
    Bo, Ho = np.zeros_like(pts), np.zeros_like(pts)
    assert ctypes.CDLL(LIB).rhc_field(ctypes.byref(desc), M.ctypes.data_as(dp), pts.ctypes.data_as(dp),
                                      ctypes.c_int64(len(pts)), ctypes.c_int32(0), Bo.ctypes.data_as(dp),
                                      Ho.ctypes.data_as(dp)) == 0
    B, H = model.field(M, pts)[:2]
    # per element 12 logarithms and 6 angles of order 1 to a few units of
    # 1.1e-16, 20 (40) elements of magnetization below 2: 40 x 18 x 4 x 2 x
    # 1.1e-16 / (4 pi)
    assert np.abs(H - Ho).max() <= 6e-14
    assert np.abs(B - Bo).max() <= 6e-14
    # the magnetization's gradient runs the same blocks
    g = rng.normal(size=pts.shape)
    gM = model.field_adjoint(None, pts, g, field="b", want_m=True)[0]
    assert abs(np.sum(g * B) - np.sum(gM * M)) <= 1e-12 * np.sqrt(np.sum(g * g) * np.sum(B * B))
    model.close()
    rad.UtiDelAll()
