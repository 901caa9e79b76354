"""Assembly at the edges of its tiling: row groups of 64, tiles of 8, 16 and 32
sources split over four waves, partial tiles, mixed element kinds (columns
that are not consecutive), transform copies and row transforms, elements far
from a wave and within it, and a collocation point inside another element."""
import ctypes
import os

import numpy as np
import pytest

from tests import models
from radiacuda_amd import _abi
from radiacuda_amd import _native as N
from radiacuda_amd import objects as O
from radiacuda_amd import rad

pytestmark = pytest.mark.gpu

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "radiacuda_amd", "_rhcheck.so")


def _host(P):
    """FP64 matrix from the host build of the general forms."""
    L = ctypes.CDLL(LIB)
    n = len(P["type"])
    desc, keep = _abi.model_desc(P)
    out = np.zeros((3 * n, 3 * n))
    rc = L.rhc_assemble(ctypes.byref(desc), ctypes.c_int64(0), ctypes.c_int64(n), 0,
                        out.ctypes.data_as(ctypes.POINTER(ctypes.c_double)))
    assert rc == 0
    return out


def _elements(n, kind, seed=3):
    """n elements in two clusters 40 sizes apart: most pairs near, many far."""
    rng = np.random.default_rng(seed)
    ids = []
    for c, count in (((0, 0, 0), n - n // 3), ((160, 20, -30), n // 3)):
        if count == 0:
            continue
        k = int(np.ceil((count / 6.0) ** (1.0 / 3.0)))
        tets = models.tet_mesh((k, k, k), 4.0, origin=c, jitter=0.1, seed=seed)[:count]
        for q, t in enumerate(tets):
            if kind == "tets" or q % 3 == 0:
                ids.append(t)
            elif q % 3 == 1:
                ids.append(rad.ObjRecMag([c[0] - 9 - 5 * (q // 3), c[1], c[2] + 4 * (q % 5)], [3, 2, 2.5], [0, 0, 1]))
            else:
                ids.append(models.hex_block([c[0] + 3 * q, c[1] - 12, c[2] + 1], [2.5, 3, 2], [0, 0, 1]))
    return ids, rng


def _check(P, prec, dense, planes=None):
    ref = _host(P)
    with N.Model(P) as m:
        Q = m.assemble(prec, dense_rows=dense)
        if planes is not None:
            assert Q.format()[0] == planes
        got = Q.export()
        Q.reassemble()
        assert np.array_equal(Q.export(), got)
        Q.close()
    scale = np.abs(ref).max(axis=1, keepdims=True)
    err = (np.abs(got - ref) / scale).max()
    # FP64: a few ulp of O(1) terms in sums of about 30; mixed: FP32 far
    # integrals and FP32 storage, the bound the assembly is held to elsewhere
    assert err <= (1e-13 if prec == N.RH_FP64 else 3e-7), err


@pytest.mark.parametrize("dense", [False, True])
@pytest.mark.parametrize("prec", [N.RH_FP64, N.RH_MIXED])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 33, 64, 65, 131])
def test_tetrahedra(n, prec, dense):
    rad.UtiDelAll()
    ids, _rng = _elements(n, "tets")
    P, _items = models.packed(rad.ObjCnt(ids))
    _check(P, prec, dense, 0 if dense else 5)
    rad.UtiDelAll()


@pytest.mark.parametrize("prec", [N.RH_FP64, N.RH_MIXED])
@pytest.mark.parametrize("n", [7, 40, 70])
def test_mixed_kinds(n, prec):
    rad.UtiDelAll()
    ids, _rng = _elements(n, "all")
    P, _items = models.packed(rad.ObjCnt(ids))
    _check(P, prec, False, 5)
    rad.UtiDelAll()


@pytest.mark.parametrize("kind", ["tets", "all"])
@pytest.mark.parametrize("rotated", [False, True])
@pytest.mark.parametrize("prec", [N.RH_FP64, N.RH_MIXED])
@pytest.mark.parametrize("n", [17, 66])
def test_transform_copies(n, prec, rotated, kind):
    rad.UtiDelAll()
    ids, _rng = _elements(n, kind)
    obj = rad.ObjCnt(ids)
    if rotated:
        rad.TrfOrnt(obj, rad.TrfRot([1, 1, 1], [0.2, 0.3, 1.0], 0.4))
    rad.TrfZerPerp(obj, [0, -60, 0], [0, 1, 0])
    rad.TrfZerPara(obj, [0, 0, -80], [0, 0, 1])
    P, _items = models.packed(obj)
    _check(P, prec, False, 0)
    rad.UtiDelAll()


@pytest.mark.parametrize("prec", [N.RH_FP64, N.RH_MIXED])
def test_point_inside_another_element(prec):
    """A small tetrahedron inside a large one: stored with six planes."""
    rad.UtiDelAll()
    ids, _rng = _elements(20, "tets")
    big = rad.ObjPolyhdr([[-30, -30, 60], [30, -30, 60], [0, 40, 60], [0, 0, 120]], models.TET_FACES, [0, 0, 1])
    small = rad.ObjPolyhdr([[-2, -2, 70], [2, -2, 70], [0, 2, 70], [0, 0, 74]], models.TET_FACES, [0, 0, 1])
    P, _items = models.packed(rad.ObjCnt(ids + [big, small]))
    _check(P, prec, False, 6)
    rad.UtiDelAll()
