"""Blocks seen from both sides of the far form's limit (every corner at least
two longest edges away): cubes, plates and sticks, points in the symmetry
planes and along the edges' lines, wavefronts that mix near and far points."""
import numpy as np
import pytest

from radiacuda_amd import _native as N
from radiacuda_amd import rad
from tests import models

pytestmark = pytest.mark.gpu


def _points(rng, dims):
    h = np.asarray(dims) / 2
    w = max(dims)
    pts = []
    for r in (0.9, 1.6, 1.95, 2.0, 2.05, 2.6, 5.0, 40.0):
        d = rng.normal(size=(24, 3))
        d /= np.linalg.norm(d, axis=1)[:, None]
        pts.append(d * r * w)
        # in the symmetry planes, and on the lines of the edges
        d = rng.normal(size=(9, 3))
        d[np.arange(9), np.arange(9) % 3] = 0.0
        pts.append(d / np.linalg.norm(d, axis=1)[:, None] * (r * w + h.max()))
        for a in range(3):
            e = np.where(np.arange(3) == a, 0.0, h)
            e[a] = h[a] + r * w
            pts.append(e[None])
    pts = np.concatenate(pts)
    inside = np.all(np.abs(pts) <= h * 1.001, axis=1)
    return rng.permutation(pts[~inside])


@pytest.mark.parametrize("dims", [(2.0, 2.0, 2.0), (5.0, 4.0, 0.3), (0.2, 0.3, 6.0), (700.0, 500.0, 900.0)])
def test_field_of_blocks(dims):
    print("case: block", dims, flush=True)
    rng = np.random.default_rng(61)
    rad.UtiDelAll()
    P, _items = models.packed(rad.ObjCnt([rad.ObjRecMag([0, 0, 0], list(dims), [0, 0, 1])]))
    pts = _points(rng, dims)
    model = N.Model(P)
    for k in range(3):
        M = np.zeros((1, 3))
        M[0, k] = 1.0
        _Bo, Ho, bad = models.oracle_field(P, M, pts)
        # an entry is the sum of at most 12 logarithms or angles of order 1,
        # each to a few units of 1.1e-16 in either program: 2 x 12 x 4 x 1.1e-16 / (4 pi)
        _B, H = model.field(M, pts)[:2]
        assert np.abs(H - Ho)[~bad].max() <= 1e-14
        # FP32 integrals: the same count of units of 6e-8
        _B, H = model.field(M, pts, precision=N.RH_MIXED)[:2]
        assert np.abs(H - Ho)[~bad].max() <= 5e-6
    model.close()
    rad.UtiDelAll()


def test_far_form_does_not_depend_on_the_wave():
    """One point per call and all points in one call give the same bits."""
    print("case: block wave independence", flush=True)
    rng = np.random.default_rng(62)
    rad.UtiDelAll()
    dims = (3.0, 2.0, 1.0)
    P, _items = models.packed(rad.ObjCnt([rad.ObjRecMag([0, 0, 0], list(dims), [0, 0, 1])]))
    pts = _points(rng, dims)
    model = N.Model(P)
    M = rng.normal(size=(1, 3))
    H = model.field(M, pts)[1]
    for i in range(0, len(pts), 5):
        assert np.array_equal(model.field(M, pts[i:i + 1])[1][0], H[i])
    model.close()
    rad.UtiDelAll()
