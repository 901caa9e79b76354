"""Field points exactly on faces of hexahedra swept one by one (no shared faces,
so no mesh form): one point and a wave of them; and the gradient by the
magnetization there."""
import ctypes

import numpy as np
import pytest

from radiacuda_amd import _native as N
from radiacuda_amd import rad
from tests import models
from tests.test_face_points_host import hexahedron, limits
from tests.test_mesh_host import LIB

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("seed", [0, 1, 2])
def test_field_on_a_face_is_a_limit(seed):
    print("case: face points", seed, flush=True)
    rad.UtiDelAll()
    obj, pts, nrm = hexahedron(seed)
    P, _items = models.packed(obj)
    lo, hi = limits(ctypes.CDLL(LIB), P, pts, nrm)
    m = N.Model(P)
    assert m.field_form() == 1
    for a in range(3):
        M = np.eye(3)[a][None]
        # each limit within 1e-7 mm x 0.1 per mm
        for x, s in [(pts, slice(None))] + [(pts[k:k + 1], slice(k, k + 1)) for k in (0, 7, 17)]:
            H = m.field(M, x)[1]
            off = np.minimum(np.abs(H - lo[s, :, a]).max(axis=1), np.abs(H - hi[s, :, a]).max(axis=1))
            assert off.max() <= 1e-6
    # sum_p g_p . H_p(M) = sum M . gM: the gradient's sweep meets the same blocks
    g = np.random.default_rng(seed).normal(size=pts.shape)
    M = np.array([[0.3, -0.7, 0.5]])
    H = m.field(M, pts)[1]
    gM = m.field_adjoint(None, pts, g, field="h", want_m=True)[0]
    assert abs(np.sum(g * H) - np.sum(gM * M)) <= 1e-12 * np.abs(g).sum()
    m.close()
    rad.UtiDelAll()
