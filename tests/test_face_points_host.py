"""Field points exactly on a face of a hexahedron: the face's solid angle is one
of its two limits there, and the block the limit from that side (CPU, the
kernels' forms; tests/test_gpu_face_points.py runs the kernels)."""
import numpy as np
import pytest

from radiacuda_amd import rad
from tests import models
from tests.test_device_forms_host import CUBE, FACES, _blocks, _field
from tests.test_mesh_host import L  # noqa: F401

DIMS = np.array([4.0, 2.0, 3.0])


def hexahedron(seed):
    """A 4 x 2 x 3 mm cuboid as a polyhedron, turned for seed > 0; points on its
    faces (off their diagonals) and the faces' normals."""
    R = np.eye(3) if seed == 0 else np.linalg.qr(np.random.default_rng(seed).normal(size=(3, 3)))[0]
    v = (CUBE * DIMS) @ R.T
    pts, nrm = [], []
    for f in FACES:
        w = v[np.array(f) - 1]
        n = np.cross(w[1] - w[0], w[2] - w[0])
        for s, t in ((0.25, 0.5), (0.75, 0.5), (0.5, 0.125)):
            pts.append(w[0] + s * (w[1] - w[0]) + t * (w[3] - w[0]))
            nrm.append(n / np.linalg.norm(n))
    return rad.ObjPolyhdr(v.tolist(), FACES, [0, 0, 1]), np.array(pts), np.array(nrm)


def limits(lib, P, pts, nrm, n=1):
    """The field matrices from either side, 1e-7 mm off the face: the field
    changes by some 0.1 per mm."""
    out = []
    for side in (1e-7, -1e-7):
        out.append(np.stack([_field(lib, "rhc_field", P, np.tile(np.eye(3)[a], (n, 1)), pts + side * nrm)[1]
                             for a in range(3)], -1))
    return out


@pytest.mark.parametrize("seed", [0, 1, 2, 3])
def test_block_on_a_face_is_a_limit(L, seed):  # noqa: F811
    rad.UtiDelAll()
    obj, pts, nrm = hexahedron(seed)
    P, _items = models.packed(obj)
    q = _blocks(L, P, 1, pts)[0][:, 0]
    lo, hi = limits(L, P, pts, nrm)
    off = np.minimum(np.abs(q - lo).max(axis=(1, 2)), np.abs(q - hi).max(axis=(1, 2)))
    assert off.max() <= 1e-6
    rad.UtiDelAll()
