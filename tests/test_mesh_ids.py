"""CPU check of the conforming-mesh form on polygons of more than four
vertices (host build): their faces are fanned into pieces, the pieces are
matched between neighbours by their vertices where both are cut the same way,
and diagonals are no edges."""
import numpy as np
import pytest

from radiacuda_amd import rad
from tests import models
from tests.test_mesh_host import L, _fields  # noqa: F401


def _prism(k, z0, z1, M, centre=(0.0, 0.0)):
    a = 2 * np.pi * np.arange(k) / k
    ring = np.stack([centre[0] + 3 * np.cos(a), centre[1] + 3 * np.sin(a)], 1)
    verts = [[x, y, z] for z in (z0, z1) for x, y in ring]
    faces = [list(range(1, k + 1)), list(range(k + 1, 2 * k + 1))]
    faces += [[i + 1, (i + 1) % k + 1, k + (i + 1) % k + 1, k + i + 1] for i in range(k)]
    return rad.ObjPolyhdr(verts, faces, list(M))


# 5: pieces of 4 and 3 vertices; 6: two of 4
@pytest.mark.parametrize("k", [5, 6])
def test_stacked_prisms_equal_per_element(L, k):  # noqa: F811
    rng = np.random.default_rng(k)
    rad.UtiDelAll()
    n = 12
    ids = [_prism(k, float(i), float(i + 1), rng.uniform(-1, 1, 3)) for i in range(n)]
    # cubes that share their sides, so that the regrouped form is taken
    ids += [rad.ObjPolyhdr([[a, b, c], [a + 1, b, c], [a + 1, b + 1, c], [a, b + 1, c],
                            [a, b, c + 1], [a + 1, b, c + 1], [a + 1, b + 1, c + 1], [a, b + 1, c + 1]],
                           [[1, 2, 3, 4], [5, 6, 7, 8], [1, 2, 6, 5], [2, 3, 7, 6], [3, 4, 8, 7], [4, 1, 5, 8]],
                           list(rng.uniform(-1, 1, 3)))
            for a in range(10, 14) for b in range(4) for c in range(4)]
    P, items = models.packed(rad.ObjCnt(ids))
    M = rng.uniform(-1, 1, (len(items), 3))
    pts = np.concatenate([rng.uniform(-4, 15, (80, 3)),
                          np.stack([np.zeros(12), np.full(12, 0.3), np.arange(12) + 0.4], 1)])
    f = _fields(L, P, M, pts)
    # every sum of ~250 terms of the field's own size: 250 roundings of 1.1e-16
    # and as many from the terms' own evaluation, with a margin of 20
    for a, b in zip(f["elem"][:2], f["mesh"][:2]):
        assert np.abs(a - b).max() <= 1e-12 * np.abs(a).max()
    # the two loops of a shared cap are each other's reverse and are fanned from
    # different vertices, so that their pieces do not match
    caps = 2 * n * ((k - 1) // 2)
    cubes = 3 * 4 * 4 * 5
    assert f["mesh"][2].tolist() == [(n + 1) * k + n * k + 3 * 4 * 5 * 5, caps + n * k + cubes, n + 64]
    rad.UtiDelAll()
