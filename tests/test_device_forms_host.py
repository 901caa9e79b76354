"""The forms that the kernels evaluate, on the CPU (host build of the same code,
every point a wave of its own): the mesh sweep, the blocks far from and near to
an element, the closed-form vertex derivatives, against the general forms and
forward-mode derivatives of the same host build."""
import ctypes

import numpy as np
import pytest

from radiacuda_amd import _abi
from radiacuda_amd import rad
from radiacuda_amd import workloads as W
from tests import models
from tests.test_mesh_host import L, dp  # noqa: F401

i64, i32 = ctypes.c_int64, ctypes.c_int32
CUBE = np.array([[0, 0, 0], [1, 0, 0], [1, 1, 0], [0, 1, 0], [0, 0, 1], [1, 0, 1], [1, 1, 1], [0, 1, 1]], float)
FACES = [[1, 4, 3, 2], [5, 6, 7, 8], [1, 2, 6, 5], [2, 3, 7, 6], [3, 4, 8, 7], [4, 1, 5, 8]]


def _p(a):
    return a.ctypes.data_as(dp)


def _field(lib, name, P, M, pts, fp32=0):
    desc, _keep = _abi.model_desc(P)
    M, pts = np.ascontiguousarray(M, float), np.ascontiguousarray(pts, float)
    B, H = np.zeros_like(pts), np.zeros_like(pts)
    assert getattr(lib, name)(ctypes.byref(desc), _p(M), _p(pts), i64(len(pts)), i32(fp32), _p(B), _p(H)) == 0
    return B, H


def _blocks(lib, P, n, pts, fp32=0):
    desc, _keep = _abi.model_desc(P)
    pts = np.ascontiguousarray(pts, float)
    q, ins = np.zeros((len(pts), n, 3, 3)), np.zeros((len(pts), n), np.int32)
    assert lib.rhc_device_blocks(ctypes.byref(desc), _p(pts), i64(len(pts)), i32(fp32), _p(q),
                                 ins.ctypes.data_as(ctypes.POINTER(i32))) == 0
    return q, ins


def _near_points(verts, n, seed, lo):
    """Points at 10^lo to 30 units of the vertices."""
    rng = np.random.default_rng(seed)
    v = verts[rng.integers(len(verts), size=n)]
    return v + 10.0 ** rng.uniform(lo, 1.5, (n, 1)) * rng.normal(size=(n, 3))


def _meshes():
    rad.UtiDelAll()
    yield "tets", rad.ObjCnt(models.tet_mesh((3, 3, 2), 4.0, jitter=0.1, seed=41))
    rad.UtiDelAll()
    yield "hexes", W.halbach(n_seg=4, n_az=2, n_rad=2, n_ax=2, n_points=1)[0]


# from 1e-3 mm of the vertices, elements being some mm
@pytest.mark.parametrize("lo", [0.5, -3])
@pytest.mark.parametrize("which", ["tets", "hexes"])
def test_sweep_forms_equal_per_element(L, which, lo):  # noqa: F811
    top = next(t for w, t in _meshes() if w == which)
    P, items = models.packed(top)
    M = np.random.default_rng(42).uniform(-1, 1, (len(items), 3))
    pts = _near_points(P["verts"], 300, 43, lo)
    Bo, Ho = _field(L, "rhc_field", P, M, pts)
    # the bounds of the device sweep's own test against the per-element form
    for fp32, tol in ((0, 1e-12), (1, 2e-6)):
        B, H = _field(L, "rhc_field_sweep", P, M, pts, fp32)
        assert np.abs(H - Ho).max() <= tol * np.abs(Ho).max()
        assert np.abs(B - Bo).max() <= tol * np.abs(Ho).max()
    rad.UtiDelAll()


def _elements():
    rng = np.random.default_rng(44)
    rad.UtiDelAll()
    ids = [rad.ObjRecMag([0, 0, 0], [2, 3, 1], [0, 0, 1]), rad.ObjRecMag([9, 0, 0], [1, 1, 6], [0, 0, 1])]
    for k in range(4):
        t = rng.normal(size=(4, 3)) + [0, 9 * k, 9]
        ids.append(rad.ObjPolyhdr(t.tolist(), [[1, 2, 3], [1, 2, 4], [1, 3, 4], [2, 3, 4]], [0, 0, 1]))
        h = (CUBE @ (np.eye(3) + rng.uniform(-0.3, 0.3, (3, 3)))) * [2, 1, 1] + [0, 9 * k, -9]
        ids.append(rad.ObjPolyhdr(h.tolist(), FACES, [0, 0, 1]))
    return models.packed(rad.ObjCnt(ids))


@pytest.mark.parametrize("lo", [0.5])
def test_block_forms_equal_the_general_ones(L, lo):  # noqa: F811
    P, items = _elements()
    n = len(items)
    blocks = np.array([[0.0, 0, 0], [9, 0, 0]])
    pts = np.concatenate([_near_points(P["verts"], 400, 45, lo), _near_points(blocks, 100, 46, lo)])
    q, _ins = _blocks(L, P, n, pts)
    q32, _ins = _blocks(L, P, n, pts, 1)
    for j in range(n):
        for a in range(3):
            M = np.zeros((n, 3))
            M[j, a] = 1.0
            H = _field(L, "rhc_field", P, M, pts)[1]
            # 12 logarithms and 6 angles of order 1 to 10, each to a few units of
            # 1.1e-16 in either form: 18 x 10 x 4 x 1.1e-16 / (4 pi)
            assert np.abs(q[:, j, :, a] - H).max() <= 1e-14
            # FP32 beyond two circumradii, where the block is below 0.1 and its
            # offsets carry 6e-8 of the distance
            assert np.abs(q32[:, j, :, a] - H).max() <= 1e-6
    rad.UtiDelAll()


def test_vertex_derivatives_equal_forward_mode(L):  # noqa: F811
    P, items = _elements()
    rng = np.random.default_rng(47)
    n, nv = len(items), len(P["verts"])
    M = rng.uniform(-1, 1, (n, 3))
    pts = np.ascontiguousarray(_near_points(P["verts"], 200, 48, -1))
    g = rng.normal(size=pts.shape)
    desc, _keep = _abi.model_desc(P)
    out = {}
    for name in ("rhc_adj_grad", "rhc_adj_grad_tri"):
        gV, gX = np.zeros((nv, 3)), np.zeros_like(pts)
        assert getattr(L, name)(ctypes.byref(desc), _p(M), _p(pts), i64(len(pts)), _p(g), _p(gV), _p(gX)) == 0
        out[name] = gV, gX
    # sums of some 200 x 12 terms, each to about 1e-14 of the largest
    for a, b in zip(out["rhc_adj_grad"], out["rhc_adj_grad_tri"]):
        assert np.abs(a - b).max() <= 1e-11 * np.abs(a).max()
    rad.UtiDelAll()


def test_tetrahedron_block_next_to_a_vertex(L):  # noqa: F811
    """At 1e-3 edges a plane distance carries 1.1e-16 / 1e-3 of itself, times
    the few operations of its dot product: 1e-12 of the angles, in either form.
    (A denominator formed as a difference of terms of the edges' size, not of
    the vertex distance's, was off by 1e-11.)"""
    rng = np.random.default_rng(49)
    rad.UtiDelAll()
    ids = []
    for k in range(20):
        t = 10 * rng.normal(size=(4, 3)) + rng.uniform(-20, 20, 3)
        ids.append(rad.ObjPolyhdr(t.tolist(), [[1, 2, 3], [1, 2, 4], [1, 3, 4], [2, 3, 4]], [0, 0, 1]))
    P, items = models.packed(rad.ObjCnt(ids))
    n = len(items)
    d = rng.normal(size=(2000, 3))
    pts = P["verts"][rng.integers(len(P["verts"]), size=2000)] + 1e-2 * d / np.linalg.norm(d, axis=1)[:, None]
    q, _ins = _blocks(L, P, n, pts)
    M = np.tile([0.0, 0.0, 1.0], (n, 1))
    H = _field(L, "rhc_field", P, M, pts)[1]
    assert np.abs(q[..., 2].sum(axis=1) - H).max() <= 1e-12
    rad.UtiDelAll()


@pytest.mark.parametrize("shape", ["flat", "needle", "sliver", "limit"])
def test_far_limit_of_thin_tetrahedra(L, shape):  # noqa: F811
    """Around the limit of the far form (distance sums of four lengths on every
    edge) for tetrahedra that are anything but regular."""
    rng = np.random.default_rng(50)
    if shape == "limit":
        # all sums at least 4.01 lengths, one vertex 1.32 longest edges away
        t = np.array([[0.624, 0.5, 0], [0.624, -0.5, 0], [0, 0, 0], [0.3, 0, 0.02]])
        pts = np.array([[-1.32, 0, 0]]) + np.concatenate([np.zeros((1, 3)), 0.05 * rng.normal(size=(400, 3))])
    else:
        t = rng.normal(size=(4, 3)) * {"flat": [1, 1, 0.01], "needle": [1, 0.01, 0.01], "sliver": [1, 0.1, 0.001]}[shape]
        u = rng.normal(size=(2000, 3))
        size = np.linalg.norm(t[:, None] - t[None], axis=2).max()
        pts = t.mean(0) + rng.uniform(1, 3, (2000, 1)) * size * u / np.linalg.norm(u, axis=1)[:, None]
    rad.UtiDelAll()
    P, _items = models.packed(rad.ObjPolyhdr(t.tolist(), [[1, 2, 3], [1, 2, 4], [1, 3, 4], [2, 3, 4]], [0, 0, 1]))
    q, ins = _blocks(L, P, 1, pts)
    assert not ins.any()
    for a in range(3):
        H = _field(L, "rhc_field", P, np.eye(3)[a][None], pts)[1]
        # weights of order 1, 6 logarithms below 1 and 3 angles below 0.5, each
        # to a few 1.1e-16 in either form: 9 x 6 x 1.1e-16 / (4 pi), doubled for
        # the normals of the thin faces
        assert np.abs(q[:, 0, :, a] - H).max() <= 1e-15
    rad.UtiDelAll()
