"""GPU adjoint sweeps at the edges of their tiles: triangles that do not fill
the last wavefront, several batches of triangles to a block, transform copies
(a mirror and a rotation), few and many points; against the host build's
forward-mode derivatives and the oracle's field columns."""

import numpy as np
import pytest

from radiacuda_amd import _native as N
from radiacuda_amd import rad
from tests import models
from tests.test_gpu_adjoint import _chk_grad, _rot

pytestmark = pytest.mark.gpu


def _model(rng, kind, sym):
    rad.UtiDelAll()
    if kind == "one":      # 4 triangles
        ids = models.tet_mesh((1, 1, 1), 3.0, jitter=0.1, seed=41)[:1]
    elif kind == "mixed":  # 24 tetrahedra and 9 hexahedra: 204 triangles, two slices
        ids = models.tet_mesh((2, 2, 1), 4.0, jitter=0.1, seed=42)
        ids += [models.hex_block([15.0 + 5 * k, 2.0, 1.0], [3.0, 2.0, 4.0], rng.uniform(-1, 1, 3), _rot(rng))
                for k in range(9)]
    top = rad.ObjCnt(ids)
    if sym:
        rad.TrfZerPara(top, [0, 0, -6], [0.1, 0.2, 1])
        rad.TrfMlt(top, rad.TrfRot([0, -20, 0], [1, 0.2, 0.3], 1.1), 3)
    P, items = models.packed(top)
    P["verts"] = np.ascontiguousarray(P["verts"] @ _rot(rng).T)
    return P, len(items)


@pytest.mark.parametrize("kind", ["one", "mixed"])
@pytest.mark.parametrize("sym", [False, True])
@pytest.mark.parametrize("np_", [1, 3, 17, 130, 1000])
def test_geometry_gradients(kind, sym, np_):
    print("case: geometry gradients %s sym %d points %d" % (kind, sym, np_), flush=True)
    rng = np.random.default_rng(43)
    P, n = _model(rng, kind, sym)
    M = rng.uniform(-1, 1, (n, 3))
    pts = rng.uniform(-30, 60, (np_, 3))
    g = rng.normal(size=pts.shape)
    # host reference copy by copy: every element has the same copies
    nc = int(P["copy_off"][1])
    assert nc == (6 if sym else 1)
    Pi = dict(P)
    Pi["copy_off"] = np.arange(n + 1, dtype=np.asarray(P["copy_off"]).dtype)
    Pi["cM"] = np.ascontiguousarray(np.tile(np.eye(3), (n, 1, 1)).reshape(np.asarray(P["cM"])[:n].shape))
    Pi["cV"], Pi["cS"] = np.zeros((n, 3)), np.ones(n)
    rV, rX = np.zeros((len(P["verts"]), 3)), np.zeros_like(pts)
    for c in range(nc):
        A = np.asarray(P["cM"])[c].reshape(3, 3)
        B = np.linalg.inv(A)
        v, x = _chk_grad(Pi, M, (pts - np.asarray(P["cV"])[c]) @ B.T, float(np.asarray(P["cS"])[c]) * (g @ A))
        rV += v
        rX += x @ B
    model = N.Model(P)
    for want_x in (False, True):
        _g, gV, gX = model.field_adjoint(M, pts, g, field="h", want_m=False, want_v=True, want_x=want_x)
        # sides are 0.02 to 0.5 of their distance: a derivative that is a
        # difference of terms 50 times its size, of up to 1,000 of them
        assert np.abs(gV - rV).max() <= 1e-10 * np.abs(rV).max()
        if want_x:
            assert np.abs(gX - rX).max() <= 1e-10 * np.abs(rX).max()
    model.close()
    rad.UtiDelAll()


# (np, n): slices of 4 to 64 elements, the last one partly filled
@pytest.mark.parametrize("np_", [1, 300, 9000])
def test_magnetization_gradient_slices(np_):
    print("case: magnetization gradient points %d" % np_, flush=True)
    rng = np.random.default_rng(44)
    rad.UtiDelAll()
    ids = models.tet_mesh((3, 3, 2), 4.0, jitter=0.1, seed=45)
    P, items = models.packed(rad.ObjCnt(ids))
    n = len(items)
    M = rng.uniform(-1, 1, (n, 3))
    pts = rng.uniform(-20, 30, (np_, 3))
    g = rng.normal(size=pts.shape)
    model = N.Model(P)
    gM, _v, _x = model.field_adjoint(None, pts, g, field="b", want_m=True)
    B = model.field(M, pts)[0]
    # <g, B(M)> = <gM, M>: both sums of np n terms of either sign
    assert abs(np.sum(g * B) - np.sum(gM * M)) <= 1e-12 * np.sqrt(np.sum(g * g) * np.sum(B * B))
    # and element by element, where the sweep of one element is the reference
    for j in (0, 3, n // 2, n - 1):
        for k in range(3):
            e = np.zeros((n, 3))
            e[j, k] = 1.0
            r = np.sum(g * model.field(e, pts)[0])
            assert abs(gM[j, k] - r) <= 1e-11 * np.abs(gM).max()
    model.close()
    rad.UtiDelAll()
