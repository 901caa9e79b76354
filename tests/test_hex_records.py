"""Hexahedron records are kept for hexahedra alone, and sweeps that read them
agree whether they were built with the model or at the call that first reads
them."""
import ctypes

import numpy as np
import pytest

from radiacuda_amd import _abi
from radiacuda_amd import _native as N
from radiacuda_amd import rad
from tests import models
from tests.test_device_forms_host import _field
from tests.test_mesh_host import LIB, L  # noqa: F401


def _prism(x, M=(0, 0, 1)):
    return rad.ObjPolyhdr([[x, 0, 0], [x + 1, 0, 0], [x, 1, 0], [x, 0, 2], [x + 1, 0, 2], [x, 1, 2]],
                          [[1, 2, 3], [4, 5, 6], [1, 2, 5, 4], [2, 3, 6, 5], [3, 1, 4, 6]], list(M))


def _model(hexes, prisms, apart):
    rad.UtiDelAll()
    ids = [models.hex_block([apart * k, 0.5, 1.0], np.array([2.0, 1.0, 2.0]), [0, 0, 1]) for k in range(hexes)]
    ids += [_prism(-20.0 - 3 * k) for k in range(prisms)]
    return models.packed(rad.ObjCnt(ids))


@pytest.mark.parametrize("hexes,prisms", [(0, 7), (5, 0), (3, 4)])
def test_records_for_hexahedra_alone(L, hexes, prisms):  # noqa: F811
    P, _items = _model(hexes, prisms, 2.0)
    desc, _keep = _abi.model_desc(P)
    L.rhc_hex_count.restype = ctypes.c_int64
    assert L.rhc_hex_count(ctypes.byref(desc)) == hexes
    rad.UtiDelAll()


# a slab of touching boxes takes the mesh form (its records wait for a reader),
# the others do not
@pytest.mark.gpu
@pytest.mark.parametrize("hexes,prisms,apart", [(40, 0, 2.0), (40, 0, 9.0), (3, 5, 9.0), (0, 5, 9.0)])
def test_sweeps_with_and_without_the_mesh_form(hexes, prisms, apart):
    print("case: hexahedron records", hexes, prisms, apart, flush=True)
    rad.UtiDelAll()
    if apart == 2.0:
        ids = [models.hex_block([2.0 * a, 1.0 * b, 2.0 * c], np.array([2.0, 1.0, 2.0]), [0, 0, 1])
               for a in range(5) for b in range(4) for c in range(2)]
        P, items = models.packed(rad.ObjCnt(ids))
    else:
        P, items = _model(hexes, prisms, apart)
    rng = np.random.default_rng(3)
    n = len(items)
    M = rng.uniform(-1, 1, (n, 3))
    pts = np.concatenate([rng.uniform(-20, 20, (150, 3)), P["verts"][:30] + 0.1 * rng.normal(size=(30, 3))])
    Bo, Ho = _field(ctypes.CDLL(LIB), "rhc_field", P, M, pts)
    g = rng.normal(size=pts.shape)
    m = N.Model(P)
    mesh = m.field_form() == 2
    assert mesh == (apart == 2.0)
    # the gradient first, so that it is what has the records built
    gM = m.field_adjoint(None, pts, g, field="h", want_m=True)[0]
    # 45 elements x 18 terms of order 1 to 10, each to a few 1.1e-16, over 4 pi
    assert abs(np.sum(g * Ho) - np.sum(gM * M)) <= 1e-12 * np.abs(g).sum()
    for form in (0, 1, 0, 1):
        m.set_field_form(form)
        B, H = m.field(M, pts)[:2]
        assert np.abs(H - Ho).max() <= 1e-12
        assert np.abs(B - Bo).max() <= 1e-12
    m.close()
    # a model whose first reader is the field
    m = N.Model(P)
    m.set_field_form(1)
    assert np.array_equal(m.field(M, pts)[1], H)
    m.close()
    rad.UtiDelAll()


@pytest.mark.gpu
def test_form_chosen_during_a_capture():
    """Choosing the per-element form touches no stream, so that it may happen
    during a capture; the records come with the next field."""
    import torch
    print("case: hexahedron records, capture", flush=True)
    rad.UtiDelAll()
    ids = [models.hex_block([2.0 * a, 1.0 * b, 2.0 * c], np.array([2.0, 1.0, 2.0]), [0, 0, 1])
           for a in range(5) for b in range(4) for c in range(2)]
    P, items = models.packed(rad.ObjCnt(ids))
    rng = np.random.default_rng(5)
    M, pts = rng.uniform(-1, 1, (len(items), 3)), rng.uniform(-20, 20, (100, 3))
    m = N.Model(P)
    x = torch.zeros(8, device="cuda")
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        x += 1.0
        m.set_field_form(1)
    Ho = _field(ctypes.CDLL(LIB), "rhc_field", P, M, pts)[1]
    for k in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(x.cpu(), torch.full((8,), k + 1.0))
        # 40 elements x 18 terms of order 1 to 10, each to a few 1.1e-16, over 4 pi
        assert np.abs(m.field(M, pts)[1] - Ho).max() <= 1e-12
        m.set_field_form(1)
    m.close()
    rad.UtiDelAll()
