"""Mesh-form field sweep at the edges of its tiling: one and two points per
lane, wave and workgroup remainders, every split class of the partial-sum
reduction, points far from the mesh and next to it (the tiers of the edge and
angle polynomials)."""
import numpy as np
import pytest

from radiacuda_amd import _native as N
from radiacuda_amd import objects as O
from radiacuda_amd import rad
from radiacuda_amd import workloads as W

pytestmark = pytest.mark.gpu

# both forms sum the same terms in FP64 (about 1e4 of them, each to a few ulp
# of the largest): 1e-12 of the field scale; FP32 integrals: the bound that the
# FP32 sweep is held to elsewhere, 2e-6
TOL = {N.RH_FP64: 1e-12, N.RH_MIXED: 2e-6}


@pytest.fixture(scope="module", params=["tets", "hexes"])
def model(request):
    rad.UtiDelAll()
    if request.param == "tets":
        _top, obj, _coil, _info = W.c_yoke(ny=1)
        lo, hi = np.array([0.0, 0.0, 0.0]), np.array([140.0, 10.0, 200.0])
    else:
        obj, _p = W.halbach(n_seg=8, n_az=4, n_rad=3, n_ax=4, n_points=1)
        lo, hi = np.array([-40.0, -40.0, -25.0]), np.array([40.0, 40.0, 25.0])
    items = list(O.walk(rad._reg, obj))
    P = O.pack_elements(items)
    rng = np.random.default_rng(4)
    m = N.Model(P)
    assert m.field_form() == 2
    M = rng.normal(size=(len(items), 3))
    ents = sum(m.mesh_counts()[:2])
    yield m, M, lo, hi, ents, P
    m.close()
    rad.UtiDelAll()


def _points(n, lo, hi, P, seed):
    """A third around the mesh, a third far off, a third within 1e-3 to 1
    element sizes of the vertices."""
    rng = np.random.default_rng(seed)
    k = n // 3
    c, d = 0.5 * (lo + hi), hi - lo
    a = c + 1.2 * d * rng.uniform(-0.5, 0.5, (k, 3))
    b = c + 20.0 * d * rng.normal(size=(k, 3))
    v = P["verts"][rng.integers(0, len(P["verts"]), n - 2 * k)]
    s = 10.0 ** rng.uniform(-3, 0, (n - 2 * k, 1)) * 5.0
    x = np.concatenate([a, b, v + s * rng.normal(size=v.shape)])
    return np.ascontiguousarray(x[rng.permutation(n)])


@pytest.mark.parametrize("prec", [N.RH_FP64, N.RH_MIXED])
@pytest.mark.parametrize("count", [1, 63, 65, 257, 513, 4001, 33000, "two"])
def test_mesh_sweep_matches_per_element(model, count, prec):
    m, M, lo, hi, ents, P = model
    # "two": just past the pair count from which a lane takes two points, the
    # last wave and its second points partly empty
    n = int(1.0e8 // ents) + 130 if count == "two" else count
    x = _points(n, lo, hi, P, 11)
    b, h = m.field(M, x, precision=prec)
    m.set_field_form(1)
    try:
        pick = np.unique(np.concatenate([np.arange(min(n, 700)), np.arange(max(0, n - 700), n)]))
        bo, ho = m.field(M, x[pick], precision=N.RH_FP64)
    finally:
        m.set_field_form(0)
    scale = np.abs(ho).max()
    assert np.abs(h[pick] - ho).max() <= TOL[prec] * scale
    assert np.abs(b[pick] - bo).max() <= TOL[prec] * scale


@pytest.mark.parametrize("count", [7, 1300])
def test_one_output_only(model, count):
    m, M, lo, hi, _ents, P = model
    x = _points(count, lo, hi, P, 12)
    b, h = m.field(M, x)
    assert np.array_equal(m.field(M, x, want_h=False)[0], b)
    assert np.array_equal(m.field(M, x, want_b=False)[1], h)
