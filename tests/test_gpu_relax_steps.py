"""The device-driven relaxation loops at the edges of their kernels: element
counts around a wavefront, histories shorter and longer than the 16
differences kept, both storage layouts of the adjoint, weak and saturating
fields of the tanh law."""
import numpy as np
import pytest

from radiacuda_amd import _native as N
from radiacuda_amd import rad
from tests import models

pytestmark = pytest.mark.gpu


def _packed(n, sym=False):
    rad.UtiDelAll()
    top = rad.ObjCnt(models.tet_mesh((4, 4, 3), 3.0, jitter=0.1, seed=51)[:n])
    if sym:
        rad.TrfZerPara(top, [0, 0, -1], [0, 0, 1])
    return models.packed(top)[0]


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 130])
@pytest.mark.parametrize("field", [1e-4, 0.05, 5.0])
def test_tanh_law_fixed_point(n, field):
    print("case: tanh law %d elements field %g" % (n, field), flush=True)
    rng = np.random.default_rng(52)
    model = N.Model(_packed(n))
    Q = model.assemble(N.RH_FP64)
    # susceptibilities of tens: the iteration needs more than 16 differences
    # on the larger models and stays well conditioned
    mats = np.zeros((n, 16))
    mats[:, 0], mats[:, 1] = 2, 3
    mats[:, 2:5] = [1.4, 0.0, 0.5]
    mats[:, 5:8] = [40.0, 3.0, 9.0]
    hext = field * rng.normal(size=(n, 3))
    res, M, H = Q.relax(mats, hext, np.zeros((n, 3)), 1e-13 * field, 400)
    assert res.converged
    Mn = models.fp64_fixed_point(Q.export(), mats, hext, M0=M, tol=1e-15)
    # RMS residual of 1e-13 of the field, times the conditioning (at most the
    # susceptibility, about 50) and sqrt(n) from RMS to maximum
    assert np.abs(M - Mn).max() <= 1e-13 * field * 50 * np.sqrt(n) + 1e-14 * np.abs(Mn).max()
    # a run that is cut off counts its iterations
    res, _M, _H = Q.relax(mats, hext, np.zeros((n, 3)), 0.0, 5)
    assert res.iters == 5 and not res.converged
    Q.close()
    model.close()
    rad.UtiDelAll()


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 130])
@pytest.mark.parametrize("sym", [False, True])
def test_adjoint_system(n, sym):
    print("case: adjoint system %d elements sym %d" % (n, sym), flush=True)
    rng = np.random.default_rng(53)
    model = N.Model(_packed(n, sym))
    Q = model.assemble(N.RH_FP64)
    mats = np.zeros((n, 16))
    mats[:, 0] = np.arange(n) % 2  # isotropic and anisotropic linear laws
    mats[:, 1] = 6.0
    A = rng.uniform(-1, 1, (n, 3, 3))
    mats[:, 4:13] = (4.0 * np.eye(3) + A + A.transpose(0, 2, 1)).reshape(n, 9) * (mats[:, :1] == 1)
    rhs = rng.normal(size=(n, 3))
    K = np.zeros((3 * n, 3 * n))
    for e in range(n):
        K[3 * e:3 * e + 3, 3 * e:3 * e + 3] = mats[e, 4:13].reshape(3, 3) if mats[e, 0] else 6.0 * np.eye(3)
    S = np.eye(3 * n) - Q.export().T @ K.T
    res, lam = Q.relax_adjoint(mats, rhs, 1e-13, 400)
    assert res.converged
    # the RMS proposal step 1e-13 times |I - K Q| <= 1 + 10 and sqrt(3 n)
    assert np.abs(S @ lam.ravel() - rhs.ravel()).max() <= 1e-13 * 11 * np.sqrt(3 * n) + 1e-13
    # started from the solution it stops at once
    res2, lam2 = Q.relax_adjoint(mats, rhs, 1e-12, 400, lam0=lam)
    assert res2.converged and res2.iters == 1
    assert np.abs(lam2 - lam).max() <= 1e-11 * np.abs(lam).max()
    res3, _l = Q.relax_adjoint(mats, rhs, 0.0, 3)
    assert res3.iters == 3 and not res3.converged
    Q.close()
    model.close()
    rad.UtiDelAll()
