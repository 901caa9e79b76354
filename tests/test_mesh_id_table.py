"""The packer's vertex table on models with round coordinates (host build): the
number of slots looked at per vertex stays that of a random table, which for one
at most half full is 1.5 by linear probing."""
import ctypes

import numpy as np
import pytest

from tests.test_mesh_host import L, dp  # noqa: F401


def _grid(shape, step, origin=(0.0, 0.0, 0.0)):
    g = np.stack(np.meshgrid(*[np.arange(n + 1.0) for n in shape], indexing="ij"), -1).reshape(-1, 3)
    return g * step + np.asarray(origin)


CASES = {"unit grid": _grid((10, 10, 10), 1.0),
         "half grid": _grid((20, 20, 20), 0.5, (-5.0, -5.0, -5.0)),
         "5 mm grid": _grid((30, 4, 30), 5.0),
         "long row": _grid((1, 1, 1000), np.array([40.0, 20.0, 5.0]), (-20.0, -10.0, -2500.0)),
         "longer row": _grid((2, 2, 2000), 5.0),
         "random": np.random.default_rng(1).normal(size=(4000, 3))}


@pytest.mark.parametrize("case", list(CASES))
def test_round_coordinates_probe_as_random_ones(L, case):  # noqa: F811
    x = np.ascontiguousarray(CASES[case])
    out = np.zeros(1)
    L.rhc_vertex_probes.restype = ctypes.c_int64
    assert L.rhc_vertex_probes(x.ctypes.data_as(dp), ctypes.c_int64(len(x)), out.ctypes.data_as(dp)) == len(x)
    # a thousand vertices or more: the mean of a random table scatters by less
    # than 0.1
    assert out[0] <= 2.0
