"""Boxes at the edges of their blocks: four particles a thread give one block
up to 1,024 particles of one system and 256 up to 262,144; above that sixteen a
thread, again 256 blocks up to 1,048,576, and never more than 1,024 (4,194,304).
The box is the coordinates' extrema with the margin of 1/10000 of the extent,
computed with the same operations, so it is compared exactly."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1023, 1024, 1025, 262143, 262144, 262145, 1048576, 1048577, 4194304,
                               4194305])
@pytest.mark.parametrize("place", ["first", "last"])
def test_box(n, place):
    from pepc_amd.solver import Solver
    p = np.random.default_rng(n).standard_normal((3, n))
    i = 0 if place == "first" else n - 1       # the extrema in the first or last block
    p[:, i] = [-9.0, 9.5, 10.0]
    p[:, i + (1 if i == 0 else -1)] = [9.25, -8.0, -11.0]
    sol = Solver(theta2=0.36, eps2=1e-4, group_size=64, group_pack=64)
    sol.grow(*p, np.ones(n))
    box = np.zeros((3, 3))
    sol._check(sol.lib.pepc_gpu_read_box(sol.h, 0, *[b.ctypes.data_as(C.c_void_p) for b in box]))
    sol.close()
    lo, hi = p.min(axis=1), p.max(axis=1)
    d = hi - lo
    assert np.array_equal(box[0], lo - d / 10000.0) and np.array_equal(box[1], hi + d / 10000.0)
