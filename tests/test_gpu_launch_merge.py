"""Boxes, levels and groups at the edges of the blocks that produce them.

Box: from one block (up to 1,024 particles of a system) to many (the block that
finishes last joins them; the edges of their rule are in
test_gpu_box_blocks.py); batches from one system per block to many blocks per
system.  The box is the coordinates' extrema with the margin of
1/10000 of the extent, computed with the same operations, so it is compared
exactly.  Groups: tiles of 4,096 marks; they cover the particles in order
without gaps.  Repeated solves equal the first bit for bit (nothing that a
launch leaves behind reaches the next one).
"""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from pepc_amd.solver import Solver
    return Solver


def _box(p):
    lo, hi = p.min(axis=1), p.max(axis=1)
    d = hi - lo
    return lo - d / 10000.0, hi + d / 10000.0


@pytest.mark.parametrize("n", [2, 255, 4095, 4096, 4097, 8193, 70000, 1048577])
def test_box_and_groups(gpu, n):
    r = np.random.default_rng(n)
    p, q = r.standard_normal((3, n)), r.standard_normal(n)
    sol = gpu(theta2=0.36, eps2=1e-4, group_size=16, group_pack=32)
    first = None
    for _ in range(3):
        st = sol.grow(*p, q)
        res = sol.traverse()
        got = (st["ngroups"], res.e.cpu().numpy(), res.pot.cpu().numpy(), sol.sync()["interactions"])
        if first is None:
            first = got
        assert got[0] == first[0] and got[3] == first[3]
        assert np.array_equal(got[1], first[1]) and np.array_equal(got[2], first[2])
    box = np.zeros((3, 3))
    sol._check(sol.lib.pepc_gpu_read_box(sol.h, 0, *[b.ctypes.data_as(C.c_void_p) for b in box]))
    lo, hi = _box(p)
    assert np.array_equal(box[0], lo) and np.array_equal(box[1], hi)
    w = sol.read_walk()
    gf, gc = w["gfirst"].astype(np.int64), w["gcount"].astype(np.int64)
    assert gf[0] == 0 and np.array_equal(gf[1:], (gf + gc)[:-1]) and gf[-1] + gc[-1] == n
    assert sol.check_tree() == 0
    p[1, n // 2] = np.inf
    with pytest.raises(Exception, match="non-finite"):
        sol.grow(*p, q)
    p[1, n // 2] = 0.0
    sol.grow(*p, q)
    sol.close()


@pytest.mark.parametrize("sizes", [[4096, 2], [70000, 3, 0, 4097], [40] * 300, [5] * 4100])
def test_batch_boxes(gpu, sizes):
    r = np.random.default_rng(len(sizes))
    off = np.concatenate([[0], np.cumsum(sizes)])
    n = int(off[-1])
    p, q = r.standard_normal((3, n)), r.standard_normal(n)
    sol = gpu(theta2=0.36, eps2=1e-4, group_size=16, group_pack=32)
    sol.grow_batch(*p, q, off)
    e = sol.traverse().e.cpu().numpy().copy()
    for s in (0, len(sizes) // 2 - 1, len(sizes) - 1):
        b, t = int(off[s]), int(off[s + 1])
        one = gpu(theta2=0.36, eps2=1e-4, group_size=16, group_pack=32)
        one.grow(*p[:, b:t], q[b:t])
        assert np.array_equal(one.traverse().e.cpu().numpy(), e[:, b:t])
        one.close()
    sol.close()
