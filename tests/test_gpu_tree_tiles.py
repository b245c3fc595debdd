"""Tree build and upward pass at the edges of their tiles (512 particles, one
tile more or less) and at larger trees of both forms, by tiles and by levels
(the edges between the forms are in test_gpu_upward_levels.py): node set and
FP64 moments bit-exact against the oracle."""
import numpy as np
import pytest

from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 511, 512, 513, 1024, 1025, 32768, 65537, 131071, 131072, 131073])
@pytest.mark.parametrize("clustered", [False, True])
def test_tiles(n, clustered):
    from pepc_amd.solver import Solver
    r = np.random.Generator(np.random.PCG64([n, int(clustered)]))
    p = r.random((n, 3))
    if clustered:   # deep chains of twigs across tile ends
        p[: n // 2] = 0.37 + 1e-4 * p[: n // 2]
    q = r.standard_normal(n)
    x, y, z = (np.ascontiguousarray(p[:, k]) for k in range(3))
    d = orc.domain_decompose(x, y, z, q)
    t = orc.tree_build(d.keys, d.x, d.y, d.z, d.q, d.box)
    sol = Solver(theta2=0.36, eps2=1e-4, precision="fp64")
    sol.grow(x, y, z, q)
    tr = sol.read_tree()
    assert sol.check_tree() == 0
    link, first, mom = tr["link"], tr["first"], tr["mom"]
    assert len(link) == t.nnodes
    gg = np.lexsort((link[:, 3], first))           # by first particle, then level
    og = np.lexsort((t.level, t.first))
    assert np.array_equal(link[gg, 3].astype(np.int64), np.asarray(t.level, np.int64)[og])
    assert np.array_equal(link[gg, 2].astype(np.int64), np.asarray(t.leaves, np.int64)[og])
    assert np.array_equal(t.mom[og][:, :15], mom[gg][:, :15])
    sol.close()


@pytest.mark.parametrize("n", [940001, 1048576, 1048577])
def test_table_capacity(n):
    """Trees on both sides of the change of tile length, in a context whose
    capacity lies on the other side, are sound."""
    from pepc_amd.solver import Solver
    r = np.random.Generator(np.random.PCG64(n))
    p = r.random((n, 3))
    sol = Solver(theta2=0.81, eps2=1e-4, precision="fp32", group_size=64, group_pack=64)
    for m in (n, 1000):
        st = sol.grow(*(np.ascontiguousarray(p[:m, k]) for k in range(3)), np.ones(m))
        assert st["nleaf"] == m and sol.check_tree() == 0
    sol.close()
