"""Upward pass on both sides of its rules: the largest trees formed by tiles
and the first formed by levels (65,536 particles), and levels of up to 98,304
twigs (four lanes per twig) and above (one).  Node set and FP64 moments are
bit-exact against the oracle."""
import numpy as np
import pytest

from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def _pairs(k):
    """One pair of particles in each of k cells of the 64^3 of level 6."""
    r = np.random.Generator(np.random.PCG64(k))
    cells = np.concatenate([[0, 64 ** 3 - 1], 1 + r.choice(64 ** 3 - 2, k - 2, replace=False)])
    c = np.stack([cells // 4096, cells // 64 % 64, cells % 64])
    p = np.concatenate([(c + 0.25) / 64, (c + 0.75) / 64], axis=1)
    d = 1.0 / (1.0 + 2e-4)          # the box [0, 1] with its margins
    p[:, 0] = d * 1e-4
    p[:, k + 1] = 1.0 - d * 1e-4
    return p


def _uniform(n):
    return np.random.Generator(np.random.PCG64(n)).random((3, n))


@pytest.mark.parametrize("kind,size", [("uniform", 65535), ("uniform", 65536), ("uniform", 65537),
                                       ("pairs", 98304), ("pairs", 98305), ("uniform", 700000)])
def test_moments(kind, size):
    from pepc_amd.solver import Solver
    p = np.ascontiguousarray(_pairs(size) if kind == "pairs" else _uniform(size))
    q = np.random.Generator(np.random.PCG64(1)).standard_normal(p.shape[1])
    d = orc.domain_decompose(*p, q)
    t = orc.tree_build(d.keys, d.x, d.y, d.z, d.q, d.box)
    level, leaves = np.asarray(t.level, np.int64), np.asarray(t.leaves, np.int64)
    twigs = np.bincount(level[leaves > 1])
    if kind == "pairs":
        assert twigs[6] == size == twigs.max()
    elif size == 700000:             # levels of both kinds
        assert twigs.max() > 98304 and np.any((twigs > 65536) & (twigs < 98304))
    sol = Solver(theta2=0.36, eps2=1e-4, precision="fp64")
    sol.grow(*p, q)
    tr = sol.read_tree()
    assert sol.check_tree() == 0
    link, first, mom = tr["link"], tr["first"], tr["mom"]
    sol.close()
    assert len(link) == t.nnodes
    gg = np.lexsort((link[:, 3], first))           # by first particle, then level
    og = np.lexsort((t.level, t.first))
    assert np.array_equal(link[gg, 3].astype(np.int64), level[og])
    assert np.array_equal(link[gg, 2].astype(np.int64), leaves[og])
    assert np.array_equal(t.mom[og][:, :15], mom[gg][:, :15])
