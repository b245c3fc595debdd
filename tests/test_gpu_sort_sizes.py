"""The particle sort at the edges of its forms (blocks of 2,048, one to four
merges, the radix passes above 524,288): keys ascending, permutation that of a
stable sort of the oracle's keys; and grouped sinks, which sort the same way."""
import numpy as np
import pytest

from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 3, 64, 127, 128, 129, 2047, 2048, 2049, 4097, 8192, 8193, 32768, 32769,
                               131073, 524288, 524289])
def test_sizes(n):
    from pepc_amd.solver import Solver
    r = np.random.Generator(np.random.PCG64(n))
    p = r.random((n, 3))
    x, y, z = (np.ascontiguousarray(p[:, k]) for k in range(3))
    keys = orc.compute_keys(x, y, z, orc.box_create(x, y, z))
    order = np.argsort(keys, kind="stable")
    assert len(np.unique(keys)) == n      # ties have their own tests
    sol = Solver(theta2=0.81, eps2=1e-4, group_size=32, group_pack=32)
    sol.grow(x, y, z, np.ones(n))
    k, perm, *_ = sol.sorted_host()
    assert np.array_equal(k, keys[order]) and np.array_equal(perm, order)
    if n <= 32769:   # grouped sinks on the sources: the grown particles' own count of sinks
        a = sol.traverse_sinks(x, y, z, grouped=True)
        one = sol.traverse_sinks(x, y, z)
        assert np.all(a.work.cpu().numpy() >= 1) or n < 3
        d = (a.e - one.e).norm(dim=0) / one.e.norm(dim=0).clamp_min(1e-30)
        assert float(d.median()) < 2e-2    # other groups, other lists: same fields to the opening angle
    sol.close()
