"""The walk's work queues: fewer groups than workgroups, about as many, and
many more; one workgroup, a number of workgroups that the queues do not
divide, and the default.  Which wave takes a group does not enter its results,
so all agree bit for bit, in a second walk of the same tree too (the queues
are ready again), for the particles and for sinks."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [5, 300, 4096, 33000, 140000])
@pytest.mark.parametrize("precision", ["fp32", "fp64"])
def test_any_number_of_workgroups(n, precision):
    from pepc_amd.solver import Solver
    r = np.random.default_rng(n)
    p, q = r.random((3, n)), r.standard_normal(n)
    m = min(n, 9000)
    want = None
    for blocks in (0, 1, 3, 13, 1000):
        if blocks in (1, 3) and n > 5000:
            continue                      # a single wave over many groups takes long
        sol = Solver(theta2=0.49, eps2=1e-4, group_size=8, precision=precision, walk_blocks=blocks)
        sol.grow(*p, q)
        got = []
        for _ in range(2):
            res = sol.traverse()
            st = sol.sync()
            got.append((res.e.cpu().numpy(), res.pot.cpu().numpy(), res.work.cpu().numpy(),
                        st["interactions"], st["walk_steps"]))
            s = sol.traverse_sinks(*p[:, :m])
            got[-1] += (s.e.cpu().numpy(), s.work.cpu().numpy())
        if want is None:
            want = got[0]
        for g in got:
            assert all(np.array_equal(a, b) for a, b in zip(g, want))
        sol.close()
