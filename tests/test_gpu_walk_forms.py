"""Forms of the walk kernel against the oracle: one or two targets per lane
(the rule changes above 16 targets per group), with and without dipole terms
(charges of one sign), kept list remainders (few or many slices)."""
import numpy as np
import pytest

from oracle import oracle as orc

pytestmark = pytest.mark.gpu

CHARGES = {
    "positive": lambda r, n: r.random(n) + 0.1,
    "negative": lambda r, n: -r.random(n) - 0.1,
    "zeros": lambda r, n: np.where(r.random(n) < 0.5, 0.0, 1.0),
    "mixed": lambda r, n: r.standard_normal(n),
    "one_negative": lambda r, n: np.concatenate([np.ones(n - 1), [-2.0]]),
}


@pytest.mark.parametrize("group,pack", [(1, 0), (2, 0), (16, 0), (17, 0), (16, 17), (32, 0), (33, 33),
                                        (64, 0), (64, 64)])
@pytest.mark.parametrize("charges", sorted(CHARGES))
def test_forms(group, pack, charges):
    from pepc_amd.solver import Solver
    n = 1500
    r = np.random.Generator(np.random.PCG64([group, pack, len(charges)]))
    p = r.random((n, 3))
    q = CHARGES[charges](r, n)
    x, y, z = (np.ascontiguousarray(p[:, k]) for k in range(3))
    eps2 = 1e-4
    d, t, w = orc.solve(x, y, z, q, 0.36, eps2, tile_size=group, pack=pack)
    # FP32 bound per target: 16 u (L sum |q|/r^3 + sum |q|/r^2), u = 2^-24,
    # for the rounding of positions relative to the group's first particle
    ds = p[:, None, :] - p[None, :, :]
    r2 = (ds * ds).sum(-1) + eps2
    np.fill_diagonal(r2, np.inf)
    scale = 16 * 2.0 ** -24 * ((np.sqrt(3.0) * np.abs(q) / r2 ** 1.5).sum(1) + (np.abs(q) / r2).sum(1))
    for precision in ("fp64", "fp32"):
        sol = Solver(theta2=0.36, eps2=eps2, group_size=group, group_pack=pack, precision=precision)
        sol.grow(x, y, z, q)
        res = sol.traverse()
        wk = sol.read_walk()
        perm = sol.sorted_host()[1]
        assert np.array_equal(wk["p2p"].astype(np.int64), np.asarray(w.p2p, np.int64))
        assert np.array_equal(wk["m2p"].astype(np.int64), np.asarray(w.m2p, np.int64))
        err = np.abs(res.e.cpu().numpy().T - w.e).max(1)
        if precision == "fp64":
            assert err.max() <= 1e-12 * np.abs(w.e).max()
        else:
            assert np.all(err <= scale[perm])
        sol.close()


def test_walk_after_replay_with_other_signs():
    """A replay may bring charges of both signs to a tree grown from charges
    of one: the walk after it has to evaluate dipoles.  The charges keep their
    magnitudes, so the centres of |charge|, and with them the lists, stay."""
    from pepc_amd.solver import Solver
    n = 2000
    r = np.random.Generator(np.random.PCG64(12))
    p = r.random((n, 3))
    x, y, z = (np.ascontiguousarray(p[:, k]) for k in range(3))
    sol = Solver(theta2=0.36, eps2=1e-4, group_size=16, precision="fp64")
    sol.grow(x, y, z, np.ones(n))
    sol.freeze()
    e = sol.replay(x, y, z, np.where(r.random(n) < 0.5, -1.0, 1.0)).e.cpu().numpy()
    got = sol.traverse().e.cpu().numpy()
    assert np.abs(got - e).max() <= 1e-12 * np.abs(e).max()
    sol.close()
