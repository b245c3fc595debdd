"""The walk of systems whose charges have one sign, over the range of
coordinate scales: positions and softening times a power of two (which leaves
every decision of the solve as it is) against the oracle at the unit scale,
whose fields scale exactly."""
import numpy as np
import pytest

from oracle import oracle as orc

pytestmark = pytest.mark.gpu


# Powers for FP32: the direct terms' r^-3 stays within its exponents, with
# r from the smallest separation (0.0055) or the softening to the diagonal (or
# the softening of 4).
@pytest.mark.parametrize("precision,powers", [("fp32", (-32, -26, -20, 0, 20, 28, 36)),
                                              ("fp64", (-220, 220))])
@pytest.mark.parametrize("group", [16, 64])   # one and two targets per lane
@pytest.mark.parametrize("eps", [0.0, 0.01, 4.0])
def test_scales(precision, powers, group, eps):
    from pepc_amd.solver import Solver
    n = 1500
    r = np.random.Generator(np.random.PCG64([group, int(100 * eps)]))
    p = r.random((n, 3))
    q = r.random(n) + 0.1
    x, y, z = (np.ascontiguousarray(p[:, k]) for k in range(3))
    d, t, w = orc.solve(x, y, z, q, 0.36, eps * eps, tile_size=group)
    ds = p[:, None, :] - p[None, :, :]
    r2 = (ds * ds).sum(-1) + eps * eps
    np.fill_diagonal(r2, np.inf)
    # FP32 per target: 16 u (L sum |q|/r^3 + sum |q|/r^2) for the field, one
    # power of r less for the potential, u = 2^-24, L the diagonal, for the
    # rounding of positions relative to the group's first particle
    rl = np.sqrt(3.0)
    u16 = 16 * 2.0 ** -24
    s1, s2, s3 = ((np.abs(q) / r2 ** (k / 2)).sum(1) for k in (1, 2, 3))
    for k in powers:
        f = 2.0 ** k
        sol = Solver(theta2=0.36, eps2=(eps * f) ** 2, group_size=group, precision=precision)
        sol.grow(x * f, y * f, z * f, q)
        res = sol.traverse()
        wk = sol.read_walk()
        perm = sol.sorted_host()[1]
        assert np.array_equal(wk["m2p"].astype(np.int64), np.asarray(w.m2p, np.int64))
        err = np.abs(res.e.cpu().numpy().T * f * f - w.e).max(1)
        perr = np.abs(res.pot.cpu().numpy() * f - w.pot)
        if precision == "fp64":
            assert err.max() <= 1e-12 * np.abs(w.e).max(), k
            assert perr.max() <= 1e-12 * np.abs(w.pot).max(), k
        else:
            assert np.all(err <= u16 * (rl * s3 + s2)[perm]), k
            assert np.all(perr <= u16 * (rl * s2 + s1)[perm]), k
        sol.close()
