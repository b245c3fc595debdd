"""The direct sum leaves the target's own pair out whatever its position: a
particle alone has no field, also one at infinity."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("x", [0.5, np.inf, -np.inf, np.nan, 1e308])
@pytest.mark.parametrize("q", [1.0, np.inf])
def test_alone(x, q):
    from pepc_amd.solver import Solver
    sol = Solver(theta2=0.36, eps2=1e-4)
    e, pot = sol.direct(*(np.array([v]) for v in (x, 0.25, -x)), np.array([q]), [0])
    assert np.array_equal(e.cpu().numpy(), np.zeros((1, 3)))
    assert np.array_equal(pot.cpu().numpy(), np.zeros(1))
    sol.close()
