"""Fields between the solver's key order and the input order, on the device.

restore_fields and sort_fields move values and compute nothing, so they are
compared with the permutation of sorted_host exactly, at the edges of a block
and below it; coulomb_field uses both, so its results equal a grow and a
traverse of its own bit for bit, and its gradients those of an adjoint call
with the same upstream values up to the order of the FP64 atomics (1e-12, as
the adjoint's own tests).
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from pepc_amd.solver import Solver
    return Solver


def _points(n, seed):
    r = np.random.default_rng(seed)
    return r.random((3, n)), r.standard_normal(n)


@pytest.mark.parametrize("n", [2, 255, 256, 257, 3001])
def test_fields_both_ways(gpu, n):
    p, q = _points(n, n)
    sol = gpu(theta2=0.36, eps2=1e-4, group_size=32, precision="fp64")
    sol.grow(*p, q)
    perm = torch.from_numpy(sol.sorted_host()[1]).cuda()
    res = sol.traverse()
    e, pot = sol.restore_fields(res.e, res.pot)
    assert e.shape == (n, 3) and torch.equal(e[perm].T, res.e) and torch.equal(pot[perm], res.pot)
    es, ps = sol.sort_fields(e, pot)
    assert torch.equal(es, res.e) and torch.equal(ps, res.pot)
    with pytest.raises(ValueError):
        sol.restore_fields(e, pot[:-1])
    with pytest.raises(ValueError):
        sol.sort_fields(e.T.contiguous()[:2], pot)
    sol.close()


def test_coulomb_field_strided_upstream_and_regrow(gpu):
    from pepc_amd.autograd import coulomb_field
    n = 2049
    p, q = _points(n, 7)
    sol = gpu(theta2=0.36, eps2=1e-4, group_size=32, precision="fp64")
    sol.grow(*p, q)
    perm = torch.from_numpy(sol.sorted_host()[1]).cuda()
    res = sol.traverse()
    w = torch.randn(3, n, dtype=torch.float64, device="cuda")
    u = torch.randn(1, dtype=torch.float64, device="cuda")
    want = sol.adjoint(w[:, perm], u.expand(n))
    want = sol.restore(*want)
    X = [torch.tensor(a, device="cuda", requires_grad=True) for a in (*p, q)]
    e, pot = coulomb_field(*X, sol)
    assert torch.equal(e[perm].T, res.e) and torch.equal(pot[perm], res.pot)
    p2, q2 = _points(1500, 8)
    sol_other = [torch.tensor(a, device="cuda") for a in (*p2, q2)]
    coulomb_field(*sol_other, sol)           # another tree before the backward
    torch.autograd.backward([e, pot], [w.T, u.expand(n)])
    for x, g in zip(X, want):
        assert torch.allclose(x.grad, g, rtol=1e-12, atol=1e-12 * g.abs().max().item())
    with pytest.raises((RuntimeError, ValueError)):
        coulomb_field(*[a.detach().cpu() for a in X], sol)
    sol.close()
