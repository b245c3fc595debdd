"""The split direct sum at the edges of its tiles, slices and source ranges,
against the sum in extended precision."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 255, 256, 257, 1023, 1024, 1025, 5000])
@pytest.mark.parametrize("m", [1, 2, 3, 64, 129, 256, 257, 900])
@pytest.mark.parametrize("periodic", [False, True])
def test_direct(n, m, periodic):
    from pepc_amd.solver import Solver
    if periodic and n * m > 300000:
        pytest.skip("27 boxes: the small sizes cover every branch")
    r = np.random.Generator(np.random.PCG64([n, m]))
    p = r.random((n, 3))
    q = r.standard_normal(n)
    idx = r.integers(0, n, m)            # any order, repeats allowed
    eps2 = 1e-4
    sol = Solver(theta2=0.36, eps2=eps2, precision="fp64", sign=-1.0)
    boxes = [np.zeros(3)]
    if periodic:
        sol.set_periodic(far_field=False)
        boxes = [np.array([i, j, k], float) for i in (-1, 0, 1) for j in (-1, 0, 1) for k in (-1, 0, 1)]
    e, pot = sol.direct(*(np.ascontiguousarray(p[:, k]) for k in range(3)), q, idx)
    e, pot = e.cpu().numpy(), pot.cpu().numpy()
    sol.close()
    ld = np.longdouble
    ex, ph = np.zeros((m, 3), ld), np.zeros(m, ld)
    sa, sp = np.zeros((m, 3), ld), np.zeros(m, ld)
    for v in boxes:
        d = ((p[idx] - v)[:, None, :] - p[None, :, :]).astype(ld)
        r2 = (d * d).sum(-1) + ld(eps2)
        w = q.astype(ld)[None, :] / np.sqrt(r2)
        if not v.any():
            w[np.arange(m), idx] = 0
        t = (w / r2)[..., None] * d
        ex += t.sum(1)
        ph += w.sum(1)
        sa += np.abs(t).sum(1)
        sp += np.abs(w).sum(1)
    # each of the n * boxes terms carries a few ulps, each addition half an ulp
    tol = (n * len(boxes) + 32) * 2.0 ** -53
    assert np.all(np.abs(e + ex) <= tol * sa + 1e-300)
    assert np.all(np.abs(pot + ph) <= tol * sp + 1e-300)
