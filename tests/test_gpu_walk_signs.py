"""FP32 walks choose their form by the signs of a system's charges, system by
system: a batch of one-signed and two-signed systems equals their separate
solves bit for bit, at group sizes with few and with many slices, and sinks of
each agree with an FP64 walk (2e-5 of the largest field: FP32 rounding in the
group frame, u L sum|q|/r^3 with u = 6e-8 and an extent of 1)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [700, 1, 3000, 64, 5000]


def _system(k, n):
    r = np.random.default_rng(100 + k)
    q = r.choice([-1.0, 1.0], n) if k % 2 == 0 else -np.ones(n)
    return r.random((3, n)), q


@pytest.mark.parametrize("group,pack", [(4, 0), (16, 32), (64, 64)])
def test_batch_of_both(group, pack):
    from pepc_amd.solver import Solver
    kw = dict(theta2=0.36, eps2=1e-4, group_size=group, group_pack=pack)
    sizes = [n for n in SIZES if n > 1]
    parts = [_system(k, n) for k, n in enumerate(sizes)]
    off = np.concatenate([[0], np.cumsum(sizes)])
    p, q = np.concatenate([a for a, _ in parts], axis=1), np.concatenate([b for _, b in parts])
    sol = Solver(**kw)
    sol.grow_batch(*p, q, off)
    res = sol.traverse()
    e, pot = res.e.cpu().numpy(), res.pot.cpu().numpy()
    sol.close()
    for k, (pk, qk) in enumerate(parts):
        one = Solver(**kw)
        one.grow(*pk, qk)
        r = one.traverse()
        b, t = int(off[k]), int(off[k + 1])
        assert np.array_equal(r.e.cpu().numpy(), e[:, b:t])
        assert np.array_equal(r.pot.cpu().numpy(), pot[b:t])
        s32 = one.traverse_sinks(*(pk[:, :200] * 1.01))
        full = Solver(precision="fp64", **kw)
        full.grow(*pk, qk)
        s64 = full.traverse_sinks(*(pk[:, :200] * 1.01))
        assert np.array_equal(s32.work.cpu().numpy(), s64.work.cpu().numpy())
        d = (s32.e - s64.e).abs().max() / s64.e.abs().max()
        assert float(d) < 2e-5
        one.close()
        full.close()
