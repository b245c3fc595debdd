"""The direct sum's partial sums live in one block of the context: calls on
several streams and replays of captured calls leave each other's alone."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _ptr(t):
    return C.c_void_p(t.data_ptr())


class Sum:
    """One direct sum of m targets over n particles on device arrays."""

    def __init__(self, torch, n, m, seed):
        r = np.random.Generator(np.random.PCG64(seed))
        self.p, self.q, self.idx = r.random((3, n)), r.standard_normal(n), r.integers(0, n, m)
        self.src = [torch.from_numpy(np.ascontiguousarray(v)).cuda() for v in (*self.p, self.q)]
        self.tgt = torch.from_numpy(self.idx).cuda()
        self.out = torch.zeros((4, m), dtype=torch.float64, device="cuda")
        self.n, self.m = n, m

    def enqueue(self, sol, stream):
        sol._check(sol.lib.pepc_gpu_set_stream(sol.h, C.c_void_p(stream.cuda_stream)))
        sol._check(sol.lib.pepc_gpu_direct_device(sol.h, self.n, *[_ptr(v) for v in self.src], self.m,
                                                  _ptr(self.tgt), 1e-4, 1.0, *[_ptr(o) for o in self.out]))

    def check(self):
        """Against extended precision at the first 50 targets: each term carries
        a few ulps, each addition half an ulp."""
        ld = np.longdouble
        i = self.idx[:50]
        d = (self.p[:, i, None] - self.p[:, None, :]).astype(ld)
        r2 = (d * d).sum(0) + ld(1e-4)
        w = self.q.astype(ld) / np.sqrt(r2)
        w[np.arange(len(i)), i] = 0
        t = np.concatenate([w / r2 * d, w[None]])
        got = self.out[:, :50].cpu().numpy()
        tol = (self.n + 32) * 2.0 ** -53
        assert np.all(np.abs(got - t.sum(-1)) <= tol * np.abs(t).sum(-1))


@pytest.mark.parametrize("sizes", [((20000, 300), (20000, 300)), ((3000, 2), (50000, 5000))])
def test_streams(sizes):
    """Two calls at a time on two streams equal the same calls one by one."""
    import torch
    from pepc_amd.solver import Solver
    sol = Solver(theta2=0.36, eps2=1e-4)
    sums = [Sum(torch, n, m, k) for k, (n, m) in enumerate(sizes)]
    streams = [torch.cuda.Stream() for _ in sums]
    torch.cuda.synchronize()
    want = []
    for s, st in zip(sums, streams):
        s.enqueue(sol, st)
        torch.cuda.synchronize()
        s.check()
        want.append(s.out.clone())
    for _ in range(3):
        for s in sums:
            s.out.zero_()
        torch.cuda.synchronize()
        for s, st in zip(sums, streams):
            s.enqueue(sol, st)
        torch.cuda.synchronize()
        for s, w in zip(sums, want):
            assert torch.equal(s.out, w)
    sol.close()


@pytest.mark.parametrize("warm", [False, True])
def test_capture(warm):
    """A captured call keeps its results when the context makes larger calls
    between its replays and beside them."""
    import torch
    from pepc_amd.solver import Solver
    sol = Solver(theta2=0.36, eps2=1e-4)
    one, large = Sum(torch, 5000, 300, 7), Sum(torch, 60000, 4096, 8)
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    if warm:
        one.enqueue(sol, side)
        torch.cuda.synchronize()
        one.check()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        one.enqueue(sol, torch.cuda.current_stream())
    first = None
    for _ in range(3):
        one.out.zero_()
        large.out.zero_()
        torch.cuda.synchronize()
        graph.replay()
        large.enqueue(sol, side)
        torch.cuda.synchronize()
        one.check()
        large.check()
        if first is None:
            first = one.out.clone()
        assert torch.equal(one.out, first)
    sol.close()
