"""Linear solves of several threads on streams of their own on one device."""
import threading
import time

import numpy as np
import pytest

from florence_amd.workloads import clamp_and_pull, clamp_and_twist, cube_hex_p4, cube_tet_p2, twisted_state

pytestmark = pytest.mark.gpu


class _System(object):
    """A masked tangent and a right-hand side on a stream of its own."""

    def __init__(self, cuda, kind, n, rtol):
        import torch
        from florence_amd.assembly import DeviceMeshData, assemble_device
        from florence_amd.multigrid import MultigridSolver
        from florence_amd.solver import LinearSolver
        if kind == "mg":
            m, fs, mat = cube_hex_p4(n)
            x, flags, self.lin = twisted_state(m, 5.0), clamp_and_twist(m), MultigridSolver(rtol=rtol)
        else:
            m, fs, mat = cube_tet_p2(n)
            x, flags, self.lin = np.asarray(m.points), clamp_and_pull(m), LinearSolver(rtol=rtol)
        self.dm = DeviceMeshData(m, fs)
        self.V, _, _ = assemble_device(self.dm, mat, x)
        self.free = torch.as_tensor(np.isnan(flags).ravel().astype(np.uint8), device=cuda)
        self.b = torch.as_tensor(np.random.default_rng(n).standard_normal(self.free.numel()), device=cuda) * self.free
        self.x = torch.empty_like(self.b)
        self.stream = torch.cuda.Stream()
        torch.cuda.synchronize()

    def solve(self):
        import torch
        with torch.cuda.stream(self.stream):
            self.lin._warm_key = None   # each solve starts from the same vectors
            self.lin.Solve(self.dm, self.V, self.free, self.b, self.x)
        self.stream.synchronize()
        return self.x.clone()


def test_solves_in_threads_equal_their_own(cuda):
    """Multigrid and block-Jacobi solves of four threads at once: every one as by itself, bitwise."""
    systems = [_System(cuda, *a) for a in (("mg", 2, 1e-10), ("pcg", 4, 1e-10), ("mg", 3, 1e-10), ("pcg", 6, 1e-10))]
    ref = [s.solve() for s in systems]
    bad = []

    def work(i):
        import torch
        for _ in range(5):
            if not torch.equal(systems[i].solve(), ref[i]):
                bad.append(i)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(systems))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


def test_short_solve_does_not_wait_for_a_long_one(cuda):
    """A thread's small solves end while another thread's long multigrid solve (some hundred
    cycles) runs: no solve holds the device from its first launch to its last."""
    long, short = _System(cuda, "mg", 6, 1e-120), _System(cuda, "pcg", 2, 1e-8)
    short.solve()
    t0 = time.perf_counter()
    long.solve()
    alone = time.perf_counter() - t0
    ended = []
    t = threading.Thread(target=lambda: (long.solve(), ended.append(time.perf_counter())))
    t.start()
    time.sleep(0.1 * alone)
    short.solve()
    mine = time.perf_counter()
    t.join()
    print("long solve {:.1f} ms, {} cycles; the short one ended {:.1f} ms before it".format(
        1e3 * alone, long.lin.iterations[-1], 1e3 * (ended[0] - mine)), flush=True)
    assert mine < ended[0] - 0.3 * alone
