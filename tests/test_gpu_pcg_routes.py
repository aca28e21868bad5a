"""FP64 Jacobi-PCG solves around the one-launch solver (pcg_grid.hip): what a
caller sees of a solve does not depend on how it is called or what runs beside it."""
import os
import threading

import numpy as np
import pytest
import torch

import se_amd

pytestmark = pytest.mark.gpu

XPER = (1, 0)


def problem(ctx, nEls, N, per=XPER, bc=(1, 1, 0, 0), seed=0):
    m = se_amd.Mesh(ctx, nEls, N, (0.0, 0.0), (1.0, 1.0), per, bc)
    h = se_amd.Helm(m, 200.0, 1.0, se_amd.DETJ_PHYSICAL)
    return m, h, np.random.default_rng(seed).standard_normal(m.n)


def test_in_place_solve_is_complete(gpu_ctx):
    """x and f the same vector: the result is there when the call returns, for
    a reader on any stream, and is that of separate vectors."""
    m, h, f = problem(gpu_ctx, (96, 96), 8)
    want, _ = h.pcg(f)
    stream = torch.cuda.ExternalStream(gpu_ctx.stream)
    for _ in range(5):
        x = torch.from_numpy(f).cuda()
        torch.cuda.synchronize()
        h.pcg_dev(x.data_ptr(), x.data_ptr())
        done = stream.query()
        got = x.cpu().numpy()
        assert done and np.array_equal(got, want)
    h.close()
    m.close()


def test_solves_beside_other_threads(gpu_ctx):
    """Solves of three contexts on one device from three threads, more workgroups
    in all than CUs: each solve the bits it has alone."""
    ctxs = [gpu_ctx, se_amd.Context(0), se_amd.Context(0)]
    probs = [problem(c, n, N, seed=N) for c, n, N in zip(ctxs, ((100, 100), (48, 40), (9, 7)), (8, 6, 5))]
    alone = [h.pcg(f) for _, h, f in probs]
    got = [[] for _ in probs]
    start = threading.Barrier(len(probs))

    def work(i):
        start.wait()
        for _ in range(4):
            got[i].append(probs[i][1].pcg(probs[i][2])[0])

    ts = [threading.Thread(target=work, args=(i,)) for i in range(len(probs))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for (x, info), xs in zip(alone, got):
        assert info["status"] == 0 and len(xs) == 4 and all(np.array_equal(x, y) for y in xs)
    for m, h, _ in probs:
        h.close()
        m.close()
    for c in ctxs[1:]:
        c.close()


def test_waits_that_ran_out_in_a_row_are_remembered(gpu_ctx):
    """One give-up changes nothing for the solve after it; from the second in a
    row on, 16 solves and then twice as many go straight to the other solver.
    A lone workgroup never waits."""
    m, h, f = problem(gpu_ctx, (24, 24), 6)
    m1, h1, f1 = problem(gpu_ctx, (4, 4), 4)

    def solve(n=1):
        a = gpu_ctx.solver_counts()
        for _ in range(n):
            h.pcg(f, maxit=2)
        b = gpu_ctx.solver_counts()
        return b[0] - a[0], b[1] - a[1]

    assert solve() == (1, 0)
    os.environ["SE_GRID_WAIT"] = "0"
    try:
        assert solve() == (0, 1)
        del os.environ["SE_GRID_WAIT"]
        assert solve() == (1, 0)
        os.environ["SE_GRID_WAIT"] = "0"
        assert solve(2) == (0, 2)
        assert solve(16) == (0, 0)
        assert solve() == (0, 1)
    finally:
        os.environ.pop("SE_GRID_WAIT", None)
    assert solve(31) == (0, 0)
    a = gpu_ctx.solver_counts()
    h1.pcg(f1)
    assert gpu_ctx.solver_counts() == (a[0] + 1, a[1])
    assert solve() == (0, 0)
    assert solve(2) == (2, 0)
    for o in (h, m, h1, m1):
        o.close()


def test_overflow_at_the_start_reports_its_residual(gpu_ctx):
    """b.b finite, r.z not: x = 0 and the relative residual is 1, in either solver."""
    m = se_amd.Mesh(gpu_ctx, (12, 10), 4, (0.0, 0.0), (1.0, 1.0), XPER, (1, 1, 0, 0))
    h = se_amd.Helm(m, 0.0, 1e-12, se_amd.DETJ_PHYSICAL)
    f = 1e151 * np.random.default_rng(1).standard_normal(m.n)
    for kw in ({}, dict(history=True, maxit=50)):
        x, i = h.pcg(f, **kw)
        assert i["status"] == se_amd.SOLVE_NONFINITE and i["iters"] == 0 and not x.any()
        assert abs(i["true_rel_residual"] - 1.0) <= 1e-12
    h.close()
    m.close()
