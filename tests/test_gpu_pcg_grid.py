"""FP64 Jacobi-PCG in one launch (pcg_grid.hip) against the launch-per-phase
solver (which a recorded history selects) and the oracle's assembled CSR."""
import os

import numpy as np
import pytest

import se_amd
from oracle import oracle as O

pytestmark = pytest.mark.gpu

PER, XPER, NONE = (1, 1), (1, 0), (0, 0)
# one tile with its own seams, one per direction, ragged last tiles, many small
# tiles, every boundary kind, orders 2..8, and tiles of 576 threads: one alone
# (orders 3, 4), and several with walls and ragged last ones, with the diagonal
# in registers (order 6) and read from memory (orders 7, 8)
CASES = [
    ((1, 1), 4, PER, (0, 0, 0, 0)), ((8, 8), 4, PER, (0, 0, 0, 0)), ((3, 40), 3, PER, (0, 0, 0, 0)),
    ((40, 3), 3, XPER, (1, 1, 0, 0)), ((23, 17), 2, NONE, (1, 1, 1, 1)), ((19, 21), 5, NONE, (1, 0, 0, 0)),
    ((31, 29), 6, XPER, (1, 1, 0, 0)), ((17, 13), 7, NONE, (0, 1, 1, 0)), ((50, 61), 8, PER, (0, 0, 0, 0)),
    ((80, 70), 6, NONE, (1, 1, 1, 1)),
    ((130, 101), 6, XPER, (1, 1, 0, 0)), ((100, 91), 7, NONE, (1, 1, 1, 1)), ((110, 90), 7, XPER, (0, 1, 0, 0)),
    ((120, 115), 8, NONE, (0, 1, 1, 0)), ((96, 96), 8, PER, (0, 0, 0, 0)),
]


@pytest.mark.parametrize("nEls,N,per,bc", CASES)
def test_grid_solve(gpu_ctx, nEls, N, per, bc):
    args = (nEls, N, (0.0, 0.0), (1.0, 1.3), per, bc)
    m = se_amd.Mesh(gpu_ctx, *args)
    h = se_amd.Helm(m, 40.0, 1.0, se_amd.DETJ_PHYSICAL)
    rng = np.random.default_rng(N)
    f = rng.standard_normal(m.n)
    launches = gpu_ctx.solver_counts()[0]
    # the same iterates: a few iterations, whose round-off grows by less than 100 eps each
    for k in (1, 6):
        x, i = h.pcg(f, maxit=k)
        y, j = h.pcg(f, maxit=k, history=True)
        assert i["iters"] == j["iters"] and i["status"] == j["status"]
        assert np.linalg.norm(x - y) <= 1e-12 * np.linalg.norm(y)
        assert abs(i["true_rel_residual"] - j["true_rel_residual"]) <= 1e-10 * (1 + j["true_rel_residual"])
    x, i = h.pcg(f)
    assert i["status"] == se_amd.SOLVE_CONVERGED and i["true_rel_residual"] <= 1e-10
    r = f - h.apply(x)
    assert np.linalg.norm(r) <= 1.01e-10 * np.linalg.norm(f)
    if m.n < 20000:
        oh = O.Helm(O.OracleMesh(*args), 40.0, 1.0, 1)
        assert np.linalg.norm(f - oh.matvec(x)) <= 1.01e-10 * np.linalg.norm(f)
    z, j = h.pcg(np.zeros(m.n))
    assert j["status"] == 0 and j["iters"] == 0 and not z.any()
    f[m.n // 2] = np.nan
    _, j = h.pcg(f)
    assert j["status"] == se_amd.SOLVE_NONFINITE
    assert gpu_ctx.solver_counts()[0] == launches + 5  # every solve without a history was one launch
    h.close()
    m.close()


def test_grid_null_space(gpu_ctx):
    m = se_amd.Mesh(gpu_ctx, (21, 18), 5, (0.0, 0.0), (1.0, 1.0), PER, (0, 0, 0, 0))
    h = se_amd.Helm(m, 0.0, -1.0, se_amd.DETJ_LITERAL)
    f = np.random.default_rng(1).standard_normal(m.n)
    launches = gpu_ctx.solver_counts()[0]
    x, i = h.pcg(f, null_space=True)
    assert gpu_ctx.solver_counts()[0] == launches + 1
    y, _ = h.pcg(f, null_space=True, history=True, maxit=5000)
    assert i["status"] == 0
    r = (f - f.mean()) - h.apply(x)
    assert np.linalg.norm(r - r.mean()) <= 1.01e-10 * np.linalg.norm(f)
    assert abs(x.mean()) <= 1e-12 * np.abs(x).max() and np.linalg.norm(x - y) <= 1e-7 * np.linalg.norm(y)
    h.close()
    m.close()


def test_grid_wait_runs_out(gpu_ctx):
    """A wait that is not granted (limit 0) leaves the solve to the other solver, unharmed."""
    m = se_amd.Mesh(gpu_ctx, (24, 24), 6, (0.0, 0.0), (1.0, 1.0), XPER, (1, 1, 0, 0))
    h = se_amd.Helm(m, -50.0, -1.0, se_amd.DETJ_LITERAL)
    f = np.random.default_rng(2).standard_normal(m.n)
    y, j = h.pcg(f, history=True, maxit=5000)
    launches, gave_up = gpu_ctx.solver_counts()
    os.environ["SE_GRID_WAIT"] = "0"
    try:
        x, i = h.pcg(f)
    finally:
        del os.environ["SE_GRID_WAIT"]
    assert gpu_ctx.solver_counts() == (launches, gave_up + 1)
    assert i["status"] == 0 and i["iters"] == j["iters"] and np.array_equal(x, y)
    x, i = h.pcg(f)  # and the next solve is whole again
    assert gpu_ctx.solver_counts() == (launches + 1, gave_up + 1)
    assert i["status"] == 0 and np.linalg.norm(f - h.apply(x)) <= 1.01e-10 * np.linalg.norm(f)
    h.close()
    m.close()


@pytest.mark.parametrize("nEls,N", [((24, 24), 6), ((96, 96), 8)])
def test_grid_restarts_from_the_true_residual(gpu_ctx, nEls, N):
    """A target below what b - A x can reach: the recursion meets it (the other
    solver's history shows where), the check fails, and the solve goes on from
    the true residual to the iteration limit with a whole x."""
    m = se_amd.Mesh(gpu_ctx, nEls, N, (0.0, 0.0), (1.0, 1.0), XPER, (1, 1, 0, 0))
    h = se_amd.Helm(m, 4e3, 1.0, se_amd.DETJ_PHYSICAL)
    f = np.random.default_rng(7).standard_normal(m.n)
    _, i = h.pcg(f, rtol=1e-12)
    assert i["status"] == 0
    limit = 2 * i["iters"]
    _, j = h.pcg(f, rtol=1e-16, maxit=limit, history=True)
    met = int(np.argmax(j["hist"] <= 1e-16))
    assert 0 < met < limit - 20 and j["status"] == se_amd.SOLVE_MAXIT
    launches = gpu_ctx.solver_counts()[0]
    x, i = h.pcg(f, rtol=1e-16, maxit=limit)
    assert gpu_ctx.solver_counts()[0] == launches + 1
    assert i["status"] == se_amd.SOLVE_MAXIT and i["iters"] == limit
    assert 1e-16 < i["true_rel_residual"] <= 1e-12
    assert np.linalg.norm(f - h.apply(x)) <= 1.01e-12 * np.linalg.norm(f)
    h.close()
    m.close()
