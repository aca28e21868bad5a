"""The semi-Lagrangian steps give a node two lanes, which read an element's rows
16 bytes at a time: every order, one to three advected components, node counts that leave a part of a workgroup, against the
oracle, bit for bit."""
import numpy as np
import pytest

import se_amd
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nd", [1, 2, 3])
@pytest.mark.parametrize("N", [2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12])
def test_sl_steps_bit_exact(gpu_ctx, N, nd):
    nEls = (7, 5) if N < 3 else (4, 3)
    args = (nEls, N, (0.0, -1.0), (2.0, 0.5), (1, 0), (1, 1, 0, 0))
    m, om = se_amd.Mesh(gpu_ctx, *args), O.OracleMesh(*args)
    rng = np.random.default_rng(10 * N + nd)
    q, qp = rng.standard_normal((2, m.nV * nd))
    vel, velp = rng.standard_normal((2, 2 * m.nV))
    vel[::11] = 0.0  # points that stay on their node
    dt = 0.07
    got, dep = m.advect(q, vel, dt, nDofs=nd)
    ref, rdep, _ = om.advect_first(q, nd, vel, dt)
    assert np.array_equal(dep, rdep)
    assert np.array_equal(np.ravel(got), ref)
    got2 = m.advect2(q, qp, vel, velp, dt, nDofs=nd)
    assert np.array_equal(np.ravel(got2), om.advect_second(q, qp, nd, vel, velp, dt))


@pytest.mark.parametrize("N", [3, 9, 12])
def test_bicubic_step_bit_exact(gpu_ctx, N):
    """The advected field by bicubic interpolation at orders that do not default to it."""
    args = ((4, 3), N, (0.0, -1.0), (2.0, 0.5), (1, 0), (1, 1, 0, 0))
    m, om = se_amd.Mesh(gpu_ctx, *args), O.OracleMesh(*args)
    m.set_sl_interp(se_amd.INTERP_BICUBIC)
    rng = np.random.default_rng(N)
    q, vel = rng.standard_normal(m.nV), rng.standard_normal(2 * m.nV)
    got, _ = m.advect(q, vel, 0.07)
    assert np.array_equal(np.ravel(got), om.advect_first_interp(q, 1, vel, 0.07, se_amd.INTERP_BICUBIC))
