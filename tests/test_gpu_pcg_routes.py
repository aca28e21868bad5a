"""FP64 Jacobi-PCG solves around the one-launch solver (pcg_grid.hip): what a
caller sees of a solve does not depend on how it is called or what runs beside it."""

import numpy as np
import pytest
import torch

import se_amd

pytestmark = pytest.mark.gpu

PER, XPER, NONE = (1, 1), (1, 0), (0, 0)


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
