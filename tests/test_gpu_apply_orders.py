"""The batched FP64 apply holds the tiles of every order in one launch: members
of all orders at the edges of their tiles (one element, a full tile, one more
element each way, several tiles) in one batch, against the operator's own apply
kernel and against each member alone."""
import numpy as np
import pytest

import se_amd

pytestmark = pytest.mark.gpu

# elements per tile of each order, in x
TILE = {2: 8, 3: 7, 4: 6, 5: 5, 6: 5, 7: 4, 8: 4}


def build(gpu_ctx, N, nEls, per):
    bc = (1, 1, 1, 1) if per == (0, 0) else (0, 0, 0, 0)
    m = se_amd.Mesh(gpu_ctx, nEls, N, (0.0, 0.0), (1.0, 1.3), per, bc)
    return m, se_amd.Helm(m, 40.0, 1.0, 1)


@pytest.mark.parametrize("seed", [0, 1])
def test_orders_in_one_apply(gpu_ctx, seed):
    shapes = {0: lambda T: [(1, 2), (T, T), (T + 1, T)], 1: lambda T: [(2, 1), (T, T + 1), (2 * T + 1, 3 * T - 1)]}
    mem = [(N, s, per) + build(gpu_ctx, N, s, per)
           for N, T in TILE.items() for s, per in zip(shapes[seed](T), [(0, 0), (1, 0), (1, 1)])]
    order = np.random.default_rng(seed).permutation(len(mem))
    mem = [mem[k] for k in order]
    fs = [np.random.default_rng(100 * seed + i).standard_normal(x[3].n) for i, x in enumerate(mem)]
    b = se_amd.Batch(gpu_ctx, [x[4] for x in mem])
    xs, infos = b.pcg(fs, rtol=1e-10, precision=se_amd.PREC_FP64, preconditioner=se_amd.PC_FDM)
    for (N, s, per, m, h), f, x, info in zip(mem, fs, xs, infos):
        assert info["status"] == se_amd.SOLVE_CONVERGED, (N, s, per, info)
        # the solve's own bound; the apply's rounding is ~1e-15 of the vectors
        assert np.linalg.norm(f - h.apply(x)) <= 1.5e-10 * np.linalg.norm(f), (N, s, per)
        x1, _ = h.pcg(f, rtol=1e-10, precision=se_amd.PREC_FP64, preconditioner=se_amd.PC_FDM)
        assert np.array_equal(x, x1), (N, s, per)
    b.close()
    for _, _, _, m, h in mem:
        h.close()
        m.close()
