"""Dense FDM transforms (lines of more than 256 elements) in the precisions and
with the null space that shorter lines solve in the plane-wave form.  Bars: the
system's own, 1e-10 against the oracle's assembled operator (1.5 of it for the
operators' different round-off)."""
import numpy as np
import pytest

import se_amd
from oracle import oracle as O

pytestmark = pytest.mark.gpu

PRECS = [se_amd.PREC_FP64, se_amd.PREC_FP32_IR, se_amd.PREC_FP64_FP32C, se_amd.PREC_FP64_BF16C]


@pytest.mark.parametrize("prec", PRECS)
@pytest.mark.parametrize("nEls,N,per,bc,null", [
    ((257, 3), 2, (1, 0), (1, 1, 0, 0), False),
    ((4, 261), 3, (0, 0), (1, 0, 0, 1), False),
    ((257, 3), 2, (1, 1), (0, 0, 0, 0), True),
    ((5, 300), 3, (1, 1), (0, 0, 0, 0), True),
])
def test_dense_solve(gpu_ctx, nEls, N, per, bc, null, prec):
    args = (nEls, N, (0.0, 0.0), (float(nEls[0]), 1.25 * nEls[1]), per, bc)
    m = se_amd.Mesh(gpu_ctx, *args)
    coef = (0.0, 1.0) if null else (1.0, 1.0)
    h = se_amd.Helm(m, *coef, se_amd.DETJ_PHYSICAL)
    oh = O.Helm(O.OracleMesh(*args), *coef, 1)
    f = np.random.default_rng(N).standard_normal(m.n)
    kw = dict(precision=prec, preconditioner=se_amd.PC_FDM, null_space=null)
    x, i = h.pcg(f, **kw)
    assert i["status"] == se_amd.SOLVE_CONVERGED and i["true_rel_residual"] <= 1e-10
    b = f - f.mean() if null else f
    r = b - oh.matvec(x)
    r = r - r.mean() if null else r
    assert np.linalg.norm(r) <= 1.5e-10 * np.linalg.norm(b)
    # it was the dense form: 2 M N K of the padded sizes in the first transform
    nU = [nEls[d] * N + 1 - (1 if per[d] else sum(bc[2:] if d == 0 else bc[:2])) for d in (0, 1)]
    P = [(n + 63) // 64 * 64 for n in nU]
    assert h.fdm_probe(reps=1)["flops_pass"][0] == 2.0 * P[0] * P[0] * P[1]
    # beside a plane-wave member, bit for bit
    m2 = se_amd.Mesh(gpu_ctx, (12, 9), 4, (0.0, 0.0), (1.0, 1.0), (1, 1), (0, 0, 0, 0))
    h2 = se_amd.Helm(m2, 0.0 if null else 2.0, 1.0, se_amd.DETJ_PHYSICAL)
    f2 = np.random.default_rng(3).standard_normal(m2.n)
    batch = se_amd.Batch(gpu_ctx, [h2, h])
    xs, infos = batch.pcg([f2, f], **kw)
    assert np.array_equal(xs[1], x) and infos[0]["status"] == 0
    batch.close()
    for o in (h, m, h2, m2):
        o.close()
