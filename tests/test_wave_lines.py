"""The wave form of the fast diagonalisation: the host tables (CPU), and the
device transforms as an inverse of the operator at the sizes where their
tiles, blocks and kernels change."""
import os
import subprocess

import numpy as np
import pytest

import se_amd

HERE = os.path.dirname(os.path.abspath(__file__))


def test_wave_tables(tmp_path):
    exe = str(tmp_path / "wave_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", os.path.join(HERE, "..", "se_amd", "csrc"),
                    os.path.join(HERE, "wave_check.cpp"), "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout


ENDS = [((1, 1), (0, 0, 0, 0)), ((1, 0), (1, 1, 0, 0)), ((0, 0), (1, 1, 1, 1)), ((0, 0), (1, 0, 0, 1)),
        ((0, 0), (0, 0, 0, 0)), ((0, 0), (0, 1, 1, 0))]


# elements per line: one tile and its edges, the change of lines per workgroup
# (64 / 65), the long kernels (128 / 129, natural ends add a slot), the last
# wave line and the first dense one (256 / 257)
@pytest.mark.gpu
@pytest.mark.parametrize("ex,ey,N", [(1, 1, 4), (2, 3, 2), (15, 17, 3), (16, 33, 5), (64, 5, 6), (65, 63, 4),
                                     (3, 127, 7), (128, 2, 8), (129, 9, 3), (7, 256, 3), (257, 2, 2)])
@pytest.mark.parametrize("per,bc", ENDS)
def test_wave_inverse(gpu_ctx, ex, ey, N, per, bc):
    # unit elements and c_mass = 1: kappa is O(N^4) at any length, so the
    # rounded inverse leaves less than 1e-9 (as the bar of the dense one)
    m = se_amd.Mesh(gpu_ctx, (ex, ey), N, (0.0, 0.0), (float(ex), 1.25 * ey), per, bc)
    if m.n == 0:
        m.close()
        return
    h = se_amd.Helm(m, 1.0, 1.0, se_amd.DETJ_PHYSICAL)
    r = np.random.default_rng(ex + ey).standard_normal(m.n)
    z = h.apply_fdm(r, se_amd.PREC_FP64)
    assert np.linalg.norm(h.apply(z) - r) <= 1e-9 * np.linalg.norm(r)
    # the whole solve, alone and beside another member, bit for bit
    x, i = h.pcg(r, precision=se_amd.PREC_FP64_BF16C, preconditioner=se_amd.PC_FDM)
    assert i["status"] == 0 and np.linalg.norm(h.apply(x) - r) <= 1.5e-10 * np.linalg.norm(r)
    m2 = se_amd.Mesh(gpu_ctx, (40, 12), 5, (0.0, 0.0), (1.0, 1.0), (1, 0), (1, 1, 0, 0))
    h2 = se_amd.Helm(m2, 2.0, 1.0, se_amd.DETJ_PHYSICAL)
    f2 = np.random.default_rng(3).standard_normal(m2.n)
    b = se_amd.Batch(gpu_ctx, [h2, h])
    xs, _ = b.pcg([f2, r], precision=se_amd.PREC_FP64_BF16C, preconditioner=se_amd.PC_FDM)
    assert np.array_equal(xs[1], x)
    b.close()
    for o in (h, m, h2, m2):
        o.close()


# the long kernels' output tiles per wave, two to seven: order 2 (no
# antisymmetric parts) and the others, lines with and without a mirror symmetry
@pytest.mark.gpu
@pytest.mark.parametrize("ex,ey,N", [(129, 2, 2), (256, 2, 2), (160, 2, 4), (2, 200, 8), (256, 1, 7), (250, 3, 5)])
@pytest.mark.parametrize("per,bc", ENDS)
def test_long_wave_inverse(gpu_ctx, ex, ey, N, per, bc):
    # bar and elements as in test_wave_inverse
    m = se_amd.Mesh(gpu_ctx, (ex, ey), N, (0.0, 0.0), (float(ex), 1.25 * ey), per, bc)
    h = se_amd.Helm(m, 1.0, 1.0, se_amd.DETJ_PHYSICAL)
    r = np.random.default_rng(ex + N).standard_normal(m.n)
    z = h.apply_fdm(r, se_amd.PREC_FP64)
    assert np.linalg.norm(h.apply(z) - r) <= 1e-9 * np.linalg.norm(r)
    h.close()
    m.close()


@pytest.mark.gpu
@pytest.mark.parametrize("order", [(0, 1), (1, 0)])
def test_probe_of_a_batch_of_both_forms(gpu_ctx, order):
    """A wave-form member beside a dense one (a line of 257 elements): the probe
    counts each with its own form's flops and times both."""
    sizes = [((40, 12), 5), ((257, 2), 2)]
    ms = [se_amd.Mesh(gpu_ctx, *sizes[k], (0.0, 0.0), (1.0, 1.0), (1, 0), (1, 1, 0, 0)) for k in order]
    hs = [se_amd.Helm(m, 2.0, 1.0, se_amd.DETJ_PHYSICAL) for m in ms]
    fs = [np.random.default_rng(k).standard_normal(m.n) for k, m in enumerate(ms)]
    kw = dict(precision=se_amd.PREC_FP64, preconditioner=se_amd.PC_FDM)
    flops = np.zeros(4)
    for h, f in zip(hs, fs):
        h.pcg(f, **kw)
        flops += h.fdm_probe(reps=2)["flops_pass"]
    b = se_amd.Batch(gpu_ctx, hs)
    b.pcg(fs, **kw)
    p = b.fdm_probe(reps=2)
    assert np.array_equal(p["flops_pass"], flops)
    assert min(p["us_pass"]) > 0.0 and p["us_apply"] > 0.0 and p["bytes_apply"] == 16.0 * sum(m.n for m in ms)
    b.close()
    for o in hs + ms:
        o.close()
