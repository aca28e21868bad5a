"""The branch-free powers of the Legendre derivative between two GLL points
(se_amd/csrc/glibc_pow.h), compiled as host code, against the C library's pow,
bit for bit, over the range that takes them."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "se_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_pow_plain_matches_libm(tmp_path):
    exe = str(tmp_path / "pow_plain_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-Wno-unknown-pragmas", "-I" + CSRC,
                    os.path.join(HERE, "pow_plain_check.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe, "1000000"], capture_output=True, text=True)
    assert r.returncode == 0 and "mismatches 0 of" in r.stdout, r.stdout
