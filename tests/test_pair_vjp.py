"""The FP64 line adjoint's pair products (flou.jl_amd/csrc/pair_vjp.hpp, built for the CPU) against extended
precision: no less exact than the general adjoint's in FP64.

Rms errors of the ρ, momentum and energy cotangents over 60,000 pairs (120,000 values or more each), for metrics
in any direction and along the line's axis, from nearly equal states to ratios of 100, over the general
adjoint's on the same pairs.  The two round in other places: 3 % are allowed, half the share of one more
rounding among the eight or so of a cotangent."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


def test_no_less_exact_than_the_general_adjoint(tmp_path):
    exe = tmp_path / "pair_vjp_check"
    cmd = ["g++", "-O2", "-std=c++17", "-mfma", "-ffp-contract=off", "-Wno-unknown-pragmas", "-D__HIP_PLATFORM_AMD__",
           "-I/opt/rocm/include", "-I", os.path.join(ROOT, "flou.jl_amd", "csrc"),
           os.path.join(HERE, "pair_vjp_check.cpp"), "-o", str(exe)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        pytest.fail("build failed:\n" + r.stderr)
    out = subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout
    rows = [line.split() for line in out.strip().splitlines()]
    assert len(rows) == 6 * 2 * 5 * 2
    for nd, tp, metric, ratio, inverse, *e in rows:
        assert max(map(float, e)) <= 1.03, (nd, tp, metric, ratio, inverse, e)
