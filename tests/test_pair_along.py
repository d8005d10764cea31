"""The two-point fluxes of the FP64 curved split form (flou.jl_amd/csrc/pair_along.hpp, built for the CPU)
against extended precision: no less exact than the reference's own FP64 arithmetic.

Rms errors of mass, momentum and energy over 100,000 pairs, for metrics in any direction and along the
line's axis, from nearly equal states to ratios of 1000, over the same pairs' rms errors in the reference's
order with correctly rounded divisions.  Each is a mean over 10^5 squares, whose ratio scatters by about
half a per cent; along an axis, where both sums have one term and differ only in the place of a
rounding or two, 3 % are allowed (one rounding more among the ten or so that the smallest of them holds
is 5 %).  Where ρ or β of the two nodes are as 11 to 9 the log-mean's branch (u = 0.01) hangs on the
rounding of its argument, and its two sides are 1e-9 apart: the branch taken is the reference's,
so deviations stay at some ten roundings, 2e-15 of the largest component."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


@pytest.fixture(scope="module")
def rows(tmp_path_factory):
    exe = tmp_path_factory.mktemp("pair") / "pair_along_check"
    cmd = ["g++", "-O2", "-std=c++17", "-mfma", "-ffp-contract=off", "-Wno-unknown-pragmas", "-D__HIP_PLATFORM_AMD__",
           "-I/opt/rocm/include", "-I", os.path.join(ROOT, "flou.jl_amd", "csrc"),
           os.path.join(HERE, "pair_along_check.cpp"), "-o", str(exe)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        pytest.fail("build failed:\n" + r.stderr)
    out = subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout
    return [line.split() for line in out.strip().splitlines()]


def test_no_less_exact_than_the_reference_order(rows):
    errors = [r for r in rows if r[0] == "error"]
    assert len(errors) == 2 * 3 * 2 * 4 * 2
    for _, nd, tp, metric, ratio, inverse, *e in errors:
        assert max(map(float, e)) <= (1.005 if metric == "0" else 1.03), (nd, tp, metric, ratio, inverse, e)


def test_branch_of_the_logarithmic_mean(rows):
    branch = [r for r in rows if r[0] == "branch"]
    assert len(branch) == 2
    for _, nd, worst in branch:
        assert float(worst) <= 2e-15, (nd, worst)
