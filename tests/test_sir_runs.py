"""The run walk of the SIR kernel (sir_runs.hpp) on the CPU: random lines of
sub-elements, ties on rounding boundaries among them, walked run by run and
index by index (tests/cxx/runs_check.cc), the same code the kernel compiles.

Bars: no sub-element in another bin than its exact index.  A bin's sum of
1/r: the lines reach 66 mm, whose accumulated positions stray from equal
spacing by at most 330 ulp(33)/4 = 6e-13 mm, at distances of 1.6 mm and more
4e-13 of the sum, far above the series' own 7e-16; without the refinement
the series to P4 leaves 2e-10."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.parametrize("seed", [1, 2])
def test_runs_equal_steps(tmp_path, seed):
    exe = str(tmp_path / "runs_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off",
                    "-I", os.path.join(HERE, "..", "dream_amd", "csrc"),
                    os.path.join(HERE, "cxx", "runs_check.cc"), "-o", exe], check=True)
    out = subprocess.run([exe, str(seed), "100000"], check=True, capture_output=True, text=True)
    lines, usable, moved, stepped, worst, worst32, _ = out.stdout.split()
    assert int(usable) > 0.8 * int(lines)
    assert int(moved) == 0
    assert float(stepped) < 0.2
    assert float(worst) <= 4e-13
    assert float(worst32) <= 2e-10
