"""The sums of 1/r of the SIR kernel's run walk (sir_runs.hpp) on the CPU,
the same code the kernel compiles, against long double.

Equally spaced positions leave the series and its rounding.  A run spans at
most r/36 (FP64 output; r/20 FP32), so half of it at most 1/72 (1/40) of r:
the first term left out, P8 (P6), is at most (1/72)^8/9 = 2e-16 ((1/40)^6/7 =
3.5e-11) of the sum.  The rounding: about ten operations of 2^-53 that carry
the whole sum, and the offset's half ulp (66 mm: 2^-47) over r >= 0.5 mm where
the offset is the larger part, |v|/r <= 1: together 4e-15.  Without the P6
term the FP64 error is 3e-13, with runs of r/16 2e-14, and of r/13 the FP32
one 1e-10.

Accumulated positions: a line is walked run by run only where their deviation
from equal spacing moves 1/r by at most 2^-47, the accuracy of a stepped
sub-element's amplitude."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("run_sums") / "run_sums_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off",
                    "-I", os.path.join(HERE, "..", "dream_amd", "csrc"),
                    os.path.join(HERE, "cxx", "run_sums_check.cc"), "-o", exe], check=True)

    def run(*args):
        out = subprocess.run([exe] + [str(a) for a in args], check=True, capture_output=True,
                             text=True)
        return [float(v) for v in out.stdout.split()]
    return run


@pytest.mark.parametrize("seed", [1, 2])
def test_series_on_equal_spacing(check, seed):
    usable, worst, worst32, stepped = check("equal", seed, 60000)
    assert usable > 40000
    assert worst <= 4e-15
    assert worst32 <= 3.5e-11
    assert stepped <= 1e-3


@pytest.mark.parametrize("shape,size,step,near,walked", [
    ("row", 10.0, 0.05, 1.0, 96),       # all lines are fit
    ("row", 50.0, 0.01, 2.0, 0),        # near and far points: 71 mm is the least
    ("row", 200.0, 0.05, 20.0, 1),
    ("row", 200.0, 0.01, 20.0, 0),
    ("disc", 7.5, 0.1, 2.0, 96),
    ("disc", 25.0, 0.05, 3.0, 1),
    ("disc", 50.0, 0.01, 2.0, 0),
    ("disc", 50.0, 0.1, 2.0, 1),
])
def test_accumulated_positions(check, shape, size, step, near, walked):
    fit, left, worst, seen, bound = check(shape, size, step, near)
    assert fit >= walked
    assert seen <= bound
    assert worst <= 2.0 ** -47 + 4e-15


def test_rest_of_a_half_is_one_stretch(check):
    """The sub-elements that no run certifies are walked once each, in
    stretches: positions accumulated from a disc row's start take at most two
    passes over the row, not one pass for each sub-element."""
    used, left, most, wrong = check("rest", 1, 4000)
    assert used > 3000 and left > 1000
    assert wrong == 0
    assert most <= 2.0


def test_price_of_runs(check):
    """The walk choice's estimate of a line's iterations against the walk's, for
    points at 0.5 to 45 mm (with the runs' longest length left out of it a near
    line was priced at a tenth of its iterations and below).  The estimate adds
    half the smaller of two rates where the true count lies between their
    larger and their sum, and takes the mean offset for all sub-elements: 1/1.6
    to 1.5."""
    used, least, most = check("price", 1, 20000)
    assert used > 18000
    assert 1 / 1.6 <= least and most <= 1.5
