"""CPU test: the terms that KVStar's softmax adds up are as exact as the 2^t they are made of."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "unified-cache-management_amd", "csrc")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = tmp_path_factory.mktemp("exp_sum") / "exp_sum"
    r = subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-I" + CSRC,
                        os.path.join(ROOT, "tests", "native", "exp_sum.cpp"), "-o", str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    return str(exe)


@pytest.mark.parametrize("lo", [-1, -10, -60, -80])
def test_terms_are_rounded_once(program, lo):
    """A term's 2^t is rounded to nearest, 2^-24 of itself at most (half a last place of a number just above a power of
    two), and its correction adds 3.2e-11: exp(x) - (1 + r) 2^t is at most r^2 / 2 with r <= 8e-6 (below
    e^-80 the correction is a denormal: the sum has a term of 1 there).  The mean of a million
    such errors, of standard deviation below 3.5e-8, is within five of its own deviations, 1.8e-10, of 0, and
    2^t's own bias and r^2 / 2 are less."""
    r = subprocess.run([program, str(lo)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
    most, mean = map(float, r.stdout.split())
    assert most <= 2.0 ** -24 + 3.2e-11
    assert abs(mean) <= 1.8e-10 + 3.2e-11
