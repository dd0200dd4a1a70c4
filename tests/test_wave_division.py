"""The wave kernel forms a bin's square root and divisions from a few double
operations on per-cell reciprocals (sqrt_near, div_near, div_by in
xbg_math.h).  They are to give the IEEE float results; checked on the host,
whose double operations are the same, for wave speeds and divisors over and
beyond the range that a model meets."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def checker(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("wdiv") / "wave_division_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off",
                    os.path.join(HERE, "native", "wave_division_check.cpp"), "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("mode,n,seed", [("near", 60000, 1), ("near", 60000, 2), ("by", 100000, 3), ("by", 100000, 4)])
def test_equal_to_the_ieee_operations(checker, mode, n, seed):
    r = subprocess.run([checker, mode, str(n), str(seed)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout
