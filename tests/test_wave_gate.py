"""Where the wave kernel forms the dissipation's quotients from reciprocals no
quotient may be subnormal (div_by and div_near in xbg_math.h are IEEE
quotients only then): the condition itself, over random cells at its limits."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.parametrize("seed", [1, 2])
def test_no_quotient_is_subnormal(tmp_path, seed):
    exe = str(tmp_path / "wave_gate_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off",
                    os.path.join(HERE, "native", "wave_gate_check.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe, "2000000", str(seed)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout
