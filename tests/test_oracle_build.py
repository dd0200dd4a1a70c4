"""The oracle uses fused multiply-add instructions only where the CPU has
them, and its elementary functions give the same bits without."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def flags(*args):
    r = subprocess.run(["make", "-n", "-B", "-C", os.path.join(HERE, "..", "oracle"), *args], capture_output=True,
                       text=True, check=True)
    return [ln for ln in r.stdout.splitlines() if "-shared" in ln]


def test_instructions_follow_the_cpu():
    has = any(ln.startswith("flags") and " fma " in ln + " " for ln in open("/proc/cpuinfo"))
    lines = flags()
    assert len(lines) == 3 and all(("-mfma" in ln) == has for ln in lines)
    assert not any("-mfma" in ln for ln in flags("FMA="))


def test_same_bits_with_and_without(tmp_path):
    got = []
    has = any(ln.startswith("flags") and " fma " in ln + " " for ln in open("/proc/cpuinfo"))
    for k, extra in enumerate([[], ["-mfma"]] if has else [[], ["-O1"]]):
        exe = str(tmp_path / f"bits{k}")
        subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", *extra, os.path.join(HERE, "native", "xmath_bits.cpp"),
                        "-o", exe], check=True)
        got.append(subprocess.run([exe], capture_output=True, text=True, check=True).stdout)
    assert got[0] == got[1] and len(got[0]) == 17
