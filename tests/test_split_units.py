"""The rule by which the decode, tile and combine kernels share a row's pages
among splits (phaseshift_amd/csrc/split_units.h) at the ends of the 32-bit
range, on the CPU: a row whose page count wraps has no split, and the combine,
which clamps its split indexes to the last used one, reads none for it."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


def test_split_units_match_64_bit_arithmetic(tmp_path):
    exe = tmp_path / "split_units_check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", os.path.join(ROOT, "phaseshift_amd", "csrc"),
                    os.path.join(HERE, "native", "split_units_check.cpp"), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "mismatches 0" in r.stdout
