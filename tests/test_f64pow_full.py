"""The power of the checksums' energy sum (`csrc/k_f64math.h`, f64_pow_full) against 113-bit arithmetic.

The header is compiled for the host (the same bits as on the device: FMA-explicit and IEEE operations only).  Bound:
0.507 ulp, half an ulp for the final rounding and 0.007 for the terms that are not carried in two parts (derived in
the header); the C library's pow is at 0.507 on the same samples.  f64_div_by, its divisions by the reference pressure
and the map factors, equals the IEEE division in every quotient, infinities and NaN included.
"""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "wrf-jax_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not found")
def test_pow_full_is_as_near_as_the_c_library(tmp_path):
    exe = str(tmp_path / "f64pow_full_check")
    subprocess.run(["g++", "-O2", "-std=gnu++17", "-ffp-contract=off", "-I", CSRC, "-o", exe,
                    os.path.join(HERE, "cf64", "f64pow_full_check.cpp"), "-lquadmath", "-lm"], check=True)
    lines = subprocess.run([exe], capture_output=True, text=True, timeout=300, check=True).stdout.strip().splitlines()
    assert len(lines) == 9
    assert lines[8].split()[0] == "div" and lines[8].endswith(" differ=0") and "checked=6" in lines[8], lines[8]
    for line in lines[:8]:
        assert float(line.split("max_ulp=")[1]) <= 0.507, line
