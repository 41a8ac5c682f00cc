"""The final passes' division by a shared reciprocal (div3_inv of the kernels), on every
quotient close enough to a midpoint for it to round wrongly, compiled for the CPU with
the same operations."""
from __future__ import annotations

import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_corrected_quotients_round_as_ieee(tmp_path):
    exe = str(tmp_path / "div_midpoints")
    subprocess.check_call([os.environ.get("CXX", "g++"), "-O2", "-mfma", "-fopenmp", "-ffp-contract=off", "-Wall",
                           os.path.join(HERE, "cpp", "div_midpoints.cpp"), "-o", exe])
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120, check=True)
    pairs, wrong, uncorrected = map(int, r.stdout.split())
    print(f"{pairs} pairs, {wrong} wrong, {uncorrected} wrong without the correction", flush=True)
    assert pairs > 90_000_000
    assert wrong == 0
    assert uncorrected > 0
