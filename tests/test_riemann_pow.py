"""The exact Riemann solver's power (PowPos in fvs_riemann.hpp), compiled for
the host: within 0.8 units in the last place of 80-bit powers for the
rarefaction and star exponents of four gases, 1.1 for those of their fans (an
exponent of 22 multiplies the logarithm's error), and its edges."""
from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent
CSRC = HERE.parent / "finitevolumesolver_amd" / "csrc"


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs a host C++ compiler")
def test_power_within_its_bound(tmp_path):
    exe = tmp_path / "riemann_pow"
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", f"-I{HERE / 'host_stub'}",
                    f"-I{CSRC}", str(HERE / "host_stub" / "riemann_pow.cpp"), "-o", str(exe)],
                   check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True).stdout
    below_one, fans, bad = out.split()
    assert float(below_one) <= 0.8 and float(fans) <= 1.1 and int(bad) == 0, out
