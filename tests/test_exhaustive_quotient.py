"""The activation quantizers' x / scale from a two-term reciprocal, and their one-step floor(q + 0.5), against the
correctly rounded division and the fp32 sum, over every fp16 value and every fp16 absmax: tests/exhaustive_quotient.c,
compiled with the host gcc."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.skipif(shutil.which("gcc") is None, reason="needs gcc")
def test_quotient_exhaustive(tmp_path):
    exe = str(tmp_path / "exhaustive_quotient")
    subprocess.run(["gcc", "-O2", "-fopenmp", "-ffp-contract=off", os.path.join(HERE, "exhaustive_quotient.c"), "-o", exe, "-lm"], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "int8 quotient 0, int4 quotient 0, rounding 0" in r.stdout
