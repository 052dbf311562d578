"""The quantising kernels' float32 division (csrc/scale_quotient.h, scale_quotient): the
product with the scale's reciprocal and two corrections, bit for bit the IEEE quotient
over the range it states. The bare product fails the same check."""
import os
import shutil
import subprocess

import pytest

SRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "native", "f32_quotient_check.c")


@pytest.mark.skipif(shutil.which("gcc") is None, reason="needs gcc")
def test_two_corrections_give_the_ieee_quotient(tmp_path):
    exe = str(tmp_path / "qc")
    subprocess.run(["gcc", "-O2", "-ffp-contract=off", "-mfma", "-fopenmp", SRC, "-o", exe, "-lm"], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0 and out.stdout.strip().endswith(" mismatches 0"), out.stdout
    assert int(out.stdout.split()[1]) > 150_000_000
    bare = subprocess.run([exe, "uncorrected"], capture_output=True, text=True, timeout=300)
    assert bare.returncode != 0 and int(bare.stdout.split()[-1]) > 1000, bare.stdout
