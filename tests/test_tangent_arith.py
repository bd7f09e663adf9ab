"""CPU check of the arithmetic of the psi and chi chains of calls with forward
tangents (tests/c/tangent_quad.c): psi_j and psi'_j in double, as the kernels form
them, against the cut recurrences differentiated in 113 bits, over x = 1e-3 to
1860, at and away from x = k pi."""
import os
import subprocess

from conftest import ROOT


def build(tmp_path):
    exe = str(tmp_path / "tangent_quad")
    subprocess.check_call(["gcc", "-std=gnu99", "-O2", "-ffp-contract=off", "-Wall",
                           os.path.join(ROOT, "tests/c/tangent_quad.c"), "-o", exe, "-lquadmath", "-lm"])
    return exe


def test_tangent_chains_against_113_bits(tmp_path):
    r = subprocess.run([build(tmp_path), "check"], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and "tangent arithmetic: ok" in r.stdout, r.stdout[-2000:] + r.stderr[-2000:]
